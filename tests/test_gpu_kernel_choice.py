"""Kernels and dispatch lines that the launchers pick by size, at the sizes where they can go wrong."""

import numpy as np
import pytest
import torch

from test_gpu_module import DEV, check_layer, make_case
from test_gpu_ops import test_dynamic_weights_forward_backward as check_dynamic_weights

pytestmark = pytest.mark.gpu

FWD = {torch.float32: (1e-5, 1e-4), torch.bfloat16: (2e-2, 2e-2), torch.float16: (2e-2, 2e-2)}


@pytest.mark.parametrize("B,S,D,dtype", [
    # the epilogue in front of branch_input: one partial tile, a tile that spans tokens, whole tiles
    # with a partial last one, several batches
    (1, 1, 8, torch.bfloat16), (3, 5, 72, torch.float16), (2, 7, 20, torch.float32), (2, 3, 2056, torch.bfloat16),
    # 1536 workgroups of one item per lane, the first of two items with a partial last one (772), and
    # 1536 of two items against the kernels apart
    (4, 768, 1024, torch.bfloat16), (4, 769, 1024, torch.bfloat16), (2, 3072, 1024, torch.float16),
    (2, 3073, 1024, torch.float16), (3, 131, 1003, torch.float32)])
def test_epilogue_in_front_of_branch_input(B, S, D, dtype):
    hc, H, bo, dHn, dbi = make_case(B, S, D, dtype, phi_std=0.02)
    check_layer(hc, H, bo, dHn, dbi, *FWD[dtype], 1e-4)


@pytest.mark.parametrize("R,K", [
    # slices of two steps (up to 224 rows at K = 16384), of four, and whole ones; K chunks that end
    # inside a slice, one step long, and with whole waves past K
    (64, 16384), (224, 16384), (225, 16384), (449, 16384), (64, 272), (70, 3088), (96, 16)])
@pytest.mark.parametrize("xdtype", [torch.bfloat16, torch.float16, torch.float32])
def test_projection_slices_of_few_rows(R, K, xdtype):
    check_dynamic_weights(R, K, xdtype)


def test_forward_reads_of_a_small_and_a_large_H_agree():
    """Static weights do not depend on the batch, so three batches (96 MB, plain loads) give the
    bits of the first three of four (128 MB, streaming loads)."""
    hc, _, _, _, _ = make_case(1, 2, 4096, torch.bfloat16, dynamic=False, res_std=1.0)
    g = torch.Generator(device=DEV).manual_seed(3)
    H = torch.randn((4, 1024, 4, 4096), generator=g, device=DEV).to(torch.bfloat16)
    bo = torch.randn((4, 1024, 4096), generator=g, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        bi4, add4 = hc(H)
        bi3, add3 = hc(H[:3])
        assert torch.equal(bi3, bi4[:3])
        assert torch.equal(add3(bo[:3]), add4(bo)[:3])


def off_by_one(t):
    """A contiguous copy of t that starts one element past a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = flat[1:].view(t.shape)
    out.copy_(t)
    return out


# Rows that are not whole 16-byte vectors, with enough elements (B S D >= 3 * 2^17) for the ragged
# vectors: one vector and one element, a vector less one past it, an even and an odd long row, rows
# one vector long; the last three start off a 16-byte boundary (whole vectors otherwise).
RAGGED = [(2, 21850, 9, torch.bfloat16, False), (3, 8750, 15, torch.float16, False),
          (2, 197, 1001, torch.bfloat16, False), (1, 265, 1500, torch.float16, False),
          (1, 78700, 5, torch.float32, False), (3, 131, 1003, torch.float32, False),
          (400, 1, 1001, torch.bfloat16, False), (70, 6, 1001, torch.float16, False),
          (1, 49200, 8, torch.bfloat16, True), (2, 200, 1024, torch.bfloat16, True),
          (1, 400, 1000, torch.float32, True)]


@pytest.mark.parametrize("B,S,D,dtype,shifted", RAGGED)
@pytest.mark.parametrize("dynamic", [True, False])
def test_layer_on_ragged_rows(B, S, D, dtype, shifted, dynamic):
    assert B * S * D >= 3 << 17
    hc, H, bo, dHn, dbi = make_case(B, S, D, dtype, dynamic=dynamic, phi_std=0.02, res_std=1.0)
    copy = off_by_one if shifted else torch.clone
    check_layer(hc, H, bo, copy(dHn), copy(dbi), *FWD[dtype], 1e-4, copy=copy)


@pytest.mark.parametrize("B,S,D,dtype,shifted", RAGGED)
def test_ops_on_ragged_rows_match_whole_vectors(B, S, D, dtype, shifted):
    """The four stream ops and their backwards give the same bits on ragged rows as on the same rows
    padded with zeros to whole vectors, and the weight gradients the same sums to fp32 rounding
    (both add at most B S D products in fp32 over fixed trees: a few 2^-24 of their largest
    partial sums; 1e-4 of the largest gradient leaves room for the trees' different shapes)."""
    import mhc
    from mhc import streams

    g = torch.Generator(device=DEV).manual_seed(11)
    P = (D + 7) // 8 * 8 + (8 if shifted else 0)

    def rows(*shape):
        return torch.randn(shape, generator=g, device=DEV).to(dtype)

    x, bo, d_bi, d_y = (rows(B, S, D) for _ in range(4))
    pre, post = torch.rand((B, 4), generator=g, device=DEV), torch.rand((B, 4), generator=g, device=DEV)
    res = torch.rand((B, 4, 4), generator=g, device=DEV)

    def run(make):
        a, b = (make(t).requires_grad_(True) for t in (x, bo))
        w = [t.clone().requires_grad_(True) for t in (pre, post, res)]
        H = streams.expand_streams(a)
        bi, hr = mhc.fused_stream_mix(make(H[..., :D]) if shifted and make is off_by_one else H, w[0], w[2])
        Hn = mhc.fused_add_residual(hr, b, w[1])
        y = streams.collapse_streams(Hn)
        torch.autograd.backward([bi, y], [make(d_bi), make(d_y)])
        return [t[..., :D] for t in (bi, Hn, y, a.grad, b.grad)], [t.grad for t in w]

    pad = lambda t: torch.nn.functional.pad(t, (0, P - D)).contiguous()  # noqa: E731
    got, got_w = run(off_by_one if shifted else torch.clone)
    want, want_w = run(pad)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i
    for i, (a, b) in enumerate(zip(got_w, want_w)):
        assert float((a - b).abs().max()) <= 1e-4 * float(b.abs().max()), i


@pytest.mark.parametrize("B,S,D,dtype", [(5, 7, 11235, torch.bfloat16), (3, 130, 1009, torch.float16),
                                         (2, 9, 21846, torch.float32),
                                         # 4 D just past a whole number of column blocks: the last block
                                         # of a row is half a vector (64-lane and 256-lane blocks)
                                         (1, 3200, 129, torch.bfloat16), (2, 200, 1025, torch.float16),
                                         (110, 7, 513, torch.bfloat16)])
@pytest.mark.parametrize("shifted", [False, True])
def test_mean_pool_on_ragged_rows(B, S, D, dtype, shifted):
    """fp32 sums of S values each: 2 S 2^-24 of the mean of |H|, at most 2^-14 here."""
    from mhc._kernels import mean_pool

    g = torch.Generator(device=DEV).manual_seed(2)
    H = torch.randn((B, S, 4, D), generator=g, device=DEV).to(dtype)
    x = mean_pool(off_by_one(H) if shifted else H)
    want = H.double().mean(dim=1).reshape(B, 4 * D)
    assert float((x.double() - want).abs().max()) <= 2.0 ** -14


@pytest.mark.parametrize("B,S,D,dtype", [
    # a workgroup per tile, a workgroup per batch, rows of one vector and an element, rows in 32 bits
    (2, 197, 1001, torch.bfloat16), (300, 5, 1001, torch.float16), (2, 21850, 9, torch.bfloat16),
    (3, 131, 1003, torch.float32)])
@pytest.mark.parametrize("factor", [0, 1])
def test_infinities_on_ragged_rows(B, S, D, dtype, factor):
    """An infinity or a NaN where the last two lanes of a row overlap reaches dH_post, dH_pre and dH_res
    once, as in plain products: +-inf stays +-inf.  The finite sums as in the test above."""
    import mhc
    from mhc import _layer

    g = torch.Generator(device=DEV).manual_seed(12)
    c = D - (4 if dtype == torch.float32 else 8)  # the last lane's first column, its neighbour's too
    H, dHn = (torch.randn((B, S, 4, D), generator=g, device=DEV).to(dtype) for _ in range(2))
    bo, dbi = (torch.randn((B, S, D), generator=g, device=DEV).to(dtype) for _ in range(2))
    inf, nan = float("inf"), float("nan")
    if factor == 0:
        dHn[0, S // 2, 1, c], dHn[1, 0, 2, c + 1], dHn[1, 0, 3, c] = inf, -inf, nan
        dbi[0, 1, c] = inf
    else:
        bo[0, S // 2, c], H[1, 1, 2, c + 1] = -inf, inf
    post, pre, res = (torch.rand(s, generator=g, device=DEV) for s in ((B, 4), (B, 4), (B, 4, 4)))
    want = [(dHn.double() * bo.double()[:, :, None]).sum((1, 3)), (H.double() * dbi.double()[:, :, None]).sum((1, 3)),
            torch.stack([torch.stack([(dHn[:, :, n].double() * H[:, :, m].double()).sum((1, 2)) for m in range(4)], -1)
                         for n in range(4)], 1)]
    hr, b, post = H.clone().requires_grad_(True), bo.clone().requires_grad_(True), post.requires_grad_(True)
    mhc.fused_add_residual(hr, b, post).backward(dHn)
    Hl, pre, res = H.clone().requires_grad_(True), pre.requires_grad_(True), res.requires_grad_(True)
    torch.autograd.backward(mhc.fused_stream_mix(Hl, pre, res), [dbi, dHn])
    _, dpre, dres = _layer.mix_backward(H, dbi, dHn, torch.rand((B, 24), generator=g, device=DEV), need_dH=False)
    for what, got, ref in (("dH_post", post.grad, want[0]), ("dH_pre", pre.grad, want[1]), ("dH_res", res.grad, want[2]),
                           ("layer dH_pre", dpre, want[1]), ("layer dH_res", dres.reshape(B, 4, 4), want[2])):
        fin = ref.isfinite()
        assert not fin.all(), what
        assert torch.equal(got[~fin].nan_to_num(1, 2, 3), ref[~fin].float().nan_to_num(1, 2, 3)), what
        assert float((got[fin] - ref[fin]).abs().max()) <= 1e-4 * float(ref[fin].abs().max()), what


def test_mixed_types_on_ragged_rows():
    """H in fp32 with a bf16 branch output (8 elements a lane): the bits of the single-element path,
    which the same rows take in pieces too small for the ragged one."""
    hc, H, bo, _, _ = make_case(2, 200, 1001, torch.float32, dynamic=False, res_std=1.0)
    bo = bo.to(torch.bfloat16)
    with torch.no_grad():
        whole = hc(H)[1](bo)
        for s in range(0, 200, 50):
            assert torch.equal(hc(H[:, s:s + 50].contiguous())[1](bo[:, s:s + 50].contiguous()), whole[:, s:s + 50])


@pytest.mark.parametrize("B,S,D,dtype", [
    # one column chunk in 384 S chunks of a few rows, rows that leave whole waves without any (S = 9:
    # one chunk of a row per wave), a partial last chunk, a column chunk of one vector
    (1, 4096, 128, torch.bfloat16), (1, 9, 64, torch.float32), (130, 9, 512, torch.bfloat16),
    (3, 1027, 130, torch.float16), (2, 517, 1032, torch.bfloat16)])
def test_mean_pool_chunks(B, S, D, dtype):
    """fp32 sums of S unit normals, each within 2^-24 of its partial sum (a few sqrt(S)): the mean is
    off by at most a few 2^-24, far inside 2^-16."""
    from mhc._kernels import mean_pool

    g = torch.Generator(device=DEV).manual_seed(4)
    H = torch.randn((B, S, 4, D), generator=g, device=DEV).to(dtype)
    want = H.double().mean(dim=1).reshape(B, 4 * D)
    assert float((mean_pool(H).double() - want).abs().max()) <= 2.0 ** -16
    hc, H, bo, dHn, dbi = make_case(min(B, 3), S, D, dtype, phi_std=0.02)
    check_layer(hc, H, bo, dHn, dbi, *FWD[dtype], 1e-4)


@pytest.mark.parametrize("B,S,D,dtype,iters", [
    # a workgroup per batch: one partial tile, exactly one and two tiles, one vector past them (where
    # few batches take the other kernels), rows in 32 bits, ragged rows
    (1, 1, 8, torch.bfloat16, 20), (3, 1, 4096, torch.bfloat16, 20), (2, 2, 4096, torch.float16, 7),
    (2, 1, 8200, torch.bfloat16, 20), (5, 3, 1368, torch.float32, 33), (300, 5, 1001, torch.bfloat16, 7),
    # 256 batches and more: three tiles with a partial last one, four, eight, and (outputs only) eight
    # of another type and one vector past eight
    (256, 3, 3000, torch.bfloat16, 20), (256, 4, 4096, torch.bfloat16, 20), (384, 4, 2040, torch.float32, 20),
    (256, 8, 2048, torch.float32, 20), (384, 8, 4096, torch.bfloat16, 20), (256, 1, 32776, torch.bfloat16, 20),
    # a last round of 256 that is less than half (the other kernels), and half
    (257, 3, 3000, torch.bfloat16, 20), (383, 3, 3000, torch.float16, 20), (384, 3, 3000, torch.float16, 20),
    # the most batches, and one more
    (1024, 2, 64, torch.float16, 20), (1025, 2, 64, torch.float16, 20)])
def test_whole_batch_workgroups(B, S, D, dtype, iters):
    hc, H, bo, dHn, dbi = make_case(B, S, D, dtype, phi_std=0.02)
    hc.sinkhorn_iters = iters
    if B * S * D > 1 << 23:  # too slow for the oracle in full: what the first batches of the same call put out
        from oracle import mhc_oracle as O
        from test_gpu_module import params_np, rel_err, run_gpu, to_np

        bi, Hn, grads = run_gpu(hc, H, bo, dHn, dbi)
        n = 2
        p = params_np(hc)
        obi, oHn, cache = O.layer_forward(p, to_np(H[:n]), to_np(bo[:n]), True, True, iters, hc.eps)
        og = O.layer_backward(p, cache, to_np(dHn[:n]), to_np(dbi[:n]))
        for got, want in ((bi[:n], obi), (Hn[:n], oHn), (grads["H"][:n], og["H"]), (grads["bo"][:n], og["bo"])):
            assert rel_err(to_np(got), want) < 2e-2
        return
    check_layer(hc, H, bo, dHn, dbi, *FWD[dtype], 1e-4)


@pytest.mark.parametrize("B,S,D,tiles", [(64, 4, 1024, 2), (256, 4, 2048, 4), (256, 8, 2048, 8)])
def test_whole_batch_sums_round_as_little_as_a_tree(B, S, D, tiles):
    """dH_post of a workgroup per batch, in fp32 from unit normals: a sum of n products is about sqrt(n), and
    a rounding at a partial sum of k of them adds sqrt(k) 2^-25 or less (rms).  Lanes chain 4 products a
    tile (2.5 n of such k in all) and add their tiles (the k / tiles of the second on), 16 lanes add in a
    tree (4 n), the 32 row sums add in fp64, and the result rounds once (n).  Summed in fp32 the rows
    would add 16.5 n."""
    import mhc

    g = torch.Generator(device=DEV).manual_seed(6)
    hr, bo = torch.randn((B, S, 4, D), generator=g, device=DEV), torch.randn((B, S, D), generator=g, device=DEV)
    post = torch.rand((B, 4), generator=g, device=DEV).requires_grad_(True)
    mhc.fused_add_residual(hr, bo, post).backward(hr)
    want = (hr.double() * bo.double()[:, :, None]).sum((1, 3))
    err = float((post.grad.double() - want).norm() / want.norm())
    bound = (2.5 + sum(range(2, tiles + 1)) / tiles + 4 + 1) ** 0.5 * 2.0 ** -25
    print(f"dH_post B={B} S={S} D={D}: {err:.2e} of {bound:.2e}", flush=True)
    assert err < 1.1 * bound


@pytest.mark.parametrize("B,S,D", [(4, 2, 512), (256, 4, 2048)])
def test_whole_batch_without_a_closure_gradient(B, S, D):
    """No dH_new and no dH_post: the same gradients as with zeros for both."""
    hc, H, bo, dHn, dbi = make_case(B, S, D, torch.bfloat16, phi_std=0.02)

    def step(zeros):
        hc.zero_grad(set_to_none=True)
        Hl = H.clone().requires_grad_(True)
        bi, add = hc(Hl)
        if zeros:
            torch.autograd.backward([add(bo), bi], [torch.zeros_like(dHn), dbi])
        else:
            bi.backward(dbi)
        return [Hl.grad] + [p.grad for p in hc.parameters()]

    for a, b in zip(step(False), step(True)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [1, 64, 257])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("eps", [0.0, 2.0 ** -26, 2.0 ** -25])
@pytest.mark.parametrize("iters", [0, 2, 33])
def test_sinkhorn_forms(n, dtype, eps, iters):
    """Partial waves of matrices whose sizes spread over eight decades, with a zero row and a zero column
    where eps keeps the sums positive.  One v_rcp and one rounding per normalised entry: 4e-7 of the
    largest."""
    import mhc
    from helpers import rel_err, to_np
    from oracle import mhc_oracle as O

    g = torch.Generator(device=DEV).manual_seed(n + iters)
    M = torch.randn((n, 4, 4), generator=g, device=DEV)
    M = (M * 10 ** (torch.rand((n, 1, 1), generator=g, device=DEV) * 8 - 4)).to(dtype)
    if eps:
        M[0, 1] = 0
        M[n // 2, :, 2] = 0
    P = mhc.sinkhorn_knopp(M, iters, eps)
    want = O.sinkhorn(to_np(M), iters, eps)
    half = {torch.float32: 0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert rel_err(to_np(P), want) < 1e-6 + half


@pytest.mark.parametrize("eps", [1e-8, 2.0 ** -26, 1e-6])
@pytest.mark.parametrize("iters", [1, 2, 3, 7, 8, 20, 33, 65])
@pytest.mark.parametrize("shifted", [False, True])
def test_sinkhorn_of_tiny_rows_and_columns(eps, iters, shifted):
    """P and dM where a row or a column is zero, or a millionth of the others, in matrices of sizes from
    0.01 to 1e20: there eps, or what it left in the column sums, outweighs that column for several
    rounds (at size 1e6 an eps term left out of the second round moves P by 4e-3, at 1e20 one left out of
    the third still moves it by more).  With eps on both sides of the line up to which its terms are
    left out from the eighth round on.  Matrix by matrix, over its largest entry: a round rounds each
    entry of P twice and its reciprocals once, so P is within a few 2^-23 whatever the round (each
    renormalises), and the backward adds two roundings a round."""
    import mhc
    from helpers import to_np
    from oracle import mhc_oracle as O

    n = 96
    g = torch.Generator(device=DEV).manual_seed(5)
    M = torch.randn((6, n, 4, 4), generator=g, device=DEV)
    M *= torch.tensor([1e-2, 1.0, 1e2, 1e4, 1e6, 1e20], device=DEV)[:, None, None, None]
    M[:, 1::6, :, 2] = 0
    M[:, 2::6, 1] = 0
    M[:, 3::6, :, 0] *= 1e-6
    M[:, 4::6, 3] *= 1e-6
    M[:, 5::6, :, 2] = 0
    M[:, 5::6, 1] = 0
    M = M.reshape(-1, 4, 4)
    dP = torch.randn(M.shape, generator=g, device=DEV)
    if shifted:
        M, dP = off_by_one(M), off_by_one(dP)
    M.requires_grad_(True)
    P = mhc.sinkhorn_knopp(M, iters, eps)
    P.backward(dP)
    eps32 = float(np.float32(eps))
    for got, want, tol in ((P, O.sinkhorn(to_np(M), iters, eps32), 8 * 2.0 ** -23),
                           (M.grad, O.sinkhorn_backward(to_np(M), to_np(dP), iters, eps32),
                            (2 * iters + 8) * 2.0 ** -23)):
        err = np.abs(to_np(got) - want).max(axis=(1, 2)) / np.abs(want).max(axis=(1, 2))
        print(f"sinkhorn eps={eps} iters={iters} shifted={shifted}: worst {err.max():.2e} of {tol:.2e}", flush=True)
        assert err.max() < tol


@pytest.mark.parametrize("R,K", [
    # two-wave column blocks (64 columns): one row chunk, several, a partial last block and column
    # block; four-wave ones from 513 rows; eight from 4097
    (64, 16384), (130, 4096), (512, 1000), (513, 1000), (1025, 8192), (4096, 1160), (4097, 264)])
@pytest.mark.parametrize("xdtype", [torch.bfloat16, torch.float16, torch.float32])
def test_weights_backward_column_blocks(R, K, xdtype):
    check_dynamic_weights(R, K, xdtype)


@pytest.mark.parametrize("R,K,xdtype", [
    # eight-wave column blocks below 4097 rows: long 16-bit rows in one round of the CUs, and where four-wave
    # ones would leave the busiest CU twice the work; fp32 with and without a full round (eight, four)
    (3584, 16384, torch.bfloat16), (3072, 3872, torch.float16), (2560, 8208, torch.float32),
    (2560, 8192, torch.float32)])
def test_weights_backward_wide_blocks_of_few_rows(R, K, xdtype):
    check_dynamic_weights(R, K, xdtype)


@pytest.mark.parametrize("B,S,D,dtype,iters", [
    # rows and wide pass in one: up to four rows, with three partials each (one past a whole batch's
    # two tiles), sixteen and seventeen, 256 and (apart again) 257 and five rows; K not a whole wave
    (1, 3, 4096, torch.bfloat16, 20), (4, 16, 4096, torch.float16, 20), (3, 17, 2050, torch.float32, 7),
    (2, 256, 4096, torch.bfloat16, 33), (2, 257, 4096, torch.bfloat16, 20), (5, 17, 2048, torch.float32, 20),
    (4, 130, 37, torch.bfloat16, 20)])
@pytest.mark.parametrize("frozen_h", [False, True])
def test_rows_in_the_wide_pass(B, S, D, dtype, iters, frozen_h):
    hc, H, bo, dHn, dbi = make_case(B, S, D, dtype, phi_std=0.02)
    hc.sinkhorn_iters = iters
    if not frozen_h:
        check_layer(hc, H, bo, dHn, dbi, *FWD[dtype], 1e-4)
        return
    grads = []
    for needs in (True, False):  # without dH the parameter gradients are the same bits
        hc.zero_grad(set_to_none=True)
        bi, add = hc(H.clone().requires_grad_(needs))
        torch.autograd.backward([add(bo), bi], [dHn, dbi])
        grads.append([p.grad for p in hc.parameters()])
    for a, b in zip(*grads):
        assert torch.equal(a, b)
