"""The C++ nodes of the eager entry points against the Python nodes, which take the calls that the
C++ ones leave alone: the same launches, so the same bits, and the same calls refused."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from test_gpu_module import DEV, make_case, run_gpu

pytestmark = pytest.mark.gpu


class _Off:
    """A binding that leaves every call to the Python nodes."""

    def __getattr__(self, name):
        return lambda *a: None


def both(monkeypatch, fn):
    from mhc import _lib

    native = _lib.native()
    seen = []

    class Spy:
        def __getattr__(self, name):
            def call(*a):
                r = getattr(native, name)(*a)
                seen.append((name, r is not None))
                return r

            return call

    monkeypatch.setattr(_lib, "native", lambda: Spy())
    got = fn()
    assert seen and all(ok for _, ok in seen), seen
    monkeypatch.setattr(_lib, "native", lambda: _Off())
    want = fn()
    monkeypatch.setattr(_lib, "native", lambda: native)
    return got, want


def same(got, want):
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a is None) == (b is None), i
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), i


@pytest.mark.parametrize("dynamic", [True, False])
@pytest.mark.parametrize("B,S,D,dtype,half_params", [(2, 24, 64, torch.float32, False), (3, 1, 72, torch.bfloat16, False),
                                                     (2, 9, 40, torch.float16, True), (0, 4, 16, torch.float32, False)])
@pytest.mark.parametrize("frozen", [(), ("H",), ("H_pre_base", "H_res_base"), ("all",)])
def test_layer_nodes_agree(monkeypatch, dynamic, B, S, D, dtype, half_params, frozen):
    hc, H, bo, dHn, dbi = make_case(B, S, D, dtype, dynamic=dynamic, phi_std=0.02, res_std=1.0)
    hc = hc.to(dtype) if half_params else hc

    def step():
        hc.zero_grad(set_to_none=True)
        for n, p in hc.named_parameters():
            p.requires_grad_(n not in frozen and "all" not in frozen)
        Hl = H.clone().requires_grad_("H" not in frozen and "all" not in frozen)
        bol = bo.clone().requires_grad_(True)
        bi, add = hc(Hl)
        Hn = add(bol)
        ends = [(Hn, dHn), (bi, dbi)]
        ends = [e for e in ends if e[0].requires_grad]
        torch.autograd.backward([e[0] for e in ends], [e[1] for e in ends])
        with torch.no_grad():
            bi0, add0 = hc(H)
            Hn0 = add0(bo)
        return [bi, Hn, bi0, Hn0, Hl.grad, bol.grad] + [p.grad for p in hc.parameters()]

    same(*both(monkeypatch, step))


def test_layer_nodes_agree_on_partial_and_repeated_backwards(monkeypatch):
    """branch_output only, then branch_input only, then two closures at once."""
    hc, H, bo, dHn, dbi = make_case(2, 12, 48, torch.float32, phi_std=0.02)

    def steps():
        Hl, bol = H.clone().requires_grad_(True), bo.clone().requires_grad_(True)
        bi, add = hc(Hl)
        Hn = add(bol)
        out = list(torch.autograd.grad(Hn, bol, dHn, retain_graph=True))
        out += torch.autograd.grad(bi, [Hl, *hc.parameters()], dbi, retain_graph=True, allow_unused=True)
        out += torch.autograd.grad([Hn, add(2 * bol), bi], [Hl, bol, *hc.parameters()], [dHn, 0.5 * dHn, dbi])
        return out

    same(*both(monkeypatch, steps))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_op_nodes_agree(monkeypatch, dtype):
    import mhc
    from mhc import streams

    g = torch.Generator(device=DEV).manual_seed(0)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    x, bo, M = r(2, 6, 24).to(dtype), r(2, 6, 24).to(dtype), r(5, 4, 4).to(dtype)
    pre, post, res = r(2, 4), r(2, 4).to(dtype), r(2, 4, 4)
    rows, phi, bias, a = r(3, 96).to(dtype), r(96, 24) * 0.1, r(24), [r(1), r(1)[0], r(1, 1)]

    def step():
        L = [t.clone().requires_grad_(True) for t in (x, bo, M, pre, post, res, rows, phi, bias, *a)]
        H = streams.expand_streams(L[0], scale=0.5)
        bi, hr = mhc.fused_stream_mix(H, L[3], L[5])
        y = streams.collapse_streams(mhc.fused_add_residual(hr, L[1], L[4]))
        P = mhc.sinkhorn_knopp(L[2], 9, 1e-6)
        W = mhc.fused_dynamic_weights(*L[6:12], 7, 1e-5)
        (bi.float().sin().sum() + y.float().sin().sum() + (P.float() ** 3).sum() + W[0].sum() +
         (W[2] ** 2).sum()).backward()
        with torch.no_grad():
            extra = [streams.expand_streams(x), mhc.sinkhorn_knopp(M), *mhc.fused_dynamic_weights(*L[6:12])]
        return [bi, y, P, *W, *extra] + [t.grad for t in L]

    same(*both(monkeypatch, step))


def test_calls_left_to_the_python_nodes():
    """Subclasses keep their type, vmap and forward-mode tangents are refused as before, float
    alphas work, and bad arguments raise what they raised."""
    import mhc
    from mhc import _lib

    hc, H, bo, dHn, dbi = make_case(2, 5, 16, torch.float32, phi_std=0.02)

    class Sub(torch.Tensor):
        pass

    assert isinstance(mhc.sinkhorn_knopp(torch.rand(2, 4, 4, device=DEV).as_subclass(Sub)), Sub)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda m: mhc.sinkhorn_knopp(m))(torch.rand(3, 2, 4, 4, device=DEV))
    for grad in (True, False):
        with torch.set_grad_enabled(grad), fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
            hc(fwAD.make_dual(H, torch.ones_like(H)))
    x, phi, bias = torch.rand(2, 16, device=DEV), torch.rand(16, 24, device=DEV), torch.rand(24, device=DEV)
    with torch.no_grad():
        assert len(_lib.native().dynamic_weights(x, phi, bias, *[torch.ones(1, device=DEV)] * 3, 20, 1e-6)) == 3
    for bad in (lambda: mhc.sinkhorn_knopp(torch.rand(2, 4, 3, device=DEV)),
                lambda: mhc.fused_dynamic_weights(x, phi[:8], bias, *[torch.ones(1, device=DEV)] * 3),
                lambda: hc(H)[1](bo[:, :2])):
        with pytest.raises(ValueError):
            bad()
    with pytest.raises(TypeError):
        mhc.sinkhorn_knopp(torch.rand(2, 4, 4, device=DEV, dtype=torch.float64))
    with pytest.raises(ValueError):
        mhc.sinkhorn_knopp(torch.rand(2, 4, 4, device=DEV), -1)


def test_saved_tensor_hooks_see_the_nodes_tensors():
    """Pack / unpack hooks run on what the nodes save (as activation offloading relies on)."""
    hc, H, bo, dHn, dbi = make_case(2, 6, 32, torch.float32, phi_std=0.02)
    _, _, want = run_gpu(hc, H, bo, dHn, dbi)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        _, _, got = run_gpu(hc, H, bo, dHn, dbi)
    assert H.shape in packed and bo.shape in packed
    for k in want:
        assert torch.equal(want[k], got[k]), k


def test_in_place_change_of_a_saved_parameter_is_refused():
    hc, H, bo, dHn, dbi = make_case(2, 6, 32, torch.float32, phi_std=0.02)
    bi, add = hc(H.clone().requires_grad_(True))
    with torch.no_grad():
        hc.phi.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.backward([add(bo), bi], [dHn, dbi])


@pytest.mark.parametrize("dtypes", [(torch.bfloat16,) * 7, (torch.float16, torch.float32, torch.bfloat16, torch.float64,
                                                            torch.float32, torch.float16, torch.float32)])
@pytest.mark.parametrize("offload", [False, True])
def test_converted_parameters(monkeypatch, dtypes, offload):
    """Parameters in 16 bits, and each in its own dtype (phi strided besides): converted in one launch
    into a buffer that the backward reads, also through hooks that change the saved layout."""
    hc, H, bo, dHn, dbi = make_case(3, 7, 20, torch.float32, phi_std=0.02, res_std=1.0)
    for p, dt in zip((hc.phi, hc.H_pre_base, hc.H_post_base, hc.H_res_base, hc.alpha_pre, hc.alpha_post, hc.alpha_res),
                     dtypes):
        p.data = p.data.to(dt)
    hc.phi.data = hc.phi.data.T.contiguous().T

    def step():
        hooks = (lambda t: t.cpu(), lambda t: t.to(DEV).contiguous()) if offload else (lambda t: t, lambda t: t)
        with torch.autograd.graph.saved_tensors_hooks(*hooks):
            bi, Hn, grads = run_gpu(hc, H, bo, dHn, dbi)
        return [bi, Hn] + [grads[k] for k in sorted(grads)]

    same(*both(monkeypatch, step))


def strided(t):
    """t's values in every second element of a storage of its own (no dimension is contiguous)."""
    return torch.stack((t, torch.full_like(t, 7)), dim=-1)[..., 0]


def turned(t):
    """t's values with its dimensions laid out in reverse order."""
    order = tuple(range(t.dim()))[::-1]
    return t.permute(order).contiguous().permute(order)


@pytest.mark.parametrize("layout", [strided, turned])
@pytest.mark.parametrize("dynamic,half_params", [(True, False), (True, True), (False, False), (False, True)])
def test_layer_backward_from_saved_tensors_in_other_strides(monkeypatch, layout, dynamic, half_params):
    """An unpack hook that hands every saved tensor back in other strides: the gradients without it, in
    the default layout."""
    hc, H, bo, dHn, dbi = make_case(3, 6, 40, torch.float32, dynamic=dynamic, phi_std=0.02, res_std=1.0)
    hc = hc.to(torch.bfloat16) if half_params else hc
    _, _, plain = run_gpu(hc, H, bo, dHn, dbi)

    def step():
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, layout):
            _, _, grads = run_gpu(hc, H, bo, dHn, dbi)
        assert all(g.is_contiguous() for g in grads.values())
        return [grads[k] for k in sorted(grads)]

    got, want = both(monkeypatch, step)
    same(got, want)
    same(got, [plain[k] for k in sorted(plain)])


def ops_step(hooks):
    """Gradients of the low-level ops with saved-tensor hooks."""
    import mhc
    from mhc import streams

    g = torch.Generator(device=DEV).manual_seed(1)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    L = [r(2, 6, 24), r(2, 6, 24), r(5, 4, 4), r(2, 4), r(2, 4).bfloat16(), r(2, 4, 4), r(6, 96), r(96, 24) * 0.1,
         r(24).bfloat16(), r(1), r(1), r(1)]
    L = [t.requires_grad_(True) for t in L]
    with torch.autograd.graph.saved_tensors_hooks(*hooks):
        bi, hr = mhc.fused_stream_mix(streams.expand_streams(L[0]), L[3], L[5])
        y = streams.collapse_streams(mhc.fused_add_residual(hr, L[1], L[4]))
        P = mhc.sinkhorn_knopp(L[2], 9, 1e-6)
        W = mhc.fused_dynamic_weights(*L[6:12], 7, 1e-5)
        out = [bi, y, P, *W]
    w = [torch.randn(t.shape, generator=g, device=DEV) for t in out]
    torch.autograd.backward(out, w)
    return [t.grad for t in L]


@pytest.mark.parametrize("layout", [strided, turned])
def test_op_backwards_from_saved_tensors_in_other_strides(layout):
    same(ops_step((lambda t: t, layout)), ops_step((lambda t: t, lambda t: t)))


@pytest.mark.parametrize("dynamic", [True, False])
def test_saved_tensors_off_the_gpu_are_refused(dynamic):
    """An unpack hook that leaves the tensors in host memory: the backward raises before any launch."""
    hc, H, bo, dHn, dbi = make_case(2, 6, 32, torch.float32, dynamic=dynamic, phi_std=0.02)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
        bi, add = hc(H.clone().requires_grad_(True))
        Hn = add(bo.clone().requires_grad_(True))
    for out, g in ((bi, dbi), (Hn, dHn)):
        with pytest.raises(RuntimeError, match="ROCm GPU"):
            out.backward(g, retain_graph=True)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        ops_step((lambda t: t.cpu(), lambda t: t))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_parameter_of_another_size_is_refused_in_the_backward(dtype):
    """phi with rows to spare: the kernels read what they need, and the gradient does not fit it."""
    hc, H, bo, dHn, dbi = make_case(2, 6, 32, torch.float32, phi_std=0.02)
    hc.phi = torch.nn.Parameter(torch.zeros((256, 24), device=DEV, dtype=dtype))
    bi, add = hc(H.clone().requires_grad_(True))
    with pytest.raises(RuntimeError, match="shape"):
        torch.autograd.backward([add(bo), bi], [dHn, dbi])
