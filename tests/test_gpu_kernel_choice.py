"""Kernels and dispatch lines that the launchers pick by size, at the sizes where they can go wrong."""

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
    # 1024 workgroups (the most that take it) and 1028
    (4, 512, 1024, torch.bfloat16), (4, 513, 1024, torch.bfloat16)])
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
