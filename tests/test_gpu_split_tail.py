"""The 256-row down-sized GEMMs split their last round from 64 K steps on, a
partial last step counted: the workspaces of the one-call forwards and of the
separate calls hold the partial sums exactly there, and at the first such sizes
the split runs and sums to the reference."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import loader, ops
from test_gpu_kernels import BF16_TOL, _experts, _routing

SIZES = [(4024, False), (4032, False), (4040, True), (4088, True), (4096, True)]


@pytest.mark.parametrize("dim_ffn,split", SIZES)
def test_workspaces_hold_the_partial_sums(dim_ffn, split):
    lib, t, dim = loader.library(), 8192, 1000
    sums = lib.astrai_moe_gemm_workspace_bytes(1) - lib.astrai_moe_gemm_workspace_bytes(0)
    rows = 2 * t * (dim + dim_ffn) * 2  # h and y
    layer = lib.astrai_moe_forward_workspace_bytes(t, 8, 2, 0, dim, dim_ffn, 1, 0)
    assert (layer > rows + sums) == split, layer
    # few tiles, which are halved and not split: none
    assert lib.astrai_moe_forward_workspace_bytes(640, 8, 2, 0, dim, dim_ffn, 1, 0) < sums
    assert lib.astrai_moe_dense_forward_workspace_bytes(1024, 4096, dim_ffn, 1) < sums
    x = torch.empty(0, dtype=torch.bfloat16)
    assert (ops._workspace(x, dim, dim_ffn, 256, down=True)[1] > sums) == split


@pytest.mark.gpu
@pytest.mark.parametrize("dim_ffn,split", SIZES)
def test_split_of_a_partial_last_step(gpu, dim_ffn, split):
    bf16, t, e, dim = torch.bfloat16, 8192, 8, 1000
    route = _routing(gpu, t, e, 2, bf16, seed=3)
    h = torch.randn(2 * t, dim_ffn, device=gpu).to(bf16)
    perm = ops.moe_permute(route, torch.zeros(t, dim, device=gpu, dtype=bf16), e, 256)
    experts = _experts(gpu, e, dim, dim_ffn, bf16, seed=6)
    td = ops.expert_weight_table([w.down for w in experts], (dim, dim_ffn))
    y = ops.moe_gemm_down(h, perm.tiles, td, perm.sorted_w, e, dim, 256)
    whole = ops.moe_gemm_down(h, perm.tiles, td, perm.sorted_w, e, dim, 256, balance=False)
    # ~68 row tiles x 4 column tiles: about 16 left for the last round, cut in eight
    assert torch.equal(y, whole) != split
    torch.testing.assert_close(y, whole, **BF16_TOL)
    offs = perm.expert_offsets.tolist()
    for w, a, b in zip(experts, offs, offs[1:]):
        ref = (h[a:b].float() @ w.down.float().t()).to(bf16) * perm.sorted_w[a:b].unsqueeze(-1)
        torch.testing.assert_close(y[a:b], ref, **BF16_TOL)
