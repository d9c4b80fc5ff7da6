"""The GEMMs for few rows (gemm_few_kernel): fewer K steps than the workgroup
has waves, partial last steps and column tiles, one run of 32 rows and several,
one token over many experts; MLP and layer against the oracle."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import ops
from astrai_amd.model.components.mlp import MLP
from oracle import moe_ref as R
from test_gpu_backward import _random_layer
from test_gpu_layer import check_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,dim_ffn", [(64, 64), (72, 328), (512, 1408), (1096, 200)])
@pytest.mark.parametrize("n_tok", [1, 16, 32, 33, 95, 128, 160, 256])
def test_mlp(gpu, n_tok, dim, dim_ffn):
    torch.manual_seed(n_tok + dim)
    mlp = MLP(dim, dim_ffn)
    for m in (mlp.up, mlp.gate, mlp.down):
        m.reset_parameters()
    mlp = mlp.to(device=gpu, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(n_tok, dim, device=gpu).to(torch.bfloat16)
    got = mlp(x)
    want = R.expert_mlp(x, R.ExpertWeights(mlp.gate.weight, mlp.up.weight, mlp.down.weight))
    # h and y are each rounded to bf16 (8 bits) at the same points; sums in another order
    torch.testing.assert_close(got, want, rtol=2e-2, atol=2e-3)


@pytest.mark.parametrize("n_tok,n_exp,top_k,n_shared", [(1, 64, 6, 1), (5, 8, 2, 2), (47, 8, 2, 0), (12, 128, 8, 0), (150, 8, 2, 1)])
def test_layer(gpu, n_tok, n_exp, top_k, n_shared):
    layer = _random_layer(gpu, 512, 640, n_exp, n_shared, top_k, torch.bfloat16, seed=n_exp).requires_grad_(False)
    x = torch.randn(1, n_tok, 512, device=gpu).to(torch.bfloat16)
    check_layer(layer, x, f"t{n_tok}_e{n_exp}_k{top_k}_s{n_shared}")
    live = layer(x)
    layer.pack_weights = True
    assert layer.uses_packed_weights(x.dtype)
    assert torch.equal(layer(x), live)  # packed copies: the same bits


@pytest.mark.parametrize("n_tok", [1200, 2000, 4400])
def test_one_call_where_the_down_list_is_shorter(gpu, n_tok):
    # listed on 256-row tiles; in one call the down GEMM has a list of 128 or 64 rows, or (4400) splits
    # the last round of 256-row ones as well: the same sums in an order of their own at most
    dim, dim_ffn = 4096, 14336
    torch.manual_seed(n_tok)
    ws = [(torch.randn(*s, device=gpu) * 0.02).bfloat16() for s in ((dim_ffn, dim), (dim_ffn, dim), (dim, dim_ffn))]
    tables = [ops.expert_weight_table([w], tuple(w.shape)) for w in ws]
    x = torch.randn(n_tok, dim, device=gpu).bfloat16()
    assert ops.dense_block_m(n_tok, dim, dim_ffn, x.dtype) == 256
    listed = ops.moe_dense_mlp(x, *tables, dim_ffn, tiles=ops.dense_tiles(n_tok, 256, x.device))
    got = ops.moe_dense_mlp(x, *tables, dim_ffn)
    torch.testing.assert_close(got, listed, rtol=2e-2, atol=2e-3)
    want = R.expert_mlp(x[-300:], R.ExpertWeights(*ws))
    torch.testing.assert_close(got[-300:], want, rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("dim,dim_ffn", [(64, 64), (72, 328), (512, 1408), (1536, 4096)])
@pytest.mark.parametrize("n_tok", [0, 1, 32, 33, 64, 65, 95, 96, 128, 129, 256, 257, 900])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_one_call_is_the_listed_calls(gpu, n_tok, dim, dim_ffn, dtype):
    # one dense expert without a tile list (few rows), or with one of each
    # GEMM's own height (900 rows of 1536, 4096: 256 and 64), and with one list:
    # the same bits
    torch.manual_seed(n_tok)
    ws = [(torch.randn(*s, device=gpu) * 0.05).to(dtype) for s in ((dim_ffn, dim), (dim_ffn, dim), (dim, dim_ffn))]
    tables = [ops.expert_weight_table([w], tuple(w.shape)) for w in ws]
    x = torch.randn(n_tok, dim, device=gpu).to(dtype)
    tiles = ops.dense_tiles(n_tok, ops.dense_block_m(n_tok, dim, dim_ffn, dtype), x.device)
    listed = ops.moe_dense_mlp(x, *tables, dim_ffn, tiles=tiles)
    out = torch.full_like(x, torch.nan)
    assert ops.moe_dense_mlp(x, *tables, dim_ffn, out=out) is out
    assert torch.equal(out, listed) and torch.equal(ops.moe_dense_mlp(x, *tables, dim_ffn), listed)
