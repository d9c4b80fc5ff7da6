"""bf16 layers whose dims are multiples of 8 but not of 64 on the matrix-core
kernels: the last K step of every GEMM is partial and staged with zeros behind
the rows. Remainders of 8, 40 and 56 of a step, one step and several, at row
counts of every tile height, against the oracle with the tolerances of
test_gpu_layer.py and test_gpu_backward.py; and what lies behind a row (the
next row) must not reach its output, NaN included."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import ops
from test_gpu_backward import _check_moe, _random_layer
from test_gpu_layer import check_layer

pytestmark = pytest.mark.gpu

DIMS = [(72, 120), (1000, 424), (184, 1080)]


@pytest.mark.parametrize("dim,dim_ffn", DIMS)
@pytest.mark.parametrize("n_tok", [3, 130, 257, 700])  # 32-, 64-, 128- and 256-row tiles at 4 experts, top-2
def test_layer(gpu, dim, dim_ffn, n_tok):
    assert ops.matrix_core_supported(dim, dim_ffn, torch.bfloat16)
    layer = _random_layer(gpu, dim, dim_ffn, 4, 1, 2, torch.bfloat16, seed=dim + n_tok).requires_grad_(False)
    x = torch.randn(1, n_tok, dim, device=gpu).to(torch.bfloat16)
    check_layer(layer, x, f"d{dim}_f{dim_ffn}_t{n_tok}")


@pytest.mark.parametrize("dim,dim_ffn", DIMS)
def test_training(gpu, dim, dim_ffn):
    layer = _random_layer(gpu, dim, dim_ffn, 4, 1, 2, torch.bfloat16, seed=dim)
    x = torch.randn(1, 333, dim, device=gpu).to(torch.bfloat16)
    _check_moe(layer, x, f"d{dim}_f{dim_ffn}")


@pytest.mark.parametrize("n_tok", [40, 700])
def test_rows_do_not_read_past_their_end(gpu, n_tok):
    layer = _random_layer(gpu, 1000, 424, 1, 0, 1, torch.bfloat16, seed=1).requires_grad_(False)
    x = torch.randn(1, n_tok, 1000, device=gpu).to(torch.bfloat16)
    clean = layer(x)
    x[0, 1::2] = float("nan")  # every even row is followed by NaN
    got = layer(x)
    assert torch.equal(got[0, ::2], clean[0, ::2])
    assert got[0, 1::2].isnan().all()


def test_unaligned_rows_still_run(gpu):
    # 8-byte aligned rows: the general kernels, as before
    layer = _random_layer(gpu, 1000, 424, 4, 0, 2, torch.bfloat16, seed=2).requires_grad_(False)
    flat = torch.randn(1 + 4 + 65 * 1000, device=gpu).to(torch.bfloat16)
    x = flat[4:4 + 65 * 1000].view(1, 65, 1000)
    assert x.data_ptr() % 16 == 8
    check_layer(layer, x, "unaligned")


def test_training_on_a_64_row_list(gpu):
    # the general kernels' lists, which such dims trained on before the matrix cores took them
    dim, dim_ffn, e = 72, 120, 4
    x = torch.randn(130, dim, device=gpu).to(torch.bfloat16)
    route = ops.moe_route(torch.randn(130, e, device=gpu).to(torch.bfloat16), 2)
    ws = [[(torch.randn(*s, device=gpu) * 0.1).bfloat16() for _ in range(e)]
          for s in ((dim_ffn, dim), (dim_ffn, dim), (dim, dim_ffn))]
    tg, tu, td = (ops.expert_weight_table(w, tuple(w[0].shape)) for w in ws)

    def step(block_m):
        perm = ops.moe_permute(route, x, e, block_m)
        h, gu = ops.moe_gemm_gate_up_train(perm.x_perm, perm.tiles, tg, tu, e, dim_ffn)
        y, y_unw = ops.moe_gemm_down_train(h, perm.tiles, td, perm.sorted_w, e, dim)
        dg, du = ops.moe_gemm_dgrad_down(y, perm.tiles, td, gu, e)
        return h, gu, y, y_unw, dg, du, ops.moe_gemm_dgrad_gate_up(dg, du, perm.tiles, tg, tu, e, dim)

    for got, want in zip(step(64), step(256)):
        # values rounded to bf16 at the same points, up to three in a chain; fp32 sums in another order
        torch.testing.assert_close(got, want, rtol=3e-2, atol=3e-2 * want.abs().max().item())
    with pytest.raises(ValueError, match="block_m"):
        step(128)


@pytest.mark.parametrize("dim,dim_ffn", [(72, 328), (1000, 424), (2056, 136)])
@pytest.mark.parametrize("n_tok", [1, 32, 33, 300, 1400])
def test_gathered_rows_are_the_copied_ones(gpu, n_tok, dim, dim_ffn):
    # the one-call forward reads the token rows itself, the separate calls copy them
    layer = _random_layer(gpu, dim, dim_ffn, 4, 0, 2, torch.bfloat16, seed=n_tok).requires_grad_(False)
    x = torch.randn(1, n_tok, dim, device=gpu).to(torch.bfloat16)
    assert not ops.gather_supported(n_tok, dim, dim_ffn, x.dtype)
    assert torch.equal(layer(x)[0], layer._routed_forward(x[0], layer._current(x.dtype, x.device)))
