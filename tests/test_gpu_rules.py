"""Which kernels a layer's GEMMs run on where the rules' lines lie: the rules
see a load's sizes only, so a choice has to hold for skewed routers too."""

from __future__ import annotations

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from astrai_amd.extension import ops
from test_gpu_backward import _random_layer
from test_gpu_layer import check_layer

pytestmark = pytest.mark.gpu


def _gemms(run):
    """Names of the GEMM kernels that ``run`` launches, in order."""
    run()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA, ProfilerActivity.CPU]) as p:
        run()
        torch.cuda.synchronize()
    names = [(e.time_range.start, torch._C._demangle(e.name)) for e in p.events() if "gemm_" in e.name and "kernel" in e.name]
    return [n for _, n in sorted(names)]


@pytest.mark.parametrize("n_tok,n_exp,top_k,n_shared,dim,dim_ffn,up,down", [
    # 8 row tiles of 128 rows if even, 9 if not: 32 columns of 128 fill one round exactly or take two
    (256, 8, 2, 0, 4096, 128, "gemm_mfma_kernel", "TileCfg<128, 256"),
    # one round of long 256-row tiles that is not split along K (more than half a round): narrower tiles
    (640, 8, 2, 0, 1000, 4096, "gemm_stream_kernel", "TileCfg<128, 128"),
    (640, 8, 2, 0, 1000, 4040, "gemm_stream_kernel", "TileCfg<128, 128"),
    # a short last round of them that is
    (8192, 8, 2, 0, 1000, 4040, "gemm_stream_kernel", "gemm_stream_kernel"),
])
def test_tiles(gpu, n_tok, n_exp, top_k, n_shared, dim, dim_ffn, up, down):
    layer = _random_layer(gpu, dim, dim_ffn, n_exp, n_shared, top_k, torch.bfloat16, seed=1).requires_grad_(False)
    x = torch.randn(1, n_tok, dim, device=gpu).to(torch.bfloat16)
    first, second = _gemms(lambda: layer(x))[:2]
    assert up in first and down in second, (first, second)


FEW, LIST = "gemm_few_kernel", "gemm_mfma_kernel"


@pytest.mark.parametrize("n_tok,n_exp,top_k,n_shared,dim,dim_ffn,up,down", [
    # 8 routed rows per expert and the next (the down GEMM has 128 tiles: half the compute units)
    (32, 8, 2, 0, 4096, 128, FEW, FEW),
    (33, 8, 2, 0, 4096, 128, FEW, LIST),
    (96, 8, 2, 0, 4096, 128, FEW, LIST),
    # shared experts: two runs of their rows, and three
    (64, 32, 2, 1, 4096, 128, FEW, FEW),
    (65, 32, 2, 1, 4096, 128, FEW, LIST),
    # small layers: a quarter of the compute units, an eighth and many K steps
    (80, 8, 2, 0, 2048, 128, FEW, FEW),
    (96, 8, 2, 0, 2048, 768, LIST, LIST),
    (192, 8, 2, 0, 1024, 768, LIST, FEW),
    (193, 8, 2, 0, 1024, 768, LIST, LIST),
])
def test_few_rows(gpu, n_tok, n_exp, top_k, n_shared, dim, dim_ffn, up, down):
    layer = _random_layer(gpu, dim, dim_ffn, n_exp, n_shared, top_k, torch.bfloat16, seed=1).requires_grad_(False)
    x = torch.randn(1, n_tok, dim, device=gpu).to(torch.bfloat16)
    first, second = _gemms(lambda: layer(x))[:2]
    assert up in first and down in second, (first, second)


@pytest.mark.parametrize("n_tok,dim_ffn,listed,rows", [
    (64, 4096, False, 32), (65, 4096, False, 64), (95, 4096, False, 64), (96, 4096, False, 64), (95, 1024, False, 32),
    (95, 4096, True, 32), (96, 4096, True, 64),
])
def test_few_row_tiles_fit_the_list(gpu, n_tok, dim_ffn, listed, rows):
    # one expert: 64-row tiles only over row tiles of that height, which a list of 65 to 95 rows has not
    ws = [(torch.randn(*s, device=gpu) * 0.02).bfloat16() for s in ((dim_ffn, 512), (dim_ffn, 512), (512, dim_ffn))]
    tables = [ops.expert_weight_table([w], tuple(w.shape)) for w in ws]
    x = torch.randn(n_tok, 512, device=gpu).bfloat16()
    tiles = ops.dense_tiles(n_tok, ops.dense_block_m(n_tok, 512, dim_ffn, x.dtype), x.device) if listed else None
    names = _gemms(lambda: ops.moe_dense_mlp(x, *tables, dim_ffn, tiles=tiles))
    assert len(names) == 2 and all(f"FewCfg<{rows}, 32>" in n for n in names), names


def test_few_rows_of_a_packed_layer_read_the_live_weights(gpu):
    layer = _random_layer(gpu, 512, 1024, 8, 1, 2, torch.bfloat16, seed=1).requires_grad_(False)
    layer.pack_weights = True
    x = torch.randn(1, 8, 512, device=gpu).to(torch.bfloat16)
    first, second = _gemms(lambda: layer(x))[:2]
    # gemm_few_kernel<..., gate/up, gather, packed, dense>
    assert "true, true, false, false>" in first and "false, false, false, false>" in second, (first, second)


@pytest.mark.parametrize("n_tok,dim,n_shared,cols", [
    (1024, 512, 0, 32),  # 36 row tiles x 8: a compute unit's share is 1.1 of 64 columns, 2.3 of 32
    (128, 4096, 0, 64),  # 8 x 64: 2 or 4
    (2048, 2048, 1, 64),  # past the shares that can gain
    (1500, 96, 1, 32),  # columns no multiple of 64
])
def test_fp32_down_columns(gpu, n_tok, dim, n_shared, cols):
    layer = _random_layer(gpu, dim, 160, 8, n_shared, 2, torch.float32, seed=1).requires_grad_(False)
    x = torch.randn(1, n_tok, dim, device=gpu)
    first, second = _gemms(lambda: layer(x))[:2]
    assert f"gemm_f32_mfma_kernel<{cols}, false" in second, second
    check_layer(layer, x, f"d{dim}_t{n_tok}_s{n_shared}")


@pytest.mark.parametrize("rows,m,n,wt", [
    ([2000, 0, 2100, 1901], 1024, 1024, 64),  # 256 tiles of 128 x 128: one round
    ([500, 0, 600, 401], 1024, 1024, 32),  # the same of fewer rows
    ([2000, 0, 2100, 1901], 1024, 512, 32),  # half a round
    ([1301, 1, 1500, 2000], 1020, 996, 64),  # partial tiles and K steps
])
def test_fp32_weight_gradient_tiles(gpu, rows, m, n, wt):
    g = torch.Generator(device=gpu).manual_seed(m + n)
    a = torch.randn(sum(rows), m, generator=g, device=gpu)
    b = torch.randn(sum(rows), n, generator=g, device=gpu)
    first = [sum(rows[:i]) for i in range(len(rows) + 1)]
    offsets = torch.tensor(first, dtype=torch.int32, device=gpu)
    names = _gemms(lambda: ops.moe_gemm_wgrad(a, b, offsets, len(rows)))
    assert [f"gemm_f32_wgrad_kernel<{wt}>" in k for k in names] == [True], names
    dw = ops.moe_gemm_wgrad(a, b, offsets, len(rows))
    for e, (i, j) in enumerate(zip(first, first[1:])):
        if j > i:
            want = a[i:j].double().t() @ b[i:j].double()
            # at most 2100 products of N(0, 1) values in fp32: error of about 1e-7 of sqrt(2100) each
            assert (dw[e] - want).abs().max().item() < 2e-6 * (j - i) ** 0.5 * 10
