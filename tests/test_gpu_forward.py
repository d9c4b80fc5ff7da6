"""The layer's one-call forward (astrai_moe_forward): shared experts as experts
of the same permutation and GEMMs, against the oracle at every tile height,
with copied rows (fp32) and gathered ones, and where it does not apply (slots
or shapes beyond it) the separate calls."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import loader, ops
from test_gpu_backward import _random_layer
from test_gpu_layer import check_layer


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_exp,n_shared,top_k", [(4, 1, 2), (8, 3, 1), (1, 2, 1), (40, 1, 31), (40, 1, 32)])
@pytest.mark.parametrize("n_tok", [1, 33, 160, 700])
def test_shared_experts_in_one_call(gpu, n_tok, n_exp, n_shared, top_k, dtype):
    layer = _random_layer(gpu, 192, 320, n_exp, n_shared, top_k, dtype, seed=n_tok + n_exp).requires_grad_(False)
    x = torch.randn(1, n_tok, 192, device=gpu).to(dtype)
    assert layer._joint(layer._current(dtype, x.device)) == (top_k + n_shared <= 32)
    check_layer(layer, x, f"e{n_exp}_s{n_shared}_k{top_k}_t{n_tok}")


@pytest.mark.gpu
def test_shared_experts_of_another_width(gpu):
    layer = _random_layer(gpu, 192, 320, 4, 1, 2, torch.bfloat16, seed=3)
    layer.shared_experts[0] = _random_layer(gpu, 192, 256, 1, 0, 1, torch.bfloat16, seed=4).routed_experts[0]
    layer.requires_grad_(False)
    x = torch.randn(1, 70, 192, device=gpu).to(torch.bfloat16)
    assert layer._current(x.dtype, x.device).joint is None
    check_layer(layer, x, "narrow shared expert")


@pytest.mark.gpu
def test_shared_experts_switched_off(gpu):
    # n_shared_experts decides, as in training and in the reference (mlp.py:75-76), not the modules there are
    layer = _random_layer(gpu, 128, 192, 4, 1, 2, torch.bfloat16, seed=7).requires_grad_(False)
    x = torch.randn(1, 50, 128, device=gpu).to(torch.bfloat16)
    with_shared = layer(x)
    layer.n_shared_experts = 0
    out = layer(x)
    assert not torch.equal(out, with_shared)
    assert torch.equal(out[0], layer._routed_forward(x[0], layer._current(x.dtype, x.device)))
    layer.n_shared_experts = 1
    assert torch.equal(layer(x), with_shared)


def test_copied_rows_need_no_place_of_their_own():
    # fp32 and ragged layers (whose unaligned x is copied), packed ones: h, y and some lists
    size = loader.library().astrai_moe_forward_workspace_bytes
    for dim, dim_ffn, dtype, packed in ((512, 1024, 0, 0), (1000, 2664, 1, 0), (512, 1024, 1, 1)):
        rows, item = 4096 * 3, 4 if dtype == 0 else 2
        assert size(4096, 8, 2, 1, dim, dim_ffn, dtype, packed) < rows * ((dim + dim_ffn) * item + 100) + (1 << 20)


@pytest.mark.gpu
def test_separate_calls_of_a_packed_layer_with_shared_experts(gpu):
    # the packed tables hold the shared experts' copies too; the separate calls take the routed ones
    layer = _random_layer(gpu, 256, 512, 4, 2, 2, torch.bfloat16, seed=5).requires_grad_(False)
    x = torch.randn(1, 300, 256, device=gpu).to(torch.bfloat16)
    st = layer._current(x.dtype, x.device)

    def apart():
        return layer._routed_forward(x[0], st, layer._shared_forward(x[0], st))

    live = apart()
    layer.pack_weights = True
    assert torch.equal(apart(), live)


@pytest.mark.gpu
@pytest.mark.parametrize("n_tok", [5, 40, 700])
def test_packed_layers_take_unaligned_rows(gpu, n_tok):
    # copied, also where few rows read the live weights: the bits of the aligned rows
    layer = _random_layer(gpu, 256, 512, 4, 1, 2, torch.bfloat16, seed=n_tok).requires_grad_(False)
    layer.pack_weights = True
    flat = torch.randn(4 + n_tok * 256, device=gpu).to(torch.bfloat16)
    x = flat[4:].view(1, n_tok, 256)
    assert x.data_ptr() % 16 == 8
    assert torch.equal(layer(x), layer(x.clone()))


def _peak(run):
    run()  # allocations that stay
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    run()
    return torch.cuda.max_memory_allocated() - before


@pytest.mark.gpu
@pytest.mark.parametrize("pack", [False, True])
@pytest.mark.parametrize("n_tok,joint", [(4096, True), (20000, False)])
def test_shared_experts_memory_is_bounded(gpu, n_tok, joint, pack):
    # two shared experts of F 2048: 32 MB of h at 4096 tokens, 156 at 20000, past
    # the line where they run by themselves before the routed experts
    layer = _random_layer(gpu, 256, 2048, 4, 2, 1, torch.bfloat16, seed=5).requires_grad_(False)
    layer.pack_weights = pack
    x = torch.randn(1, n_tok, 256, device=gpu).to(torch.bfloat16)
    assert ops.layer_forward_pays(n_tok, 2, 1, 2048, 2) == joint
    st = layer._current(x.dtype, x.device)

    def apart():
        return layer._routed_forward(x[0], st, layer._shared_forward(x[0], st))

    extra = _peak(lambda: layer(x)) - _peak(apart)
    assert extra <= (ops.SHARED_ROWS_BYTES if joint else 1 << 20), extra
    assert torch.allclose(layer(x)[0].float(), apart().float(), rtol=2e-2, atol=2e-2)
    check_layer(layer, x[:, :256], "first tokens")


def test_one_call_takes_the_rows_that_fit_31_bits():
    assert ops.layer_forward_pays((1 << 31) // 3 - 1, 1, 2, 0, 2) and not ops.layer_forward_pays((1 << 31) // 3 + 1, 1, 2, 0, 2)


def test_arguments_are_checked_on_the_host():
    lib = loader.library()
    size = lib.astrai_moe_forward_workspace_bytes
    assert size(10, 8, 2, 1, 64, 128, 1, 0) > 0
    for args, word in (((10, 8, 9, 0, 64, 128, 1, 0), "top_k"), ((10, 40, 32, 1, 64, 128, 1, 0), "top_k + n_shared"),
                       ((10, 1024, 2, 1, 64, 128, 1, 0), "n_experts + n_shared"), ((10, 8, 2, 0, 64, 128, 7, 0), "dtype"),
                       ((10, 8, 2, 0, 0, 128, 1, 0), "dims"), ((1 << 30, 8, 2, 0, 64, 128, 1, 0), "n_tokens")):
        assert size(*args) == -1 and word in loader.last_error()

    def call(workspace=256, nbytes=1 << 40, gate=16, tokens=10):
        return lib.astrai_moe_forward(16, 16, gate, 16, 16, None, None, 1, tokens, 8, 2, 1, 64, 128, workspace, nbytes,
                                      16, None)

    assert call(tokens=0) == 0
    assert call(gate=None) == -1 and "null" in loader.last_error()
    assert call(workspace=16) == -1 and "256-byte aligned" in loader.last_error()
    assert call(nbytes=100) == -1 and "needs" in loader.last_error()
    assert not ops.layer_forward_supported(8, 1, 32) and ops.layer_forward_supported(8, 1, 31)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n_exp,top_k", [(1, 1), (3, 2), (64, 6), (130, 32), (1000, 8)])
@pytest.mark.parametrize("n_tok", [1, 31, 32, 33])
def test_one_chunk_is_routed_and_listed_by_one_kernel(gpu, n_tok, n_exp, top_k, dtype):
    # up to 32 tokens: the same bits as the separate route and permute kernels
    # (zero rows among the tokens: every probability tied)
    layer = _random_layer(gpu, 64, 64, n_exp, 0, top_k, dtype, seed=n_tok + n_exp).requires_grad_(False)
    x = torch.randn(1, n_tok, 64, device=gpu).to(dtype)
    x[0, ::5] = 0
    st = layer._current(dtype, x.device)
    for _ in range(2):
        assert torch.equal(layer(x)[0], layer._routed_forward(x[0], st))


@pytest.mark.gpu
@pytest.mark.parametrize("n_tok", [5, 32])
def test_one_chunk_of_long_rows(gpu, n_tok):
    # rows of 3072, whose permutation lists whole groups of tiles first: one chunk has none
    layer = _random_layer(gpu, 3072, 64, 8, 0, 2, torch.bfloat16, seed=n_tok).requires_grad_(False)
    x = torch.randn(1, n_tok, 3072, device=gpu).to(torch.bfloat16)
    assert torch.equal(layer(x)[0], layer._routed_forward(x[0], layer._current(x.dtype, x.device)))
    check_layer(layer, x, f"t{n_tok}")
