"""GEMMs of few 256-row tiles, which take 128-row halves of them and narrower
columns: the same bits as the training forward's kernels, which take whole
tiles, at experts of no row up to three tiles, half tiles full and one over,
partial column tiles and partial K steps, copied and gathered rows."""

from __future__ import annotations

import pytest
import torch

from astrai_amd.extension import ops

ROWS = [0, 1, 127, 128, 129, 255, 256, 257, 385, 700]


@pytest.mark.gpu
@pytest.mark.parametrize("dim,dim_ffn", [
    (512, 1024),  # both GEMMs on 128 x 128 tiles
    (2048, 128),  # down on halves of 256 columns where 128 columns take two rounds
    (200, 456),  # partial K steps and column tiles
])
@pytest.mark.parametrize("rows", [ROWS, ROWS[::-1], [300], [1100], [40] * 12])
def test_same_bits_as_whole_tiles(gpu, dim, dim_ffn, rows):
    bf16 = torch.bfloat16
    e, t = len(rows), sum(rows)
    g = torch.Generator(device=gpu).manual_seed(dim + t)
    owner = torch.repeat_interleave(torch.arange(e, device=gpu), torch.tensor(rows, device=gpu))
    owner = owner[torch.randperm(t, generator=g, device=gpu)]
    logits = torch.zeros(t, e, device=gpu, dtype=bf16)
    logits[torch.arange(t, device=gpu), owner] = 8.0
    x = torch.randn(t, dim, generator=g, device=gpu).to(bf16)

    def weights(out, inp):
        return [(torch.randn(out, inp, generator=g, device=gpu) * inp ** -0.5).to(bf16) for _ in range(e)]

    ws = weights(dim_ffn, dim), weights(dim_ffn, dim), weights(dim, dim_ffn)
    tg, tu, td = (ops.expert_weight_table(w, tuple(w[0].shape)) for w in ws)
    perm = ops.moe_permute(ops.moe_route(logits, 1), x, e, 256)
    h_ref, _ = ops.moe_gemm_gate_up_train(perm.x_perm, perm.tiles, tg, tu, e, dim_ffn)
    y_ref, _ = ops.moe_gemm_down_train(h_ref, perm.tiles, td, perm.sorted_w, e, dim)
    for _ in range(2):
        assert torch.equal(ops.moe_gemm_gate_up(perm.x_perm, perm.tiles, tg, tu, e, dim_ffn, 256), h_ref)
        if ops.gather_supported(t, dim, dim_ffn, bf16):
            assert torch.equal(ops.moe_gemm_gate_up_gather(x, perm.sorted_token, perm.tiles, tg, tu, e, dim_ffn, 256),
                               h_ref)
        assert torch.equal(ops.moe_gemm_down(h_ref, perm.tiles, td, perm.sorted_w, e, dim, 256), y_ref)
    first = perm.expert_offsets.tolist()
    for i in range(e):
        a = slice(first[i], first[i + 1])
        ref = perm.x_perm[a].float() @ ws[0][i].float().t(), perm.x_perm[a].float() @ ws[1][i].float().t()
        ref = torch.nn.functional.silu(ref[0].to(bf16).float()).to(bf16).float() * ref[1].to(bf16).float()
        # h in bf16 from projections and silu rounded to bf16: a unit or two
        assert torch.allclose(h_ref[a].float(), ref, rtol=2e-2, atol=2e-2)
        ref = (h_ref[a].float() @ ws[2][i].float().t()).to(bf16).float() * perm.sorted_w[a].float()[:, None]
        assert torch.allclose(y_ref[a].float(), ref, rtol=2e-2, atol=2e-2)
