// The layer's forward behind the router as one call (mlp.py:71-77, :84-100):
// routing, permutation, the grouped GEMMs and the combine, with the shared
// experts as experts n_experts .. n_experts + n_shared - 1 of the same
// permutation and GEMMs. Every token's last n_shared slots are theirs, with
// weight 1, so their rows of y lie behind the routed ones as [n_shared,
// n_tokens, dim], which is what the combine takes as the shared outputs.
//
// One host call and one workspace in place of nine to twelve wrapped calls and
// about twenty allocations, and two launches fewer for each shared expert plus
// one for their tile list: at one token of D 512, F 1024, 8 experts, top-2 and
// a shared expert the host, not the GPU, set the time (125 us a layer, of
// which the kernels take 63).
#include "moe_common.h"
#include "moe_gemm.h"

namespace astrai_moe {
namespace {

struct Sizes {
  int64_t n_tokens;
  int n_experts, top_k, n_shared;
  int64_t dim, dim_ffn;
  int dtype;
  bool packed;
};

// Byte offsets of the workspace's parts, 256-byte aligned.
struct Plan {
  int experts, slots, block_m;
  bool packed_up, packed_down;  // the GEMM reads the packed copies
  int64_t rows, tiles_len;
  bool gather, gather_ragged, gather_f32;
  int64_t topk_idx, topk_w, chunk_hist, chunk_base, offsets, sorted_token, sorted_w, token_pos, tiles, x_perm, h, y,
      gemm_ws, gemm_ws_bytes, bytes;
};

RowCounts row_counts(const Sizes& z) { return {z.n_tokens * z.top_k, z.n_experts, z.n_shared, z.n_tokens}; }

int check_sizes(const Sizes& z) {
  ASTRAI_REQUIRE(z.dtype == ASTRAI_MOE_BF16 || z.dtype == ASTRAI_MOE_F32, "forward: unsupported dtype %d", z.dtype);
  ASTRAI_REQUIRE(z.n_shared >= 0 && z.n_shared <= ASTRAI_MOE_MAX_TOPK, "forward: bad n_shared %d", z.n_shared);
  ASTRAI_REQUIRE(z.n_experts >= 1 && z.n_experts + z.n_shared <= ASTRAI_MOE_MAX_EXPERTS,
                 "forward: n_experts + n_shared must be in [1, %d] (got %d + %d)", ASTRAI_MOE_MAX_EXPERTS, z.n_experts,
                 z.n_shared);
  ASTRAI_REQUIRE(z.top_k >= 1 && z.top_k <= z.n_experts && z.top_k + z.n_shared <= ASTRAI_MOE_MAX_TOPK,
                 "forward: top_k must be in [1, n_experts] and top_k + n_shared at most %d (got %d + %d)",
                 ASTRAI_MOE_MAX_TOPK, z.top_k, z.n_shared);
  ASTRAI_REQUIRE(z.dim >= 1 && z.dim_ffn >= 1, "forward: dims must be >= 1");
  ASTRAI_REQUIRE(z.n_tokens >= 0 && z.n_tokens * (int64_t)(z.top_k + z.n_shared) < (1ll << 31),
                 "forward: n_tokens * (top_k + n_shared) must be in [0, 2^31)");
  return ASTRAI_MOE_OK;
}

Plan make_plan(const Sizes& z) {
  Plan p{};
  const int64_t size = z.dtype == ASTRAI_MOE_BF16 ? 2 : 4, T = z.n_tokens;
  p.experts = z.n_experts + z.n_shared;
  p.slots = z.top_k + z.n_shared;
  p.rows = T * p.slots;
  p.block_m = astrai_moe_select_block_m(T, z.n_experts, z.top_k, z.dim, z.dim_ffn, z.dtype);
  p.tiles_len = astrai_moe_tile_list_len(T, p.experts, p.slots, p.block_m);
  // Few rows read the live weights: the same bits, and their tiles of 32 weight
  // rows stream these better than the copies' blocks of 256 (8 experts, top-2, D
  // 4096, F 14336, 8 tokens 538 / 502 us a layer, 32 545 / 500).
  p.packed_up = z.packed && !few_rows(row_counts(z), p.block_m, z.dim, z.dim_ffn, true);
  p.packed_down = z.packed && !few_rows(row_counts(z), p.block_m, z.dim_ffn, z.dim, false);
  // the bf16 gate/up GEMM reads the token rows itself where its kernels do
  // (32-bit row offsets: x under 4 GiB)
  p.gather = z.dtype == ASTRAI_MOE_BF16 && !p.packed_up && mfma_shape_supported(z.dim, z.dim_ffn) && z.dim % 64 == 0 &&
             z.dim_ffn % 64 == 0 && T * z.dim * 2 < (1ll << 32);
  // (other dims: where x is aligned, below; 1500 tokens of D 1000, F 2664 with a
  // shared expert 162 us a layer with copied rows, 149 without)
  p.gather_ragged = z.dtype == ASTRAI_MOE_BF16 && !p.packed_up && mfma_shape_supported(z.dim, z.dim_ffn) && !p.gather &&
                    T * z.dim * 2 < (1ll << 32);
  p.gather_f32 = z.dtype == ASTRAI_MOE_F32 && T * z.dim * 4 < (1ll << 32) &&
                 mfma_f32_supported(z.dim, z.dim_ffn, true, p.block_m, nullptr, nullptr, nullptr);
  int64_t at = 0;
  auto part = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  p.topk_idx = part(p.rows * 4);
  p.topk_w = part(p.rows * size);
  p.chunk_hist = part(n_chunks(T) * p.experts * 4);
  p.chunk_base = part(n_chunks(T) * p.experts * 4);
  p.offsets = part((p.experts + 1) * 4);
  p.sorted_token = part(p.rows * 4);
  p.sorted_w = part(p.rows * size);
  p.token_pos = part(p.rows * 4);
  p.tiles = part(p.tiles_len * 4);
  p.h = part(p.rows * z.dim_ffn * size);
  p.y = part(p.rows * z.dim * size);
  p.x_perm = p.y;  // copied rows are read by the gate/up GEMM, before the down GEMM writes y
  // the 256-row GEMMs' scheduling block, and partial sums where the down GEMM
  // splits its last round (layer of D 1000, F 4040, 8 experts, top 2, 1000
  // tokens: halved tiles, 19.3 MiB in all where unused sums made it 83.3)
  if (p.block_m == kMfmaBigBM)
    p.gemm_ws_bytes = gemm_workspace_bytes(down_splits(row_counts(z), p.block_m, z.dim_ffn, z.dim, p.packed_down));
  p.gemm_ws = part(p.gemm_ws_bytes);
  p.bytes = at;
  return p;
}

}  // namespace
}  // namespace astrai_moe

using namespace astrai_moe;

extern "C" int64_t astrai_moe_forward_workspace_bytes(int64_t n_tokens, int n_experts, int top_k, int n_shared,
                                                      int64_t dim, int64_t dim_ffn, int dtype, int packed) {
  clear_error();
  const Sizes z{n_tokens, n_experts, top_k, n_shared, dim, dim_ffn, dtype, packed != 0};
  if (int rc = check_sizes(z)) return rc;
  return make_plan(z).bytes;
}

extern "C" int astrai_moe_forward(const void* x, const void* logits, const void* const* w_gate,
                                  const void* const* w_up, const void* const* w_down, const void* const* packed_gate_up,
                                  const void* const* packed_down, int dtype, int64_t n_tokens, int n_experts,
                                  int top_k, int n_shared, int64_t dim, int64_t dim_ffn, void* workspace,
                                  int64_t workspace_bytes, void* out, void* stream) {
  clear_error();
  const Sizes z{n_tokens, n_experts, top_k, n_shared, dim, dim_ffn, dtype, packed_gate_up != nullptr};
  int rc = check_sizes(z);
  if (rc) return rc;
  if (n_tokens == 0) return ASTRAI_MOE_OK;
  ASTRAI_REQUIRE(x && logits && w_gate && w_up && w_down && workspace && out, "forward: null buffer");
  ASTRAI_REQUIRE((packed_gate_up == nullptr) == (packed_down == nullptr), "forward: one packed table without the other");
  ASTRAI_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 256 == 0, "forward: workspace must be 256-byte aligned");
  const Plan p = make_plan(z);
  ASTRAI_REQUIRE(!z.packed || (dtype == ASTRAI_MOE_BF16 && dim % 256 == 0 && dim_ffn % 128 == 0 &&
                               mfma_shape_supported(dim, dim_ffn)),
                 "forward: unsupported shape for packed weights (dim %lld, dim_ffn %lld) or dtype", (long long)dim,
                 (long long)dim_ffn);
  ASTRAI_REQUIRE(workspace_bytes >= p.bytes, "forward: workspace holds %lld bytes, needs %lld",
                 (long long)workspace_bytes, (long long)p.bytes);
  // (a layer with packed copies copies such rows, whichever weights its GEMMs read)
  const bool x_aligned = reinterpret_cast<uintptr_t>(x) % 16 == 0;
  ASTRAI_REQUIRE(!p.gather || z.packed || x_aligned,
                 "forward: unsupported alignment (x must start on a 16-byte boundary)");
  char* const base = static_cast<char*>(workspace);
  auto i32 = [&](int64_t off) { return reinterpret_cast<int32_t*>(base + off); };
  int32_t *topk_idx = i32(p.topk_idx), *hist = i32(p.chunk_hist), *sorted_token = i32(p.sorted_token),
          *token_pos = i32(p.token_pos), *tiles = i32(p.tiles);
  void *topk_w = base + p.topk_w, *sorted_w = base + p.sorted_w, *h = base + p.h, *y = base + p.y;
  const bool gather = (p.gather || p.gather_ragged) && x_aligned, gather_f32 = p.gather_f32 && x_aligned;
  void* const x_perm = gather || gather_f32 ? nullptr : base + p.x_perm;
  void* const gws = p.gemm_ws_bytes > 0 ? base + p.gemm_ws : nullptr;
  hipStream_t s = static_cast<hipStream_t>(stream);

  // One chunk of tokens whose rows the GEMM reads itself: routing and
  // permutation in one workgroup. (Rows to copy want the permutation's grid, more
  // tokens its many workgroups.)
  if (n_tokens <= ASTRAI_MOE_CHUNK_TOKENS && x_perm == nullptr) {
    const RouteList list{sorted_token, sorted_w, token_pos, tiles,
                         (p.tiles_len - ASTRAI_MOE_TILE_HEADER) / ASTRAI_MOE_TILE_STRIDE, p.block_m};
    rc = launch_route_list(logits, dtype, n_tokens, n_experts, top_k, n_shared, list, s);
  } else if ((rc = launch_route(logits, dtype, n_tokens, n_experts, top_k, n_shared, topk_idx, topk_w, hist, s)) == 0) {
    rc = astrai_moe_permute(topk_idx, topk_w, hist, x, dtype, n_tokens, p.experts, p.slots, dim, p.block_m,
                            i32(p.offsets), sorted_token, sorted_w, token_pos, x_perm, tiles, p.tiles_len,
                            i32(p.chunk_base), stream);
  }
  if (rc) return rc;
  const RowCounts rows = row_counts(z);
  const GemmWorkspace ws{gws, p.gemm_ws_bytes};
  if (gather)
    rc = launch_gate_up_gather(x, sorted_token, tiles, p.tiles_len, w_gate, w_up, rows, dim, dim_ffn, p.block_m, h, ws,
                               s);
  else if (gather_f32)
    rc = launch_mfma_f32_gate_up(x, tiles, (p.tiles_len - ASTRAI_MOE_TILE_HEADER) / ASTRAI_MOE_TILE_STRIDE, w_gate, w_up,
                                 rows, dim, dim_ffn, h, nullptr, s, sorted_token);
  else
    rc = launch_gate_up(x_perm, tiles, p.tiles_len, p.packed_up ? packed_gate_up : w_gate,
                        p.packed_up ? packed_gate_up : w_up, dtype, rows, dim, dim_ffn, p.block_m, p.packed_up, h, ws, s);
  if (rc) return rc;
  rc = launch_down(h, tiles, p.tiles_len, p.packed_down ? packed_down : w_down, sorted_w, dtype, rows, dim_ffn, dim,
                   p.block_m, p.packed_down, y, ws, s);
  if (rc) return rc;
  const int64_t size = dtype == ASTRAI_MOE_BF16 ? 2 : 4;
  const void* shared = n_shared > 0 ? static_cast<const char*>(y) + n_tokens * top_k * dim * size : nullptr;
  return launch_combine(y, token_pos, nullptr, shared, n_shared, dtype, n_tokens, top_k, p.slots, dim, out, s);
}

// One dense expert (MLP.forward, mlp.py:22-25) in one call. A decoding batch
// needs neither the tile list (5 us to write and wait for, of 82 us at 24 rows
// of D 4096, F 14336) nor its allocations (8 rows of D 2048, F 5632, bound by the
// host with the separate calls, 28 -> 23 us; D 704, F 576, 800 rows 27 -> 18). More
// rows have a list for each GEMM, of the height it runs fastest on.
namespace astrai_moe {
namespace {

struct DensePlan {
  int block_m, block_m_down;
  bool few;  // (x and out allowing) both GEMMs on the few-row kernels
  int64_t len, len_down, tiles, tiles_down, h, gemm_ws, gemm_ws_bytes, bytes;
};

int check_dense(int64_t n_rows, int64_t dim, int64_t dim_ffn, int dtype) {
  ASTRAI_REQUIRE(dtype == ASTRAI_MOE_BF16 || dtype == ASTRAI_MOE_F32, "dense_forward: unsupported dtype %d", dtype);
  ASTRAI_REQUIRE(dim >= 1 && dim_ffn >= 1, "dense_forward: dims must be >= 1");
  ASTRAI_REQUIRE(n_rows >= 0 && n_rows < (1ll << 31), "dense_forward: n_rows must be in [0, 2^31)");
  return ASTRAI_MOE_OK;
}

DensePlan dense_plan(int64_t n_rows, int64_t dim, int64_t dim_ffn, int dtype) {
  DensePlan p{};
  p.block_m = p.block_m_down = astrai_moe_select_block_m(n_rows, 1, 1, dim, dim_ffn, dtype);
  if (dtype == ASTRAI_MOE_BF16 && mfma_shape_supported(dim, dim_ffn)) {
    const bool few_up = few_rows({n_rows, 1}, p.block_m, dim, dim_ffn, true);
    const bool few_down = few_rows({n_rows, 1}, p.block_m, dim_ffn, dim, false);
    p.few = few_up && few_down;
    if (p.block_m > kMfmaSmallBM) {
      if (!few_up) p.block_m = dense_gemm_block_m(n_rows, dim, dim_ffn, true);
      if (!few_down) p.block_m_down = dense_gemm_block_m(n_rows, dim_ffn, dim, false);
    }
  }
  p.len = astrai_moe_tile_list_len(n_rows, 1, 1, p.block_m);
  p.len_down = p.block_m_down == p.block_m ? 0 : astrai_moe_tile_list_len(n_rows, 1, 1, p.block_m_down);
  auto part = [&](int64_t bytes) {
    const int64_t here = p.bytes;
    p.bytes += (bytes + 255) / 256 * 256;
    return here;
  };
  p.tiles = part(p.len * 4);
  p.tiles_down = p.len_down > 0 ? part(p.len_down * 4) : p.tiles;
  p.h = part(n_rows * dim_ffn * (dtype == ASTRAI_MOE_BF16 ? 2 : 4));
  if (p.block_m == kMfmaBigBM || p.block_m_down == kMfmaBigBM)
    p.gemm_ws_bytes = gemm_workspace_bytes(down_splits({n_rows, 1}, p.block_m_down, dim_ffn, dim, false));
  p.gemm_ws = part(p.gemm_ws_bytes);
  return p;
}

}  // namespace
}  // namespace astrai_moe

extern "C" int64_t astrai_moe_dense_forward_workspace_bytes(int64_t n_rows, int64_t dim, int64_t dim_ffn, int dtype) {
  clear_error();
  if (int rc = check_dense(n_rows, dim, dim_ffn, dtype)) return rc;
  return dense_plan(n_rows, dim, dim_ffn, dtype).bytes;
}

extern "C" int astrai_moe_dense_forward(const void* x, const void* const* w_gate, const void* const* w_up,
                                        const void* const* w_down, int dtype, int64_t n_rows, int64_t dim,
                                        int64_t dim_ffn, void* workspace, int64_t workspace_bytes, void* out,
                                        void* stream) {
  clear_error();
  int rc = check_dense(n_rows, dim, dim_ffn, dtype);
  if (rc) return rc;
  if (n_rows == 0) return ASTRAI_MOE_OK;
  ASTRAI_REQUIRE(x && w_gate && w_up && w_down && workspace && out, "dense_forward: null buffer");
  ASTRAI_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 256 == 0,
                 "dense_forward: workspace must be 256-byte aligned");
  const DensePlan p = dense_plan(n_rows, dim, dim_ffn, dtype);
  ASTRAI_REQUIRE(workspace_bytes >= p.bytes, "dense_forward: workspace holds %lld bytes, needs %lld",
                 (long long)workspace_bytes, (long long)p.bytes);
  char* const base = static_cast<char*>(workspace);
  int32_t* const tiles = reinterpret_cast<int32_t*>(base + p.tiles);
  int32_t* const tiles_down = reinterpret_cast<int32_t*>(base + p.tiles_down);
  void* const h = base + p.h;
  void* const gws = p.gemm_ws_bytes > 0 ? base + p.gemm_ws : nullptr;
  if (p.few && mfma_gate_up_supported(dim, dim_ffn, p.block_m, x, h) &&
      mfma_down_supported(dim_ffn, dim, p.block_m, h, out))
    return launch_few_dense(x, w_gate, w_up, w_down, n_rows, dim, dim_ffn, p.block_m, h, out,
                            static_cast<hipStream_t>(stream));
  const int64_t len_down = p.len_down > 0 ? p.len_down : p.len;
  if ((rc = launch_dense_tiles(n_rows, p.block_m, p.len, tiles, p.block_m_down, p.len_down, tiles_down,
                               static_cast<hipStream_t>(stream))))
    return rc;
  if ((rc = astrai_moe_gemm_gate_up(x, tiles, p.len, w_gate, w_up, dtype, n_rows, 1, dim, dim_ffn, p.block_m, h, gws,
                                    p.gemm_ws_bytes, stream)))
    return rc;
  return astrai_moe_gemm_down(h, tiles_down, len_down, w_down, nullptr, dtype, n_rows, 1, dim_ffn, dim, p.block_m_down,
                              out, gws, p.gemm_ws_bytes, stream);
}
