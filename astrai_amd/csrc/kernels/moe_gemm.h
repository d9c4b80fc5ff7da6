// Internal interface between the entry points (moe_gemm.hip, moe_forward.hip)
// and the kernels of the other files.
#pragma once

#include "moe_common.h"

#include <algorithm>
#include <cmath>

namespace astrai_moe {

// Row-tile heights of the bf16 matrix-core kernels. The large tile serves
// prefill-sized expert loads; the small one serves decode-sized loads, where
// the work is streaming expert weights and padding rows to 256 would make the
// kernel compute-bound on empty rows.
constexpr int kMfmaBigBM = 256;
constexpr int kMfmaSmallBM = 32;
// Mid-sized expert loads (about 48-128 rows per expert): one 64-row tile per
// expert reads its weights once, where 32-row tiles would stream them twice or
// more and 256-row tiles would compute mostly padding.
constexpr int kMfmaMidBM = 64;
// Loads of up to about 128 rows per expert: one 128-row tile per expert reads
// its weights once where two 64-row tiles would stream them twice.
constexpr int kMfmaMid2BM = 128;

// Scratch of the 256-row streaming kernels (none: every work item is dealt
// statically and the tiles left over after the last whole round run whole).
// The first kSchedBytes hold the run-time work claims (a counter the launch
// clears, and one mailbox ring per workgroup); the down GEMMs' split-tail
// partial sums follow, one 256 x 256 fp32 tile per workgroup.
// gemm_workspace_bytes(down) is the size that enables both on the current
// device.
struct GemmWorkspace {
  void* base = nullptr;
  int64_t bytes = 0;
};
constexpr int64_t kSchedBytes = 65536;
// Tiles of fewer K steps (of 64) are never split: the reduce launch and the
// partial sums' traffic (~15 us at 16 tiles) cost about what splitting a short
// tile saves (the fine-grained shape's 22-step down tiles take ~31 us).
constexpr int kSplitMinTileSteps = 64;
// Whether a 256-row GEMM over k inputs splits its last round of tiles along K.
// The one test of the kernels' launches, of what sizes their workspace and of
// the choice of tiles; a partial last step counts as one.
inline bool splits_tail(int64_t k) { return ceil_div(k, 64) >= kSplitMinTileSteps; }
int64_t gemm_workspace_bytes(bool down);

// K of the bf16 kernels: a multiple of 8, at least one 64-K step. (Below it,
// a tile is mostly padding and the general kernels stay.)
inline bool mfma_k_supported(int64_t k) { return k >= 64 && k % 8 == 0; }
// Expert shapes whose bf16 GEMMs, forward and backward, all run on the matrix
// cores.
inline bool mfma_shape_supported(int64_t dim, int64_t dim_ffn) {
  return mfma_k_supported(dim) && mfma_k_supported(dim_ffn) && dim <= (1ll << 22) && dim_ffn <= (1ll << 22);
}

// Shape constraints of the bf16 kernels: K as above, the output columns a
// multiple of 8, 16-byte aligned operands.
bool mfma_gate_up_supported(int64_t dim, int64_t dim_ffn, int block_m,
                            const void* a, const void* c);
bool mfma_down_supported(int64_t dim_ffn, int64_t dim, int block_m,
                         const void* a, const void* c);

// Row-tile height of the list for one GEMM of a dense expert (96 rows or more).
int dense_gemm_block_m(int64_t n_rows, int64_t k, int64_t n, bool gate_up);

// Rows of a grouped GEMM as far as the host knows them: `rows` over `experts`
// experts, divided by the router, and `exact` experts (shared ones, a dense
// expert) of exactly `exact_rows` rows each. The rules that choose kernels and
// tiles by the load take it; results depend on it only through those.
struct RowCounts {
  int64_t rows;
  int experts;
  int exact = 0;
  int64_t exact_rows = 0;
  RowCounts(int64_t rows_, int experts_, int exact_ = 0, int64_t exact_rows_ = 0)
      : rows(rows_), experts(experts_), exact(exact_), exact_rows(exact_rows_) {
    if (experts == 1 && (exact == 0 || exact_rows == rows)) {  // the only routed expert has every row
      exact_rows = rows;
      ++exact;
      rows = experts = 0;
    }
  }
  int64_t total() const { return rows + exact * exact_rows; }
  bool dense() const { return experts == 0 && exact == 1; }
};

// Whether a down GEMM takes whole 256-row tiles and splits its last round of them
// (its workspace then holds the partial sums).
bool down_splits(const RowCounts& rows, int block_m, int64_t k, int64_t n, bool packed);

// Row tiles of `bm` rows that a load makes: expected under even routing (an
// expert's rows about normal, with their mean as variance); under a skewed one
// (the last tile of nearly every expert nearly empty: routers biased by Zipf
// weights of exponents 0.4 to 4 over 8 to 128 experts gave rows / bm + 0.1 to 0.85
// per expert); and the most that any routing makes, the list's capacity. The
// same number where the host knows every expert's rows.
struct RowTileCount {
  double even, skewed, most;
};
inline RowTileCount count_row_tiles(const RowCounts& rows, int bm) {
  const double exact = (double)rows.exact * (double)ceil_div(rows.exact_rows, bm);
  if (rows.experts == 0) return {exact, exact, exact};
  const double r = (double)rows.rows / rows.experts, sd = std::sqrt(std::max(r, 1.0));
  double tiles = 0.0;
  for (int64_t j = 0; j * bm < r + 8.0 * sd; ++j) tiles += 0.5 * std::erfc(((double)(j * bm) - r) / (sd * 1.41421356));
  const int64_t most = std::min(rows.rows, (rows.rows + (int64_t)rows.experts * (bm - 1)) / bm);
  const double even = std::min(rows.experts * tiles, (double)most);
  const double skewed = std::min(std::max(even, (double)rows.rows / bm + 0.8 * rows.experts), (double)most);
  return {exact + even, exact + skewed, exact + (double)most};
}

// `packed`: the weight tables point at packed copies written by launch_pack
// (bf16, 256-row tiles of K / 64 contiguous 32 KB blocks in staged order).
int launch_mfma_gate_up(const void* x_perm, const int32_t* tiles,
                        int64_t capacity, const void* const* w_gate,
                        const void* const* w_up, const RowCounts& rows,
                        int64_t dim, int64_t dim_ffn, int block_m, bool packed, void* h, hipStream_t s,
                        const GemmWorkspace& ws = {});
int launch_mfma_down(const void* h, const int32_t* tiles, int64_t capacity,
                     const void* const* w_down, const void* sorted_w,
                     const RowCounts& rows, int64_t dim_ffn,
                     int64_t dim, int block_m, bool packed,
                     void* y, hipStream_t s,
                     const GemmWorkspace& ws = {});

// The same for K that is no multiple of 64 (moe_gemm_mfma_ragged.hip,
// moe_gemm_bwd_ragged.hip), where the functions of these names go by
// themselves; unpacked weights only.
namespace ragged {
int launch_mfma_gate_up(const void* x_perm, const int32_t* tiles,
                        int64_t capacity, const void* const* w_gate,
                        const void* const* w_up, const RowCounts& rows,
                        int64_t dim, int64_t dim_ffn, int block_m, bool packed, void* h, hipStream_t s,
                        const GemmWorkspace& ws);
int launch_mfma_down(const void* h, const int32_t* tiles, int64_t capacity,
                     const void* const* w_down, const void* sorted_w,
                     const RowCounts& rows, int64_t dim_ffn,
                     int64_t dim, int block_m, bool packed,
                     void* y, hipStream_t s, const GemmWorkspace& ws);
int launch_mfma_gate_up_gather(const void* x, const int32_t* sorted_token,
                               const int32_t* tiles, int64_t capacity,
                               const void* const* w_gate,
                               const void* const* w_up, const RowCounts& rows,
                               int64_t dim, int64_t dim_ffn, int block_m, void* h,
                               hipStream_t s,
                               const GemmWorkspace& ws);
int launch_mfma_gate_up_save(const void* x_perm, const int32_t* tiles,
                             int64_t capacity, const void* const* w_gate,
                             const void* const* w_up, int64_t dim,
                             int64_t dim_ffn, void* h, void* gu,
                             hipStream_t s, const GemmWorkspace& ws);
int launch_mfma_down_save(const void* h, const int32_t* tiles,
                          int64_t capacity, const void* const* w_down,
                          const void* sorted_w, int64_t dim_ffn, int64_t dim,
                          void* y, void* y_unweighted, hipStream_t s,
                          const GemmWorkspace& ws);
int launch_dgrad_down(const void* dy, const int32_t* tiles, int64_t capacity,
                      const void* const* w_down, const void* gu, int64_t dim,
                      int64_t dim_ffn, void* dg, void* du, hipStream_t s);
int launch_dgrad_in(const void* d, const int32_t* tiles, int64_t capacity,
                    const void* const* w, int64_t k, int64_t n,
                    const void* add, void* dx, hipStream_t s,
                    const GemmWorkspace& ws);
}  // namespace ragged

// As launch_mfma_gate_up, reading the activation rows as x[sorted_token[r]]
// (x: [n_tokens, dim]) instead of a copied x_perm.
int launch_mfma_gate_up_gather(const void* x, const int32_t* sorted_token,
                               const int32_t* tiles, int64_t capacity,
                               const void* const* w_gate,
                               const void* const* w_up, const RowCounts& rows,
                               int64_t dim, int64_t dim_ffn, int block_m, void* h,
                               hipStream_t s,
                               const GemmWorkspace& ws = {});

// The GEMMs on the kernels their sizes take (moe_gemm.hip). packed: the tables
// hold packed copies.
int launch_gate_up(const void* x_perm, const int32_t* tiles, int64_t tiles_len,
                   const void* const* w_gate, const void* const* w_up,
                   int dtype, const RowCounts& rows, int64_t dim,
                   int64_t dim_ffn, int block_m, bool packed, void* h,
                   const GemmWorkspace& ws, hipStream_t s);
int launch_down(const void* h, const int32_t* tiles, int64_t tiles_len,
                const void* const* w_down, const void* sorted_w, int dtype,
                const RowCounts& rows, int64_t dim_ffn, int64_t dim,
                int block_m, bool packed, void* y, const GemmWorkspace& ws,
                hipStream_t s);
// gathering (bf16); x and h aligned to 16 bytes, x under 4 GiB
int launch_gate_up_gather(const void* x, const int32_t* sorted_token,
                          const int32_t* tiles, int64_t tiles_len,
                          const void* const* w_gate, const void* const* w_up,
                          const RowCounts& rows, int64_t dim,
                          int64_t dim_ffn, int block_m, void* h,
                          const GemmWorkspace& ws, hipStream_t s);

// Few rows (moe_gemm_few.hip), tiles below 256 rows: whether the kernels there
// take a GEMM with k inputs and n output columns, and the GEMMs (row_src: the
// gathered rows' tokens, or null; packed: the tables hold packed copies).
bool few_rows(const RowCounts& rows, int block_m, int64_t k, int64_t n,
              bool gate_up);
int launch_few_gate_up(const void* x, const int32_t* row_src,
                       const int32_t* tiles, int64_t capacity,
                       const void* const* w_gate, const void* const* w_up,
                       const RowCounts& rows, int64_t dim, int64_t dim_ffn,
                       int block_m, bool packed, void* h, hipStream_t s);
int launch_few_down(const void* h, const int32_t* tiles, int64_t capacity,
                    const void* const* w_down, const void* sorted_w,
                    const RowCounts& rows, int64_t dim_ffn, int64_t dim,
                    int block_m, bool packed, void* y, hipStream_t s);
// Both GEMMs of one dense expert whose GEMMs few_rows both takes, without a
// tile list.
int launch_few_dense(const void* x, const void* const* w_gate,
                     const void* const* w_up, const void* const* w_down,
                     int64_t n_rows, int64_t dim, int64_t dim_ffn, int block_m,
                     void* h, void* out, hipStream_t s);

// The tile lists of one dense expert for two GEMMs (moe_permute.hip); the second
// only where len_down > 0.
int launch_dense_tiles(int64_t n_rows, int block_m, int64_t len, int32_t* tiles,
                       int block_m_down, int64_t len_down, int32_t* tiles_down,
                       hipStream_t s);

// Training forward (256-row tiles): as launch_mfma_gate_up / launch_mfma_down,
// also storing the bf16 gate and up projections (gu: [rows, 2 dim_ffn],
// blocks of 4 gate columns then the same 4 up columns) or the unweighted bf16
// expert output (y_unweighted: [rows, dim]).
int launch_mfma_gate_up_save(const void* x_perm, const int32_t* tiles,
                             int64_t capacity, const void* const* w_gate,
                             const void* const* w_up, int64_t dim,
                             int64_t dim_ffn, void* h, void* gu,
                             hipStream_t s,
                        const GemmWorkspace& ws = {});
int launch_mfma_down_save(const void* h, const int32_t* tiles,
                          int64_t capacity, const void* const* w_down,
                          const void* sorted_w, int64_t dim_ffn, int64_t dim,
                          void* y, void* y_unweighted, hipStream_t s,
                          const GemmWorkspace& ws = {});

// fp32 on the matrix cores (moe_gemm_mfma_f32.hip), 64-row tile lists, K and
// the output columns multiples of 32, 16-byte aligned operands. A non-null gu / y_unweighted selects the training
// forward, which also stores the gate and up projections (blocked layout of
// gu_index) or the output before the routing weight. row_src (inference only):
// x_perm is x and row r is x[row_src[r]] (x under 4 GiB).
bool mfma_f32_supported(int64_t k, int64_t n, bool gate_up, int block_m,
                        const void* a, const void* c, const void* s0);
int launch_mfma_f32_gate_up(const void* x_perm, const int32_t* tiles,
                            int64_t capacity, const void* const* w_gate,
                            const void* const* w_up, const RowCounts& rows,
                            int64_t dim, int64_t dim_ffn, void* h, void* gu,
                            hipStream_t s, const int32_t* row_src = nullptr);
int launch_mfma_f32_down(const void* h, const int32_t* tiles, int64_t capacity,
                         const void* const* w_down, const void* sorted_w,
                         const RowCounts& rows, int64_t dim_ffn, int64_t dim,
                         void* y, void* y_unweighted, hipStream_t s);

// fp32 backward on the matrix cores (moe_gemm_mfma_f32_bwd.hip): the dgrad
// GEMMs over 64-row tile lists with K a multiple of 32 and N of 4, wgrad with
// M and N multiples of 4; same contracts as the general-shape ones below.
bool mfma_f32_bwd_supported(int64_t k, int64_t n, int block_m, const void* a,
                            const void* c0, const void* c1, const void* e0);
bool mfma_f32_wgrad_supported(int64_t m, int64_t n, const void* a,
                              const void* b, const void* dw);
int launch_mfma_f32_dgrad_down(const void* dy, const int32_t* tiles,
                               int64_t capacity, const void* const* w_down,
                               const void* gu, int64_t dim, int64_t dim_ffn,
                               void* dg, void* du, hipStream_t s);
int launch_mfma_f32_dgrad_in(const void* d, const int32_t* tiles,
                             int64_t capacity, const void* const* w, int64_t k,
                             int64_t n, const void* add, void* dx,
                             hipStream_t s);
int launch_mfma_f32_wgrad(const void* a, const void* b, const int32_t* offsets,
                          int64_t n_rows, int n_experts, int64_t m, int64_t n,
                          void* dw, hipStream_t s);

// Routing with n_shared always-chosen experts behind the n_experts routed ones
// (moe_route.hip): topk_idx, topk_w [n_tokens, top_k + n_shared], chunk_hist
// [n_chunks, n_experts + n_shared].
int launch_route(const void* logits, int dtype, int64_t n_tokens,
                 int n_experts, int top_k, int n_shared, int32_t* topk_idx,
                 void* topk_w, int32_t* chunk_hist, hipStream_t s);

// The same for at most ASTRAI_MOE_CHUNK_TOKENS tokens, straight to what
// astrai_moe_permute writes of the decisions (tiles of block_m >= 32 rows, so one
// for every expert that has any); neither x_perm nor expert offsets.
struct RouteList {
  int32_t* sorted_token;
  void* sorted_w;
  int32_t* token_pos;
  int32_t* tiles;
  int64_t tile_capacity;
  int block_m;
};
int launch_route_list(const void* logits, int dtype, int64_t n_tokens,
                      int n_experts, int top_k, int n_shared,
                      const RouteList& list, hipStream_t s);

// astrai_moe_combine with token_pos rows pos_stride >= top_k wide, of which
// the first top_k are combined (moe_combine.hip).
int launch_combine(const void* y, const int32_t* token_pos, const void* row_w,
                   const void* shared, int n_shared, int dtype,
                   int64_t n_tokens, int top_k, int pos_stride, int64_t dim,
                   void* out, hipStream_t s);

// Backward (moe_gemm_bwd.hip), bf16, 256-row tile lists:
// dy = dout[sorted_token] * sorted_w and dw_rows = sum(dout[tok] * y) per row;
int launch_row_grad(const void* dout, const int32_t* sorted_token,
                    const void* sorted_w, const void* y, int64_t n_rows,
                    int64_t dim, void* dy, void* dw_rows, hipStream_t s);
// dg, du [rows, dim_ffn] from dy [rows, dim], W_down [dim, dim_ffn] and the
// saved interleaved gu;
int launch_dgrad_down(const void* dy, const int32_t* tiles, int64_t capacity,
                      const void* const* w_down, const void* gu, int64_t dim,
                      int64_t dim_ffn, void* dg, void* du, hipStream_t s);
// dx [rows, n] = bf16(d . W[e]) (+ add, rounded again), W[e] [k, n]; ws as
// the down GEMM's (gemm_workspace_bytes(true)): the last round's tiles split
// along K;
int launch_dgrad_in(const void* d, const int32_t* tiles, int64_t capacity,
                    const void* const* w, int64_t k, int64_t n,
                    const void* add, void* dx, hipStream_t s,
                    const GemmWorkspace& ws = {});
// dw[e] [m, n] = a[rows_e]^T . b[rows_e] for every expert with rows
// (a: [rows, m], b: [rows, n]); experts without rows are not written.
int launch_wgrad(const void* a, const void* b, const int32_t* offsets,
                 int n_experts, int64_t m, int64_t n, void* dw,
                 hipStream_t s);

// General-shape backward (moe_gemm_generic_bwd.hip): fp32 or bf16, any dim
// and dim_ffn, any row-tile height; same contracts as the matrix-core ones
// above, the saved gu in the blocked layout of gu_index.
int launch_generic_dgrad_down(int dtype, const void* dy, const int32_t* tiles,
                              int64_t capacity, const void* const* w_down,
                              const void* gu, int64_t dim, int64_t dim_ffn,
                              void* dg, void* du, hipStream_t s);
int launch_generic_dgrad_in(int dtype, const void* d, const int32_t* tiles,
                            int64_t capacity, const void* const* w, int64_t k,
                            int64_t n, const void* add, void* dx,
                            hipStream_t s);
int launch_generic_wgrad(int dtype, const void* a, const void* b,
                         const int32_t* offsets, int n_experts, int64_t m,
                         int64_t n, void* dw, hipStream_t s);
int launch_generic_row_grad(int dtype, const void* dout,
                            const int32_t* sorted_token, const void* sorted_w,
                            const void* y, int64_t n_rows, int64_t dim,
                            void* dy, void* dw_rows, hipStream_t s);

// Packs one expert's weight for the packed GEMMs: gate/up (w0 = gate, w1 =
// up, each [rows, k]) or down (w0 = [rows, k]).
int launch_pack(const void* w0, const void* w1, int64_t rows, int64_t k,
                bool gate_up, void* out, hipStream_t s);

}  // namespace astrai_moe
