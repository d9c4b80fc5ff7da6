// bf16 grouped expert GEMMs for few rows (single-sequence and small-batch
// decode) on CDNA4 matrix cores (gfx950): same contracts as the kernels of
// moe_gemm_mfma.hip.
//
// Bound by reading each live expert's weights once, which needs every compute
// unit to hold reads in flight. The 256-column tiles of gemm_mfma_kernel give
// a down GEMM of D 4096 only 16 workgroups per row tile: one MLP of D 4096,
// F 14336 over 24 rows streamed its 117 MB at 0.8 TB/s (150 us), two experts
// of one token at 1.6 TB/s (145 us). Here a column tile is 32 weight rows
// (down) or 16 gate and 16 up rows, eight times as many workgroups, and the
// four waves of a workgroup share a tile by taking every fourth 64-K step of
// it: each wave streams its steps through an LDS ring of its own, DMA'd and
// swizzled as in moe_gemm_mfma.hip, with no barrier in the K loop and across
// tile ends. Three sizes of a stage (activation by weight rows of 128 bytes):
// 32 x 32, four stages; 32 x 16, six; 64 x 32, three. Then the waves' fp32 sums
// meet in LDS, summed in wave order, 32 rows at a time: one barrier for each 32,
// the place they meet in alternating between two halves, or two barriers and one
// place for the 64 x 32 stages, whose rings leave no room for more.
//
// Persistent, workgroup b taking tiles b, b + G, ...: consecutive workgroups
// read consecutive weight rows of one expert. A row tile is walked in runs of
// the stage's rows. The K order of a column tile's sums, which step each wave
// starts at and the order of the waves, depends only on the expert and the column
// tile (see gemm_mfma_kernel), so results are the same for every row tile height
// and run, for packed and gathered operands.
//
// Measured at few_rows below; an MLP of D 4096, F 14336 over 24 rows streams its
// 352 MB of weights at 4.4 TB/s (205 -> 80 us).
#include <algorithm>
#include <cmath>

#include "mfma_tile.h"

namespace astrai_moe {
namespace {

template <int BM_, int BN_>
struct FewCfg {
  static constexpr int BM = BM_, BN = BN_, WAVES = 4, STAGES = BM == 64 ? 3 : BN == 32 ? 4 : 6;
  static constexpr int NR = BM / 16, NC = BN / 16;  // 16-row and 16-column blocks
  static constexpr int A_BYTES = BM * kRowBytes, B_BYTES = BN * kRowBytes, STAGE = A_BYTES + B_BYTES;
  static constexpr int OPS = STAGE / 1024;                     // DMA ops per wave and step
  static constexpr int RED_ROWS = 32;                          // rows whose sums meet at a time
  static constexpr int RED_WAVE = RED_ROWS * BN * 4;           // one wave's fp32 sums of these
  static constexpr int RED_OFF = WAVES * STAGES * STAGE;       // 128 or 144 KB of rings
  static constexpr int RED_BUFS = BM == 64 ? 1 : 2;            // places they meet in
  static constexpr int LDS = RED_OFF + RED_BUFS * WAVES * RED_WAVE;  // 160 KB
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert(OPS * (STAGES - 1) <= 63, "vmcnt range");
};

// The row tiles a launch walks: those of the list, or (kDense) one expert's
// n_rows rows in tiles of block_m, with no list to write and wait for.
template <bool kDense>
struct RowTiles {
  const int32_t* tiles;
  int n_rows, block_m;
  __device__ int live(int capacity) const {
    if constexpr (kDense) return capacity;
    return min(load_scalar(tiles), min(load_scalar(tiles + 2), capacity));
  }
  __device__ void get(int mt, int& e, int& row0, int& rows) const {
    if constexpr (kDense) {
      e = 0;
      row0 = mt * block_m;
      rows = min(block_m, n_rows - row0);
    } else {
      const int32_t* ti = tiles + ASTRAI_MOE_TILE_HEADER + (int64_t)mt * ASTRAI_MOE_TILE_STRIDE;
      e = load_scalar(ti);
      row0 = load_scalar(ti + 1);
      rows = min(load_scalar(tiles + 1), load_scalar(ti + 2) - row0);
    }
  }
};

// Position of a wave in its sequence of K steps: run `sub` of 32 rows of tile
// `unit`, the wave's step j of n.
template <typename Cfg, bool kGateUp, bool kGather, bool kPacked>
struct FewCursor {
  int unit, mt, nt, row0, rows, sub, j, n, rot;
  bool live;
  const char *a, *b0, *b1;
  uint32_t off[Cfg::BM / 8];  // byte offsets of the rows a lane loads of the activation tile
  int b_rows;

  // tile and weights of `unit` (< total)
  template <bool kDense>
  __device__ void enter(const RowTiles<kDense>& tiles, const void* const* W0, const void* const* W1, int K, int N, int n_cols) {
    constexpr int kCols = kGateUp ? Cfg::BN / 2 : Cfg::BN;
    mt = unit / n_cols;
    nt = unit - mt * n_cols;
    int e;
    tiles.get(mt, e, row0, rows);
    const int KT = k_steps(K);
    b_rows = min(kCols, N - nt * kCols);
    const char* w0 = static_cast<const char*>(load_scalar(W0 + e));
    if constexpr (kPacked) {
      // rows of the packed 256-row tile (128 gate and 128 up rows) that holds these columns
      constexpr int kTile = kGateUp ? 128 : 256;
      const int t = nt * kCols / kTile, r = nt * kCols - t * kTile;
      b0 = w0 + ((int64_t)t * KT * 256 + r) * kRowBytes;
      b1 = b0 + 128 * kRowBytes;
    } else {
      b0 = w0 + (int64_t)nt * kCols * K * 2;
      b1 = kGateUp ? static_cast<const char*>(load_scalar(W1 + e)) + (int64_t)nt * kCols * K * 2 : b0;
    }
    rot = n > 0 ? (7 * e + 3 * nt) % n : 0;
    sub = 0;
  }
  __device__ void enter_rows(const bf16_t* A, const int32_t* row_src, int K, int lane) {
    j = 0;
    const uint32_t k2 = (uint32_t)K * 2u;
    a = reinterpret_cast<const char*>(kGather ? A : A + (int64_t)(row0 + sub * Cfg::BM) * K);
    const int last = rows - sub * Cfg::BM - 1;  // pad rows re-read the last row
#pragma unroll
    for (int q = 0; q < Cfg::BM / 8; ++q) {
      const int r = min(q * 8 + (lane >> 3), last);
      off[q] = kGather ? (uint32_t)row_src[row0 + sub * Cfg::BM + r] * k2 : (uint32_t)r * k2;
    }
  }
  template <bool kDense>
  __device__ void advance(int total, int G, const RowTiles<kDense>& tiles, const bf16_t* A, const void* const* W0,
                          const void* const* W1, const int32_t* row_src, int K, int N, int n_cols, int lane) {
    if (++j < n) return;
    const int old_mt = mt, old_sub = sub;
    if ((sub + 1) * Cfg::BM < rows) {
      ++sub;
    } else {
      unit += G;
      live = unit < total;
      if (!live) return;
      enter(tiles, W0, W1, K, N, n_cols);
    }
    // (the same rows: only the step restarts; their list is read again only where it changes)
    if (mt == old_mt && sub == old_sub)
      j = 0;
    else
      enter_rows(A, row_src, K, lane);
  }
  // the wave's next step into LDS at `lds`
  __device__ void issue(int wave, int lane, int K, char* lds) const {
    int jr = j + rot;
    if (jr >= n) jr -= n;
    const int ks = wave + Cfg::WAVES * jr;
    const uint32_t k2 = (uint32_t)K * 2u;
    const DmaLane dl(lane, ks);
    const bool tail = (ks + 1) * kBK > K;
#pragma unroll
    for (int q = 0; q < Cfg::BM / 8; ++q) {
      if (tail)
        dma_16_or_zero(a, off[q] + dl.chunk(q), dl.chunk(q), k2, lds + q * 1024);
      else
        lds_dma_16(a + (off[q] + dl.chunk(q)), lds + q * 1024);
    }
    lds += Cfg::A_BYTES;
#pragma unroll
    for (int q = 0; q < Cfg::BN / 8; ++q) {
      constexpr int kHalf = Cfg::BN / 16;  // gate/up: ops of the gate rows, then of the up rows
      const bool up = kGateUp && q >= kHalf;
      const int q_in = kGateUp ? q % kHalf : q;
      const char* b = up ? b1 : b0;
      if constexpr (kPacked) {
        // the copy's chunks are swizzled by its own rows: 8 gate or up rows
        // may lie at the other parity of 8 than their place in the stage
        const uint32_t flip = (kGateUp && Cfg::BN == 16) ? 64u * (uint32_t)((nt ^ q) & 1) : 0u;
        const uint32_t at = (uint32_t)ks * (256u * kRowBytes) + (uint32_t)q_in * 1024u + ((uint32_t)lane * 16u ^ flip);
        lds_dma_16(b + at, lds + q * 1024);
      } else {
        const uint32_t o = (uint32_t)min(q_in * 8 + dl.row, b_rows - 1) * k2 + dl.chunk(q);
        if (tail)
          dma_16_or_zero(b, o, dl.chunk(q), k2, lds + q * 1024);
        else
          lds_dma_16(b + o, lds + q * 1024);
      }
    }
  }
};

template <typename Cfg, bool kGateUp, bool kGather, bool kPacked, bool kDense>
__global__ __launch_bounds__(Cfg::WAVES * 64, 1) void gemm_few_kernel(
    const bf16_t* __restrict__ A, const RowTiles<kDense> tiles, const void* const* __restrict__ W0,
    const void* const* __restrict__ W1, const bf16_t* __restrict__ row_w, int K, int N, int n_cols, int capacity,
    bf16_t* __restrict__ C, const int32_t* __restrict__ row_src) {
  constexpr int NR = Cfg::NR, NC = Cfg::NC;
  __shared__ __attribute__((aligned(1024))) char smem[Cfg::LDS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int G = gridDim.x;
  const int total = tiles.live(capacity) * n_cols;
  if ((int)blockIdx.x >= total) return;
  char* const ring = smem + wave * (Cfg::STAGES * Cfg::STAGE);

  FewCursor<Cfg, kGateUp, kGather, kPacked> ld;  // the next step to load
  const int KT = k_steps(K);
  const int n_steps = KT > wave ? (KT - wave + Cfg::WAVES - 1) / Cfg::WAVES : 0;
  ld.n = n_steps;
  ld.unit = blockIdx.x;
  ld.enter(tiles, W0, W1, K, N, n_cols);
  ld.enter_rows(A, row_src, K, lane);
  ld.live = n_steps > 0;
  int issued = 0, used = 0;  // steps loaded and consumed so far; step i sits in stage i % STAGES
  auto issue = [&]() {
    ld.issue(wave, lane, K, ring + (issued % Cfg::STAGES) * Cfg::STAGE);
    ++issued;
    ld.advance(total, G, tiles, A, W0, W1, row_src, K, N, n_cols, lane);
  };
#pragma unroll 1
  for (int i = 0; i < Cfg::STAGES; ++i)
    if (ld.live) issue();

  const int frag_row = lane & 15, fq = lane >> 4, fsw = (frag_row >> 1) & 7;
  int parity = 0;
  for (int unit = blockIdx.x; unit < total; unit += G) {
    const int mt = unit / n_cols, nt = unit - mt * n_cols;
    int e, row0, rows;
    tiles.get(mt, e, row0, rows);
    for (int r0 = 0; r0 < rows; r0 += Cfg::BM) {
      f32x4_t acc[NR][NC];
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[i][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      for (int step = 0; step < n_steps; ++step) {
        wait_groups<Cfg::OPS, Cfg::STAGES - 1>(issued - used - 1);  // this step has landed
        const char* sa = ring + (used % Cfg::STAGES) * Cfg::STAGE + frag_row * kRowBytes;
        bf16x8_t fa[2][NR], fb[2][NC];
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
          const int chunk = ((kh * 4 + fq) ^ fsw) << 4;
#pragma unroll
          for (int i = 0; i < NR; ++i)
            fa[kh][i] = *reinterpret_cast<const bf16x8_t*>(sa + i * 16 * kRowBytes + chunk);
#pragma unroll
          for (int c = 0; c < NC; ++c)
            fb[kh][c] = *reinterpret_cast<const bf16x8_t*>(sa + Cfg::A_BYTES + c * 16 * kRowBytes + chunk);
        }
        wait_lds();  // the stage has been read: it may be loaded again
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        ++used;
        if (ld.live) issue();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
#pragma unroll
          for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int c = 0; c < NC; ++c)
              acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[kh][c], fa[kh][i], acc[i][c], 0, 0, 0);
      }
      // the waves' sums meet, 32 rows at a time: row r's 16-byte piece c at piece
      // c ^ (r % pieces)
      static_for<Cfg::BM / Cfg::RED_ROWS>([&](auto half) {
      constexpr int i0 = decltype(half)::value * 2;  // the first of these rows' two 16-row blocks
      const int rh = r0 + i0 * 16;
      if (rh >= rows) return;
      constexpr int PIECES = Cfg::BN / 4, ROW = Cfg::BN * 4;
      char* const red = smem + Cfg::RED_OFF + parity * (Cfg::WAVES * Cfg::RED_WAVE);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int r = i * 16 + frag_row;
          *reinterpret_cast<f32x4_t*>(red + wave * Cfg::RED_WAVE + r * ROW +
                                      (((c * 4 + fq) ^ (r & (PIECES - 1))) << 4)) = acc[i0 + i][c];
        }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      auto sum = [&](int r, int piece) {
        f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < Cfg::WAVES; ++w)
          v += *reinterpret_cast<const f32x4_t*>(red + w * Cfg::RED_WAVE + r * ROW + ((piece ^ (r & (PIECES - 1))) << 4));
        return v;
      };
      if constexpr (kGateUp) {
        constexpr int HP = PIECES / 2;  // pieces of the gate columns, then of the up columns
        const int r = threadIdx.x / HP, p = threadIdx.x % HP, n = nt * (Cfg::BN / 2) + p * 4;
        if (r < Cfg::RED_ROWS && rh + r < rows && n < N) {
          const f32x4_t g4 = sum(r, p), u4 = sum(r, HP + p);
          bf16x4_t o;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float g = (float)(__bf16)g4[q], u = (float)(__bf16)u4[q];
            const float ex = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
            o[q] = (__bf16)(u * (float)(__bf16)(g * __builtin_amdgcn_rcpf(1.0f + ex)));
          }
          *reinterpret_cast<bf16x4_t*>(C + (int64_t)(row0 + rh + r) * N + n) = o;
        }
      } else {
        const int r = threadIdx.x / PIECES, p = threadIdx.x % PIECES, n = nt * Cfg::BN + p * 4;
        if (r < Cfg::RED_ROWS && rh + r < rows && n < N) {
          const int64_t row = row0 + rh + r;
          const f32x4_t y4 = sum(r, p);
          const float w = row_w != nullptr ? bf16_bits_to_f32(row_w[row]) : 1.0f;
          bf16x4_t o;
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] = (__bf16)((float)(__bf16)y4[q] * w);
          *reinterpret_cast<bf16x4_t*>(C + row * N + n) = o;
        }
      }
      if constexpr (Cfg::RED_BUFS == 2)
        parity ^= 1;
      else  // the next sums go to the same place
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      });
    }
  }
}

template <typename Cfg, bool kGateUp, bool kGather, bool kPacked, bool kDense>
int launch_few_cfg(const void* A, const RowTiles<kDense>& tiles, int64_t capacity, const void* const* W0, const void* const* W1,
               const void* row_w, int64_t K, int64_t N, void* C, hipStream_t s, const int32_t* row_src) {
  if (capacity == 0) return ASTRAI_MOE_OK;
  const int64_t n_cols = ceil_div(N, kGateUp ? Cfg::BN / 2 : Cfg::BN);  // the last may be partial
  int64_t grid = 0;
  if (int rc = persistent_grid(capacity, n_cols, &grid)) return rc;
  hipLaunchKernelGGL((gemm_few_kernel<Cfg, kGateUp, kGather, kPacked, kDense>), dim3((unsigned)grid), dim3(Cfg::WAVES * 64),
                     0, s, static_cast<const bf16_t*>(A), tiles, W0, W1, static_cast<const bf16_t*>(row_w), (int)K,
                     (int)N, (int)n_cols, (int)capacity, static_cast<bf16_t*>(C), row_src);
  return check_launch(kGateUp ? "gemm_few_kernel<gate_up>" : "gemm_few_kernel<down>");
}

// Experts that meet one of n_rows rows, expected under even routing.
double live_experts(int64_t n_rows, int n_experts) {
  return n_experts > 0 ? n_experts * (1.0 - std::pow(1.0 - 1.0 / n_experts, (double)n_rows)) : 0.0;
}

// Share of the compute-unit time that `tiles` equal tiles fill, a partial last
// round included.
double fill(double tiles) {
  const double rounds = tiles / cu_count();
  return rounds / std::ceil(rounds);
}

// Limits of few_rows (below), which has the figures.
constexpr int kFewRowsPerExpert = 8, kFewExactRows = 64, kFewSmallRows = 24, kFewDenseRows = 128, kFewLongSteps = 12;
constexpr double kFewMaxFill = 0.88, kFewMaxFillLong = 0.86, kFewLongRounds = 3.0;

// Tiles of 64 activation rows on lists of at least that height, where most
// experts, or more than two runs of 32 of one expert, have more than 32 rows
// (MLP of D 4096, F 14336: 96 rows 197 -> 149 us, 64 rows 133 -> 138). One
// expert without a list takes rows of 64 from 65 rows on (80 rows 196 -> 132,
// 64-row tiles over 32-row ones before; D 2048, F 5632 46 -> 37) unless its
// 32-row tiles all run at once (D 512, F 1024 9.7 / 10.4).
//
// One expert's single run of 32 rows (an MLP decoding) takes tiles of 16 weight
// rows where those fill the rounds of tiles better: D 4096, F 14336, 24 rows,
// gate/up 3.5 rounds of 32-row tiles or 7 of 16, down half a round or one, 100
// -> 89 us; D 1536, F 4096 20.5 -> 19.6. A 16-row tile reads as many
// activation bytes as one of 32, which costs more elsewhere: more runs (48
// rows 131 -> 163 us) and routed rows (8 experts of that size, 24 tokens 541
// -> 560; 64 of D 2048, F 1408, 8 tokens 144 -> 188).
template <bool kGateUp, bool kGather, bool kPacked, bool kDense>
int launch_few_tiles(const void* A, const RowTiles<kDense>& tiles, int64_t capacity, const void* const* W0, const void* const* W1,
               const void* row_w, const RowCounts& load, int block_m, int64_t K, int64_t N, void* C, hipStream_t s,
               const int32_t* row_src) {
  if (block_m >= FewCfg<64, 32>::BM &&
      load.total() > (load.dense() ? 2 * FewCfg<32, 32>::BM : (int64_t)kFewSmallRows * (load.experts + load.exact)))
    return launch_few_cfg<FewCfg<64, 32>, kGateUp, kGather, kPacked, kDense>(A, tiles, capacity, W0, W1, row_w, K, N, C, s,
                                                                     row_src);
  if (load.dense() && load.total() <= FewCfg<32, 16>::BM &&
      fill((double)ceil_div(N, kGateUp ? 8 : 16)) > 1.05 * fill((double)ceil_div(N, kGateUp ? 16 : 32)))
    return launch_few_cfg<FewCfg<32, 16>, kGateUp, kGather, kPacked, kDense>(A, tiles, capacity, W0, W1, row_w, K, N, C, s, row_src);
  return launch_few_cfg<FewCfg<32, 32>, kGateUp, kGather, kPacked, kDense>(A, tiles, capacity, W0, W1, row_w, K, N, C, s, row_src);
}

template <bool kGateUp, bool kGather, bool kPacked>
int launch_few(const void* A, const int32_t* tiles, int64_t capacity, const void* const* W0, const void* const* W1,
               const void* row_w, const RowCounts& load, int block_m, int64_t K, int64_t N, void* C, hipStream_t s,
               const int32_t* row_src) {
  return launch_few_tiles<kGateUp, kGather, kPacked>(A, RowTiles<false>{tiles, 0, 0}, capacity, W0, W1, row_w, load, block_m, K,
                                                     N, C, s, row_src);
}

}  // namespace

// Where these kernels replace the 256-column tiles of moe_gemm_mfma.hip. An
// expert of more than 32 rows reads its weights once for each run, so the lines
// lie where a skewed router, of which the host sees nothing, loses nothing
// either (a Zipf bias of exponent 1.44 below; us per layer or MLP without and
// with, replayed from a graph):
// - up to kFewRowsPerExpert routed rows per expert, where the other kernel's
//   last round of tiles would leave more than kFewMaxFill of its compute-unit
//   time idle (kFewMaxFillLong past kFewLongRounds rounds, of which one more
//   costs less). 8 experts, top-2, D 4096, F 14336: 1 token 264 / 165, 8 532 /
//   495; past the line, 33 tokens 539 / 520, skewed 555 / 522, but 48 538 / 590
//   skewed, 80 553 / 673 and 96 552 / 711. 64 experts, top-6, D 2048, F 1408: 1
//   token 74 / 60, 32 (2.6 rounds, 0.87) 229 / 217; 128 experts, top-8, D 4096, F
//   1536, 33 tokens (5.2 rounds, 0.87) 797 / 813, skewed 298 / 311. Shared
//   experts run along with up to two runs of rows each (kFewExactRows; 128
//   experts and a shared one, 256 tokens 908 / 961, skewed 615 / 742);
// - small layers, whose tiles occupy at most a quarter of the compute units and
//   whose weights the caches hold: below kFewSmallRows rows per expert, and twice
//   as many where they occupy an eighth in kFewLongSteps K steps or more. 8
//   experts, top-2, D 1000, F 2664, 64 tokens 73 / 53, 192 77 / 68, skewed 76 / 59
//   and 77 / 75; D 512, F 4096, 64 66 / 43, 192 72 / 55; a quarter, D 2048, F 8192:
//   64 212 / 178, skewed 189 / 145; past the line 192 skewed 219 / 262;
// - one expert, whose rows are known, up to kFewDenseRows of them by the first
//   rule, and twice as many where its tiles occupy at most half the compute units
//   in kFewLongSteps K steps or more. D 4096, F 14336: 1 row 201 / 81, 24 217 /
//   90, 64 214 / 133, 128 235 / 156, 256 (the down GEMM; its gate/up GEMM has 448
//   tiles) 255 / 191; D 2048, F 5632: 24 66 / 28, 128 72 / 43, 256 73 / 44.
// The same for tiles of 32, 64 and 128 rows, so that these give the same bits;
// lists of 256-row tiles keep their kernels, whose bits the training forward
// shares.
bool few_rows(const RowCounts& rows, int block_m, int64_t k, int64_t n, bool gate_up) {
  if (block_m == kMfmaBigBM) return false;
  const double cols = (double)ceil_div(n, gate_up ? 128 : 256), cu = cu_count();
  const bool long_steps = k_steps(k) >= kFewLongSteps;
  if (rows.dense()) {
    const int64_t n_rows = rows.exact_rows;
    if (n_rows <= kFewDenseRows) return fill(cols) < kFewMaxFill;
    return n_rows <= 2 * kFewDenseRows && long_steps && 2.0 * ceil_div(n_rows, kMfmaMidBM) * cols <= cu;
  }
  if (rows.rows <= (int64_t)kFewRowsPerExpert * rows.experts && rows.exact_rows <= kFewExactRows) {
    const double tiles = (live_experts(rows.rows, rows.experts) + rows.exact * ceil_div(rows.exact_rows, kMfmaSmallBM)) * cols;
    if (fill(tiles) < (tiles <= kFewLongRounds * cu ? kFewMaxFill : kFewMaxFillLong)) return true;
  }
  const double tiles = std::max(rows.experts, rows.exact) * cols;
  const int64_t small = (int64_t)kFewSmallRows * (rows.experts + rows.exact);
  return (rows.total() < small && 4.0 * tiles <= cu) || (rows.total() <= 2 * small && long_steps && 8.0 * tiles <= cu);
}

int launch_few_gate_up(const void* x, const int32_t* row_src, const int32_t* tiles, int64_t capacity,
                       const void* const* w_gate, const void* const* w_up, const RowCounts& rows, int64_t dim,
                       int64_t dim_ffn, int block_m, bool packed, void* h, hipStream_t s) {
  if (packed) return launch_few<true, false, true>(x, tiles, capacity, w_gate, w_gate, nullptr, rows, block_m, dim, dim_ffn, h, s, nullptr);
  if (row_src != nullptr)
    return launch_few<true, true, false>(x, tiles, capacity, w_gate, w_up, nullptr, rows, block_m, dim, dim_ffn, h, s, row_src);
  return launch_few<true, false, false>(x, tiles, capacity, w_gate, w_up, nullptr, rows, block_m, dim, dim_ffn, h, s, nullptr);
}

int launch_few_down(const void* h, const int32_t* tiles, int64_t capacity, const void* const* w_down,
                    const void* sorted_w, const RowCounts& rows, int64_t dim_ffn, int64_t dim, int block_m, bool packed,
                    void* y, hipStream_t s) {
  if (packed)
    return launch_few<false, false, true>(h, tiles, capacity, w_down, w_down, sorted_w, rows, block_m, dim_ffn, dim, y, s, nullptr);
  return launch_few<false, false, false>(h, tiles, capacity, w_down, w_down, sorted_w, rows, block_m, dim_ffn, dim, y, s, nullptr);
}

int launch_few_dense(const void* x, const void* const* w_gate, const void* const* w_up, const void* const* w_down,
                     int64_t n_rows, int64_t dim, int64_t dim_ffn, int block_m, void* h, void* out, hipStream_t s) {
  using Low = FewCfg<32, 32>;
  if (n_rows > 2 * Low::BM && ceil_div(n_rows, Low::BM) * ceil_div(dim_ffn, Low::BN / 2) > cu_count())
    block_m = std::max(block_m, FewCfg<64, 32>::BM);
  const RowTiles<true> rows{nullptr, (int)n_rows, block_m};
  const RowCounts load(n_rows, 1);
  const int64_t n_tiles = ceil_div(n_rows, block_m);
  if (int rc = launch_few_tiles<true, false, false>(x, rows, n_tiles, w_gate, w_up, nullptr, load, block_m, dim, dim_ffn, h,
                                                    s, nullptr))
    return rc;
  return launch_few_tiles<false, false, false>(h, rows, n_tiles, w_down, nullptr, nullptr, load, block_m, dim_ffn, dim, out,
                                               s, nullptr);
}

}  // namespace astrai_moe
