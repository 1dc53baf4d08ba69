// gemm.hip: the prefill projection y[m, n] = bf16(x)[m, k] . w[n, k]^T
// (+ bias[n]) on gfx950's bf16 matrix cores, fp32 accumulation and output:
// the reference's cuda::linear for m > 1 (src/backend/cuda/ops.h:14-17,
// ops.cu:268-287, which rounds x to bf16 in its own pass and calls a bf16
// cuBLAS GEMM with fp32 compute, then adds the bias).
//
// Both operands are k-contiguous (x rows, w rows), so one layout serves both:
// tile rows in LDS are chunks of 8 bf16 (16 bytes), a chunk's slot XOR-swizzled
// by its row so that the rows one operand read spans fall on different banks.
// Two kernels, both on v_mfma_f32_32x32x16_bf16:
//   * linear_pipe_k, x already bf16 and k a multiple of 64: the tiles go from
//     memory straight into LDS (16-byte global_load_lds, each lane's chunk
//     picked so that it lands in its swizzled slot), one or two steps of k
//     ahead of the products. Its forms, small tiles to large, are chosen by
//     the tile count (form_of below);
//   * linear_staged_k otherwise (fp32 x, or k not a multiple of 64): 128 x 128
//     tiles of 4 waves, chunks staged through registers, x rounded to bf16
//     with the hardware's nearest-even conversion on the way, chunks past k
//     zero-filled; a k that is not a multiple of 8 (or unaligned rows) loads
//     element by element. A product with few tiles and a long k may split k
//     over a caller's workspace: each split writes its partial products and
//     one more launch sums them in split order, then adds the bias.
// Workgroups are dealt to the 8 XCDs round-robin; each XCD takes a
// contiguous run of tiles, ordered in groups of 8 tile-rows sweeping the
// columns, so the tiles resident on one XCD share x rows and w rows in its
// L2. The bias is added to each finished sum (one fp32 rounding, as the
// reference's separate bias pass). Products of bf16 rows with no epilogue
// beyond the bias and the add into y, at least 128 rows and too many tiles
// for the small forms, go to hipBLASLt instead (gemm_library.hip).

#include <type_traits>

#include "act_math.hpp"
#include "common.hpp"

namespace uocr_rocm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTileM = 128;
constexpr int kTileN = 128;
constexpr int kTileK = 64;
constexpr int kGemmThreads = 256;
constexpr int kRowChunks = kTileK / 8;                                     // 16-byte chunks per tile row
constexpr int kTileChunks = kTileM * kRowChunks;                           // per operand tile
constexpr int kChunksPerThread = kTileChunks / kGemmThreads;               // 4
static_assert(kTileM == kTileN, "one staging pattern for both operands");

// The LDS slot of 16-byte chunk `chunk` of tile row `row`. A 128-bit LDS
// read serves 16 lanes a pass from 64 four-byte banks (16 chunk-wide bank
// groups, 256 bytes); the products' reads take one chunk column of 16
// consecutive rows per pass, whose row bases fall on 2 bank groups (rows are
// 128 bytes). XOR-ing the chunk with (row / 2) mod 8 spreads the 8 rows of
// each parity over the 8 groups of its half: the 16 reads land on 16
// different groups. (With row mod 8, rows r and r + 8 met in one group:
// measured 4 conflict cycles per LDS instruction on MI355X.)
__device__ __forceinline__ int swz(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int slot(int row, int chunk) { return row * kRowChunks + (chunk ^ swz(row)); }

constexpr int kXcds = 8;
constexpr int kGroupRows = 8;

// The tile (tm, tn) of workgroup bid: a contiguous run of tiles per XCD
// (workgroups go to the XCDs in turn, bid mod 8; XCD x holds total / 8
// tiles, one more for the first total mod 8), groups of kGroupRows
// tile-rows sweeping the columns inside a run.
__device__ __forceinline__ void tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  const int per_xcd = total / kXcds, extra = total % kXcds, xcd = bid % kXcds;
  const int t = xcd * per_xcd + (xcd < extra ? xcd : extra) + bid / kXcds;
  const int per = kGroupRows * tiles_n, group = t / per, first = group * kGroupRows;
  const int rows = tiles_m - first < kGroupRows ? tiles_m - first : kGroupRows;
  const int in = t - group * per;
  tm = first + in % rows;
  tn = in / rows;
}

struct LinearArgs {
  const void* x;  // float or bf16 rows
  const uint16_t* w;
  const float* bias;
  float* y;
  int64_t m, n;
  int k;
  int tiles_m, tiles_n;
  // Split k: workgroup b takes tile b % tiles of split b / tiles, columns
  // [split * k_len, min(k, (split + 1) * k_len)) of the sums, into part +
  // split * m * n (no bias); part null: one split, into y with the bias.
  int k_len;
  float* part;
  // y += the product (+ bias): each element y + (sum + bias), as the
  // product followed by an in-place add
  bool accumulate;
  // Non-null: product row r goes to y row row_map[r], dropped when that is
  // y_rows or more (a scatter of window slots back into a grid); linear_pipe_k
  // only.
  const int64_t* row_map;
  int64_t y_rows;
  // the activation epilogues' output: y16 = bf16(act(sum + bias)), no split,
  // no accumulate
  uint16_t* y16;
  // n a multiple of 4 and bias, y and y16 allow 16-byte (y16: 8-byte) accesses
  bool vec;
  int runs;  // linear_staged_k: runs of k, 1 with a split
};

// What the epilogue writes: the fp32 sums, or an MLP's activation of them
// rounded to bf16, bitwise the fp32 product followed by the elementwise
// activation into bf16 (the same arithmetic, from act_math.hpp).
enum class Epi { kPlain, kGeluBf16, kQuickGeluBf16 };

template <Epi kEpi>
__device__ __forceinline__ float activate(float v) {
  return kEpi == Epi::kGeluBf16 ? gelu_f<10>(v) : quick_gelu_f(v);
}

template <Epi kEpi>
__device__ __forceinline__ void store_act(const LinearArgs& a, int64_t row, int64_t col, float v) {
  a.y16[row * a.n + col] = f32_to_bf16(activate<kEpi>(v));
}

// 16 elements of one output column, product rows row0 + 8 (r / 4) + r % 4
// (r < 16), into y through the row map.
__device__ __forceinline__ void store_mapped(const LinearArgs& a, int64_t row0, int64_t col, float bv, bool add,
                                             const float (&val)[16]) {
  int64_t at[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t row = row0 + 8 * (r / 4) + (r % 4);
    const int64_t to = row < a.m ? a.row_map[row] : a.y_rows;
    at[r] = to < a.y_rows ? to * a.n + col : -1;
  }
  float base[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) base[r] = a.accumulate && at[r] >= 0 ? a.y[at[r]] : 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if (at[r] >= 0) {
      const float v = add ? val[r] + bv : val[r];
      a.y[at[r]] = a.accumulate ? base[r] + v : v;
    }
  }
}

// The tile, split and k range of this workgroup.
struct Work {
  int64_t m0, n0;
  int split, k_begin, k_end;
};

__device__ __forceinline__ Work work_of(const LinearArgs& a) {
  const int tiles = a.tiles_m * a.tiles_n;
  const int split = static_cast<int>(blockIdx.x) / tiles;
  int tm, tn;
  tile_of(static_cast<int>(blockIdx.x) - split * tiles, a.tiles_m, a.tiles_n, tm, tn);
  const int kb = split * a.k_len;
  return {static_cast<int64_t>(tm) * kTileM, static_cast<int64_t>(tn) * kTileN, split, kb,
          a.k - kb < a.k_len ? a.k : kb + a.k_len};
}

// The registers one k step stages: per thread kChunksPerThread chunks of the
// x tile (8 elements each: fp32, rounded on the way to LDS, or bf16) and of
// the w tile.
template <bool kF32X>
struct Staged {
  u32x4 xa[kChunksPerThread][kF32X ? 2 : 1];
  u32x4 wb[kChunksPerThread];
};

template <bool kF32X>
__device__ __forceinline__ void load_step(const LinearArgs& a, int64_t m0, int64_t n0, int k0, int k_end,
                                          Staged<kF32X>& s) {
#pragma unroll
  for (int i = 0; i < kChunksPerThread; ++i) {
    const int id = static_cast<int>(threadIdx.x) + kGemmThreads * i;
    const int row = id / kRowChunks, c = id % kRowChunks;
    const int kc = k0 + 8 * c;
    const bool kin = kc < k_end;
    const int64_t xr = m0 + row, wr = n0 + row;
#pragma unroll
    for (int h = 0; h < (kF32X ? 2 : 1); ++h) s.xa[i][h] = u32x4{0u, 0u, 0u, 0u};
    s.wb[i] = u32x4{0u, 0u, 0u, 0u};
    if (kin && xr < a.m) {
      if constexpr (kF32X) {
        const u32x4* p = reinterpret_cast<const u32x4*>(static_cast<const float*>(a.x) + xr * a.k + kc);
        s.xa[i][0] = p[0];
        s.xa[i][1] = p[1];
      } else {
        s.xa[i][0] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.x) + xr * a.k + kc);
      }
    }
    if (kin && wr < a.n) s.wb[i] = *reinterpret_cast<const u32x4*>(a.w + wr * a.k + kc);
  }
}

// A k that is not a multiple of 8 (rows not 16-byte aligned): each chunk's
// 8 elements are loaded one by one, those at or past k read as zero.
template <bool kF32X>
__device__ __forceinline__ void load_step_ragged(const LinearArgs& a, int64_t m0, int64_t n0, int k0, int k_end,
                                                 Staged<kF32X>& s) {
#pragma unroll
  for (int i = 0; i < kChunksPerThread; ++i) {
    const int id = static_cast<int>(threadIdx.x) + kGemmThreads * i;
    const int row = id / kRowChunks, c = id % kRowChunks;
    const int kc = k0 + 8 * c;
    const int64_t xr = m0 + row, wr = n0 + row;
    uint32_t xv[8], wv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool in = kc + e < k_end;
      xv[e] = 0u;
      wv[e] = 0u;
      if (in && xr < a.m) {
        if constexpr (kF32X) {
          xv[e] = __float_as_uint(static_cast<const float*>(a.x)[xr * a.k + kc + e]);
        } else {
          xv[e] = static_cast<const uint16_t*>(a.x)[xr * a.k + kc + e];
        }
      }
      if (in && wr < a.n) wv[e] = a.w[wr * a.k + kc + e];
    }
    if constexpr (kF32X) {
      s.xa[i][0] = u32x4{xv[0], xv[1], xv[2], xv[3]};
      s.xa[i][1] = u32x4{xv[4], xv[5], xv[6], xv[7]};
    } else {
      s.xa[i][0] = u32x4{xv[0] | (xv[1] << 16), xv[2] | (xv[3] << 16), xv[4] | (xv[5] << 16), xv[6] | (xv[7] << 16)};
    }
    s.wb[i] = u32x4{wv[0] | (wv[1] << 16), wv[2] | (wv[3] << 16), wv[4] | (wv[5] << 16), wv[6] | (wv[7] << 16)};
  }
}

template <bool kF32X>
__device__ __forceinline__ void store_step(const Staged<kF32X>& s, u32x4* xs, u32x4* ws) {
#pragma unroll
  for (int i = 0; i < kChunksPerThread; ++i) {
    const int id = static_cast<int>(threadIdx.x) + kGemmThreads * i;
    const int row = id / kRowChunks, c = id % kRowChunks;
    if constexpr (kF32X) {
      const u32x4 lo = s.xa[i][0], hi = s.xa[i][1];
      xs[slot(row, c)] = u32x4{pack_bf16(__uint_as_float(lo.x), __uint_as_float(lo.y)),
                               pack_bf16(__uint_as_float(lo.z), __uint_as_float(lo.w)),
                               pack_bf16(__uint_as_float(hi.x), __uint_as_float(hi.y)),
                               pack_bf16(__uint_as_float(hi.z), __uint_as_float(hi.w))};
    } else {
      xs[slot(row, c)] = s.xa[i][0];
    }
    ws[slot(row, c)] = s.wb[i];
  }
}

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// The 16 matrix products of one 64-wide k step of a wave's 64 x 64 quarter
// from the tiles in LDS. The operand reads of slice kk + 1 go out one
// between each two products of slice kk: a wave never waits on LDS with
// products it could have issued (the group barriers pin that order; left to
// itself the scheduler bunches the reads and waits for them before the
// products).
__device__ __forceinline__ void mfma_step(const u32x4* xs, const u32x4* ws, int wm, int wn, int half, int r32,
                                          f32x16 (&acc)[2][2]) {
  constexpr int kMfma = 0x008, kDsRead = 0x100;
  bf16x8 fa[2][2], fb[2][2];
  auto read = [&](int kk, int b) {
    const int c = 2 * kk + half;
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[b][i] = as_bf16x8(xs[slot(64 * wm + 32 * i + r32, c)]);
#pragma unroll
    for (int j = 0; j < 2; ++j) fb[b][j] = as_bf16x8(ws[slot(64 * wn + 32 * j + r32, c)]);
  };
  read(0, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int kk = 0; kk < kTileK / 16; ++kk) {
    if (kk + 1 < kTileK / 16) read(kk + 1, (kk + 1) & 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kk & 1][i], fb[kk & 1][j], acc[i][j], 0, 0, 0);
      }
    }
    if (kk + 1 < kTileK / 16) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// One 32 x 32 product tile into `out`: v[r] is row row0 + 8 (r / 4) + r % 4
// (row0 the tile's first row + 4 half), column col (of this lane). The bias,
// the add into y, the row map and the activation apply unless `split`.
template <Epi kEpi>
__device__ __forceinline__ void store_frag(const LinearArgs& a, float* out, bool split, int64_t row0, int64_t col,
                                           const f32x16& v) {
  if (col >= a.n) return;
  const bool add = !split && a.bias != nullptr;
  const bool accumulate = !split && a.accumulate;
  const float bv = add ? a.bias[col] : 0.0f;
  if constexpr (kEpi != Epi::kPlain) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = row0 + 8 * (r / 4) + (r % 4);
      if (row < a.m) store_act<kEpi>(a, row, col, add ? v[r] + bv : v[r]);
    }
    return;
  }
  if (a.row_map != nullptr) {
    float val[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) val[r] = v[r];
    store_mapped(a, row0, col, bv, add, val);
    return;
  }
  float* const o = out + row0 * a.n + col;  // element r: row row0 + 8 (r / 4) + r % 4
  auto live = [&](int r) { return row0 + 8 * (r / 4) + (r % 4) < a.m; };
  auto off = [&](int r) { return static_cast<int64_t>(8 * (r / 4) + (r % 4)) * a.n; };
  // accumulate: the 16 y values are requested before the first store (a
  // load issued after a store could alias it and would wait for it)
  float base[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) base[r] = accumulate && live(r) ? o[off(r)] : 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if (live(r)) {
      const float s = add ? v[r] + bv : v[r];
      o[off(r)] = accumulate ? base[r] + s : s;
    }
  }
}

// y = the sum of the splits' partial products in split order (+ bias);
// accumulate: y += that.
__global__ __launch_bounds__(kBlock) void split_sum_k(const float* __restrict__ part, int splits, int64_t m, int64_t n,
                                                       const float* __restrict__ bias, float* __restrict__ y,
                                                       bool accumulate) {
  const int64_t total = m * n;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * kBlock) {
    float v = part[i];
    for (int sp = 1; sp < splits; ++sp) v += part[sp * total + i];
    v = bias != nullptr ? v + bias[i % n] : v;
    y[i] = accumulate ? y[i] + v : v;
  }
}

__device__ __forceinline__ void zero(f32x16 (&acc)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    }
  }
}

// Chunks staged through registers (fp32 x, or a k that is not a multiple of
// 64; kRagged: not a multiple of 8).
template <bool kF32X, bool kRagged>
__global__ __launch_bounds__(kGemmThreads) void linear_staged_k(const LinearArgs a) {
  __shared__ u32x4 xs[2][kTileChunks];
  __shared__ u32x4 ws[2][kTileChunks];
  const Work wk = work_of(a);
  const int lane = threadIdx.x & (kWave - 1), wave = wave_in_block();
  const int wm = wave >> 1, wn = wave & 1;
  const int half = lane >> 5, r32 = lane & 31;
  f32x16 acc[2][2];
  zero(acc);
  const int steps = (wk.k_end - wk.k_begin + kTileK - 1) / kTileK;
  // a.runs > 1: the k steps in that many runs, as the split forms of
  // linear_pipe_k sum theirs (the same rows in fp32 and in bf16 then give the
  // same sums up to the order of the last additions)
  f32x16 total[2][2];
  zero(total);
  int run = 0, run_end = steps / a.runs;
  auto fold = [&] {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) total[i][j] += acc[i][j];
    }
    zero(acc);
  };
  Staged<kF32X> s;
  auto load = [&](int k0) {
    if constexpr (kRagged) {
      load_step_ragged(a, wk.m0, wk.n0, k0, wk.k_end, s);
    } else {
      load_step(a, wk.m0, wk.n0, k0, wk.k_end, s);
    }
  };
  load(wk.k_begin);
  store_step(s, xs[0], ws[0]);
  lds_barrier();
  for (int t = 0; t < steps; ++t) {
    const int buf = t & 1;
    const bool more = t + 1 < steps;
    if (more) load(wk.k_begin + (t + 1) * kTileK);
    mfma_step(xs[buf], ws[buf], wm, wn, half, r32, acc);
    if (a.runs > 1 && t + 1 >= run_end) {
      fold();
      do {
        ++run;
        run_end = static_cast<int>(static_cast<int64_t>(steps) * (run + 1) / a.runs);
      } while (run + 1 < a.runs && t + 1 >= run_end);
    }
    if (more) store_step(s, xs[buf ^ 1], ws[buf ^ 1]);
    lds_barrier();
  }
  const bool split = a.part != nullptr;
  float* out = split ? a.part + static_cast<int64_t>(wk.split) * a.m * a.n : a.y;
  if (a.runs > 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = total[i][j];
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      store_frag<Epi::kPlain>(a, out, split, wk.m0 + 64 * wm + 32 * i + 4 * half, wk.n0 + 64 * wn + 32 * j + r32,
                              acc[i][j]);
    }
  }
}

// A tile of TM x TN outputs by WM x WN x WK waves; kKC columns of k a step,
// kS steps of tiles in LDS, kS - 1 of them in flight ahead of the products.
//
// WK = 1: the WM x WN waves share the tiles, one barrier a step (behind it
// every wave's loads of the step are in LDS and every wave has read the step
// before, whose tiles the next loads overwrite).
//
// WM = WN = 1: each of the WK waves takes the whole tile over a WK-th of k
// with tiles of its own: no barrier, no operand read twice, and WK times the
// loads in flight of a tile that few workgroups share the chip for. The
// partial sums meet in LDS (rows kP floats apart: the two halves of a wave,
// four rows apart, write different banks) and are added in pairs.
//
// What bounds the small forms is the latency from the first load to the last
// store and, past that, a CU's 64 bytes a clock from L2: 64 x 896 x 1280
// 17.7 us by the earlier 32 x 128 tiles (one step's loads waited for a step)
// to 4.9, 64 x 1280 x 6848 91 to 16.5, 65 x 1024 x 4096 43 to 7.8; the
// library's best without a workspace 7.6 us at 384 x 896 x 1280 against 6.5,
// 13.6 at 257 x 1024 x 4096 against 10.9.
//
// kFar: row offsets of 64 bits (rows of 2^23 columns or more).
template <int TM, int TN, int WM, int WN, int WK, int kKC, int kS, bool kFar, Epi kEpi>
__global__ __launch_bounds__(kWave* WM* WN* WK) void linear_pipe_k(const LinearArgs a) {
  constexpr int kRC = kKC / 8, kGroup = WM * WN;  // chunks a tile row, waves sharing tiles
  constexpr int kXLoads = TM * kRC / kWave, kLoads = (TM + TN) * kRC / kWave / kGroup;
  constexpr int FM = TM / WM / 32, FN = TN / WN / 32;
  constexpr int kStage = (TM + TN) * kRC;
  constexpr int kP = TN + 8;
  constexpr int kTiles = WK * kS * kStage, kSums = WK > 1 ? WK * TM * kP / 4 : 0;
  static_assert((kXLoads + TN * kRC / kWave) % kGroup == 0 && (kGroup == 1 || WK == 1) && kS >= 2 && kS <= 3);
  static_assert(4 * kP % 64 == 32);
  using Off = std::conditional_t<kFar, uint64_t, uint32_t>;
  __shared__ u32x4 lds[kTiles > kSums ? kTiles : kSums];
  const int lane = threadIdx.x & (kWave - 1), wave = wave_in_block();
  const int grp = wave / kGroup, wg = wave % kGroup, wm = wg / WN, wn = wg % WN;
  const int half = lane >> 5, r32 = lane & 31;
  int tm, tn;
  tile_of(static_cast<int>(blockIdx.x), a.tiles_m, a.tiles_n, tm, tn);
  const int64_t m0 = static_cast<int64_t>(tm) * TM, n0 = static_cast<int64_t>(tn) * TN;
  const int steps = a.k / kKC;
  const int first = static_cast<int>(static_cast<int64_t>(steps) * grp / WK);
  const int n = static_cast<int>(static_cast<int64_t>(steps) * (grp + 1) / WK) - first;
  const char* const xb = static_cast<const char*>(a.x) + (m0 * a.k + static_cast<int64_t>(first) * kKC) * 2;
  const char* const wb = reinterpret_cast<const char*>(a.w) + (n0 * a.k + static_cast<int64_t>(first) * kKC) * 2;
  const int xlast = static_cast<int>(a.m - 1 - m0 < TM ? a.m - 1 - m0 : TM - 1);
  const int wlast = static_cast<int>(a.n - 1 - n0 < TN ? a.n - 1 - n0 : TN - 1);
  // 16 rows of 128 (64) bytes span 32 (16) bank groups of 16 bytes, of which
  // there are 16: the chunk moves with the row where the rows repeat
  auto swizzle = [](int row) { return kRC == 8 ? (row >> 1) & 7 : (row >> 2) & 3; };
  // load i of this wave: 64 slots of the x tile, then of the w tile; rows
  // past m or n read the last one (their sums are never stored)
  Off off[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int q = wg * kLoads + i;
    const bool isx = q < kXLoads;
    const int s = (isx ? q : q - kXLoads) * kWave + lane, row = s / kRC, c = (s % kRC) ^ swizzle(row);
    const int last = isx ? xlast : wlast;
    off[i] = static_cast<Off>(row < last ? row : last) * a.k * 2 + c * 16;
  }
  u32x4* const mine = lds + grp * kS * kStage;
  const uint32_t lds0 = lds_address(mine);
  auto issue = [&](int t, int buf) {
    const int64_t at = static_cast<int64_t>(t) * kKC * 2;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int q = wg * kLoads + i;
      dma16(lds0 + (buf * kStage + q * kWave) * 16, (q < kXLoads ? xb : wb) + at, off[i]);
    }
  };
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    }
  }
  auto products = [&](int buf) {
    const u32x4* xs = mine + buf * kStage;
    const u32x4* ws = xs + TM * kRC;
    bf16x8 fa[kRC / 2][FM], fb[kRC / 2][FN];
#pragma unroll
    for (int kk = 0; kk < kRC / 2; ++kk) {
      const int c = 2 * kk + half;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int row = 32 * (wm * FM + i) + r32;
        fa[kk][i] = as_bf16x8(xs[row * kRC + (c ^ swizzle(row))]);
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int row = 32 * (wn * FN + j) + r32;
        fb[kk][j] = as_bf16x8(ws[row * kRC + (c ^ swizzle(row))]);
      }
    }
#pragma unroll
    for (int kk = 0; kk < kRC / 2; ++kk) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[kk][i], fb[kk][j], acc[i][j], 0, 0, 0);
        }
      }
    }
  };
#pragma unroll
  for (int t = 0; t < kS - 1; ++t) {
    if (t < n) issue(t, t);
  }
  int buf = 0, next = kS - 1, t = 0;
  for (; t + kS - 1 < n; ++t) {
    wait_loads<(kS - 2) * kLoads, (kGroup > 1)>();
    issue(t + kS - 1, next);
    products(buf);
    buf = buf + 1 == kS ? 0 : buf + 1;
    next = next + 1 == kS ? 0 : next + 1;
  }
  if (kS == 3 && n > 1) {  // the last step's loads still in flight
    wait_loads<kLoads, (kGroup > 1)>();
    products(buf);
    buf = buf + 1 == kS ? 0 : buf + 1;
  }
  if (n > 0) {
    wait_loads<0, (kGroup > 1)>();
    products(buf);
  }

  if constexpr (WK == 1) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        store_frag<kEpi>(a, a.y, false, m0 + 32 * (wm * FM + i) + 4 * half, n0 + 32 * (wn * FN + j) + r32, acc[i][j]);
      }
    }
    return;
  }
  float* const part = reinterpret_cast<float*>(lds);
  __syncthreads();  // every wave has read its tiles
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        part[(grp * TM + 32 * i + 8 * (r / 4) + 4 * half + r % 4) * kP + 32 * j + r32] = acc[i][j][r];
      }
    }
  }
  __syncthreads();
  constexpr int kQuads = TN / 4, kThreads = kWave * WK;
  static_assert(TM * kQuads % kThreads == 0);
  const bool add = a.bias != nullptr;
#pragma unroll
  for (int it = 0; it < TM * kQuads / kThreads; ++it) {
    const int id = static_cast<int>(threadIdx.x) + kThreads * it, row = id / kQuads, q = id % kQuads;
    static_assert(WK == 1 || WK == 4);
    float4 u[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) u[g] = *reinterpret_cast<const float4*>(part + (g * TM + row) * kP + 4 * q);
    float v[4] = {(u[0].x + u[1].x) + (u[2].x + u[3].x), (u[0].y + u[1].y) + (u[2].y + u[3].y),
                  (u[0].z + u[1].z) + (u[2].z + u[3].z), (u[0].w + u[1].w) + (u[2].w + u[3].w)};
    const int64_t at = m0 + row, col = n0 + 4 * q;
    if (at >= a.m || col >= a.n) continue;
    int64_t to = at;
    if (a.row_map != nullptr) {
      to = a.row_map[at];
      if (to >= a.y_rows) continue;
    }
    const int cols = a.n - col < 4 ? static_cast<int>(a.n - col) : 4;
    if (a.vec) {
      if (add) {
        const float4 b = *reinterpret_cast<const float4*>(a.bias + col);
        v[0] += b.x;
        v[1] += b.y;
        v[2] += b.z;
        v[3] += b.w;
      }
      if constexpr (kEpi != Epi::kPlain) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = activate<kEpi>(v[e]);
        *reinterpret_cast<uint2*>(a.y16 + to * a.n + col) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      } else {
        float4* const o = reinterpret_cast<float4*>(a.y + to * a.n + col);
        if (a.accumulate) {
          const float4 y = *o;
          *o = make_float4(y.x + v[0], y.y + v[1], y.z + v[2], y.w + v[3]);
        } else {
          *o = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e >= cols) continue;
        if (add) v[e] += a.bias[col + e];
        if constexpr (kEpi != Epi::kPlain) {
          store_act<kEpi>(a, at, col + e, v[e]);
        } else {
          float* const o = a.y + to * a.n + col + e;
          *o = a.accumulate ? *o + v[e] : v[e];
        }
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void round_bf16_k(const float* __restrict__ src, int64_t n,
                                                        uint16_t* __restrict__ dst) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 8;
  if (i + 8 <= n) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(src + i), hi = *reinterpret_cast<const u32x4*>(src + i + 4);
    *reinterpret_cast<u32x4*>(dst + i) = u32x4{pack_bf16(__uint_as_float(lo.x), __uint_as_float(lo.y)),
                                               pack_bf16(__uint_as_float(lo.z), __uint_as_float(lo.w)),
                                               pack_bf16(__uint_as_float(hi.x), __uint_as_float(hi.y)),
                                               pack_bf16(__uint_as_float(hi.z), __uint_as_float(hi.w))};
  } else {
    for (int64_t j = i; j < n; ++j) dst[j] = f32_to_bf16(src[j]);
  }
}

// The forms of linear_pipe_k. Split forms: four waves over k, a tile to each
// CU; shared forms: waves over the tile.
enum class Form { kSplit32, kSplit64x32, kSplit64, kShared64, kShared128, kFar };

// Workgroups the split forms want at most: one a CU. A CU holds one of their
// workgroups (96 to 147 KB of tiles), so one more tile than this costs a
// second pass over the chip.
constexpr int64_t kChipTiles = 256;
// Past this many 64 x 64 tiles (three a CU, what it holds at once) the 128 x
// 128 ones by eight waves are ahead: 4900 x 768 x 768 (924) 25.4 against 16.7
// us, 3136 x 2304 x 768 (1764) 29 against 20.8, 4096 x 2304 x 768 (2304) 34.6
// against 33.8; 4096 x 768 x 3072 (768) 40.2 against 44.9.
constexpr int64_t kSharedTiles = 3 * kChipTiles;
// Rows of this many columns or more: 256 of them are 2^32 bytes.
constexpr int64_t kFarColumns = int64_t{1} << 23;

int64_t tiles_of(int64_t m, int64_t n, int64_t tm, int64_t tn) { return ((m + tm - 1) / tm) * ((n + tn - 1) / tn); }

// The smallest tiles that the chip holds at once (us at 16 / 64 / 384 / 900 x
// 896 x 1280, 32 x 32 / 64 x 32 / 64 x 64 split: 4.5 / 5.2 / 6.6; 4.9 / 6.2 /
// 8.2; 8.0 / 6.5 / 8.2; 17 / 10.7 / 8.4), past them the shared tiles (900 x
// 1280 x 896, 300 tiles: 64 x 64 split 12.0, shared 9.6). A rule on m, n and k
// alone, so that a product has the same sums whatever its epilogue.
// Up to kChain columns there is little to split, and the sums stay one chain
// over k in column order.
constexpr int64_t kChain = 256;

Form form_of(int64_t m, int64_t n, int64_t k) {
  if (k >= kFarColumns) return Form::kFar;
  if (k <= kChain) return tiles_of(m, n, 64, 64) <= kSharedTiles ? Form::kShared64 : Form::kShared128;
  if (tiles_of(m, n, 32, 32) <= kChipTiles) return Form::kSplit32;
  if (tiles_of(m, n, 64, 32) <= kChipTiles) return Form::kSplit64x32;
  if (tiles_of(m, n, 64, 64) <= kChipTiles) return Form::kSplit64;
  return tiles_of(m, n, 64, 64) <= kSharedTiles ? Form::kShared64 : Form::kShared128;
}

// The runs of k a form sums apart.
int runs_of(Form form) { return form == Form::kShared64 || form == Form::kShared128 ? 1 : 4; }

// Where the library's larger tiles are the faster ones (us, here / library):
// past the split forms with a long k (1600 x 768 x 3072, 300 tiles 23.4 /
// 20.3; 2500 x 768 x 3072 25.3 / 22.2; 1024 x 1280 x 6848 54 / 45) and, with
// a short one, past two passes of the chip (257 x 4096 x 1024, 320 tiles 10.7
// / 12.0, 400 x 3584 x 1280 14.9 / 15.7, 577 x 3072 x 1024 12.1 / 13.2, 2500 x
// 768 x 768, 480 tiles 10.1 / 10.6; 577 x 4096 x 1024, 640 tiles 15.4 / 14.6,
// 4096 x 768 x 768 14.1 / 13.0). A call into the library is 16 us of host
// time against 3.3, and a shape's first call times its candidates, which
// these sizes (a prompt's rows, an expert's share of them) hardly ever repeat.
// Products narrower than one tile stay with the library too (of 128 rows and
// more): most of a tile would be padding, and the features the small vision
// model is held to hang on which side of a bf16 rounding such a sum falls.
bool library_faster(int64_t m, int64_t n, int64_t k) {
  const int64_t tiles = tiles_of(m, n, 64, 64);
  return n < 32 || tiles > 2 * kChipTiles || (tiles > kChipTiles && k > 1280);
}

template <Epi kEpi>
void launch_pipe(LinearArgs& a, Form form, hipStream_t st) {
  auto launch = [&]<int TM, int TN, int WM, int WN, int WK, int kKC, int kS, bool kFar>() {
    a.tiles_m = static_cast<int>((a.m + TM - 1) / TM);
    a.tiles_n = static_cast<int>((a.n + TN - 1) / TN);
    linear_pipe_k<TM, TN, WM, WN, WK, kKC, kS, kFar, kEpi>
        <<<static_cast<unsigned>(a.tiles_m) * static_cast<unsigned>(a.tiles_n), kWave * WM * WN * WK, 0, st>>>(a);
  };
  switch (form) {
    case Form::kSplit32: launch.template operator()<32, 32, 1, 1, 4, 64, 3, false>(); break;
    case Form::kSplit64x32: launch.template operator()<64, 32, 1, 1, 4, 64, 3, false>(); break;
    case Form::kSplit64: launch.template operator()<64, 64, 1, 1, 4, 64, 2, false>(); break;
    case Form::kShared64: launch.template operator()<64, 64, 2, 2, 1, 64, 3, false>(); break;
    case Form::kShared128: launch.template operator()<128, 128, 2, 4, 1, 64, 2, false>(); break;
    case Form::kFar: launch.template operator()<32, 32, 1, 1, 4, 64, 3, true>(); break;
  }
}

}  // namespace

// The splits of k worth taking for an m x n x k product on the staged tiles:
// a product of fewer than 64 tiles with k >= 1024 gets enough workgroups to
// cover the 256 CUs twice, each split at least 4 steps of 64 columns; any
// other runs unsplit. (Measured at the vision encoder's shapes: 16-24 tiles
// with k of 2304-4608 run 1.3-1.9x faster split; 72-234 tiles, or k of
// 768-1024, lose 5-100% to the partial sums' traffic and the extra launch.)
int64_t splits_for(int64_t m, int64_t k, int64_t n) {
  const int64_t tiles = ((m + kTileM - 1) / kTileM) * ((n + kTileN - 1) / kTileN);
  if (tiles >= 64 || k < 16 * kTileK) return 1;
  int64_t s = (512 + tiles - 1) / tiles;
  s = s < k / (4 * kTileK) ? s : k / (4 * kTileK);
  return s < 32 ? s : 32;
}

int linear_entry(const char* what, void* stream, const void* x, bool f32x, int64_t m, int64_t k, const uint16_t* w,
                 int64_t n, const float* bias, float* y, float* workspace = nullptr, int64_t workspace_floats = 0,
                 bool accumulate = false, const int64_t* row_map = nullptr, int64_t y_rows = 0,
                 Epi epi = Epi::kPlain, uint16_t* y16 = nullptr) {
  UOCR_REQUIRE(m >= 0 && n >= 0 && k >= 0, what, "m, n and k must be >= 0");
  if (m == 0 || n == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(k >= 1 && k < (int64_t{1} << 30), what, "k must be in [1, 2^30)");
  UOCR_REQUIRE(x != nullptr && w != nullptr && (epi == Epi::kPlain ? y != nullptr : y16 != nullptr), what,
               "null x, w or y");
  const bool ragged = k % 8 != 0 || !aligned16(x) || !aligned16(w);
  const bool pipe = !ragged && !f32x && k % kTileK == 0;
  // products of bf16 rows with no epilogue beyond the bias (and the add
  // into y) go to the BLAS library where it is the faster and takes them
  if (!f32x && epi == Epi::kPlain && row_map == nullptr && (!pipe || library_faster(m, n, k))) {
    const int st =
        library_linear_bf16(what, as_stream(stream), static_cast<const uint16_t*>(x), m, k, w, n, bias, y, accumulate);
    if (st != kLibraryDeclined) return st;
  }
  UOCR_REQUIRE(tiles_of(m, n, 32, 32) < (int64_t{1} << 31), what, "too many tiles");
  LinearArgs a{x, w, bias, y, m, n, static_cast<int>(k), 0, 0, static_cast<int>(k), nullptr, accumulate, row_map,
               y_rows, y16, n % 4 == 0 && (bias == nullptr || aligned16(bias)) && aligned16(y) && aligned16(y16), 1};
  clear_launch_error();
  const hipStream_t st = as_stream(stream);
  if (pipe) {
    const Form form = form_of(m, n, k);
    if (epi == Epi::kGeluBf16) {
      launch_pipe<Epi::kGeluBf16>(a, form, st);
    } else if (epi == Epi::kQuickGeluBf16) {
      launch_pipe<Epi::kQuickGeluBf16>(a, form, st);
    } else {
      launch_pipe<Epi::kPlain>(a, form, st);
    }
    return check_launch(what);
  }
  // split k into the workspace when it holds the partial products
  int64_t splits = workspace != nullptr ? splits_for(m, k, n) : 1;
  if (splits > 1 && workspace_floats < splits * m * n) splits = 1;
  const int64_t k_len = splits > 1 ? (k / splits + kTileK - 1) / kTileK * kTileK : k;
  splits = (k + k_len - 1) / k_len;
  const int64_t tiles_m = (m + kTileM - 1) / kTileM, tiles_n = (n + kTileN - 1) / kTileN;
  UOCR_REQUIRE(tiles_m * tiles_n * splits < (int64_t{1} << 31), what, "too many tiles");
  a.tiles_m = static_cast<int>(tiles_m);
  a.tiles_n = static_cast<int>(tiles_n);
  a.k_len = static_cast<int>(k_len);
  a.part = splits > 1 ? workspace : nullptr;
  if (splits == 1) a.runs = runs_of(form_of(m, n, k));
  const unsigned grid = static_cast<unsigned>(tiles_m * tiles_n * splits);
  if (ragged) {
    if (f32x) {
      linear_staged_k<true, true><<<grid, kGemmThreads, 0, st>>>(a);
    } else {
      linear_staged_k<false, true><<<grid, kGemmThreads, 0, st>>>(a);
    }
  } else if (f32x) {
    linear_staged_k<true, false><<<grid, kGemmThreads, 0, st>>>(a);
  } else {
    linear_staged_k<false, false><<<grid, kGemmThreads, 0, st>>>(a);
  }
  if (splits > 1) {
    const int64_t blocks = (m * n + kBlock - 1) / kBlock;
    split_sum_k<<<static_cast<unsigned>(blocks < 65536 ? blocks : 65536), kBlock, 0, st>>>(
        workspace, static_cast<int>(splits), m, n, bias, y, accumulate);
  }
  return check_launch(what);
}

}  // namespace uocr_rocm

using namespace uocr_rocm;

extern "C" {

int uocr_rocm_linear(void* stream, const float* x, int64_t m, int64_t k, const uint16_t* w, int64_t n,
                     const float* bias, float* y) {
  // One row streams the weights once through the GEMV (the reference's
  // m == 1 path, ops.cu:271-274).
  if (m == 1 && k % 8 == 0 && k <= 12288 && aligned16(x) && aligned16(w)) {
    return uocr_rocm_gemv_bf16(stream, x, k, w, n, bias, y);
  }
  return linear_entry("uocr_rocm_linear", stream, x, true, m, k, w, n, bias, y);
}

int uocr_rocm_linear_bf16x(void* stream, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w, int64_t n,
                           const float* bias, float* y) {
  return linear_entry("uocr_rocm_linear_bf16x", stream, x, false, m, k, w, n, bias, y);
}

int64_t uocr_rocm_linear_workspace_floats(int64_t m, int64_t k, int64_t n) {
  if (m <= 1 || n <= 0 || k <= 0) return 0;
  const int64_t s = splits_for(m, k, n);
  return s > 1 ? s * m * n : 0;
}

int uocr_rocm_linear_ws(void* stream, const float* x, int64_t m, int64_t k, const uint16_t* w, int64_t n,
                        const float* bias, float* y, float* workspace, int64_t workspace_floats) {
  if (m == 1 && k % 8 == 0 && k <= 12288 && aligned16(x) && aligned16(w)) {
    return uocr_rocm_gemv_bf16(stream, x, k, w, n, bias, y);
  }
  return linear_entry("uocr_rocm_linear_ws", stream, x, true, m, k, w, n, bias, y, workspace, workspace_floats);
}

int uocr_rocm_linear_bf16x_ws(void* stream, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w, int64_t n,
                              const float* bias, float* y, float* workspace, int64_t workspace_floats) {
  return linear_entry("uocr_rocm_linear_bf16x_ws", stream, x, false, m, k, w, n, bias, y, workspace,
                      workspace_floats);
}

int uocr_rocm_linear_bf16x_add_ws(void* stream, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w, int64_t n,
                                  const float* bias, float* y, float* workspace, int64_t workspace_floats) {
  return linear_entry("uocr_rocm_linear_bf16x_add_ws", stream, x, false, m, k, w, n, bias, y, workspace,
                      workspace_floats, true);
}

int uocr_rocm_linear_bf16x_add_rows(void* stream, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w,
                                    int64_t n, const float* bias, float* y, const int64_t* y_row, int64_t y_rows) {
  constexpr const char* kWhat = "uocr_rocm_linear_bf16x_add_rows";
  UOCR_REQUIRE(y_row != nullptr || m == 0, kWhat, "null row map");
  UOCR_REQUIRE(y_rows >= 0, kWhat, "y_rows must be >= 0");
  UOCR_REQUIRE(k % kTileK == 0 && aligned16(x) && aligned16(w), kWhat,
               "k must be a multiple of 64 and x, w 16-byte aligned");
  return linear_entry(kWhat, stream, x, false, m, k, w, n, bias, y, nullptr, 0, true, y_row, y_rows);
}

int uocr_rocm_linear_bf16x_gelu_erf_bf16(void* stream, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w,
                                         int64_t n, const float* bias, uint16_t* y) {
  constexpr const char* kWhat = "uocr_rocm_linear_bf16x_gelu_erf_bf16";
  UOCR_REQUIRE(k % kTileK == 0 && aligned16(x) && aligned16(w), kWhat,
               "k must be a multiple of 64 and x, w 16-byte aligned");
  return linear_entry(kWhat, stream, x, false, m, k, w, n, bias, nullptr, nullptr, 0, false, nullptr, 0,
                      Epi::kGeluBf16, y);
}

int uocr_rocm_linear_bf16x_quick_gelu_bf16(void* stream, const uint16_t* x, int64_t m, int64_t k,
                                           const uint16_t* w, int64_t n, const float* bias, uint16_t* y) {
  constexpr const char* kWhat = "uocr_rocm_linear_bf16x_quick_gelu_bf16";
  UOCR_REQUIRE(k % kTileK == 0 && aligned16(x) && aligned16(w), kWhat,
               "k must be a multiple of 64 and x, w 16-byte aligned");
  return linear_entry(kWhat, stream, x, false, m, k, w, n, bias, nullptr, nullptr, 0, false, nullptr, 0,
                      Epi::kQuickGeluBf16, y);
}

int uocr_rocm_round_bf16(void* stream, const float* src, int64_t n, uint16_t* dst) {
  constexpr const char* kWhat = "uocr_rocm_round_bf16";
  UOCR_REQUIRE(n >= 0, kWhat, "n must be >= 0");
  if (n == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(src != nullptr && dst != nullptr, kWhat, "null pointer");
  UOCR_REQUIRE(aligned16(src) && aligned16(dst), kWhat, "src and dst must be 16-byte aligned");
  const int64_t blocks = (n + 8 * kBlock - 1) / (8 * kBlock);
  UOCR_REQUIRE(blocks < (int64_t{1} << 31), kWhat, "n too large");
  clear_launch_error();
  round_bf16_k<<<static_cast<unsigned>(blocks), kBlock, 0, as_stream(stream)>>>(src, n, dst);
  return check_launch(kWhat);
}

}  // extern "C"
