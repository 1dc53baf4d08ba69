// prefill_ops.hip: the fp32 products and row moves of a prefill pass for
// gfx950 (the reference's gemm_nt, gemm_nn, gather_rows and
// scatter_add_rows, src/backend/cuda/ops.h:19-27,56-60, ops.cu:185-190,
// 289-309, 377-391).
//
// gemm_nt / gemm_nn: c[b] = alpha a[b] . b[b]^T (b rows k-contiguous) or
// a[b] . b[b] (b rows n-contiguous), batched over slices `stride_*` elements
// apart, leading dimensions given, on the fp32 matrix cores
// (v_mfma_f32_32x32x2f32: fp32 products and sums, two columns of k each, lane
// half h supplying column 2 i + h of product i). No LDS for the operands: a
// lane reads 16 consecutive bytes of its k-contiguous row (half h columns
// 8 j + 4 h ..) and two half swaps put them in the products' order; the
// n-contiguous operand is read as 32 consecutive floats per half. The next
// span of k is in flight in registers while the current one multiplies.
// Sums run over k in order, one fused multiply-add a column (past kGemmChain
// columns: four such runs added in order), alpha applied to the finished
// sum. Any m, n, k.
//
// gather_rows: dst[i] = src[index[i]]; scatter_add_rows: dst[index[i]] +=
// weight[i] * src[i] for i in order (each column walks the rows in order, so
// an index that repeats accumulates deterministically, as in the reference).

#include "common.hpp"

namespace uocr_rocm {
namespace {

constexpr int kGemmTile = 32;  // rows and columns of one matrix-core product
constexpr int kGemmWaves = 4;

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct GemmArgs {
  const float* a;
  const float* b;
  float* c;
  int64_t m, n, k;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;
  float alpha;
  int tiles_n;          // workgroup tiles along n
  int64_t tiles;        // workgroup tiles of a slice
};

// Columns 8 j + 4 h + (0..3) of lane half h to columns 2 i + h of products
// i = 0..3 of the eight (v_permlane32_swap exchanges the first's high half
// with the second's low half).
__device__ __forceinline__ float4 product_order(float4 v) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.x), __float_as_uint(v.y), false, false);
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.z), __float_as_uint(v.w), false, false);
  return make_float4(__uint_as_float(p[0]), __uint_as_float(q[0]), __uint_as_float(p[1]), __uint_as_float(q[1]));
}

// Four consecutive floats: one 16-byte read, or four.
template <bool kVec>
__device__ __forceinline__ float4 load4(const float* p) {
  if constexpr (kVec) return *reinterpret_cast<const float4*>(p);
  return make_float4(p[0], p[1], p[2], p[3]);
}

// Wave tiles of 32 TM x 32 TN outputs. kSplitK: the workgroup's 4 waves take
// one tile's k in four runs (summed in wave order through LDS); else four
// tiles, two by two. kKC: columns of k held per span. kVecA / kVecB: the
// operand's rows allow 16-byte reads (kVecB for gemm_nt).
template <bool kNT, int TM, int TN, bool kSplitK, int kKC, bool kVecA, bool kVecB>
__global__ __launch_bounds__(kGemmWaves * kWave) void gemm_f32_k(const GemmArgs g) {
  constexpr int kJ = kKC / 8;
  __shared__ float part[kSplitK ? kGemmWaves * TN * 16 * kWave : 1];
  const int lane = static_cast<int>(threadIdx.x) % kWave, wave = wave_in_block();
  const int hl = lane >> 5, c = lane & 31;
  const unsigned id = xcd_block(blockIdx.x, gridDim.x);
  const int64_t slice = id / g.tiles;
  const int tile = static_cast<int>(id - slice * g.tiles);
  const int tm = tile / g.tiles_n, tn = tile - tm * g.tiles_n;
  const float* A = g.a + slice * g.sa;
  const float* B = g.b + slice * g.sb;
  float* C = g.c + slice * g.sc;
  const int64_t m0 = (kSplitK ? static_cast<int64_t>(tm) : 2 * static_cast<int64_t>(tm) + wave / 2) * kGemmTile * TM;
  const int64_t n0 = (kSplitK ? static_cast<int64_t>(tn) : 2 * static_cast<int64_t>(tn) + wave % 2) * kGemmTile * TN;
  if (!kSplitK && (m0 >= g.m || n0 >= g.n)) return;  // no barrier on this path
  int64_t k = 0, ke = g.k;
  if (kSplitK) {
    const int64_t run = (g.k + 8 * kGemmWaves - 1) / (8 * kGemmWaves) * 8;
    k = run * wave < g.k ? run * wave : g.k;
    ke = k + run < g.k ? k + run : g.k;
  }
  // rows and columns past the end repeat the last one; their sums are not stored
  const float* ap[TM];
  const float* bp[TN];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int64_t row = m0 + kGemmTile * t + c;
    ap[t] = A + (row < g.m ? row : g.m - 1) * g.lda;
  }
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const int64_t col = n0 + kGemmTile * t + c;
    bp[t] = kNT ? B + (col < g.n ? col : g.n - 1) * g.ldb : B + (col < g.n ? col : g.n - 1);
  }
  auto load_b = [&](int t, int64_t k8) -> float4 {
    if constexpr (kNT) {
      return load4<kVecB>(bp[t] + k8 + 4 * hl);
    } else {
      const float* p = bp[t] + (k8 + hl) * g.ldb;  // already in the products' order
      return make_float4(p[0], p[2 * g.ldb], p[4 * g.ldb], p[6 * g.ldb]);
    }
  };
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    }
  }
  auto multiply = [&](const float4 (&xs)[TM], const float4 (&ys)[TN]) {
    float4 x[TM], y[TN];
#pragma unroll
    for (int t = 0; t < TM; ++t) x[t] = product_order(xs[t]);
#pragma unroll
    for (int t = 0; t < TN; ++t) y[t] = kNT ? product_order(ys[t]) : ys[t];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i].x, y[j].x, acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i].y, y[j].y, acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i].z, y[j].z, acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i].w, y[j].w, acc[i][j], 0, 0, 0);
      }
    }
  };
  float4 x[kJ][TM], y[kJ][TN], xn[kJ][TM], yn[kJ][TN];
  auto load_span = [&](int64_t at, float4 (&xs)[kJ][TM], float4 (&ys)[kJ][TN]) {
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
#pragma unroll
      for (int t = 0; t < TM; ++t) xs[j][t] = load4<kVecA>(ap[t] + at + 8 * j + 4 * hl);
#pragma unroll
      for (int t = 0; t < TN; ++t) ys[j][t] = load_b(t, at + 8 * j);
    }
  };
  if (k + kKC <= ke) {
    load_span(k, x, y);
    while (k + 2 * kKC <= ke) {
      load_span(k + kKC, xn, yn);
      __builtin_amdgcn_sched_barrier(0);  // the next span's reads go out before this span's products
#pragma unroll
      for (int j = 0; j < kJ; ++j) multiply(x[j], y[j]);
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
#pragma unroll
        for (int t = 0; t < TM; ++t) x[j][t] = xn[j][t];
#pragma unroll
        for (int t = 0; t < TN; ++t) y[j][t] = yn[j][t];
      }
      k += kKC;
    }
#pragma unroll
    for (int j = 0; j < kJ; ++j) multiply(x[j], y[j]);
    k += kKC;
  }
  for (; k + 8 <= ke; k += 8) {
#pragma unroll
    for (int t = 0; t < TM; ++t) x[0][t] = load4<kVecA>(ap[t] + k + 4 * hl);
#pragma unroll
    for (int t = 0; t < TN; ++t) y[0][t] = load_b(t, k);
    multiply(x[0], y[0]);
  }
  if (k < ke) {  // the last columns one by one, zeros past them on both sides
    auto tail = [&](const float* p, int64_t step, int64_t first, int64_t apart) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t at = k + first + e * apart;
        v[e] = at < ke ? p[at * step] : 0.0f;
      }
      return make_float4(v[0], v[1], v[2], v[3]);
    };
#pragma unroll
    for (int t = 0; t < TM; ++t) x[0][t] = tail(ap[t], 1, 4 * hl, 1);
#pragma unroll
    for (int t = 0; t < TN; ++t) y[0][t] = kNT ? tail(bp[t], 1, 4 * hl, 1) : tail(bp[t], g.ldb, hl, 2);
    multiply(x[0], y[0]);
  }

  // register r of lane half h: row 8 (r / 4) + 4 h + r % 4, column c
  if constexpr (kSplitK) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i > 0) __syncthreads();  // part is read
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int r = 0; r < 16; ++r) part[((wave * TN + j) * 16 + r) * kWave + lane] = acc[i][j][r];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = n0 + kGemmTile * j + c;
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // this wave's quarter of the registers
          float sum = part[(j * 16 + 4 * wave + r) * kWave + lane];
#pragma unroll
          for (int w = 1; w < kGemmWaves; ++w) sum += part[((w * TN + j) * 16 + 4 * wave + r) * kWave + lane];
          const int64_t row = m0 + kGemmTile * i + 8 * wave + 4 * hl + r;
          if (row < g.m && col < g.n) C[row * g.ldc + col] = g.alpha * sum;
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = n0 + kGemmTile * j + c;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int64_t row = m0 + kGemmTile * i + 8 * (r / 4) + 4 * hl + r % 4;
          if (row < g.m && col < g.n) C[row * g.ldc + col] = g.alpha * acc[i][j][r];
        }
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void gather_rows_f32_k(const float* __restrict__ src,
                                                            const int64_t* __restrict__ index, int64_t rows,
                                                            int64_t cols, float* __restrict__ dst) {
  const int64_t total = rows * cols;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * kBlock) {
    const int64_t r = i / cols, c = i - r * cols;
    dst[i] = src[index[r] * cols + c];
  }
}

__global__ __launch_bounds__(kBlock) void scatter_add_rows_k(float* __restrict__ dst, const int64_t* __restrict__ index,
                                                             const float* __restrict__ weight,
                                                             const float* __restrict__ src, int64_t rows,
                                                             int64_t cols) {
#pragma clang fp contract(off)
  const int64_t c = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
  if (c >= cols) return;
  for (int64_t r = 0; r < rows; ++r) {
    float* d = dst + index[r] * cols + c;
    *d = *d + weight[r] * src[r * cols + c];
  }
}

// scatter_add_rows with the rows in parallel: a wave per (source row i, span
// of columns). The wave of the first row of an index owns its destination: it
// adds every row of that index in row order in registers (the same steps as
// the walk above, so the same bits) and stores once; the wave of a later row
// of the same index finds the earlier one in its scan of index[0..i) and
// leaves. Bound by latency (the index scan, rows / 64 coalesced reads a lane,
// four in flight, beside its own rows' loads issued first): 372 rows of 1280
// took 105 us as a walk by 5 workgroups, one dependent load and store a row.
// VW floats per lane and access: 4 (rows of whole, aligned 16-byte chunks) or 1.
constexpr int kScatterPer = 2;  // accesses per lane: 512 columns a wave at VW 4

template <int VW>
__global__ __launch_bounds__(kWave) void scatter_rows_once_k(float* dst, const int64_t* __restrict__ index,
                                                             const float* __restrict__ weight,
                                                             const float* __restrict__ src, int rows, int64_t cols) {
#pragma clang fp contract(off)
  constexpr int kScan = 4;
  const int i = static_cast<int>(blockIdx.x), lane = static_cast<int>(threadIdx.x);
  const int64_t c0 = (static_cast<int64_t>(blockIdx.y) * kScatterPer * kWave + lane) * VW;
  const int64_t mine = index[i];
  float* drow = dst + mine * cols;
  float v[kScatterPer][VW], t[kScatterPer][VW];
  auto load = [&](const float* row, float (&to)[kScatterPer][VW]) {
#pragma unroll
    for (int e = 0; e < kScatterPer; ++e) {
      const int64_t c = c0 + e * kWave * VW;
      if (c < cols) load_f32<VW>(row + c, to[e]);
    }
  };
  auto add = [&](float w) {
#pragma unroll
    for (int e = 0; e < kScatterPer; ++e) {
#pragma unroll
      for (int x = 0; x < VW; ++x) v[e][x] = v[e][x] + w * t[e][x];
    }
  };
  load(src + i * cols, t);
  load(drow, v);
  for (int j0 = 0; j0 < i; j0 += kScan * kWave) {
    bool hit = false;
#pragma unroll
    for (int u = 0; u < kScan; ++u) {
      const int j = j0 + u * kWave + lane;
      hit = hit || index[j < i ? j : i - 1] == mine;
    }
    if (__ballot(hit) != 0) return;
  }
  add(weight[i]);
  for (int j0 = i + 1; j0 < rows; j0 += kScan * kWave) {
    uint64_t m[kScan], any = 0;
#pragma unroll
    for (int u = 0; u < kScan; ++u) {
      const int j = j0 + u * kWave + lane;
      m[u] = __ballot(index[j < rows ? j : rows - 1] == mine && j < rows);
      any |= m[u];
    }
    if (any == 0) continue;
#pragma unroll
    for (int u = 0; u < kScan; ++u) {
      for (uint64_t b = m[u]; b != 0; b &= b - 1) {
        const int j = j0 + u * kWave + __builtin_ctzll(b);
        load(src + j * cols, t);
        add(weight[j]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < kScatterPer; ++e) {
    const int64_t c = c0 + e * kWave * VW;
    if (c < cols) {
      if constexpr (VW == 4) {
        *reinterpret_cast<float4*>(drow + c) = make_float4(v[e][0], v[e][1], v[e][2], v[e][3]);
      } else {
        drow[c] = v[e][0];
      }
    }
  }
}

// Rows up to which the scans (rows^2 index reads over the waves) stay cheaper
// than the walk, whose one dependent load and store a row takes 0.28 us.
constexpr int64_t kScatterScanRows = 65536;

constexpr int64_t kGemmGrid = int64_t{1} << 23;  // workgroups a launch (of 256 threads, below 2^32 in all)

// The four forms a product takes: 64 x 64 or 32 x 32 wave tiles with k whole,
// 64 x 32 or 32 x 32 tiles with k over the workgroup's four waves.
enum class GemmForm { kWide, kWhole32, kSplit64, kSplit32 };

// Products of at most this many columns are summed in column order as one
// chain; longer ones as four.
constexpr int64_t kGemmChain = 256;

template <bool kNT, bool kVecA, bool kVecB>
void launch_gemm(const GemmArgs& g, unsigned grid, GemmForm form, hipStream_t st) {
  constexpr int kThreads = kGemmWaves * kWave;
  if (form == GemmForm::kWide) {
    gemm_f32_k<kNT, 2, 2, false, 8, kVecA, kVecB><<<grid, kThreads, 0, st>>>(g);
  } else if (form == GemmForm::kWhole32) {
    gemm_f32_k<kNT, 1, 1, false, 32, kVecA, kVecB><<<grid, kThreads, 0, st>>>(g);
  } else if (form == GemmForm::kSplit64) {
    gemm_f32_k<kNT, 2, 1, true, 16, kVecA, kVecB><<<grid, kThreads, 0, st>>>(g);
  } else {
    gemm_f32_k<kNT, 1, 1, true, 32, kVecA, kVecB><<<grid, kThreads, 0, st>>>(g);
  }
}

int gemm_entry(const char* what, bool nt, void* stream, int64_t m, int64_t n, int64_t k, float alpha, const float* a,
               int64_t lda, int64_t stride_a, const float* b, int64_t ldb, int64_t stride_b, float* c, int64_t ldc,
               int64_t stride_c, int64_t batch) {
  UOCR_REQUIRE(m >= 0 && n >= 0 && k >= 0 && batch >= 0, what, "m, n, k and batch must be >= 0");
  if (m == 0 || n == 0 || batch == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(a != nullptr && b != nullptr && c != nullptr, what, "null pointer");
  UOCR_REQUIRE(lda >= k && ldc >= n && ldb >= (nt ? k : n), what, "a leading dimension is below the row width");
  UOCR_REQUIRE(stride_a >= 0 && stride_b >= 0 && stride_c >= 0, what, "strides must be >= 0");
  UOCR_REQUIRE((m + 63) / 64 < 65536 && batch < 65536, what, "grid too large");
  clear_launch_error();
  const auto up = [](int64_t x, int64_t d) { return (x + d - 1) / d; };
  // Short k: the wide tiles read least a product, where there are enough of
  // them to give every SIMD one (us, wide / 32 x 32: 10 x 1003 x 1520 k 96
  // 47 / 61, 16 x 512 x 512 k 128 17 / 24, 16 x 257 x 257 k 96 11.6 / 9.5).
  // Long k over four waves, with the larger tile once it gives every CU a
  // workgroup (whole / 64 x 32 / 32 x 32: 10 x 1003 x 96 k 1520 94 / 46 / 56,
  // 4096 x 64 k 1280 38 / 17.8 / 12.7). A thread per 4 x 4 outputs over
  // operands staged in LDS, the form before these, took 67, 31, 14.1, 272 and
  // 161 us on the same five. Outputs past 2^34 take the wide tiles, whose
  // grid then still fits.
  const int64_t wide = up(m, 64) * up(n, 64);
  const GemmForm form = wide >= kGemmGrid / 2 || (k <= kGemmChain && wide * batch >= 1024) ? GemmForm::kWide
                        : k <= kGemmChain                                              ? GemmForm::kWhole32
                        : up(m, 64) * up(n, 32) * batch >= 256                         ? GemmForm::kSplit64
                                                                                       : GemmForm::kSplit32;
  const int64_t tile_m = form == GemmForm::kWide ? 128 : form == GemmForm::kSplit32 ? 32 : 64;
  const int64_t tile_n = form == GemmForm::kWide ? 128 : form == GemmForm::kWhole32 ? 64 : 32;
  const int64_t tiles_n = up(n, tile_n), tiles = up(m, tile_m) * tiles_n;
  UOCR_REQUIRE(tiles < kGemmGrid, what, "grid too large");
  const auto rows16 = [](const float* p, int64_t ld, int64_t stride, int64_t slices) {
    return aligned16(p) && ld % 4 == 0 && (slices == 1 || stride % 4 == 0);
  };
  const bool va = rows16(a, lda, stride_a, batch), vb = nt && rows16(b, ldb, stride_b, batch);
  const int64_t per = kGemmGrid / tiles;  // slices a launch
  for (int64_t s = 0; s < batch; s += per) {
    const int64_t count = batch - s < per ? batch - s : per;
    const GemmArgs g{a + s * stride_a, b + s * stride_b, c + s * stride_c, m, n, k, lda, ldb, ldc,
                     stride_a, stride_b, stride_c, alpha, static_cast<int>(tiles_n), tiles};
    const unsigned grid = static_cast<unsigned>(tiles * count);
    const hipStream_t st = as_stream(stream);
    if (nt) {
      if (va && vb) {
        launch_gemm<true, true, true>(g, grid, form, st);
      } else {
        launch_gemm<true, false, false>(g, grid, form, st);
      }
    } else if (va) {
      launch_gemm<false, true, false>(g, grid, form, st);
    } else {
      launch_gemm<false, false, false>(g, grid, form, st);
    }
  }
  return check_launch(what);
}

unsigned flat_blocks(int64_t total) {
  const int64_t b = (total + kBlock - 1) / kBlock;
  return static_cast<unsigned>(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

}  // namespace
}  // namespace uocr_rocm

using namespace uocr_rocm;

extern "C" {

int uocr_rocm_gemm_nt(void* stream, int64_t m, int64_t n, int64_t k, float alpha, const float* a, int64_t lda,
                      int64_t stride_a, const float* b, int64_t ldb, int64_t stride_b, float* c, int64_t ldc,
                      int64_t stride_c, int64_t batch) {
  return gemm_entry("uocr_rocm_gemm_nt", true, stream, m, n, k, alpha, a, lda, stride_a, b, ldb, stride_b, c, ldc,
                    stride_c, batch);
}

int uocr_rocm_gemm_nn(void* stream, int64_t m, int64_t n, int64_t k, const float* a, int64_t lda, int64_t stride_a,
                      const float* b, int64_t ldb, int64_t stride_b, float* c, int64_t ldc, int64_t stride_c,
                      int64_t batch) {
  return gemm_entry("uocr_rocm_gemm_nn", false, stream, m, n, k, 1.0f, a, lda, stride_a, b, ldb, stride_b, c, ldc,
                    stride_c, batch);
}

int uocr_rocm_gather_rows(void* stream, const float* src, const int64_t* index, int64_t rows, int64_t cols,
                          float* dst) {
  constexpr const char* kWhat = "uocr_rocm_gather_rows";
  UOCR_REQUIRE(rows >= 0 && cols >= 0, kWhat, "rows and cols must be >= 0");
  if (rows == 0 || cols == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(src != nullptr && index != nullptr && dst != nullptr, kWhat, "null pointer");
  clear_launch_error();
  gather_rows_f32_k<<<flat_blocks(rows * cols), kBlock, 0, as_stream(stream)>>>(src, index, rows, cols, dst);
  return check_launch(kWhat);
}

int uocr_rocm_scatter_add_rows(void* stream, float* dst, const int64_t* index, const float* weight, const float* src,
                               int64_t rows, int64_t cols) {
  constexpr const char* kWhat = "uocr_rocm_scatter_add_rows";
  UOCR_REQUIRE(rows >= 0 && cols >= 0, kWhat, "rows and cols must be >= 0");
  if (rows == 0 || cols == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(dst != nullptr && index != nullptr && weight != nullptr && src != nullptr, kWhat, "null pointer");
  UOCR_REQUIRE(cols < (int64_t{1} << 40), kWhat, "cols too large");
  clear_launch_error();
  const bool vec = cols % 4 == 0 && aligned16(dst) && aligned16(src);
  const int64_t span = kScatterPer * kWave * (vec ? 4 : 1), spans = (cols + span - 1) / span;
  if (rows <= kScatterScanRows && spans < 65536) {
    const dim3 grid(static_cast<unsigned>(rows), static_cast<unsigned>(spans));
    if (vec) {
      scatter_rows_once_k<4><<<grid, kWave, 0, as_stream(stream)>>>(dst, index, weight, src, static_cast<int>(rows),
                                                                    cols);
    } else {
      scatter_rows_once_k<1><<<grid, kWave, 0, as_stream(stream)>>>(dst, index, weight, src, static_cast<int>(rows),
                                                                    cols);
    }
    return check_launch(kWhat);
  }
  scatter_add_rows_k<<<static_cast<unsigned>((cols + kBlock - 1) / kBlock), kBlock, 0, as_stream(stream)>>>(
      dst, index, weight, src, rows, cols);
  return check_launch(kWhat);
}

}  // extern "C"
