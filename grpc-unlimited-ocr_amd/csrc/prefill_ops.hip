// prefill_ops.hip: the fp32 products and row moves of a prefill pass for
// gfx950 (the reference's gemm_nt, gemm_nn, gather_rows and
// scatter_add_rows, src/backend/cuda/ops.h:19-27,56-60, ops.cu:185-190,
// 289-309, 377-391).
//
// gemm_nt / gemm_nn: c[b] = alpha a[b] . b[b]^T (b rows k-contiguous) or
// a[b] . b[b] (b rows n-contiguous), batched over slices `stride_*` elements
// apart, leading dimensions given. A workgroup of 256 threads computes a
// 64 x 64 tile of one slice; each thread a 4 x 4 block. k advances 16 at a
// time through LDS, both operands held k-major there so that a thread reads
// its 4 a values and 4 b values as two 16-byte loads per k. Sums are fp32
// (fused multiply-adds), alpha applied to the finished sum. Any m, n, k.
//
// gather_rows: dst[i] = src[index[i]]; scatter_add_rows: dst[index[i]] +=
// weight[i] * src[i] for i in order (each column walks the rows in order, so
// an index that repeats accumulates deterministically, as in the reference).

#include "common.hpp"

namespace uocr_rocm {
namespace {

constexpr int kGM = 64, kGN = 64, kGK = 16;
constexpr int kGemmBlock = 256;

struct GemmArgs {
  const float* a;
  const float* b;
  float* c;
  int64_t m, n, k;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;
  float alpha;
};

template <bool kNT>
__global__ __launch_bounds__(kGemmBlock) void gemm_f32_k(const GemmArgs g) {
  __shared__ __attribute__((aligned(16))) float as[kGK][kGM + 4];
  __shared__ __attribute__((aligned(16))) float bs[kGK][kGN + 4];
  const int64_t slice = blockIdx.z;
  const float* A = g.a + slice * g.sa;
  const float* B = g.b + slice * g.sb;
  float* C = g.c + slice * g.sc;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kGM, n0 = static_cast<int64_t>(blockIdx.x) * kGN;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
  }
  for (int64_t k0 = 0; k0 < g.k; k0 += kGK) {
#pragma unroll
    for (int i = 0; i < kGM * kGK / kGemmBlock; ++i) {
      const int id = static_cast<int>(threadIdx.x) + kGemmBlock * i;
      const int r = id / kGK, kk = id % kGK;
      const int64_t row = m0 + r, kc = k0 + kk;
      as[kk][r] = row < g.m && kc < g.k ? A[row * g.lda + kc] : 0.0f;
    }
    if constexpr (kNT) {
#pragma unroll
      for (int i = 0; i < kGN * kGK / kGemmBlock; ++i) {
        const int id = static_cast<int>(threadIdx.x) + kGemmBlock * i;
        const int r = id / kGK, kk = id % kGK;
        const int64_t col = n0 + r, kc = k0 + kk;
        bs[kk][r] = col < g.n && kc < g.k ? B[col * g.ldb + kc] : 0.0f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kGN * kGK / kGemmBlock; ++i) {
        const int id = static_cast<int>(threadIdx.x) + kGemmBlock * i;
        const int kk = id / kGN, cc = id % kGN;
        const int64_t col = n0 + cc, kc = k0 + kk;
        bs[kk][cc] = col < g.n && kc < g.k ? B[kc * g.ldb + col] : 0.0f;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kGK; ++kk) {
      const u32x4 av = *reinterpret_cast<const u32x4*>(&as[kk][4 * ty]);
      const u32x4 bv = *reinterpret_cast<const u32x4*>(&bs[kk][4 * tx]);
      const float a4[4] = {__uint_as_float(av.x), __uint_as_float(av.y), __uint_as_float(av.z), __uint_as_float(av.w)};
      const float b4[4] = {__uint_as_float(bv.x), __uint_as_float(bv.y), __uint_as_float(bv.z), __uint_as_float(bv.w)};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a4[i], b4[j], acc[i][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t row = m0 + 4 * ty + i;
    if (row >= g.m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t col = n0 + 4 * tx + j;
      if (col < g.n) C[row * g.ldc + col] = g.alpha * acc[i][j];
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

int gemm_entry(const char* what, bool nt, void* stream, int64_t m, int64_t n, int64_t k, float alpha, const float* a,
               int64_t lda, int64_t stride_a, const float* b, int64_t ldb, int64_t stride_b, float* c, int64_t ldc,
               int64_t stride_c, int64_t batch) {
  UOCR_REQUIRE(m >= 0 && n >= 0 && k >= 0 && batch >= 0, what, "m, n, k and batch must be >= 0");
  if (m == 0 || n == 0 || batch == 0) return UOCR_ROCM_OK;
  UOCR_REQUIRE(a != nullptr && b != nullptr && c != nullptr, what, "null pointer");
  UOCR_REQUIRE(lda >= k && ldc >= n && ldb >= (nt ? k : n), what, "a leading dimension is below the row width");
  UOCR_REQUIRE(stride_a >= 0 && stride_b >= 0 && stride_c >= 0, what, "strides must be >= 0");
  const int64_t gx = (n + kGN - 1) / kGN, gy = (m + kGM - 1) / kGM;
  UOCR_REQUIRE(gx < (int64_t{1} << 31) && gy < 65536 && batch < 65536, what, "grid too large");
  GemmArgs g{a, b, c, m, n, k, lda, ldb, ldc, stride_a, stride_b, stride_c, alpha};
  const dim3 grid(static_cast<unsigned>(gx), static_cast<unsigned>(gy), static_cast<unsigned>(batch));
  clear_launch_error();
  if (nt) {
    gemm_f32_k<true><<<grid, kGemmBlock, 0, as_stream(stream)>>>(g);
  } else {
    gemm_f32_k<false><<<grid, kGemmBlock, 0, as_stream(stream)>>>(g);
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
