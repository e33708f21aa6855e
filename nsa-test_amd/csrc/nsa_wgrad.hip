// Weight gradient of a token-wise linear layer, dW = dY^T X over every token row: the
// compression MLP's first layer reduces over all B*G*T tokens (32768 rows against a
// 384 x 192 weight at the paper configuration), a shape whose output has too few tiles
// for one GEMM to fill the GPU.  The rows are split into S chunks: workgroup (i, j, c)
// sums chunk c of the output tile (i, j) (64 rows by up to 192 columns) on the matrix
// cores (fp32), and a second pass adds the S partial tiles in chunk order
// (deterministic) and rounds once.
//
// Both operands are read row-major (token rows, features contiguous) into LDS; the MFMA
// fragments, whose K slots run along the token axis, come from LDS transpose loads.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/nsa_hip.h"
#include "nsa_device.h"
#include "nsa_kernels.h"

namespace nsa {

constexpr int kWgTile = 64;   // output rows per workgroup (dY features); n1, n2 multiples of it
constexpr int kWgRows = 64;   // token rows staged per step

// the widest column block (192, 128 or 64 columns) that divides n2
static int wgrad_block_cols(int n2) { return n2 % 192 == 0 ? 192 : n2 % 128 == 0 ? 128 : 64; }

// rows per chunk, a multiple of the staging step: enough chunks for about 512 workgroups
// over the output tiles, at most 64 (each chunk writes a partial of the whole output)
static int wgrad_chunk_rows(int rows, int n1, int n2) {
  const int tiles = (n1 / kWgTile) * (n2 / wgrad_block_cols(n2));
  int s = (512 + tiles - 1) / tiles;
  s = s < 1 ? 1 : s > 64 ? 64 : s;
  const int per = (rows + s - 1) / s;
  return ((per + kWgRows - 1) / kWgRows) * kWgRows;
}

// Workgroup (i, j, c): output rows 64 i .. + 63 and columns 16 NS j .. + 16 NS - 1 over the
// token rows of chunk c; wave w owns output rows 64 i + 16 w .. + 15 and all NS column
// subtiles, so every staged X row is read from HBM once per 64 output rows.  Logical row r is
// physical row r / rows_per * row_pitch + r % rows_per of both operands (the padded block
// rows of the compressed tokens).  With BIAS the column blocks j = 0 also sum dY over the
// rows (a product with ones), n1 values after the tile's n1 x n2.
// fp32: half the rows a step (the same LDS), one k slot per token in the operands' place.
template <typename T, int NS>
__global__ __launch_bounds__(256) void wgrad_partial_kernel(const typename Store<T>::type* __restrict__ dy,
                                                            int64_t ld_dy,
                                                            const typename Store<T>::type* __restrict__ x, int64_t ld_x,
                                                            int rows, IntDiv rows_per, int row_pitch, int n1, int n2,
                                                            int chunk_rows, int bias, float* __restrict__ part) {
  using S = typename Store<T>::type;
  constexpr bool kBf = sizeof(S) == 2;
  constexpr int EPF = Elem<T>::kPerFrag;
  constexpr int RS = kBf ? kWgRows : kWgRows / 2;  // rows staged per step
  constexpr int WB = 16 * NS;         // output columns of the workgroup
  constexpr int PB = WB + EPF;        // X tile pitch
  constexpr int PA = kWgTile + EPF;   // dY tile pitch
  constexpr int NPA = RS * kWgTile / EPF / 256;  // 16-byte pieces per thread and step
  constexpr int NPB = RS * WB / EPF / 256;
  __shared__ __attribute__((aligned(16))) S sa[2][RS * PA];
  __shared__ __attribute__((aligned(16))) S sb[2][RS * PB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, j = lane & 15;
  const int c1 = blockIdx.x * kWgTile, c2 = blockIdx.y * WB;
  const int r_lo = blockIdx.z * chunk_rows, r_hi = min(rows, r_lo + chunk_rows);
  uint4 va[NPA], vb[NPB];
  auto phys = [&](int r) __attribute__((always_inline)) -> int64_t {
    const int q = rows_per.div(r);
    return (int64_t)q * row_pitch + (r - q * rows_per.d);
  };
  auto load = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NPA; ++u) {
      const int p = tid + 256 * u, rr = p / (kWgTile / EPF), cc = (p % (kWgTile / EPF)) * EPF;
      const int r = r0 + rr;
      va[u] = r < r_hi ? *reinterpret_cast<const uint4*>(dy + phys(r) * ld_dy + c1 + cc) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < NPB; ++u) {
      const int p = tid + 256 * u, rr = p / (WB / EPF), cc = (p % (WB / EPF)) * EPF;
      const int r = r0 + rr;
      vb[u] = r < r_hi ? *reinterpret_cast<const uint4*>(x + phys(r) * ld_x + c2 + cc) : make_uint4(0, 0, 0, 0);
    }
  };
  auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NPA; ++u) {
      const int p = tid + 256 * u, rr = p / (kWgTile / EPF), cc = (p % (kWgTile / EPF)) * EPF;
      *reinterpret_cast<uint4*>(&sa[buf][rr * PA + cc]) = va[u];
    }
#pragma unroll
    for (int u = 0; u < NPB; ++u) {
      const int p = tid + 256 * u, rr = p / (WB / EPF), cc = (p % (WB / EPF)) * EPF;
      *reinterpret_cast<uint4*>(&sb[buf][rr * PB + cc]) = vb[u];
    }
  };
  f32x4 acc[NS], accb = zero4();
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = zero4();
  const bool sum_rows = bias && blockIdx.y == 0;
  int buf = 0;
  if (r_lo < r_hi) {
    load(r_lo);
    stage(0);
  }
  for (int r0 = r_lo; r0 < r_hi; r0 += RS) {
    __syncthreads();  // step r0 is staged in buf; the other buffer is free
    const bool more = r0 + RS < r_hi;
    if (more) load(r0 + RS);
    if constexpr (kBf) {
#pragma unroll
      for (int kc = 0; kc < RS / 32; ++kc) {
        // K slots 8g..8g+7 of a fragment are token rows kc*32 + 8g .. + 7: lanes 4 rho ..
        // 4 rho + 3 of a 16-lane group address row rho of a 4 x 16 block (transpose load)
        const int row = kc * 32 + 8 * g + (j >> 2), col = 4 * (j & 3);
        const uint4 a = ld_tr_pair(&sa[buf][row * PA + wave * 16 + col], 4 * PA);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const uint4 b = ld_tr_pair(&sb[buf][row * PB + s * 16 + col], 4 * PB);
          acc[s] = Mma<bf16>::run(acc[s], a, b);
        }
        if (sum_rows) accb = Mma<bf16>::run(accb, a, make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u));
      }
    } else {
#pragma unroll
      for (int k4 = 0; k4 < RS; k4 += 4) {
        const float a = sa[buf][(k4 + g) * PA + wave * 16 + j];
#pragma unroll
        for (int s = 0; s < NS; ++s)
          acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, sb[buf][(k4 + g) * PB + s * 16 + j], acc[s], 0, 0, 0);
        if (sum_rows) accb = __builtin_amdgcn_mfma_f32_16x16x4f32(a, 1.0f, accb, 0, 0, 0);
      }
    }
    if (more) stage(buf ^ 1);
    buf ^= 1;
  }
  // acc[s][i]: output (c1 + 16 wave + 4 g + i, c2 + 16 s + j)
  float* pt = part + (int64_t)blockIdx.z * n1 * (n2 + bias);
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int i = 0; i < 4; ++i) pt[(int64_t)(c1 + wave * 16 + 4 * g + i) * n2 + c2 + s * 16 + j] = acc[s][i];
  if (sum_rows && j == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) pt[(int64_t)n1 * n2 + c1 + wave * 16 + 4 * g + i] = accb[i];
}

// dW (db) = the chunks' partial tiles added in chunk order (reproducible), rounded once; eight
// chunks' loads in flight per step
template <typename T>
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const float* __restrict__ part, int nchunks, int n1, int n2,
                                                        int bias, typename Store<T>::type* __restrict__ dw,
                                                        int64_t ld_dw, typename Store<T>::type* __restrict__ db) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t nw = (int64_t)n1 * n2, ne = (int64_t)n1 * (n2 + bias);
  if (e >= ne) return;
  float s = 0.f;
  int c = 0;
  for (; c + 8 <= nchunks; c += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(part + (c + u) * ne + e);
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; c < nchunks; ++c) s += part[c * ne + e];
  if (e >= nw) db[e - nw] = Elem<T>::from_f32(s);
  else if (dw) dw[(e / n2) * ld_dw + e % n2] = Elem<T>::from_f32(s);
}

size_t wgrad_bytes(int rows, int n1, int n2) {
  const int per = wgrad_chunk_rows(rows, n1, n2);
  return (size_t)((rows + per - 1) / per) * n1 * (n2 + 1) * sizeof(float);
}

template <typename T>
static void launch_wgrad_t(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, int rows, int rows_per,
                           int row_pitch, int n1, int n2, void* dw, int64_t ld_dw, void* db, float* part,
                           hipStream_t st) {
  using S = typename Store<T>::type;
  const int per = rows > 0 ? wgrad_chunk_rows(rows, n1, n2) : 1, nchunks = (rows + per - 1) / per;
  const int bias = db != nullptr;
  if (rows > 0) {
    const int wb = wgrad_block_cols(n2);
    const dim3 grid(n1 / kWgTile, n2 / wb, nchunks);
    const IntDiv rp = IntDiv::make(rows_per);
    auto fn = wb == 192 ? wgrad_partial_kernel<T, 12> : wb == 128 ? wgrad_partial_kernel<T, 8> : wgrad_partial_kernel<T, 4>;
    hipLaunchKernelGGL(fn, grid, dim3(256), 0, st, (const S*)dy, ld_dy, (const S*)x, ld_x, rows, rp, row_pitch, n1, n2,
                       per, bias, part);
  }
  hipLaunchKernelGGL(wgrad_sum_kernel<T>, dim3((unsigned)(((int64_t)n1 * (n2 + bias) + 255) / 256)), dim3(256), 0, st,
                     (const float*)part, nchunks, n1, n2, bias, (S*)dw, ld_dw, (S*)db);
}

void launch_wgrad(int dtype, const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, int rows, int rows_per,
                  int row_pitch, int n1, int n2, void* dw, int64_t ld_dw, void* db, float* part, hipStream_t st) {
  auto fn = dtype == kF32 ? launch_wgrad_t<float> : launch_wgrad_t<bf16>;
  fn(dy, ld_dy, x, ld_x, rows, rows_per, row_pitch, n1, n2, dw, ld_dw, db, part, st);
}

}  // namespace nsa

extern "C" size_t nsa_wgrad_workspace_size(int rows, int n1, int n2) {
  if (rows <= 0 || n1 <= 0 || n2 <= 0 || n1 % nsa::kWgTile || n2 % nsa::kWgTile) return 0;
  const int per = nsa::wgrad_chunk_rows(rows, n1, n2);
  const size_t nchunks = (size_t)((rows + per - 1) / per);
  return nchunks * (size_t)n1 * (size_t)n2 * sizeof(float);
}

extern "C" int nsa_wgrad(const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, int rows, int n1, int n2,
                         void* dw, int64_t ld_dw, int dtype, void* workspace, size_t workspace_bytes,
                         nsa_stream_t stream) {
  using namespace nsa;
  if (dtype != NSA_BF16) return set_error(NSA_ERR_UNSUPPORTED, "nsa_wgrad: bf16 only");
  if (rows < 0 || n1 <= 0 || n2 <= 0 || n1 % kWgTile || n2 % kWgTile)
    return set_error(NSA_ERR_INVALID, "nsa_wgrad: n1 and n2 must be positive multiples of 64, rows >= 0");
  if ((rows > 0 && (!dy || !x)) || !dw) return set_error(NSA_ERR_INVALID, "nsa_wgrad: null pointer");
  if ((uintptr_t)dy % 16 || (uintptr_t)x % 16 || ld_dy % 8 || ld_x % 8 || ld_dy < n1 || ld_x < n2 || ld_dw < n2)
    return set_error(NSA_ERR_LAYOUT, "nsa_wgrad: rows must be 16-byte aligned with unit feature stride");
  if (rows > 0) {
    const size_t need = nsa_wgrad_workspace_size(rows, n1, n2);
    if (!workspace || workspace_bytes < need) {
      char msg[128];
      snprintf(msg, sizeof msg, "nsa_wgrad: workspace %zu bytes < required %zu", workspace_bytes, need);
      return set_error(NSA_ERR_WORKSPACE, msg);
    }
  }
  launch_wgrad(kBF16, dy, ld_dy, x, ld_x, rows, rows > 0 ? rows : 1, rows, n1, n2, dw, ld_dw, nullptr,
               reinterpret_cast<float*>(workspace), (hipStream_t)stream);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? NSA_OK : set_error(NSA_ERR_HIP, hipGetErrorString(e));
}
