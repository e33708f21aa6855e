// Linear layers over a few token rows (a decode step's projections) on gfx950: up to
// kLinJobs weight matrices applied to the same rows in one launch, each result written
// where it belongs (the query buffer, a token's slot of a K / V cache).
//
// y[r][n] = act(sum_k x[r][k] W[n][k] + b[n]) for up to 64 rows: every weight is read
// once, so the step is bound by the weight stream, and for small layers by launches.  A
// workgroup takes 16 features for all rows (W rows as the A operand of 16 x 16 x 32 MFMAs, the
// token rows as B); its eight waves take the K chunks in turn (together 512 contiguous bytes
// of each weight row), kLinU loads per wave in flight, and add their sums in wave order
// through LDS: fp32 throughout, rounded once.  Every 16 features read the rows once more (from
// L2), so past some rows x weights a library GEMM is faster: the callers say where (linear_one,
// OWN_OUT).
#include <stdio.h>

#include "../../include/nsa_hip.h"
#include "nsa_attn.h"
#include "nsa_device.h"
#include "nsa_kernels.h"

namespace nsa {

constexpr int kLinJobs = 8, kLinWaves = 8, kLinU = 10, kLinMaxRows = 64;

struct LinearArgs {
  const void* x;
  int64_t ldx;
  int rows, k, njobs;               // rows of one batch (grid z); 16 RT of them per workgroup (grid y)
  int64_t x_batch, out_batch;
  int tile0[kLinJobs + 1];  // first 16-feature tile of each job
  nsa_linear_job job[kLinJobs];
};

template <typename T, int RT>
__global__ __launch_bounds__(64 * kLinWaves) void linear_few_kernel(LinearArgs a) {
  using S = typename Store<T>::type;
  constexpr int EPF = Elem<T>::kPerFrag, KC = Elem<T>::kKChunk;
  constexpr int U = RT == 1 ? kLinU : RT == 2 ? 6 : 4;
  __shared__ f32x4 s_acc[kLinWaves][RT][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g4 = lane >> 4, c16 = lane & 15;
  int j = 0;
  while (j + 1 < a.njobs && (int)blockIdx.x >= a.tile0[j + 1]) ++j;
  const nsa_linear_job& jb = a.job[j];
  const int n0 = ((int)blockIdx.x - a.tile0[j]) * 16;
  const S* w = reinterpret_cast<const S*>(jb.w) + (int64_t)min(n0 + c16, jb.n - 1) * jb.ldw;
  const int row0 = blockIdx.y * 16 * RT;
  const S* xr[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
    xr[rt] = reinterpret_cast<const S*>(a.x) + blockIdx.z * a.x_batch + (int64_t)min(row0 + rt * 16 + c16, a.rows - 1) * a.ldx;
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = zero4();
  const int nk = (a.k + KC - 1) / KC;
  for (int c0 = wave; c0 < nk; c0 += kLinWaves * U) {
    uint4 wf[U], xf[U][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // unconditional loads (clamped), so that none of them waits at a branch; the pieces
      // past k (a last chunk's lane groups) are zeros in both operands
      const int e = min(c0 + u * kLinWaves, nk - 1) * KC + g4 * EPF;
      const int ec = min(e, a.k - EPF);
      wf[u] = *reinterpret_cast<const uint4*>(w + ec);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) xf[u][rt] = *reinterpret_cast<const uint4*>(xr[rt] + ec);
      if (e >= a.k) {
        wf[u] = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) xf[u][rt] = make_uint4(0, 0, 0, 0);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c0 + u * kLinWaves < nk)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = Mma<T>::run(acc[rt], wf[u], xf[u][rt]);
  }
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) s_acc[wave][rt][lane] = acc[rt];
  __syncthreads();
  if (wave >= RT) return;
  const int row = row0 + wave * 16 + c16;
  if (row >= a.rows) return;
  f32x4 v = s_acc[0][wave][lane];
#pragma unroll
  for (int i = 1; i < kLinWaves; ++i) v += s_acc[i][wave][lane];
  // lane (g4, c16): features n0 + 4 g4 + i of row c16; a group holds whole 16-feature tiles
  const S* bias = reinterpret_cast<const S*>(jb.bias);
  S* o = reinterpret_cast<S*>(jb.out) + blockIdx.z * a.out_batch + row * jb.stride_row + (n0 / jb.group) * jb.stride_group + n0 % jb.group + 4 * g4;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 4 * g4 + i;
    if (n >= jb.n) break;
    float y = v[i] + (bias ? Elem<T>::to_f32(bias[n]) : 0.f);
    if (jb.relu) y = y < 0.f ? 0.f : y;  // NaN stays NaN
    o[i] = Elem<T>::from_f32(y);
  }
}

template <typename T>
static void launch_linear(const LinearArgs& a, int batches, hipStream_t st) {
  const dim3 grid(a.tile0[a.njobs], (a.rows + 63) / 64, batches), block(64 * kLinWaves);
  if (a.rows <= 16) hipLaunchKernelGGL((linear_few_kernel<T, 1>), grid, block, 0, st, a);
  else if (a.rows <= 32) hipLaunchKernelGGL((linear_few_kernel<T, 2>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((linear_few_kernel<T, 4>), grid, block, 0, st, a);
}

int launch_linear_rows(const void* x, int64_t ldx, int rows, int k, int batches, int64_t x_batch, int64_t out_batch,
                       const nsa_linear_job& job, int dtype, hipStream_t st) {
  LinearArgs a{};
  a.x = x;
  a.ldx = ldx;
  a.rows = rows;
  a.k = k;
  a.njobs = 1;
  a.x_batch = x_batch;
  a.out_batch = out_batch;
  a.job[0] = job;
  a.tile0[1] = (job.n + 15) / 16;
  if (dtype == NSA_F32) launch_linear<float>(a, batches, st);
  else launch_linear<bf16>(a, batches, st);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NSA_OK : set_error(NSA_ERR_HIP, hipGetErrorString(e));
}

}  // namespace nsa

extern "C" int nsa_linear_few(const void* x, int64_t ld_x, int rows, int k, const nsa_linear_job* jobs, int n_jobs,
                              int dtype, nsa_stream_t stream) {
  using namespace nsa;
  if (dtype != NSA_F32 && dtype != NSA_BF16) return set_error(NSA_ERR_INVALID, "dtype not supported");
  if (!x || !jobs || n_jobs < 1 || n_jobs > kLinJobs || rows < 1 || rows > kLinMaxRows || k < 1)
    return set_error(NSA_ERR_INVALID, "need 1 to 64 rows, 1 to 8 jobs and k >= 1");
  const int esz = dtype == NSA_F32 ? 4 : 2;
  if (((uintptr_t)x) % 16 || (k * esz) % 16 || (rows > 1 && (ld_x * esz) % 16))
    return set_error(NSA_ERR_LAYOUT, "x needs 16-byte aligned rows of whole 16-byte pieces");
  LinearArgs a{};
  a.x = x;
  a.ldx = ld_x;
  a.rows = rows;
  a.k = k;
  a.njobs = n_jobs;
  for (int j = 0; j < n_jobs; ++j) {
    const nsa_linear_job& b = jobs[j];
    if (!b.w || !b.out || b.n < 1 || b.group < 1 || (b.group < b.n && b.group % 16) || (b.group < b.n && b.n % b.group))
      return set_error(NSA_ERR_INVALID, "a job needs w, out, n >= 1 and whole groups of a multiple of 16 features");
    if (((uintptr_t)b.w) % 16 || (b.n > 1 && (b.ldw * esz) % 16) || ((uintptr_t)b.out) % esz)
      return set_error(NSA_ERR_LAYOUT, "weights need 16-byte aligned rows");
    a.job[j] = b;
    a.tile0[j + 1] = a.tile0[j] + (b.n + 15) / 16;
  }
  if (dtype == NSA_F32) launch_linear<float>(a, 1, (hipStream_t)stream);
  else launch_linear<bf16>(a, 1, (hipStream_t)stream);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NSA_OK : set_error(NSA_ERR_HIP, hipGetErrorString(e));
}
