// One decode step's attention on gfx950: the query rows of one timestep per batch entry at
// absolute position t over the cached keys and values, all three branches and the gated mix.
//
// The prefill kernels re-pack a branch's whole K / V into fragment-native copies, which
// amortises over many query rows; a decode step reads each visible key once, so the copy
// alone moved several times the bytes the step needs (16 x 32000 cached tokens, H32 G2 dk =
// dv = 128: 378 us of re-packs a step).  Here the keys are read from the cache as they lie, and
// the keys of every branch are split over many workgroups: one workgroup takes 256 keys of
// one branch for up to 16 heads of a KV group (a wave 64 keys), merges its four waves'
// softmax states in LDS and writes one partial {max, sum, O} to the workspace;
// decode_mix_kernel folds the partials of each head, normalises, and mixes the branches with
// the activated gates in fp32.  Bound by the latency of one pass over a wave's loads, which
// are all in flight at once, and by launches: 18 us for the 58 MB of that step (12 us at the
// card's copy rate), 8 us at B1 H8 G2 T1000 dk = dv = 64; the re-packs, three forwards, index
// clean-up and mix it replaces took 506 and 45 us.
//
// Per wave: S^T = K Q^T with the K rows read straight into MFMA operand registers (lane
// (g, r) reads 16 bytes of key r), V rows through LDS (bf16: read back by the LDS transpose
// load as V^T fragments; fp32: V^T elements straight from memory), O^T += V^T P^T.
#include "nsa_attn.h"
#include "nsa_device.h"
#include "nsa_kernels.h"

namespace nsa {

constexpr int kDecWaveKeys = 64, kDecKeys = 256;  // keys of one wave, of one workgroup

// fp32 values of one partial: max[16], sum[16], O [16][DV]
__host__ __device__ inline int decode_part(int dv) { return 16 * (dv + 2); }

template <typename T, int DK, int DV>
__global__ __launch_bounds__(256) void decode_attn_kernel(DecodeArgs a) {
  using S = typename Store<T>::type;
  constexpr int EPF = Elem<T>::kPerFrag, KC = Elem<T>::kKChunk, NKC = DK / KC;
  constexpr bool kBf = sizeof(S) == 2;
  constexpr int VP = DV + 16;  // staged V row pitch: row + 32 bytes, conflict-free transpose reads
  constexpr int VBYTES = kBf ? 4 * kDecWaveKeys * VP * 2 : 0;
  constexpr int OBYTES = 4 * 16 * DV * 4;
  __shared__ __attribute__((aligned(16))) char s_buf[VBYTES > OBYTES ? VBYTES : OBYTES];
  __shared__ float s_m[4][16], s_l[4][16];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g4 = lane >> 4, c16 = lane & 15;
  const int bg = blockIdx.y, b = bg / a.G, grp = bg % a.G;
  // the workgroup's branch and its first key
  int wg = blockIdx.x, br = 0;
  while (br < 2 && wg >= a.nwg[br]) wg -= a.nwg[br++];
  const int pos0 = wg * kDecKeys + wave * kDecWaveKeys;

  const int hc = blockIdx.z * 16 + c16;  // the lane's head within the group
  const bool colv = hc < a.hpg;
  const S* qp = reinterpret_cast<const S*>(a.q) + b * a.sq_b + (int64_t)(grp * a.hpg + (colv ? hc : 0)) * a.sq_h;
  uint4 qf[NKC];
#pragma unroll
  for (int kc = 0; kc < NKC; ++kc)
    qf[kc] = colv ? *reinterpret_cast<const uint4*>(qp + kc * KC + g4 * EPF) : make_uint4(0, 0, 0, 0);

  // the wave's four 16-key groups: first key and number of visible keys
  int key0[4], nv[4];
  if (br == kDecSel) {
    int lv = lane < a.nslots ? (int)a.idx[(int64_t)bg * a.nslots + lane] : -1;
    if (__ballot(lv >= 0) == 0 && lane == 0) lv = a.t / a.lprime;  // no block chosen: the query's own
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = pos0 + 16 * u, slot = p / a.lprime;
      const int blk = slot < a.nslots ? __builtin_amdgcn_readlane(lv, slot) : -1;
      const int64_t k0 = (int64_t)blk * a.lprime + p % a.lprime;
      // a block counts at the first slot that names it (the cleaned lists are sets as well)
      const bool ok = blk >= 0 && k0 <= a.t && __builtin_ctzll(__ballot(lv == blk)) == slot;
      key0[u] = ok ? (int)k0 : 0;
      nv[u] = ok ? min(16, a.t + 1 - (int)k0) : 0;
    }
  } else {
    const int lo = br == kDecWin ? max(0, a.t - a.window + 1) : 0;
    const int n = br == kDecWin ? a.t + 1 : a.n_cmp;  // end of the visible keys
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k0 = lo + pos0 + 16 * u;
      key0[u] = k0 < n ? k0 : 0;
      nv[u] = max(0, min(16, n - k0));
    }
  }
  const S* kb = reinterpret_cast<const S*>(a.k[br]) + b * a.sk_b[br] + grp * a.sk_g[br];
  const S* vb = reinterpret_cast<const S*>(a.v[br]) + b * a.sv_b[br] + grp * a.sv_g[br];

  // V rows to LDS (bf16), the loads ahead of the S products; rows that are not visible are
  // zeros, so what they hold never meets a zero probability
  constexpr int LPR = DV * (int)sizeof(S) / 16;  // lanes per V row
  constexpr int RPI = 64 / LPR;                  // rows per load
  constexpr int NVI = kDecWaveKeys / RPI;
  uint4 vr[kBf ? NVI : 1];
  if constexpr (kBf) {
#pragma unroll
    for (int i = 0; i < NVI; ++i) {
      const int u = i * RPI / 16, r = (i * RPI) % 16 + lane / LPR;
      const S* p = vb + (int64_t)(key0[u] + min(r, max(nv[u] - 1, 0))) * a.sv_t[br] + (lane % LPR) * 8;
      const uint4 x = *reinterpret_cast<const uint4*>(p);
      vr[i] = r < nv[u] ? x : make_uint4(0, 0, 0, 0);
    }
  }
  f32x4 st[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const S* kp = kb + (int64_t)(key0[u] + min(c16, max(nv[u] - 1, 0))) * a.sk_t[br];
    uint4 kf[NKC];
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) kf[kc] = *reinterpret_cast<const uint4*>(kp + kc * KC + g4 * EPF);
    st[u] = zero4();
#pragma unroll
    for (int kc = 0; kc < NKC; ++kc) st[u] = Mma<T>::run(st[u], kf[kc], qf[kc]);
  }
  S* vs = reinterpret_cast<S*>(s_buf) + wave * kDecWaveKeys * VP;
  if constexpr (kBf) {
#pragma unroll
    for (int i = 0; i < NVI; ++i)
      *reinterpret_cast<uint4*>(vs + (i * RPI + lane / LPR) * VP + (lane % LPR) * 8) = vr[i];
  }

  // softmax of the wave's keys (lane: head c16, keys 4 g4 + i of each group)
  const float scale2 = a.scale * kLog2e;
  float mx = -INFINITY;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      st[u][i] = 4 * g4 + i < nv[u] ? st[u][i] : -INFINITY;
      mx = fmaxf(mx, st[u][i]);
    }
  mx = wave_max16(mx) * scale2;
  const float nref = mx == -INFINITY ? 0.f : -mx;
  float ls = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = fast_exp2(mul_add_rounded(st[u][i], scale2, nref));
      st[u][i] = p;
      ls += p;
    }
  ls = wave_sum16(ls);

  f32x4 oacc[DV / 16];
#pragma unroll
  for (int j = 0; j < DV / 16; ++j) oacc[j] = zero4();
  if constexpr (kBf) {
    wave_lds_sync();
    const S* vt = vs + (4 * g4 + (c16 >> 2)) * VP + (c16 & 3) * 4;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const uint4 pf = CFrag<T>::pack(st[2 * c], st[2 * c + 1]);
#pragma unroll
      for (int j = 0; j < DV / 16; ++j)
        oacc[j] = Mma<T>::run(oacc[j], ld_tr_pair(reinterpret_cast<const uint16_t*>(vt + 32 * c * VP + 16 * j), 16 * VP), pf);
    }
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint4 pf = CFrag<T>::pack(st[u], st[u]);
#pragma unroll
      for (int j = 0; j < DV / 16; ++j) {
        float x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 4 * g4 + i;
          const float y = Elem<T>::to_f32(vb[(int64_t)(key0[u] + min(r, max(nv[u] - 1, 0))) * a.sv_t[br] + 16 * j + c16]);
          x[i] = r < nv[u] ? y : 0.f;
        }
        oacc[j] = Mma<T>::run(oacc[j], CFrag<float>::pack(f32x4{x[0], x[1], x[2], x[3]}, zero4()), pf);
      }
    }
  }

  // the four waves' states merged through LDS (over the V rows, once every wave is past
  // them)
  if (g4 == 0) {
    s_m[wave][c16] = mx;
    s_l[wave][c16] = ls;
  }
  __syncthreads();
  float* so = reinterpret_cast<float*>(s_buf);
#pragma unroll
  for (int j = 0; j < DV / 16; ++j)
    *reinterpret_cast<f32x4*>(so + (wave * 16 + c16) * DV + 16 * j + 4 * g4) = oacc[j];
  __syncthreads();
  float* part = a.part + (((int64_t)bg * gridDim.z + blockIdx.z) * a.nparts + blockIdx.x) * decode_part(DV);
  for (int e = threadIdx.x; e < 16 * DV; e += 256) {
    const int c = e / DV;
    const float M = fmaxf(fmaxf(s_m[0][c], s_m[1][c]), fmaxf(s_m[2][c], s_m[3][c]));
    float o = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = s_m[w][c] == -INFINITY ? 0.f : fast_exp2(s_m[w][c] - M);
      o += f * so[w * 16 * DV + e];
      l += f * s_l[w][c];
    }
    part[32 + e] = o;
    if (e % DV == 0) {
      part[c] = M;
      part[16 + c] = l;
    }
  }
}

// One workgroup per (head, batch entry), a thread per output feature: the branches'
// partials folded, normalised and mixed.
template <typename T>
__global__ void decode_mix_kernel(DecodeArgs a, int nheadtiles) {
  using S = typename Store<T>::type;
  const int h = blockIdx.x, b = blockIdx.y, f = threadIdx.x, dv = blockDim.x;
  const int grp = h / a.hpg, hc = h % a.hpg, c = hc & 15;
  const int np = decode_part(dv);
  const float* p = a.part + (((int64_t)(b * a.G + grp) * nheadtiles + (hc >> 4)) * a.nparts) * np;
  float gate[3];
  const S* z = reinterpret_cast<const S*>(a.gates) + b * a.sg_b + h * a.sg_h;
#pragma unroll
  for (int k = 0; k < 3; ++k) gate[k] = Elem<T>::to_f32(z[k * a.sg_k]);
  if (a.act == 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) gate[k] = 1.f / (1.f + expf(-gate[k]));
  } else if (a.act == 2) {
    const float m = fmaxf(gate[0], fmaxf(gate[1], gate[2]));
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) s += gate[k] = expf(gate[k] - m);
#pragma unroll
    for (int k = 0; k < 3; ++k) gate[k] /= s;
  }
  float out = 0.f;
  for (int br = 0; br < 3; ++br) {
    float M = -INFINITY;
    for (int i = 0; i < a.nwg[br]; ++i) M = fmaxf(M, p[i * np + c]);
    float o = 0.f, l = 0.f;
    for (int i = 0; i < a.nwg[br]; ++i) {
      const float m = p[i * np + c];
      const float w = m == -INFINITY ? 0.f : fast_exp2(m - M);
      l += w * p[i * np + 16 + c];
      o += w * p[i * np + 32 + c * dv + f];
    }
    // no visible key: 0 (the sum is exactly 0); a NaN sum is one of a visible key and stays
    out += gate[br] * (l == 0.f ? 0.f : o / l);
    p += a.nwg[br] * np;
  }
  reinterpret_cast<S*>(a.out)[b * a.so_b + (int64_t)h * a.so_h + f] = Elem<T>::from_f32(out);
}

void decode_split(DecodeArgs& a) {
  a.nwg[kDecCmp] = (a.n_cmp + kDecKeys - 1) / kDecKeys;
  a.nwg[kDecSel] = (a.nslots * a.lprime + kDecKeys - 1) / kDecKeys;
  a.nwg[kDecWin] = (min(a.window, a.t + 1) + kDecKeys - 1) / kDecKeys;
  a.nparts = a.nwg[0] + a.nwg[1] + a.nwg[2];
}

size_t decode_part_bytes(const DecodeArgs& a, int dv) {
  return (size_t)a.B * a.G * ((a.hpg + 15) / 16) * a.nparts * decode_part(dv) * 4;
}

template <typename T, int DK, int DV>
static void launch_decode(const DecodeArgs& a, hipStream_t st) {
  const int nht = (a.hpg + 15) / 16;
  hipLaunchKernelGGL((decode_attn_kernel<T, DK, DV>), dim3(a.nparts, a.B * a.G, nht), dim3(256), 0, st, a);
  hipLaunchKernelGGL(decode_mix_kernel<T>, dim3(a.G * a.hpg, a.B), dim3(DV), 0, st, a, nht);
}

bool dispatch_decode(int dtype, int dk, int dv, const DecodeArgs& a, hipStream_t st) {
#define NSA_CASE(DKV, DVV)                                       \
  if (dk == DKV && dv == DVV) {                                  \
    if (dtype == kF32) launch_decode<float, DKV, DVV>(a, st);    \
    else launch_decode<bf16, DKV, DVV>(a, st);                   \
    return true;                                                 \
  }
  NSA_HEAD_DIMS(NSA_CASE)
#undef NSA_CASE
  return false;
}

}  // namespace nsa
