// Host-side launchers behind the C ABI (internal, not exported).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/nsa_hip.h"
#include "nsa_attn.h"

// Head-dimension pairs (DK, DV) with compiled kernels.  Other widths are served by
// zero-padding to the next pair in the host shim (padding q/k columns with zeros
// leaves q.k unchanged; padded v columns are dropped).
#define NSA_HEAD_DIMS(X) X(32, 32) X(64, 64) X(128, 128) X(192, 128)

namespace nsa {

void launch_repack(int dtype, const void* src, int64_t s_b, int64_t s_g, int64_t s_r, int64_t s_c, int B, int G,
                   int R, int C, int Rp, void* rowm, void* colm, void* rowf, void* colf, hipStream_t st);
// K and V fragment copies of one call (one launch when both suit the fragment kernel);
// sk / sv: (b, g, row, feature) strides
void launch_repack_kv(int dtype, const void* k, const int64_t* sk, int dk, void* krf, void* kcf, const void* v,
                      const int64_t* sv, int dv, void* vrf, void* vcf, int B, int G, int R, int Rp, hipStream_t st);

// return false when (dtype, dk, dv, branch) has no compiled kernel
bool dispatch_attn_fwd(int dtype, int dk, int dv, int br, const AttnArgs& a, hipStream_t st);
bool dispatch_attn_bwd_dq(int dtype, int dk, int dv, int br, const AttnArgs& a, hipStream_t st);
bool dispatch_attn_bwd_dkdv(int dtype, int dk, int dv, int br, const AttnArgs& a, hipStream_t st);
// lse2 / delta (/ row_dot) of every query row before a dK/dV kernel that runs first
bool launch_row_stats(int dtype, int dv, const AttnArgs& a, hipStream_t st);
void launch_partial_reduce(int dtype, int dk, int dv, int br, const AttnArgs& a, hipStream_t st);
// the compression dK/dV work list (a.cmp_plan) of at most a.items_per_bg items
void launch_cmp_plan(const AttnArgs& a, int* plan, hipStream_t st);
// dK / dV [B, G, Tkv, dk | dv] (a.dk / a.dv, any strides) set to zero
void launch_zero_dkdv(int dtype, int dk, int dv, const AttnArgs& a, hipStream_t st);

// selection index cleaning and block -> query CSR
void launch_sel_clean(const void* idx, int idx_is64, int64_t si_b, int64_t si_g, int64_t si_t, int64_t si_n, int B,
                      int G, int Tq, int n_in, int nslots, int lprime, int Tkv, int fallback, int causal, int* clean,
                      int* chunk_cnt, int nblk, int q0, hipStream_t st);
// csr_s (nullable) receives each entry's slot in its timestep's cleaned list
void launch_sel_csr(const int* clean, int* chunk_cnt, int B, int G, int Tq, int nslots, int nblk, int* csr_off,
                    int* csr_t, int* csr_s, int* seg_off, int seg, hipStream_t st);
int sel_csr_chunks(int Tq);

// one decode step's attention (nsa_decode.hip); branch order of the gates
enum DecodeBranch : int { kDecCmp = 0, kDecSel = 1, kDecWin = 2 };
struct DecodeArgs {
  const void* q;  // [B,H,DK]
  int64_t sq_b, sq_h;
  const void* k[3];  // per branch, strides (b, g, token)
  const void* v[3];
  int64_t sk_b[3], sk_g[3], sk_t[3], sv_b[3], sv_g[3], sv_t[3];
  const int64_t* idx;  // [B*G][nslots]
  const void* gates;   // [B,H,3]
  int64_t sg_b, sg_h, sg_k;
  void* out;  // [B,H,DV]
  int64_t so_b, so_h;
  float* part;  // workspace: [B*G][head tiles][nparts] partials
  int nwg[3];   // workgroups (partials) of each branch
  int nparts;
  int B, G, hpg, t, n_cmp, nslots, lprime, window, act;
  float scale;
};
void decode_split(DecodeArgs& a);  // nwg / nparts from the key counts
size_t decode_part_bytes(const DecodeArgs& a, int dv);
bool dispatch_decode(int dtype, int dk, int dv, const DecodeArgs& a, hipStream_t st);

// one linear layer over `batches` groups of `rows` rows (x / out batch strides in elements;
// row strides ldx and job.stride_row); returns NSA_OK or an error code
int launch_linear_rows(const void* x, int64_t ldx, int rows, int k, int batches, int64_t x_batch, int64_t out_batch,
                       const nsa_linear_job& job, int dtype, hipStream_t st);
// dW (and, when not null, db = the column sums of dY) over `rows` rows, logical row r being
// physical row r / rows_per * row_pitch + r % rows_per of both operands; n1, n2 multiples of
// 64; part: wgrad_bytes of fp32 workspace
size_t wgrad_bytes(int rows, int n1, int n2);
void launch_wgrad(int dtype, const void* dy, int64_t ld_dy, const void* x, int64_t ld_x, int rows, int rows_per,
                  int row_pitch, int n1, int n2, void* dw, int64_t ld_dw, void* db, float* part, hipStream_t st);

// record an error message for nsa_last_error(); returns `code`
int set_error(int code, const char* msg);

// Kernel ids for nsa_timing_begin (fwd / dq / dkdv are offset by the branch).
enum KernelId : int {
  kIdFwd = 0,    // + branch
  kIdDq = 3,     // + branch
  kIdDkdv = 6,   // + branch
  kIdReduce = 9,
  kIdScore = 10,
  kIdPoolFwd = 11,
  kIdPoolBwd = 12,
  kIdPrep = 13,  // K/V repack, row statistics, selection index CSR
};

// Records a HIP event pair around its lifetime when timing of `kind` is armed.
class TimingScope {
 public:
  TimingScope(int kind, hipStream_t st);
  ~TimingScope();

 private:
  bool active_;
  hipStream_t stream_;
};

}  // namespace nsa
