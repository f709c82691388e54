// Scaled dot-product attention (cv3cpu/ops.py:244-310) on strided q/k/v.
//
//   out[b, h, n, :] = softmax_m((q[b, h, n] * scale) . k[b, h', m]  + mask) . v[b, h', m]
//   with h' = h / (H / Hk) (grouped-query attention, ops.py:279-283) and masks
//   none / ("causal", offset) / ("chunk", size, left) (ops.py:244-264).
//
// The reference takes one ordinary softmax per query tile; here the softmax is
// streamed over key tiles (online max/sum rescaling), which changes only
// rounding.  The head_dim == 64 path runs on the matrix cores with
// v_mfma_f32_16x16x4_f32.  It computes S^T = K . Q^T so that each lane's
// accumulator registers already hold P^T in the B-operand layout of the next
// MFMA, O^T += V^T . P^T: no LDS round trip for the probabilities.
#include "bf16x3.hpp"
#include "common.hpp"

using namespace cv3;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct AttnParams {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  int64_t q_sb, q_sh, q_sn;
  int64_t k_sb, k_sh, k_sm;
  int64_t v_sb, v_sh, v_sm;
  int64_t o_sb, o_sh, o_sn;
  int h, hk;
  int64_t n, m;
  int d;
  float scale;
  int mask_kind;  // 0 none, 1 causal(a = offset), 2 chunk(a = size, b = left)
  int64_t mask_a, mask_b;
  uint2* op;      // k_flash64x: the output's bfloat16 planes in fragment order instead of o, or null
  int64_t opl;    // 8-byte halves per plane
};

// Every mask spec leaves query qi an interval of visible keys [lo, hi):
//   none  -> [0, m);   ("causal", a) -> [0, qi + a + 1);
//   ("chunk", size, left) -> [max((qi/size - left) * size, 0), (qi/size + 1) * size), left < 0: from 0.
// (ops.py:244-264.)  Computed once per query, applied with selects.
__device__ __forceinline__ void visible_keys(const AttnParams& p, int64_t qi, int64_t& lo, int64_t& hi) {
  lo = 0;
  hi = p.m;
  if (p.mask_kind == 1) {
    hi = min(hi, qi + p.mask_a + 1);
  } else if (p.mask_kind == 2) {
    const int64_t c = qi / p.mask_a;
    hi = min(hi, (c + 1) * p.mask_a);
    if (p.mask_b >= 0) lo = max((int64_t)0, (c - p.mask_b) * p.mask_a);
  }
}

constexpr int KT = 64;        // keys per LDS tile
constexpr float kLog2E = 1.4426950408889634f;
constexpr int KS = 68;        // LDS row stride (floats) for K and V tiles
constexpr int QW = 16;        // queries per wave
constexpr int QT = 64;        // queries per workgroup
constexpr int kNumCU = 256;

// 4 * NKG waves: wave w takes queries (w % 4) * 16 .. +15 of the workgroup's 64 and
// key group kg = w / 4.  Each stage stages NKG tiles of 64 keys; key group kg works
// on tile NKG * stage + kg, so every SIMD runs NKG waves (one per key group) and the
// key range is split between them.  Each wave keeps its own online softmax
// (max, sum, output) and the groups merge in LDS at the end:
//   M = max_g m_g, l = sum_g l_g e^{m_g-M}, o = sum_g o_g e^{m_g-M}.
// NKG = 4 (1024 threads, 139 KB of LDS) hides the per-tile latency chain better on
// long key ranges (1024 keys and up); shorter ones keep NKG = 2.
// Per tile a wave scores all 64 keys (64 MFMAs), rescales its running state once,
// then accumulates P V (64 MFMAs).  V is staged transposed ([dim][key]) so the
// P V operands of four consecutive keys are one 16-byte LDS read.
// Scores are kept in base-2 units: q is scaled by log2(e) after the reference's
// (q * scale), so every exponential is one v_exp_f32 (2^x) instead of an expf
// range reduction; e^{s - m} = 2^{s log2 e - m log2 e}, to within a few ulp.
//
// The grid is one-dimensional, nq query tiles x h heads x batch.  Workgroup w runs on XCD w % 8
// (round-robin dispatch), and each XCD has its own L2: when the tile count divides by 8, XCD x
// takes the x-th eighth of the tiles in (batch, head)-major order, so each head's K / V rows
// are fetched into one L2 and re-read from there by that head's query tiles (otherwise every
// XCD would hold a query tile of every head and fetch all of K / V).
template <int NKG>
__global__ __launch_bounds__(256 * NKG) void k_flash64(AttnParams p, int nq) {
  __shared__ float Ks[NKG][KT * KS];
  __shared__ float Vs[NKG][KT * KS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int qw = wave & 3, kg = wave >> 2;
  const int ntiles = (int)gridDim.x;
  const int wg = (int)blockIdx.x;
  const int tile = (ntiles & 7) == 0 ? (wg & 7) * (ntiles >> 3) + (wg >> 3) : wg;
  const int qt = tile % nq, bh = tile / nq;
  const int b = bh / p.h, hq = bh % p.h;
  const int hkv = hq / (p.h / p.hk);
  const int64_t q0 = (int64_t)qt * QT + qw * QW;
  const int c16 = lane & 15, g = lane >> 4;
  const int64_t qi = q0 + c16;
  const bool qvalid = qi < p.n;
  int64_t klo64, khi64;
  visible_keys(p, qi, klo64, khi64);
  const int klo = (int)klo64, khi = (int)khi64;  // the host bounds m below 2^31 - 64

  // Q fragments, pre-scaled like the reference's (q * scale) (ops.py:292)
  f32x4 qf[4];
  const float* qrow = p.q + b * p.q_sb + hq * p.q_sh + (qvalid ? qi : 0) * p.q_sn;
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
    const float4 t = qvalid ? *reinterpret_cast<const float4*>(qrow + s4 * 16 + g * 4) : make_float4(0, 0, 0, 0);
    qf[s4] = f32x4{(t.x * p.scale) * kLog2E, (t.y * p.scale) * kLog2E, (t.z * p.scale) * kLog2E,
                   (t.w * p.scale) * kLog2E};
  }

  f32x4 oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) oacc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  const float* kbase = p.k + b * p.k_sb + hkv * p.k_sh;
  const float* vbase = p.v + b * p.v_sb + hkv * p.v_sh;
  const int64_t nstages = ceil_div(p.m, NKG * KT);
  // The next stage's NKG * 64 K/V rows are loaded into registers while the current stage
  // is computed.  Rows past m are clamped to m - 1 (always in bounds); their scores
  // are masked to -inf below, so the loads carry no predicates.
  // K: thread -> tile tid/256, keys (tid%256)/16 + 16r (r < 4), dims (tid%16)*4 .. +3.
  // V: thread -> tile tid/256, key tid%64, dims ((tid/64)%4)*16 .. +15, so the transposed
  // LDS stores of one wave hit 64 consecutive keys of a dim row.
  const int ltile = tid >> 8, lkey = (tid & 255) >> 4, ld4 = (tid & 15) * 4;
  const int vkey = tid & 63, vd = ((tid >> 6) & 3) * 16;
  float4 k0r, k1r, k2r, k3r, v0r, v1r, v2r, v3r;
#define CV3_KV_LOAD(KOFF)                                                                        \
  {                                                                                              \
    const int64_t kb0 = (KOFF) + ltile * KT + lkey;                                              \
    const int64_t j0 = min(kb0, p.m - 1), j1 = min(kb0 + 16, p.m - 1);                           \
    const int64_t j2 = min(kb0 + 32, p.m - 1), j3 = min(kb0 + 48, p.m - 1);                      \
    k0r = *reinterpret_cast<const float4*>(kbase + j0 * p.k_sm + ld4);                           \
    k1r = *reinterpret_cast<const float4*>(kbase + j1 * p.k_sm + ld4);                           \
    k2r = *reinterpret_cast<const float4*>(kbase + j2 * p.k_sm + ld4);                           \
    k3r = *reinterpret_cast<const float4*>(kbase + j3 * p.k_sm + ld4);                           \
    const float* vr_ = vbase + min((KOFF) + ltile * KT + vkey, p.m - 1) * p.v_sm + vd;            \
    v0r = *reinterpret_cast<const float4*>(vr_);                                                 \
    v1r = *reinterpret_cast<const float4*>(vr_ + 4);                                             \
    v2r = *reinterpret_cast<const float4*>(vr_ + 8);                                             \
    v3r = *reinterpret_cast<const float4*>(vr_ + 12);                                            \
  }
  CV3_KV_LOAD((int64_t)0)
  for (int64_t st = 0; st < nstages; ++st) {
    const int k0i = (int)(st * NKG * KT + kg * KT);  // first key of this wave's tile
    __syncthreads();
    float* kt_ = Ks[ltile];
    float* vt_ = Vs[ltile];
    *reinterpret_cast<float4*>(&kt_[lkey * KS + ld4]) = k0r;
    *reinterpret_cast<float4*>(&kt_[(lkey + 16) * KS + ld4]) = k1r;
    *reinterpret_cast<float4*>(&kt_[(lkey + 32) * KS + ld4]) = k2r;
    *reinterpret_cast<float4*>(&kt_[(lkey + 48) * KS + ld4]) = k3r;
    {
      const float vv[16] = {v0r.x, v0r.y, v0r.z, v0r.w, v1r.x, v1r.y, v1r.z, v1r.w,
                            v2r.x, v2r.y, v2r.z, v2r.w, v3r.x, v3r.y, v3r.z, v3r.w};
#pragma unroll
      for (int e = 0; e < 16; ++e) vt_[(vd + e) * KS + vkey] = vv[e];
    }
    __syncthreads();
    if (st + 1 < nstages) CV3_KV_LOAD((st + 1) * NKG * KT)
    __builtin_amdgcn_sched_barrier(0);  // the prefetch is issued before this stage's math
    const float* Kt = Ks[kg];
    const float* Vt = Vs[kg];

    // S^T for the tile: sub-tile sub holds keys sub*16 + 4g + i (i < 4) for query column c16
    // the four sub-tiles' accumulators are independent: consecutive MFMAs go to different ones
    f32x4 s[KT / 16];
#pragma unroll
    for (int sub = 0; sub < KT / 16; ++sub) s[sub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      float4 kf[KT / 16];
#pragma unroll
      for (int sub = 0; sub < KT / 16; ++sub)
        kf[sub] = *reinterpret_cast<const float4*>(&Kt[(sub * 16 + c16) * KS + g * 4 + s4 * 16]);
#pragma unroll
      for (int sub = 0; sub < KT / 16; ++sub) s[sub] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[sub].x, qf[s4].x, s[sub], 0, 0, 0);
#pragma unroll
      for (int sub = 0; sub < KT / 16; ++sub) s[sub] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[sub].y, qf[s4].y, s[sub], 0, 0, 0);
#pragma unroll
      for (int sub = 0; sub < KT / 16; ++sub) s[sub] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[sub].z, qf[s4].z, s[sub], 0, 0, 0);
#pragma unroll
      for (int sub = 0; sub < KT / 16; ++sub) s[sub] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[sub].w, qf[s4].w, s[sub], 0, 0, 0);
    }
    // copy out of the accumulators and mask with selects (no divergent writes into them)
    float sc[KT / 16][4];
    float mx = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < KT / 16; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kj = k0i + sub * 16 + 4 * g + i;
        const bool ok = kj >= klo && kj < khi;
        sc[sub][i] = ok ? s[sub][i] : -INFINITY;
        mx = fmaxf(mx, sc[sub][i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    // Branch-free so the wave-wide MFMAs below see uniform control flow: a query
    // column with nothing visible yet keeps alpha = 1 and p = 0.
    const float m_new = fmaxf(m_run, mx);
    const bool none = m_new == -INFINITY;
    const float m_use = none ? 0.f : m_new;
    const float alpha = none ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
    float psum = 0.f;
#pragma unroll
    for (int sub = 0; sub < KT / 16; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[sub][i] = __builtin_amdgcn_exp2f(sc[sub][i] - m_use);
        psum += sc[sub][i];
      }
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < 4; ++db) oacc[db] *= alpha;
    // O^T += V^T P^T: the A operand of key group i is V^T[db*16 + c16][sub*16 + 4g + i]
#pragma unroll
    for (int sub = 0; sub < KT / 16; ++sub) {
      float4 vf[4];
#pragma unroll
      for (int db = 0; db < 4; ++db)
        vf[db] = *reinterpret_cast<const float4*>(&Vt[(db * 16 + c16) * KS + sub * 16 + 4 * g]);
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db].x, sc[sub][0], oacc[db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db].y, sc[sub][1], oacc[db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db].z, sc[sub][2], oacc[db], 0, 0, 0);
#pragma unroll
      for (int db = 0; db < 4; ++db) oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[db].w, sc[sub][3], oacc[db], 0, 0, 0);
    }
  }
#undef CV3_KV_LOAD
  // merge the key groups through LDS (each lane's state is per query column)
  __syncthreads();
  float* mb = &Ks[0][0];  // (NKG - 1) x 4 waves x 64 lanes x 18 floats <= NKG * 64 * 68
  static_assert((NKG - 1) * 4 * 64 * 18 <= NKG * KT * KS, "merge slots fit the K tiles");
  if (kg > 0) {
    float* slot = mb + (((kg - 1) * 4 + qw) * 64 + lane) * 18;
    slot[0] = m_run;
    slot[1] = l_run;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) slot[2 + db * 4 + i] = oacc[db][i];
  }
  __syncthreads();
  if (kg > 0) return;
  float M = m_run;
#pragma unroll
  for (int g2 = 1; g2 < NKG; ++g2) M = fmaxf(M, mb[(((g2 - 1) * 4 + qw) * 64 + lane) * 18]);
  const float a0 = M == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - M);
  l_run = l_run * a0;
#pragma unroll
  for (int db = 0; db < 4; ++db) oacc[db] *= a0;
#pragma unroll
  for (int g2 = 1; g2 < NKG; ++g2) {
    const float* slot = mb + (((g2 - 1) * 4 + qw) * 64 + lane) * 18;
    const float ag = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(slot[0] - M);
    l_run += slot[1] * ag;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[db][i] += slot[2 + db * 4 + i] * ag;
  }
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  if (!qvalid) return;
  float* orow = p.o + b * p.o_sb + hq * p.o_sh + qi * p.o_sn;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) orow[db * 16 + 4 * g + i] = oacc[db][i] / l_tot;
}

// One query of any head dim <= 256 by one wave, 64 keys per step; qs: the scaled query in LDS.
__device__ __forceinline__ void attend_row(const AttnParams& p, int b, int hq, int hkv, int64_t qi, int lane, const float* qs) {
  const float* kbase = p.k + b * p.k_sb + hkv * p.k_sh;
  const float* vbase = p.v + b * p.v_sb + hkv * p.v_sh;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;
  int64_t klo, khi;
  visible_keys(p, qi, klo, khi);
  for (int64_t c0 = 0; c0 < p.m; c0 += 64) {
    const int64_t kj = c0 + lane;
    float s = -INFINITY;
    if (kj >= klo && kj < khi) {
      const float* kr = kbase + kj * p.k_sm;
      float t = 0.f;
      for (int d = 0; d < p.d; ++d) t = fmaf(qs[d], kr[d], t);
      s = t;
    }
    const float mx = wave_max(s);
    const float m_new = fmaxf(m_run, mx);
    if (m_new == -INFINITY) continue;
    const float alpha = expf(m_run - m_new);
    const float pj = expf(s - m_new);
    l_run = l_run * alpha + wave_sum(pj);
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] *= alpha;
    const int64_t cnt = p.m - c0 < 64 ? p.m - c0 : 64;
    for (int jj = 0; jj < cnt; ++jj) {
      const float pb = __shfl(pj, jj, 64);
      const float* vr = vbase + (c0 + jj) * p.v_sm;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = lane + 64 * r;
        if (d < p.d) acc[r] = fmaf(pb, vr[d], acc[r]);
      }
    }
    m_run = m_new;
  }
  float* orow = p.o + b * p.o_sb + hq * p.o_sh + qi * p.o_sn;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int d = lane + 64 * r;
    if (d < p.d) orow[d] = acc[r] / l_run;
  }
}

// k_flash64x's second pass: one query from the floats, 64 dims in 16-byte aligned rows, by one wave, with sums in
// 64 bits (a lone wave's serial sums in 32 were off by 1.4e-6, the tiles' are by 4e-7).  qs: the scaled query in
// LDS.  Every value counts, those of masked keys with probability zero.  Scores: a lane per key; values: 16 lanes
// across a row, four keys at a time.  16 heads, 1500 rows, every query: 14.2 ms a key at a time, 2.4 so.
__device__ __forceinline__ double wave_max_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
  return v;
}

__device__ __forceinline__ void attend_again(const AttnParams& p, int b, int hq, int hkv, int64_t qi, int lane,
                                             const float4* qs) {
  const float* kbase = p.k + b * p.k_sb + hkv * p.k_sh;
  const float* vbase = p.v + b * p.v_sb + hkv * p.v_sh;
  const int dq = lane & 15, sub = lane >> 4;
  double acc[4] = {0., 0., 0., 0.}, m_run = -INFINITY, l_run = 0.;
  int64_t klo, khi;
  visible_keys(p, qi, klo, khi);
  for (int64_t c0 = 0; c0 < p.m; c0 += 64) {
    const int64_t kj = c0 + lane;
    double s = -INFINITY;
    if (kj >= klo && kj < khi) {
      const float4* kr = reinterpret_cast<const float4*>(kbase + kj * p.k_sm);
      s = 0.;
#pragma unroll 4
      for (int d = 0; d < 16; ++d) {
        const float4 k4 = kr[d], q4 = qs[d];
        s = fma((double)q4.x, (double)k4.x, s);
        s = fma((double)q4.y, (double)k4.y, s);
        s = fma((double)q4.z, (double)k4.z, s);
        s = fma((double)q4.w, (double)k4.w, s);
      }
    }
    const double m_new = fmax(m_run, wave_max_d(s));
    const bool none = m_new == -INFINITY;
    const float alpha = none ? 1.f : expf((float)(m_run - m_new));
    const float pj = none ? 0.f : expf((float)(s - m_new));
    l_run = l_run * alpha + wave_sum_d((double)pj);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= alpha;
#pragma unroll 8
    for (int j = 0; j < 16; ++j) {
      const int key = 4 * j + sub;
      const float pb = __shfl(pj, key, kWave);
      float4 v = *reinterpret_cast<const float4*>(vbase + min(c0 + key, p.m - 1) * p.v_sm + 4 * dq);
      if (c0 + key >= p.m) v = make_float4(0.f, 0.f, 0.f, 0.f);
      acc[0] = fma((double)pb, (double)v.x, acc[0]);
      acc[1] = fma((double)pb, (double)v.y, acc[1]);
      acc[2] = fma((double)pb, (double)v.z, acc[2]);
      acc[3] = fma((double)pb, (double)v.w, acc[3]);
    }
    m_run = m_new;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    acc[e] += __shfl_xor(acc[e], 16, kWave);
    acc[e] += __shfl_xor(acc[e], 32, kWave);
  }
  const double own = sub == 0 ? acc[0] : sub == 1 ? acc[1] : sub == 2 ? acc[2] : acc[3];
  p.o[b * p.o_sb + hq * p.o_sh + qi * p.o_sn + 4 * dq + sub] = (float)(own / l_run);
}

// The same flash attention on the bfloat16 matrix cores (v_mfma_f32_16x16x32_bf16): q, k, v
// and the probabilities split into three bfloat16 planes each (bf16x3.hpp), every product
// as the six plane products of weight >= 2^-16, hh into one accumulator and the other five
// into a second, added where the float32 kernel reads its accumulator.  Eight waves of 16
// queries each, QWN of them side by side and 8 / QWN key groups; a stage stages 128 keys and a
// key group takes 16 NS of them (NS = QWN sub-tiles of 16).
//   QWN = 4: 64 queries a workgroup, two key groups of 64 keys.
//   QWN = 2: 32 queries, four key groups of 32 keys: twice the workgroups with half the products
//   and LDS reads each, for launches that leave half of the chip idle.
//
// LDS holds each 64-key tile's planes as 64 rows of 128 bytes (8 chunks of 8 bf16, chunk c of
// row r in slot r * 8 + (c ^ (r / 2) % 8)): K as [key][dim], key NS c + s of a group's keys in row
// 16 s + c of its rows, V^T as [dim][key].  Score sub-tile s (MFMA rows r = LDS rows 16 s + r) then
// holds keys NS r + s, so lane (c16, g) ends with keys 4 NS g + NS i + s (i < 4, s < NS): 4 NS
// consecutive keys of its query column.  P V step j takes keys 4 NS g + 8 j + t (t < 8) from lane
// group g, which are the lane's own values (i, s) = divmod(8 j + t, NS) as the B operand (k index
// 8 g + t), and V^T row d, chunk NS g / 2 + j of the group's as the A operand: no data moves
// between the two products.
__device__ __forceinline__ int xkv(int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); }
// V^T rows (64 dims of 8 16-byte key chunks) of k_flash64x: chunk c of row d at slot
// (d / 2) 16 + ((8 (d % 2) + c) ^ f(d)), f(d) = 8 b5 + ((d / 2) % 8 ^ b4) with b4, b5 bits 4 and 5 of d.
// A row pair fills 16 slots (256 bytes, one bank window).  The P.V reads (16 consecutive rows, one
// chunk) and the staging writes (rows 4 q + e for q = 0..15, one chunk, 8 bytes each) both land on
// 16 distinct slots of a window.
__device__ __forceinline__ int vslot(int d, int c) {
  const int f = (((d >> 5) & 1) << 3) | (((d >> 1) & 7) ^ ((d >> 4) & 1));
  return (d >> 1) * 16 + (((d & 1) * 8 + c) ^ f);
}

__device__ __forceinline__ void mfma6(const bf16x8_t& ah, const bf16x8_t& am, const bf16x8_t& al,
                                      const bf16x8_t& bh, const bf16x8_t& bm, const bf16x8_t& bl, f32x4& big,
                                      f32x4& small) {
  big = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, big, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm, small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh, small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, small, 0, 0, 0);
}

// A stage that no query of the workgroup sees is skipped, but for its values' exponents: a masked key counts with
// probability zero, and zero times an infinity or NaN is NaN in that dim of every output, whichever tile it is in.
// AGAIN: outputs that come out not finite, or smaller than planes of the values hold in full, are formed again from
// the floats (attend_again).
template <int QWN, bool AGAIN>
__global__ __launch_bounds__(512) void k_flash64x(AttnParams p, int nq) {
  constexpr int NKG = 8 / QWN, NS = QWN, WKT = 16 * NS;  // key groups; a group's sub-tiles and keys
  constexpr int TILES = 2, STAGE = TILES * KT;
  static_assert(NKG * WKT == STAGE, "the key groups share a stage");
  __shared__ uint4 Ks[TILES][3][KT * 8];
  __shared__ uint4 Vs[TILES][3][KT * 8];
  __shared__ uint32_t skipped[2];  // dims with an infinity or NaN among the values of the skipped stages
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid < 2) skipped[tid] = 0;
  const int qw = wave % QWN, kg = wave / QWN;
  const int wt = kg * WKT / KT, wr = kg * WKT % KT;  // the group's tile and its first key there
  const int ntiles = (int)gridDim.x;
  const int wg = (int)blockIdx.x;
  const int tile = (ntiles & 7) == 0 ? (wg & 7) * (ntiles >> 3) + (wg >> 3) : wg;
  const int qt = tile % nq, bh = tile / nq;
  const int b = bh / p.h, hq = bh % p.h;
  const int hkv = hq / (p.h / p.hk);
  const int64_t q0 = (int64_t)qt * (QWN * QW) + qw * QW;
  const int c16 = lane & 15, g = lane >> 4;
  const int64_t qi = q0 + c16;
  const bool qvalid = qi < p.n;
  int64_t klo64, khi64;
  visible_keys(p, qi, klo64, khi64);
  const int klo = (int)klo64, khi = (int)khi64;  // the host bounds m below 2^31 - 64

  // Q^T fragments: query c16, dims 32 ks + 8 g .. + 7, pre-scaled like the reference's
  // (q * scale) (ops.py:292), in base-2 units, as planes
  bf16x8_t qh[2], qm[2], ql[2];
  const float* qrow = p.q + b * p.q_sb + hq * p.q_sh + (qvalid ? qi : 0) * p.q_sn;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    float4 t0 = qvalid ? *reinterpret_cast<const float4*>(qrow + 32 * ks + 8 * g) : make_float4(0, 0, 0, 0);
    float4 t1 = qvalid ? *reinterpret_cast<const float4*>(qrow + 32 * ks + 8 * g + 4) : make_float4(0, 0, 0, 0);
    t0 = make_float4((t0.x * p.scale) * kLog2E, (t0.y * p.scale) * kLog2E, (t0.z * p.scale) * kLog2E,
                     (t0.w * p.scale) * kLog2E);
    t1 = make_float4((t1.x * p.scale) * kLog2E, (t1.y * p.scale) * kLog2E, (t1.z * p.scale) * kLog2E,
                     (t1.w * p.scale) * kLog2E);
    uint4 h4, m4, l4;
    split_x3(t0, t1, h4, m4, l4);
    qh[ks] = __builtin_bit_cast(bf16x8_t, h4);
    qm[ks] = __builtin_bit_cast(bf16x8_t, m4);
    ql[ks] = __builtin_bit_cast(bf16x8_t, l4);
  }

  f32x4 ob[4], os[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) ob[db] = os[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  const float* kbase = p.k + b * p.k_sb + hkv * p.k_sh;
  const float* vbase = p.v + b * p.v_sb + hkv * p.v_sh;
  // the stages that hold a key which some query of the workgroup sees (both bounds grow with the query)
  int64_t first, last, unused;
  visible_keys(p, (int64_t)qt * (QWN * QW), first, unused);
  visible_keys(p, min((int64_t)(qt + 1) * (QWN * QW), p.n) - 1, unused, last);
  const int64_t st0 = first / STAGE, nstages = max(ceil_div(max(last, (int64_t)0), STAGE), st0);
  // Staging (next stage's rows in registers while this one is computed; rows past m clamp
  // to m - 1 and are masked to -inf below):
  // K: thread -> tile tid/256, key (tid%256)/4, dims 16 (tid%4) .. + 15 (two chunks);
  // V: thread -> tile tid/256, keys 4 kq .. + 3 (kq = (tid%256)/16), dims 4 dq .. + 3 (dq = tid%16):
  //    each dim's four keys are one 8-byte half-chunk of a V^T row.
  const int ltile = tid >> 8, lkey = (tid & 255) >> 2, ld16 = (tid & 3) * 16;
  const int lrow = lkey / WKT * WKT + lkey % NS * 16 + lkey % WKT / NS;
  const int dq = tid & 15, kq = (tid & 255) >> 4;
  float4 kr[4], vv[4];
#define CV3_KVX_LOAD(KOFF)                                                                 \
  {                                                                                        \
    const int64_t jk = min((KOFF) + ltile * KT + lkey, p.m - 1);                           \
    const float* kr_ = kbase + jk * p.k_sm + ld16;                                         \
    kr[0] = *reinterpret_cast<const float4*>(kr_);                                         \
    kr[1] = *reinterpret_cast<const float4*>(kr_ + 4);                                     \
    kr[2] = *reinterpret_cast<const float4*>(kr_ + 8);                                     \
    kr[3] = *reinterpret_cast<const float4*>(kr_ + 12);                                    \
    _Pragma("unroll") for (int r_ = 0; r_ < 4; ++r_) {                                     \
      const int64_t jv = min((KOFF) + ltile * KT + 4 * kq + r_, p.m - 1);                  \
      vv[r_] = *reinterpret_cast<const float4*>(vbase + jv * p.v_sm + 4 * dq);             \
    }                                                                                      \
  }
  CV3_KVX_LOAD(st0 * STAGE)
  for (int64_t st = st0; st < nstages; ++st) {
    const int k0i = (int)(st * STAGE + kg * WKT);  // first key of this wave's group
    __syncthreads();
    {
      uint4 h4, m4, l4;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        split_x3(kr[2 * half], kr[2 * half + 1], h4, m4, l4);
        const int slot = xkv(lrow, (ld16 >> 3) + half);
        Ks[ltile][0][slot] = h4;
        Ks[ltile][1][slot] = m4;
        Ks[ltile][2][slot] = l4;
      }
      const float vr[4][4] = {{vv[0].x, vv[0].y, vv[0].z, vv[0].w}, {vv[1].x, vv[1].y, vv[1].z, vv[1].w},
                              {vv[2].x, vv[2].y, vv[2].z, vv[2].w}, {vv[3].x, vv[3].y, vv[3].z, vv[3].w}};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint2 hh, mm, ll;
        split_x3(vr[0][e], vr[1][e], hh.x, mm.x, ll.x);  // keys 4 kq, 4 kq + 1
        split_x3(vr[2][e], vr[3][e], hh.y, mm.y, ll.y);  // keys 4 kq + 2, 4 kq + 3
        const int sl = vslot(4 * dq + e, kq >> 1);
        reinterpret_cast<uint2*>(&Vs[ltile][0][sl])[kq & 1] = hh;
        reinterpret_cast<uint2*>(&Vs[ltile][1][sl])[kq & 1] = mm;
        reinterpret_cast<uint2*>(&Vs[ltile][2][sl])[kq & 1] = ll;
      }
    }
    __syncthreads();
    if (st + 1 < nstages) CV3_KVX_LOAD((st + 1) * STAGE)
    __builtin_amdgcn_sched_barrier(0);  // the prefetch is issued before this stage's math

    // S^T sub-tiles: sub-tile s holds keys NS r + s in MFMA row r; k = dims
    f32x4 sb[NS], ss[NS];
#pragma unroll
    for (int sub = 0; sub < NS; ++sub) sb[sub] = ss[sub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int sub = 0; sub < NS; ++sub) {
        const int slot = xkv(wr + sub * 16 + c16, 4 * ks + g);
        const bf16x8_t kh = __builtin_bit_cast(bf16x8_t, Ks[wt][0][slot]);
        const bf16x8_t km = __builtin_bit_cast(bf16x8_t, Ks[wt][1][slot]);
        const bf16x8_t kl = __builtin_bit_cast(bf16x8_t, Ks[wt][2][slot]);
        mfma6(kh, km, kl, qh[ks], qm[ks], ql[ks], sb[sub], ss[sub]);
      }
    }
    // lane (c16, g): sc[s][i] = score of key k0i + 4 NS g + NS i + s for query c16; a group that
    // every query of the wave sees whole skips the per-key selects
    float sc[NS][4];
    float mx = -INFINITY;
    if (__all(k0i >= klo && k0i + WKT <= khi)) {
#pragma unroll
      for (int sub = 0; sub < NS; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sc[sub][i] = sb[sub][i] + ss[sub][i];
          mx = fmaxf(mx, sc[sub][i]);
        }
    } else {
#pragma unroll
      for (int sub = 0; sub < NS; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kj = k0i + NS * (4 * g + i) + sub;
          const bool ok = kj >= klo && kj < khi;
          sc[sub][i] = ok ? sb[sub][i] + ss[sub][i] : -INFINITY;
          mx = fmaxf(mx, sc[sub][i]);
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const bool none = m_new == -INFINITY;
    const float m_use = none ? 0.f : m_new;
    const float alpha = none ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
    float psum = 0.f;
#pragma unroll
    for (int sub = 0; sub < NS; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[sub][i] = __builtin_amdgcn_exp2f(sc[sub][i] - m_use);
        psum += sc[sub][i];
      }
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      ob[db] *= alpha;
      os[db] *= alpha;
    }
    // O^T += V^T P^T over keys 4 NS g + 8 j + t: P^T's B operand is the lane's own values
#pragma unroll
    for (int j = 0; j < NS / 2; ++j) {
      float pv[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) pv[t] = sc[(8 * j + t) % NS][(8 * j + t) / NS];
      const float4 p0 = make_float4(pv[0], pv[1], pv[2], pv[3]), p1 = make_float4(pv[4], pv[5], pv[6], pv[7]);
      uint4 h4, m4, l4;
      split_x3(p0, p1, h4, m4, l4);
      const bf16x8_t ph = __builtin_bit_cast(bf16x8_t, h4);
      const bf16x8_t pm = __builtin_bit_cast(bf16x8_t, m4);
      const bf16x8_t pl = __builtin_bit_cast(bf16x8_t, l4);
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const int slot = vslot(db * 16 + c16, wr / 8 + NS / 2 * g + j);
        const bf16x8_t vh = __builtin_bit_cast(bf16x8_t, Vs[wt][0][slot]);
        const bf16x8_t vm = __builtin_bit_cast(bf16x8_t, Vs[wt][1][slot]);
        const bf16x8_t vl = __builtin_bit_cast(bf16x8_t, Vs[wt][2][slot]);
        mfma6(vh, vm, vl, ph, pm, pl, ob[db], os[db]);
      }
    }
  }
#undef CV3_KVX_LOAD
  f32x4 oacc[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) oacc[db] = ob[db] + os[db];
  // merge the key groups through LDS, as k_flash64
  __syncthreads();
  if (p.mask_kind != 0) {
    // thread -> dims 4 dq .. + 3 of every 32nd row; rows past the end clamp to the last one
    const int rows0 = (int)(st0 * STAGE), at1 = (int)(nstages * STAGE), rows1 = max((int)p.m - at1, 0);
    float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    auto scan = [&](int from, int rows) {
      for (int r = tid >> 4; r < rows; r += 4 * 32) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 v = *reinterpret_cast<const float4*>(vbase + (int64_t)(from + min(r + 32 * u, rows - 1)) * p.v_sm + 4 * dq);
          z = make_float4(fmaf(v.x, 0.f, z.x), fmaf(v.y, 0.f, z.y), fmaf(v.z, 0.f, z.z), fmaf(v.w, 0.f, z.w));
        }
      }
    };
    scan(0, min(rows0, (int)p.m));
    scan(at1, rows1);
    const uint32_t bits = (z.x != z.x) | (z.y != z.y) << 1 | (z.z != z.z) << 2 | (z.w != z.w) << 3;
    if (bits) atomicOr(&skipped[dq >> 3], bits << (4 * (dq & 7)));
  }
  float* mb = reinterpret_cast<float*>(&Ks[0][0][0]);
  static_assert((NKG - 1) * QWN * 64 * 18 * 4 <= (int)sizeof(Ks), "merge slots fit the K tiles");
  if (kg > 0) {
    float* slot = mb + (((kg - 1) * QWN + qw) * 64 + lane) * 18;
    slot[0] = m_run;
    slot[1] = l_run;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) slot[2 + db * 4 + i] = oacc[db][i];
  }
  __syncthreads();
  if (kg > 0) return;
  float M = m_run;
#pragma unroll
  for (int g2 = 1; g2 < NKG; ++g2) M = fmaxf(M, mb[(((g2 - 1) * QWN + qw) * 64 + lane) * 18]);
  const float a0 = M == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - M);
  l_run = l_run * a0;
#pragma unroll
  for (int db = 0; db < 4; ++db) oacc[db] *= a0;
#pragma unroll
  for (int g2 = 1; g2 < NKG; ++g2) {
    const float* slot = mb + (((g2 - 1) * QWN + qw) * 64 + lane) * 18;
    const float ag = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(slot[0] - M);
    l_run += slot[1] * ag;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) oacc[db][i] += slot[2 + db * 4 + i] * ag;
  }
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  if (p.mask_kind != 0 && (skipped[0] | skipped[1])) {
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (skipped[db >> 1] >> (16 * (db & 1) + 4 * g + i) & 1) oacc[db][i] = __builtin_nanf("");
  }
  if (p.op && qvalid) {
    // row b n + qi of [batch n, 64 h] rows as the fragments a plane linear reads: four neighbouring
    // columns are half of a lane's 16 bytes
    const int64_t row = b * p.n + qi;
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      const int64_t col = hq * 64 + db * 16 + 4 * g;
      const int64_t at = (((row >> 5) * (4 * p.h) + (col >> 4)) * 64 + (row & 31) + 32 * ((col >> 3) & 1)) * 2 +
                         ((col >> 2) & 1);
      uint2 hi, mid, lo;
      split_x3(oacc[db][0] / l_tot, oacc[db][1] / l_tot, hi.x, mid.x, lo.x);
      split_x3(oacc[db][2] / l_tot, oacc[db][3] / l_tot, hi.y, mid.y, lo.y);
      p.op[at] = hi;
      p.op[at + p.opl] = mid;
      p.op[at + 2 * p.opl] = lo;
    }
  }
  if (p.op) return;
  [[maybe_unused]] float y[4][4];
  [[maybe_unused]] uint32_t most = 0, least = 0xffffffffu;   // least: of the magnitudes but zero, less one
  if (qvalid) {
    float* orow = p.o + b * p.o_sb + hq * p.o_sh + qi * p.o_sn;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        y[db][i] = oacc[db][i] / l_tot;
        orow[db * 16 + 4 * g + i] = y[db][i];
        most = max(most, magnitude(y[db][i]));
        least = min(least, magnitude(y[db][i]) - 1u);
      }
  }
  if constexpr (AGAIN) {
    // infinities and the largest floats have no planes here (inf - inf), values below 2^-110 not all their bits: the
    // whole wave does those queries again, but for dims with a NaN among the values and queries with one or with no
    // key to see, which are NaN as they stand
    uint32_t bad = 0;   // bit 4 db + i
    if (__any(!in_range(most) || !in_range(least + 1u))) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) bad |= (uint32_t)(qvalid && !in_range(magnitude(y[db][i]))) << (4 * db + i);
      const int sub = lane >> 4;
      uint32_t nan = 0;
      for (int r = sub; r < (int)p.m; r += 4) {
        const float4 v = *reinterpret_cast<const float4*>(vbase + (int64_t)r * p.v_sm + 4 * c16);
        nan |= (v.x != v.x) | (v.y != v.y) << 1 | (v.z != v.z) << 2 | (v.w != v.w) << 3;
      }
      nan |= __shfl_xor(nan, 16, 64);
      nan |= __shfl_xor(nan, 32, 64);
#pragma unroll
      for (int db = 0; db < 4; ++db) bad &= ~(__shfl(nan, 4 * db + g, 64) << (4 * db));
    }
    uint64_t todo = __ballot(bad != 0);
    todo = (todo | todo >> 16 | todo >> 32 | todo >> 48) & 0xffff;
    float* qs = reinterpret_cast<float*>(&Vs[0][0][0]) + 64 * qw;
    while (todo) {
      const int64_t row = q0 + __builtin_ctzll(todo);
      todo &= todo - 1;
      const float x = p.q[b * p.q_sb + hq * p.q_sh + row * p.q_sn + lane] * p.scale;
      int64_t lo, hi;
      visible_keys(p, row, lo, hi);
      if (hi <= lo || __any(x != x)) continue;
      qs[lane] = x;
      __builtin_amdgcn_wave_barrier();
      attend_again(p, b, hq, hkv, row, lane, reinterpret_cast<const float4*>(qs));
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// Generic path for any head dim <= 256: one wave per query row, 64 keys per step.
__global__ __launch_bounds__(256) void k_attn_generic(AttnParams p) {
  extern __shared__ float qs_all[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = blockIdx.z, hq = blockIdx.y;
  const int hkv = hq / (p.h / p.hk);
  const int64_t qi = (int64_t)blockIdx.x * 4 + wave;
  float* qs = qs_all + wave * p.d;
  const bool qvalid = qi < p.n;
  const float* qrow = p.q + b * p.q_sb + hq * p.q_sh + (qvalid ? qi : 0) * p.q_sn;
  for (int d = lane; d < p.d; d += 64) qs[d] = qvalid ? qrow[d] * p.scale : 0.f;
  __syncthreads();
  if (!qvalid) return;
  attend_row(p, b, hq, hkv, qi, lane, qs);
}

}  // namespace

static int attention(bool x3, const float* q, const float* k, const float* v, float* out, int64_t batch, int h,
                     int hk, int64_t n, int64_t m, int d, const int64_t* q_strides, const int64_t* k_strides,
                     const int64_t* v_strides, const int64_t* o_strides, float scale, int mask_kind, int64_t mask_a,
                     int64_t mask_b, cv3_stream_t s, uint16_t* out_planes = nullptr, int64_t plan_batch = 2, bool again = false) {
  CV3_REQUIRE(h > 0 && hk > 0, CV3_EINVAL, "head counts must be positive");
  CV3_REQUIRE(h % hk == 0, CV3_EINVAL, "%d query heads is not a multiple of %d kv heads", h, hk);
  CV3_REQUIRE(d > 0 && d <= 256, CV3_EUNSUPPORTED, "head dim %d not supported (max 256)", d);
  CV3_REQUIRE(mask_kind >= 0 && mask_kind <= 2, CV3_EINVAL, "unknown mask spec kind %d", mask_kind);
  CV3_REQUIRE(mask_kind != 2 || mask_a > 0, CV3_EINVAL, "chunk mask needs a positive chunk size");
  if (batch <= 0 || n <= 0) return CV3_OK;
  CV3_REQUIRE(m > 0, CV3_EINVAL, "attention over zero keys");
  AttnParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.o = out;
  p.q_sb = q_strides[0]; p.q_sh = q_strides[1]; p.q_sn = q_strides[2];
  p.k_sb = k_strides[0]; p.k_sh = k_strides[1]; p.k_sm = k_strides[2];
  p.v_sb = v_strides[0]; p.v_sh = v_strides[1]; p.v_sm = v_strides[2];
  if (o_strides) p.o_sb = o_strides[0], p.o_sh = o_strides[1], p.o_sn = o_strides[2];
  p.op = reinterpret_cast<uint2*>(out_planes);
  p.opl = ceil_div(batch * n, 32) * (4 * h) * 128;
  p.h = h;
  p.hk = hk;
  p.n = n;
  p.m = m;
  p.d = d;
  p.scale = scale;
  p.mask_kind = mask_kind;
  p.mask_a = mask_a;
  p.mask_b = mask_b;
  hipStream_t st = stream_of(s);
  const bool aligned16 = ((uintptr_t)q % 16 == 0) && ((uintptr_t)k % 16 == 0) && ((uintptr_t)v % 16 == 0) &&
                         (p.q_sb % 4 == 0) && (p.q_sh % 4 == 0) && (p.q_sn % 4 == 0) && (p.k_sb % 4 == 0) &&
                         (p.k_sh % 4 == 0) && (p.k_sm % 4 == 0) && (p.v_sb % 4 == 0) && (p.v_sh % 4 == 0) &&
                         (p.v_sm % 4 == 0);
  CV3_REQUIRE(!out_planes || (d == 64 && aligned16 && (uintptr_t)out_planes % 16 == 0), CV3_EUNSUPPORTED,
              "attention into planes needs head dim 64 and 16-byte aligned rows");
  if (d == 64 && aligned16) {
    CV3_REQUIRE(m < (1ll << 31) - 4 * 64, CV3_EUNSUPPORTED, "attention over 2^31 keys or more");
    const int64_t nq = ceil_div(n, QT);
    CV3_REQUIRE(nq * h * batch < (int64_t)1 << 31, CV3_EUNSUPPORTED, "attention grid too large");
    const dim3 grid((unsigned)(nq * h * batch));
    // 32-query workgroups where they fit the chip at once (one to a CU: 96 KB of LDS), counted for plan_batch
    // rows so that both halves of a guidance batch run what the whole batch runs.  64- against 32-query:
    // [2, 16, 151, 64] 11.9 / 10.1 us, causal [14 on 2, 333, 64] 14.9 / 12.2 us; past one round they cost more.
    const int64_t nq2 = ceil_div(n, QT / 2);
    const bool small = nq2 * h * std::max(batch, plan_batch) <= kNumCU;
    const dim3 grid2((unsigned)(nq2 * h * batch));
    if (x3 && small && again)
      hipLaunchKernelGGL((k_flash64x<2, true>), grid2, dim3(512), 0, st, p, (int)nq2);
    else if (x3 && small)
      hipLaunchKernelGGL((k_flash64x<2, false>), grid2, dim3(512), 0, st, p, (int)nq2);
    else if (x3 && again)
      hipLaunchKernelGGL((k_flash64x<4, true>), grid, dim3(512), 0, st, p, (int)nq);
    else if (x3)
      hipLaunchKernelGGL((k_flash64x<4, false>), grid, dim3(512), 0, st, p, (int)nq);
    else if (m >= 16 * KT)  // 1024 keys and up: 8 % faster at 1500 keys, no gain at 500
      hipLaunchKernelGGL(k_flash64<4>, grid, dim3(1024), 0, st, p, (int)nq);
    else
      hipLaunchKernelGGL(k_flash64<2>, grid, dim3(512), 0, st, p, (int)nq);
  } else {
    const dim3 grid((unsigned)ceil_div(n, 4), (unsigned)h, (unsigned)batch);
    hipLaunchKernelGGL(k_attn_generic, grid, dim3(256), 4 * d * sizeof(float), st, p);
  }
  CV3_LAUNCHED();
  return CV3_OK;
}

extern "C" int cv3_attention(const float* q, const float* k, const float* v, float* out, int64_t batch, int h,
                             int hk, int64_t n, int64_t m, int d, const int64_t* q_strides,
                             const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                             float scale, int mask_kind, int64_t mask_a, int64_t mask_b, cv3_stream_t s) {
  CV3_ALIVE();
  return attention(false, q, k, v, out, batch, h, hk, n, m, d, q_strides, k_strides, v_strides, o_strides, scale,
                   mask_kind, mask_a, mask_b, s);
}

extern "C" int cv3_attention_x3(const float* q, const float* k, const float* v, float* out, int64_t batch, int h,
                                int hk, int64_t n, int64_t m, int d, const int64_t* q_strides,
                                const int64_t* k_strides, const int64_t* v_strides, const int64_t* o_strides,
                                float scale, int mask_kind, int64_t mask_a, int64_t mask_b, cv3_stream_t s) {
  CV3_ALIVE();
  return attention(true, q, k, v, out, batch, h, hk, n, m, d, q_strides, k_strides, v_strides, o_strides, scale,
                   mask_kind, mask_a, mask_b, s);
}

extern "C" int cv3_attention_x3_planes(const float* q, const float* k, const float* v, uint16_t* out_planes,
                                       int64_t batch, int h, int hk, int64_t n, int64_t m, int d,
                                       const int64_t* q_strides, const int64_t* k_strides, const int64_t* v_strides,
                                       float scale, int mask_kind, int64_t mask_a, int64_t mask_b, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(out_planes, CV3_EINVAL, "attention into planes needs its output");
  return attention(true, q, k, v, nullptr, batch, h, hk, n, m, d, q_strides, k_strides, v_strides, nullptr, scale,
                   mask_kind, mask_a, mask_b, s, out_planes);
}

extern "C" int cv3_sdpa(const float* q, const float* k, const float* v, float* out, int h, int hk, int64_t n, int64_t m,
                        int d, float scale, int mask_kind, int64_t mask_a, int64_t mask_b, cv3_stream_t s) {
  CV3_ALIVE();
  const int64_t sq[3] = {0, n * d, d}, sk[3] = {0, m * d, d};
  return attention(true, q, k, v, out, 1, h, hk, n, m, d, sq, sk, sk, sq, scale, mask_kind, mask_a, mask_b, s, nullptr,
                   1, true);
}
