// Linears with both operands as bfloat16 planes in the matrix cores' fragment order.
//
// The float32 linear as six bfloat16 plane products (bf16x3.hpp) and the q8 linear as three
// (a code is exact in bfloat16), y = epi(x . W^T + bias), with the activation split into its
// planes once, by the kernel that produces it (a norm, the attention, the activation epilogue of
// the linear before), instead of by every tile that reads it.  A plane fragment is one contiguous
// kilobyte: frag[p][b][t][l] is the 16 bytes lane l feeds to v_mfma_f32_32x32x16_bf16 for the
// 16-k step t of the 32-row block b (row 32 b + l % 32, k = 16 t + 8 (l / 32) .. + 7), for weights
// and activations alike, so loads need no address arithmetic, no swizzle and no split.
//
// The weight is the matrix core's A operand and the activation its B: a lane's accumulator
// registers 4 g .. 4 g + 3 are four neighbouring outputs n of one row m = 32 b + l % 32, so the
// epilogue reads and writes float4, holds a rotary pair in one lane, and writes its result's own
// planes in whole 512-byte runs.
//
// Two kernels, chosen per shape by plane_variant():
//  * k_pg_reg: the K range split over the WK waves of a workgroup, each wave the whole RM x RN
//    block tile, fragments straight from L2 into registers, no barrier in the loop, the partial
//    sums met in LDS.  A small grid has WK times the waves and 1 / WK of the serial K steps.
//  * k_pg_lds: the tile split over the waves, fragments through a ring of LDS stages (two 16-k
//    steps each) filled by global -> LDS DMA, each loaded once per workgroup.  Fewer bytes from
//    L2 per product, which bounds the large grids.
// In both, the compiler sinks every load to the end of the MFMA block it may move past and then
// waits for all of them at once; sched_group_barrier pins one load between every one or two MFMAs
// (K = 2048 x [3000] rows: 73 -> 63 us, one 128 x 128 tile per 16-k step 1390 -> 900 cycles, 768
// of them MFMAs).
#include <algorithm>

#include "bf16x3.hpp"
#include "common.hpp"
#include "epilogue.hpp"

namespace cv3 {
int split_x3_frag(const float* w, int64_t n, int64_t k, int64_t ldw, uint16_t* frag, hipStream_t st);
}  // namespace cv3

using namespace cv3;

namespace {

typedef f32x16_t f32x16;

struct PlaneParams {
  const uint4* w;   // weight fragments [planes][nbw][S][64]
  int64_t wpl;      // fragments (16 bytes) per weight plane
  const uint4* x;   // activation fragments [3][nbx][S][64]
  int64_t xpl;
  int nbw, nbx, S;  // 32-row blocks of each operand, 16-k steps
  const float* scales;  // q8: [blocks][32 nbw]
  int m, n;
  const float* bias;
  float* c;         // float32 rows, or null
  int64_t ldc;
  uint2* yp;        // result planes in fragment order, or null
  int64_t ypl;      // 8-byte halves per result plane
  cv3_epilogue epi;
  // A_QKV: c holds q rows; the caches are at this layer's row pos0 of head 0
  float *kc, *vc;
  int heads, kv_heads, cap, pos0;
  const float *cos, *sin;  // [cap][64]
  // the float32 rows x was split from, or null (AGAIN kernels read them).  Outputs that come out not finite are
  // formed again from these: an infinity times a plane of zero is NaN, and code products may pass the range before
  // their scale.  So are those below 2^-90: rows below 2^-110 have fewer than 24 bits in their planes, which shows
  // (2^-134 an element) only in outputs this small, unless an output's weights sum to more than 2^20.
  const float* fx;
  int64_t ldfx;
  int tiles_m, tiles_n, gm;
};

// weights as three planes; as codes with one scale a row, per 64 codes, per 32 codes
enum { W_F32 = 0, W_ROW = 1, W_B64 = 2, W_B32 = 3 };
constexpr int planes_of(int kind) { return kind == W_F32 ? 3 : 1; }
constexpr int fold_steps(int kind) { return kind == W_B64 ? 4 : kind == W_B32 ? 2 : 0; }  // 16-k steps per scale

// Epilogues beyond the activations of cv3_epilogue, for the LM's prompt:
//  A_SWIGLU  outputs 2 j, 2 j + 1 are gate j and up j (the weight's rows interleaved): silu(g) u, N / 2 wide
//  A_QKV     bias, half-split rotary on q and k (each head's rows interleaved so that dims j and j + 32 are
//            outputs 2 j, 2 j + 1 of the head), q to rows, k and v to their cache rows
enum { A_SWIGLU = 100, A_QKV = 101 };

// Tile of workgroup L: XCD L % 8 takes a contiguous run of tiles, walked gm row tiles high.
__device__ __forceinline__ void plane_tile(const PlaneParams& p, int& tm, int& tn) {
  const int T = gridDim.x, L = blockIdx.x, x = L & 7, q = T >> 3, r = T & 7;
  const int t = x * q + min(x, r) + (L >> 3);
  const int per = p.gm * p.tiles_n, g = t / per, o = t - g * per;
  const int first = g * p.gm, gh = min(p.gm, p.tiles_m - first);
  tm = first + o % gh;
  tn = o / gh;
}

// The products of one 16-k step: hh (of q8: hq) into `big`, the small ones into `small`, each
// kind over all blocks before the next so no MFMA waits for the one before it.  FIRST starts both
// sums at zero.
template <int KIND, int RM, int RN, bool FIRST>
__device__ __forceinline__ void mma_step(f32x16 (&big)[RM][RN], f32x16 (&small)[RM][RN], const uint4 (&x)[RM][3],
                                         const uint4 (&w)[RN][planes_of(KIND)]) {
  const f32x16 zero = {0.f};
#define CV3_PRODUCT(ACC, PW, PX, ZERO)                                                   \
  _Pragma("unroll") for (int i = 0; i < RM; ++i) _Pragma("unroll") for (int j = 0; j < RN; ++j) \
      ACC[i][j] = mfma_bf16(w[j][PW], x[i][PX], (ZERO) ? zero : ACC[i][j]);
  CV3_PRODUCT(big, 0, 0, FIRST)
  if constexpr (KIND == W_F32) {
    CV3_PRODUCT(small, 1, 0, FIRST)
    CV3_PRODUCT(small, 0, 1, false)
    CV3_PRODUCT(small, 2, 0, false)
    CV3_PRODUCT(small, 1, 1, false)
    CV3_PRODUCT(small, 0, 2, false)
  } else {
    CV3_PRODUCT(small, 0, 1, FIRST)
    CV3_PRODUCT(small, 0, 2, false)
  }
#undef CV3_PRODUCT
}

// The scales of one 64-k block for this lane's outputs: register 4 g + e of block j is output
// 32 (tn RN + j) + 8 g + 4 (lane / 32) + e.
template <int RN>
struct BlockScales {
  float4 v[RN][4];
};

template <int RN>
__device__ __forceinline__ void load_scales(BlockScales<RN>& s, const float* base, int64_t ld, int blk, const int (&nb)[RN],
                                            int h) {
#pragma unroll
  for (int j = 0; j < RN; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      s.v[j][g] = *reinterpret_cast<const float4*>(base + blk * ld + nb[j] * 32 + 8 * g + 4 * h);
}

template <int RM, int RN>
__device__ __forceinline__ void fold_scales(f32x16 (&acc)[RM][RN], const f32x16 (&big)[RM][RN],
                                            const f32x16 (&small)[RM][RN], const BlockScales<RN>& s) {
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float sc[4] = {s.v[j][g].x, s.v[j][g].y, s.v[j][g].z, s.v[j][g].w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[i][j][4 * g + e] = fmaf(sc[e], big[i][j][4 * g + e] + small[i][j][4 * g + e], acc[i][j][4 * g + e]);
      }
}

template <int ACT>
__device__ __forceinline__ float act_of(float v) {
  if constexpr (ACT == CV3_ACT_GELU_TANH) return act_gelu_tanh(v);
  return v;
}

// Epilogue of G groups of four neighbouring outputs: group q of this lane is v[q], outputs
// n[q] .. n[q] + 3 of row m[q].  Every operand is loaded before the first store (C may be the
// residual itself), in k_pg_reg before the waves meet.  Order of operations as store_tile's
// (gemm.hip): bias, rotary, activation, gate, residual.  GATED kernels take a gate and a residual,
// AGAIN kernels the float rows of fx; the others spend no registers on them (which leaves the q8
// 64 x 128 tiles two workgroups per CU).
template <int ACT, int KIND, bool GATED, bool AGAIN, int G>
struct PlaneEpilogue {
  int m[G], n[G];
  float4 scale[G], bias[G], gate[G], res[G];

  __device__ __forceinline__ void load(const PlaneParams& p) {
    const cv3_epilogue& e = p.epi;
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int mm = min(m[q], p.m - 1), nn = min(n[q], p.n - 4);
      if constexpr (KIND == W_ROW) scale[q] = *reinterpret_cast<const float4*>(p.scales + nn);
      if (p.bias) bias[q] = *reinterpret_cast<const float4*>(p.bias + nn);
      if constexpr (GATED) {
        if (e.gate)
          gate[q] = *reinterpret_cast<const float4*>(
              e.gate + (int64_t)(e.rows_per_gate > 1 ? mm / (int)e.rows_per_gate : mm) * e.gate_stride + nn);
        if (e.residual) res[q] = *reinterpret_cast<const float4*>(e.residual + (int64_t)mm * e.ld_res + nn);
      }
    }
  }

  // The rotary of one block's groups q0 .. q0 + NQ - 1 (dit.py:40-54): a pair is two of a lane's four
  // outputs.  Few waves hold a rotated column; the others skip the table loads (a wave-uniform vote).
  template <int NQ>
  __device__ __forceinline__ void rotate(const PlaneParams& p, float4 (&v)[G], int q0) const {
    const cv3_epilogue& e = p.epi;
    bool rot[NQ], any = false;
    uint32_t cp[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      cp[q] = (uint32_t)n[q0 + q] % (uint32_t)e.rope_period;
      rot[q] = n[q0 + q] < e.rope_limit && cp[q] < (uint32_t)e.rope_width;
      any |= rot[q];
    }
    if (!__any(any)) return;
    float4 cs[NQ], sn[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const uint32_t row = (uint32_t)min(m[q0 + q], p.m - 1) % (uint32_t)e.rope_rows;
      const uint32_t ti = row * (uint32_t)e.rope_width + (rot[q] ? cp[q] : 0u);
      cs[q] = *reinterpret_cast<const float4*>(e.rope_cos + ti);
      sn[q] = *reinterpret_cast<const float4*>(e.rope_sin + ti);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const float4 u = v[q0 + q];
      if (rot[q])
        v[q0 + q] = make_float4(u.x * cs[q].x + (-u.y) * sn[q].x, u.y * cs[q].y + u.x * sn[q].y,
                                u.z * cs[q].z + (-u.w) * sn[q].z, u.w * cs[q].w + u.z * sn[q].w);
    }
  }

  // Row mm of fx times the weight's outputs nn .. nn + 3 in float32, by the whole wave: a lane takes every 64th run
  // of eight k, which is its 16 bytes of each plane.
  __device__ __forceinline__ float4 again(const PlaneParams& p, int mm, int nn, float4 row) const {
    constexpr int NPW = planes_of(KIND), FOLD = fold_steps(KIND);
    const int lane = threadIdx.x & 63;
    const float rs[4] = {row.x, row.y, row.z, row.w};
    float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int c = lane; c < p.S * 2; c += 64) {
      const float4 x0 = *reinterpret_cast<const float4*>(p.fx + (int64_t)mm * p.ldfx + 8 * c);
      const float4 x1 = *reinterpret_cast<const float4*>(p.fx + (int64_t)mm * p.ldfx + 8 * c + 4);
      const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __builtin_amdgcn_sched_barrier(0);   // one output's weights at a time: the tile's registers are few
        const int r = nn + e;
        const int64_t at = ((int64_t)(r >> 5) * p.S + (c >> 1)) * 64 + (r & 31) + 32 * (c & 1);
        uint4 f[NPW];
#pragma unroll
        for (int pl = 0; pl < NPW; ++pl) f[pl] = p.w[at + pl * p.wpl];
        float scale = 1.f;
        if constexpr (KIND == W_ROW) scale = rs[e];
        if constexpr (FOLD > 0) scale = p.scales[(int64_t)((c >> 1) / FOLD) * p.nbw * 32 + r];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float w = 0.f;   // lo + mid + hi: exact in this order
#pragma unroll
          for (int pl = NPW - 1; pl >= 0; --pl) {
            const uint32_t two = j < 2 ? f[pl].x : j < 4 ? f[pl].y : j < 6 ? f[pl].z : f[pl].w;
            w += __uint_as_float(j & 1 ? two & 0xffff0000u : two << 16);
          }
          if constexpr (KIND != W_F32) w *= scale;
          a[e] = fmaf(x[j], w, a[e]);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = wave_sum(a[e]);
    return make_float4(a[0], a[1], a[2], a[3]);
  }

  // Whether row mm of fx holds a NaN (by the whole wave): its outputs are NaN as they stand.
  __device__ __forceinline__ bool row_is_nan(const PlaneParams& p, int mm) const {
    bool nan = false;
#pragma unroll 1
    for (int k = 4 * (threadIdx.x & 63); k < p.S * 16; k += 256) {
      const float4 x = *reinterpret_cast<const float4*>(p.fx + (int64_t)mm * p.ldfx + k);
      nan |= x.x != x.x || x.y != x.y || x.z != x.z || x.w != x.w;
    }
    return __any(nan);
  }

  // Forms the groups that are out of the planes' range again.  Float32 [3000, 1024] x 3072, 0.12 ms: with one NaN
  // row as long, nothing but such rows 0.22 ms, nothing but rows of 1e-30 8.8 ms (each lane alone: 3.0, 8.2, 8.2).
  __device__ __forceinline__ void mend(const PlaneParams& p, float4 (&v)[G]) const {
    const int lane = threadIdx.x & 63;
    enum { UNREAD, NUMBERS, LOST };
    int mine = UNREAD;   // what the lane's row is
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const bool bad = !in_range(v[q]) && m[q] < p.m && n[q] < p.n;
      if (q == 0 || __builtin_amdgcn_readfirstlane(m[q]) != __builtin_amdgcn_readfirstlane(m[q - (q > 0)])) mine = UNREAD;
      uint64_t todo = __ballot(bad && mine != LOST);
      while (todo) {
        const int src = __builtin_ctzll(todo);
        const int mm = __builtin_amdgcn_readlane(m[q], src), nn = __builtin_amdgcn_readlane(n[q], src);
        if (__builtin_amdgcn_readlane(mine, src) == UNREAD) {
          const bool nan = row_is_nan(p, mm);
          if (m[q] == mm) mine = nan ? LOST : NUMBERS;
          if (nan) {
            todo &= ~__ballot(m[q] == mm);
            continue;
          }
        }
        todo &= todo - 1;
        float4 row = make_float4(1.f, 1.f, 1.f, 1.f);
        if constexpr (KIND == W_ROW) {
          auto at = [&](float f) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), src)); };
          row = make_float4(at(scale[q].x), at(scale[q].y), at(scale[q].z), at(scale[q].w));
        }
        const float4 again4 = again(p, mm, nn, row);
        if (lane == src) v[q] = again4;
      }
    }
  }

  __device__ __forceinline__ void store_swiglu(const PlaneParams& p, const float4 (&v)[G]) const {
    uint32_t* y = reinterpret_cast<uint32_t*>(p.yp);
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if (m[q] >= p.m || n[q] >= p.n) continue;
      uint32_t hi, mid, lo;
      split_x3(v[q].y * act_silu(v[q].x), v[q].w * act_silu(v[q].z), hi, mid, lo);
      const int c = n[q] >> 1;  // outputs c, c + 1: a quarter of a lane's 16 bytes
      const int64_t at =
          (((int64_t)(m[q] >> 5) * (p.n >> 5) + (c >> 4)) * 64 + (m[q] & 31) + 32 * ((c >> 3) & 1)) * 4 + ((c >> 1) & 3);
      y[at] = hi;
      y[at + 2 * p.ypl] = mid;
      y[at + 4 * p.ypl] = lo;
    }
  }

  // qwen2.py:64-71,155-168
  __device__ __forceinline__ void store_qkv(const PlaneParams& p, const float4 (&v)[G]) const {
    float2 cs[G], sn[G];
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int64_t t = (int64_t)(p.pos0 + min(m[q], p.m - 1)) * 64 + ((n[q] & 63) >> 1);
      cs[q] = *reinterpret_cast<const float2*>(p.cos + t);
      sn[q] = *reinterpret_cast<const float2*>(p.sin + t);
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if (m[q] >= p.m || n[q] >= p.n) continue;
      const int head = n[q] >> 6, r = n[q] & 63, kv = head - p.heads;
      if (kv >= p.kv_heads) {
        *reinterpret_cast<float4*>(p.vc + ((int64_t)(kv - p.kv_heads) * p.cap + m[q]) * 64 + r) = v[q];
        continue;
      }
      float* row = kv < 0 ? p.c + (int64_t)m[q] * p.ldc + head * 64 : p.kc + ((int64_t)kv * p.cap + m[q]) * 64;
      const float4 u = v[q];
      *reinterpret_cast<float2*>(row + (r >> 1)) = make_float2(u.x * cs[q].x + (-u.y) * sn[q].x, u.z * cs[q].y + (-u.w) * sn[q].y);
      *reinterpret_cast<float2*>(row + (r >> 1) + 32) = make_float2(u.y * cs[q].x + u.x * sn[q].x, u.w * cs[q].y + u.z * sn[q].y);
    }
  }

  __device__ __forceinline__ void store(const PlaneParams& p, float4 (&v)[G]) const {
    const cv3_epilogue& e = p.epi;
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if constexpr (KIND == W_ROW)
        v[q] = make_float4(v[q].x * scale[q].x, v[q].y * scale[q].y, v[q].z * scale[q].z, v[q].w * scale[q].w);
    }
    if constexpr (AGAIN) {  // a row too small makes its outputs small together (weights with such rows have no planes)
      bool fine = true;
#pragma unroll
      for (int q = 0; q < G; ++q) fine &= in_range(v[q]);
      if (__any(!fine)) mend(p, v);
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      if (p.bias) v[q] = make_float4(v[q].x + bias[q].x, v[q].y + bias[q].y, v[q].z + bias[q].z, v[q].w + bias[q].w);
    }
    if constexpr (ACT == A_QKV) return store_qkv(p, v);
    if constexpr (ACT == A_SWIGLU) return store_swiglu(p, v);
    if (e.rope_cos) {
      constexpr int NQ = G < 4 ? G : 4;
#pragma unroll
      for (int q0 = 0; q0 < G; q0 += NQ) rotate<NQ>(p, v, q0);
    }
#pragma unroll
    for (int q = 0; q < G; ++q) {
      float o[4] = {act_of<ACT>(v[q].x), act_of<ACT>(v[q].y), act_of<ACT>(v[q].z), act_of<ACT>(v[q].w)};
      if constexpr (GATED) {
        if (e.gate) {
          o[0] = gate[q].x * o[0];
          o[1] = gate[q].y * o[1];
          o[2] = gate[q].z * o[2];
          o[3] = gate[q].w * o[3];
        }
        if (e.residual) {
          o[0] = res[q].x + o[0];
          o[1] = res[q].y + o[1];
          o[2] = res[q].z + o[2];
          o[3] = res[q].w + o[3];
        }
      }
      if (m[q] >= p.m || n[q] >= p.n) continue;
      if (p.c) *reinterpret_cast<float4*>(p.c + (int64_t)m[q] * p.ldc + n[q]) = make_float4(o[0], o[1], o[2], o[3]);
      if (p.yp) {
        uint2 hi, mid, lo;
        split_x3(o[0], o[1], hi.x, mid.x, lo.x);
        split_x3(o[2], o[3], hi.y, mid.y, lo.y);
        // fragment of block m / 32, step n / 16; lane (m % 32) + 32 (n / 8 % 2); half n / 4 % 2
        const int64_t at =
            (((int64_t)(m[q] >> 5) * (p.n >> 4) + (n[q] >> 4)) * 64 + (m[q] & 31) + 32 * ((n[q] >> 3) & 1)) * 2 +
            ((n[q] >> 2) & 1);
        p.yp[at] = hi;
        p.yp[at + p.ypl] = mid;
        p.yp[at + 2 * p.ypl] = lo;
      }
    }
  }
};

// ---- fragments straight into registers, K split over the workgroup's waves ----
// PF register stages (PF - 1 steps in flight); a block-scaled weight's ranges are whole 64-k blocks.
template <int KIND, int ACT, bool GATED, bool AGAIN, int RM, int RN, int WK, int PF>
__global__ __launch_bounds__(64 * WK) void k_pg_reg(PlaneParams p) {
  constexpr int NPW = planes_of(KIND), FOLD = fold_steps(KIND), UNIT = FOLD ? FOLD : 1, LOADS = RM * 3 + RN * NPW;
  static_assert(UNIT == 1 || PF % 4 == 0, "a turn of the register ring is whole blocks");
  
  __shared__ float4 red[WK][RM * RN * 4 * 64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  plane_tile(p, tm, tn);
  const int units = p.S / UNIT;
  const int s0 = units * wave / WK * UNIT, s1 = units * (wave + 1) / WK * UNIT;
  // blocks past the last read it again; their outputs are dropped
  const uint4 *xp[RM], *wp[RN];
  int nb[RN];
#pragma unroll
  for (int i = 0; i < RM; ++i) xp[i] = p.x + (int64_t)min(tm * RM + i, p.nbx - 1) * p.S * 64 + lane;
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    nb[j] = min(tn * RN + j, p.nbw - 1);
    wp[j] = p.w + (int64_t)nb[j] * p.S * 64 + lane;
  }
  f32x16 big[RM][RN], small[RM][RN], acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) big[i][j] = small[i][j] = acc[i][j] = f32x16{0.f};
  uint4 bx[PF][RM][3], bw[PF][RN][NPW];
  auto load = [&](int buf, int s) {
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      if (pl < NPW) {
#pragma unroll
        for (int j = 0; j < RN; ++j) bw[buf][j][pl] = wp[j][pl * p.wpl + (int64_t)s * 64];
      }
#pragma unroll
      for (int i = 0; i < RM; ++i) bx[buf][i][pl] = xp[i][pl * p.xpl + (int64_t)s * 64];
    }
  };
#pragma unroll
  for (int j = 0; j < PF - 1; ++j) load(j, max(min(s0 + j, s1 - 1), 0));  // (an empty range loads step 0)
  __builtin_amdgcn_sched_barrier(0);
  constexpr int MF = RM * RN * (KIND == W_F32 ? 6 : 3), PER = MF / LOADS > 0 ? MF / LOADS : 1;
  const int h = lane >> 5;
  const int64_t lds = (int64_t)p.nbw * 32;
  BlockScales<RN> sc;
  // one step: its MFMAs with the loads of the step PF - 1 ahead between them (a uniform branch: the
  // wave's last turn of the ring may be short)
#define CV3_STEP(J, FIRST)                                                          \
  if (s + (J) < s1) {                                                               \
    load(((J) + PF - 1) % PF, min(s + (J) + PF - 1, s1 - 1));                       \
    mma_step<KIND, RM, RN, FIRST>(big, small, bx[J], bw[J]);                        \
    interleave<0x20, 1, 0x8, PER, LOADS>();                                         \
    __builtin_amdgcn_sched_barrier(0);                                              \
  }
  if constexpr (FOLD > 0) {
    for (int s = s0; s < s1; s += PF) {
#pragma unroll
      for (int c = 0; c < PF; c += FOLD) {
        if (s + c >= s1) break;
        load_scales<RN>(sc, p.scales, lds, (s + c) / FOLD, nb, h);
        CV3_STEP(c, true)
        CV3_STEP(c + 1, false)
        if constexpr (FOLD == 4) {
          CV3_STEP(c + 2, false)
          CV3_STEP(c + 3, false)
        }
        fold_scales<RM, RN>(acc, big, small, sc);
      }
    }
  } else {
    for (int s = s0; s < s1; s += PF) {
#pragma unroll
      for (int j = 0; j < PF; ++j) CV3_STEP(j, false)
    }
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j) acc[i][j] = big[i][j] + small[i][j];
  }
#undef CV3_STEP
  // the waves' partial sums meet in LDS, in wave order; each wave finishes its share of the groups
  constexpr int GROUPS = RM * RN * 4, G = GROUPS > WK ? GROUPS / WK : 1;
  PlaneEpilogue<ACT, KIND, GATED, AGAIN, G> ep;
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int id = min(wave * G + q, GROUPS - 1), blk = id >> 2, g = id & 3;
    ep.m[q] = (tm * RM + blk / RN) * 32 + (lane & 31);
    ep.n[q] = (tn * RN + blk % RN) * 32 + 8 * g + 4 * h;
  }
  ep.load(p);
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        red[wave][((i * RN + j) * 4 + g) * 64 + lane] =
            make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
  __syncthreads();
  if (wave * G >= GROUPS) return;  // more waves than groups: the first ones finish
  float4 v[G];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int id = wave * G + q;
    v[q] = red[0][id * 64 + lane];
#pragma unroll
    for (int u = 1; u < WK; ++u) {
      const float4 t = red[u][id * 64 + lane];
      v[q] = make_float4(v[q].x + t.x, v[q].y + t.y, v[q].z + t.z, v[q].w + t.w);
    }
  }
  ep.store(p, v);
}

// ---- fragments through a ring of LDS stages ----
// WM x WN waves of RM x RN blocks.  Stage s (16-k steps 2 s, 2 s + 1) sits in ring slot s % NST.  Per stage:
//   read the step's second fragments while the first's MFMAs run; wait until the next stage has
//   landed and every wave has read this one (vmcnt counts this wave's DMAs, which land in order);
//   refill this slot NST stages ahead and read the next stage's first fragments under the second
//   step's MFMAs.
template <int KIND, int ACT, bool GATED, bool AGAIN, int WM, int WN, int RM, int RN, int NST>
__global__ __launch_bounds__(64 * WM * WN) void k_pg_lds(PlaneParams p) {
  constexpr int NPW = planes_of(KIND), NW = WM * WN, TM = WM * RM, TN = WN * RN;
  constexpr int F = (TM * 3 + TN * NPW) * 2, FP = (F + NW - 1) / NW;  // fragments per stage, per wave
  __shared__ uint4 sh0[F * 64];
  __shared__ uint4 sh1[F * 64];
  __shared__ uint4 sh2[F * 64];
  __shared__ uint4 sh3[NST == 4 ? F * 64 : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  plane_tile(p, tm, tn);
  const int wm = wave / WN, wn = wave % WN, h = lane >> 5;
  // fragment f of a stage: f / 2 = (block, plane) of the activation's 3 TM, then the weight's, f % 2 = step
  const char* src[FP];
#pragma unroll
  for (int f = 0; f < FP; ++f) {
    const int id = min(wave * FP + f, F - 1), ks = id & 1, r = id >> 1;
    const uint4* base;
    if (r < 3 * TM)
      base = p.x + (r % 3) * p.xpl + (int64_t)min(tm * TM + r / 3, p.nbx - 1) * p.S * 64;
    else
      base = p.w + ((r - 3 * TM) % NPW) * p.wpl + (int64_t)min(tn * TN + (r - 3 * TM) / NPW, p.nbw - 1) * p.S * 64;
    src[f] = reinterpret_cast<const char*>(base + ks * 64);
  }
  const uint32_t loff = lane * 16;
  auto dma = [&](uint4* sh, int st) {
#pragma unroll
    for (int f = 0; f < FP; ++f)
      dma16(reinterpret_cast<const uint4*>(src[f] + (uint64_t)(uint32_t)st * 2048 + loff),
            sh + min(wave * FP + f, F - 1) * 64);
  };
  auto read = [&](const uint4* sh, int ks, uint4 (&x)[RM][3], uint4 (&w)[RN][NPW]) {
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
      if (pl < NPW) {
#pragma unroll
        for (int j = 0; j < RN; ++j) w[j][pl] = sh[((3 * TM + (wn * RN + j) * NPW + pl) * 2 + ks) * 64 + lane];
      }
#pragma unroll
      for (int i = 0; i < RM; ++i) x[i][pl] = sh[(((wm * RM + i) * 3 + pl) * 2 + ks) * 64 + lane];
    }
  };
  int nb[RN];
#pragma unroll
  for (int j = 0; j < RN; ++j) nb[j] = min(tn * TN + wn * RN + j, p.nbw - 1);
  f32x16 big[RM][RN], small[RM][RN], acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) big[i][j] = small[i][j] = acc[i][j] = f32x16{0.f};
  uint4 x0[RM][3], w0[RN][NPW], x1[RM][3], w1[RN][NPW];
  constexpr int NRD = RM * 3 + RN * NPW, NMF = RM * RN * (KIND == W_F32 ? 6 : 3);
  constexpr int RDP = (NRD + NMF / 2 - 1) / (NMF / 2);  // LDS reads per MFMA so that they fill its first half
  const int NS = p.S / 2;
  const int64_t lds = (int64_t)p.nbw * 32;
  BlockScales<RN> sc;
  dma(sh0, 0);
  dma(sh1, min(1, NS - 1));
  dma(sh2, min(2, NS - 1));
  if constexpr (NST == 4) dma(sh3, min(3, NS - 1));
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(CV3_VM((NST - 1) * FP));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read(sh0, 0, x0, w0);
#define CV3_STAGE(CUR, NXT, ST, FIRST)                                                              \
  {                                                                                                 \
    read(CUR, 1, x1, w1);                                                                           \
    mma_step<KIND, RM, RN, FIRST>(big, small, x0, w0);                                              \
    interleave<0x8, 1, 0x100, RDP, NRD / RDP>();                                                    \
    __builtin_amdgcn_sched_barrier(0);                                                              \
    __builtin_amdgcn_s_waitcnt(CV3_VM((NST - 2) * FP) & ~(0xF << 8));                               \
    __builtin_amdgcn_s_barrier();                                                                   \
    __builtin_amdgcn_sched_barrier(0);                                                              \
    read(NXT, 0, x0, w0);                                                                           \
    dma(CUR, min((ST) + NST, NS - 1));                                                              \
    mma_step<KIND, RM, RN, false>(big, small, x1, w1);                                              \
    interleave<0x8, 1, 0x100, RDP, NRD / RDP>();                                                    \
    interleave<0x20, 1, 0x8, 1, FP>();                                                              \
    __builtin_amdgcn_sched_barrier(0);                                                              \
  }
  int s = 0;
  if constexpr (KIND == W_B64) {
    // a 64-k block is two stages (K % 64 == 0: NS even)
#define CV3_BLOCK(A, B, C, ST)                               \
  load_scales<RN>(sc, p.scales, lds, (ST) >> 1, nb, h);      \
  CV3_STAGE(A, B, ST, true)                                  \
  CV3_STAGE(B, C, (ST) + 1, false)                           \
  fold_scales<RM, RN>(acc, big, small, sc);
    for (; s + 4 <= NS; s += 4) {
      CV3_BLOCK(sh0, sh1, sh2, s)
      CV3_BLOCK(sh2, sh3, sh0, s + 2)
    }
    if (s < NS) {
      CV3_BLOCK(sh0, sh1, sh2, s)
    }
#undef CV3_BLOCK
  } else if constexpr (KIND == W_B32) {
    // a 32-k block is one stage
#define CV3_BLOCK(A, B, ST)                          \
  load_scales<RN>(sc, p.scales, lds, ST, nb, h);     \
  CV3_STAGE(A, B, ST, true)                          \
  fold_scales<RM, RN>(acc, big, small, sc);
    for (; s + 4 <= NS; s += 4) {
      CV3_BLOCK(sh0, sh1, s)
      CV3_BLOCK(sh1, sh2, s + 1)
      CV3_BLOCK(sh2, sh3, s + 2)
      CV3_BLOCK(sh3, sh0, s + 3)
    }
    if (s < NS) {  // NS is even
      CV3_BLOCK(sh0, sh1, s)
      CV3_BLOCK(sh1, sh2, s + 1)
    }
#undef CV3_BLOCK
  } else if constexpr (NST == 4) {
    for (; s + 4 <= NS; s += 4) {
      CV3_STAGE(sh0, sh1, s, false)
      CV3_STAGE(sh1, sh2, s + 1, false)
      CV3_STAGE(sh2, sh3, s + 2, false)
      CV3_STAGE(sh3, sh0, s + 3, false)
    }
    if (s < NS) {
      CV3_STAGE(sh0, sh1, s, false)
      if (s + 1 < NS) {
        CV3_STAGE(sh1, sh2, s + 1, false)
        if (s + 2 < NS) CV3_STAGE(sh2, sh3, s + 2, false)
      }
    }
  } else {
    for (; s + 3 <= NS; s += 3) {
      CV3_STAGE(sh0, sh1, s, false)
      CV3_STAGE(sh1, sh2, s + 1, false)
      CV3_STAGE(sh2, sh0, s + 2, false)
    }
    if (s < NS) {
      CV3_STAGE(sh0, sh1, s, false)
      if (s + 1 < NS) CV3_STAGE(sh1, sh2, s + 1, false)
    }
  }
#undef CV3_STAGE
  __builtin_amdgcn_s_waitcnt(CV3_VM(0));  // no DMA outlives the workgroup's LDS
  constexpr int G = RM * RN * 4;
  PlaneEpilogue<ACT, KIND, GATED, AGAIN, G> ep;
  float4 v[G];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      if constexpr (fold_steps(KIND) == 0) acc[i][j] = big[i][j] + small[i][j];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int q = (i * RN + j) * 4 + g;
        v[q] = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        ep.m[q] = (tm * TM + wm * RM + i) * 32 + (lane & 31);
        ep.n[q] = (tn * TN + wn * RN + j) * 32 + 8 * g + 4 * h;
      }
    }
  ep.load(p);
  ep.store(p, v);
}

// Packed row r is source row r, but within the first `limit` rows each run of `span` rows is its two
// halves interleaved (span 0: none).
__device__ __forceinline__ int64_t source_row(int64_t r, int64_t span, int64_t limit) {
  return r < limit ? r / span * span + (r & 1) * (span / 2) + (r % span) / 2 : r;
}

// frag[nb][t][l] = the codes q[32 nb + l % 32][16 t + 8 (l / 32) .. + 7] as bfloat16 (exact; rows past n
// zero), and scales transposed to float32 [blocks][32 nbw].  q4: byte j of a 32-code block's 16 holds codes
// j (low nibble) and j + 16 (high), each + 8.
__global__ __launch_bounds__(256) void k_pack_codes(const uint8_t* q, bool q4, int64_t n, int64_t k, int64_t row_bytes,
                                                    int64_t span, int64_t limit, uint4* frag, int64_t total) {
  const int64_t T = k / 16;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(i & 63);
    const int64_t t = (i >> 6) % T, row = (i >> 6) / T * 32 + (l & 31), k0 = 16 * t + 8 * (l >> 5);
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = 0.f;
    if (row < n) {
      const uint8_t* src = q + source_row(row, span, limit) * row_bytes;
      if (q4) {
        const uint2 w = *reinterpret_cast<const uint2*>(src + k0 / 32 * 16 + (k0 & 8));
        const int sh = (k0 & 16) ? 4 : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float)((int)(((j < 4 ? w.x : w.y) >> (8 * (j & 3) + sh)) & 15u) - 8);
      } else {
        const uint2 w = *reinterpret_cast<const uint2*>(src + k0);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (float)((int32_t)((j < 4 ? w.x : w.y) << (24 - 8 * (j & 3))) >> 24);
      }
    }
    uint4 r;
    uint32_t* o = &r.x;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x2_t p2 = {v[2 * j], v[2 * j + 1]};
      o[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(p2, bf16x2_t));
    }
    frag[i] = r;
  }
}

__global__ __launch_bounds__(256) void k_scales_t(const void* scales, int sf16, int64_t n, int64_t npad, int64_t nb,
                                                  int64_t use, int64_t span, int64_t limit, float* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < use * npad; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / npad, r = i - b * npad;
    const int64_t src = r < n ? source_row(r, span, limit) * nb + b : 0;
    out[i] = r >= n ? 0.f
             : sf16 ? __half2float(reinterpret_cast<const __half*>(scales)[src])
                    : reinterpret_cast<const float*>(scales)[src];
  }
}

// The kernel and tile for a shape: a few rows take small tiles with K split over the waves (a lone
// wave's serial steps are the time), many rows the tiles that load the fewest bytes per product.  A
// variant's time on `tiles` tiles over S 16-k steps is modelled as
//   k_pg_lds: f0 + rounds (f1 + S max(a, b u)), rounds of 256 `occ` workgroups, u = tiles per CU and round
//   k_pg_reg: f0 + f1 u + S max(a, b u), u = the tiles of the busiest CU
// (a: one workgroup's step, b: a step with every CU busy; us).  The constants are least-squares fits to
// every variant timed at [40 .. 3000] rows x (N, K) = (3072, 1024), (2048, 1024), (1024, 1024),
// (1024, 2048), weights from HBM, within 4-9 %; the pick is the fastest variant or on average 0.9 % behind
// it.  Weights of 32-code blocks fold twice as often and have no fit of their own: they take the 64-code row.  The
// LM's shapes (K or N 896, 4864, 9728) were not in the fit either.  For both the pick is known to beat the float32
// kernels it took the place of, at 5 .. 3000 rows (q4 by 1.15 to 6 times), not to be the best of the six.  E.g.
// float32, us: [40, 1024] x 1024: 10.3 (1 x 1) against 17.3 (2 x 2) and 31 (128 x 128);
// [1000, 3072] x 1024: 36.9 (128 x 96) against 43.5 (2 x 2) and 66.7 (1 x 1).
struct Variant {
  int tm, tn;  // blocks of 32
  int occ;     // k_pg_lds: workgroups per CU; k_pg_reg: 0
  float f0, f1, a, b;
};
enum { V_R11, V_R12, V_R22, V_L12, V_L22, V_L13, V_COUNT };
constexpr Variant kVariants[3][V_COUNT] = {
    // float32 weights
    {{1, 1, 0, 3.89f, 1.06f, 0.087f, 0.065f}, {1, 2, 0, 3.05f, 2.05f, 0.117f, 0.095f},
     {2, 2, 0, 1.12f, 4.72f, 0.156f, 0.146f}, {2, 4, 1, 3.98f, 6.19f, 0.248f, 0.297f},
     {4, 4, 1, 0.86f, 8.31f, 0.397f, 0.650f}, {4, 3, 1, 0.97f, 11.73f, 0.321f, 0.362f}},
    // q8 weights, one scale a row
    {{1, 1, 0, 2.79f, 1.07f, 0.008f, 0.037f}, {1, 2, 0, 1.45f, 2.63f, 0.050f, 0.051f},
     {2, 2, 0, 1.28f, 3.56f, 0.091f, 0.091f}, {2, 4, 2, 7.27f, 0.00f, 0.115f, 0.193f},
     {4, 4, 1, 3.16f, 7.28f, 0.206f, 0.338f}, {4, 3, 1, 1.56f, 5.84f, 0.212f, 0.247f}},
    // q8 weights, one scale per 64 codes (and per 32)
    {{1, 1, 0, 2.15f, 1.70f, 0.040f, 0.043f}, {1, 2, 0, 1.58f, 2.65f, 0.058f, 0.062f},
     {2, 2, 0, 1.89f, 2.63f, 0.103f, 0.135f}, {2, 4, 2, 10.54f, 0.00f, 0.216f, 0.241f},
     {4, 4, 1, 5.85f, 0.00f, 0.503f, 0.571f}, {4, 3, 1, 5.93f, 0.00f, 0.424f, 0.445f}},
};

int plane_variant(int kind, int nbm, int nbn, int S) {
  kind = std::min(kind, (int)W_B64);
  int best = V_R11;
  float bt = 1e30f;
  for (int i = 0; i < V_COUNT; ++i) {
    const Variant& v = kVariants[kind][i];
    const int64_t tiles = ceil_div(nbm, v.tm) * ceil_div(nbn, v.tn);
    const int64_t rounds = v.occ ? ceil_div(tiles, 256 * v.occ) : 1;
    const float u = v.occ ? (float)tiles / (256.f * (float)rounds) : (float)ceil_div(tiles, 256);
    const float step = (float)S * std::max(v.a, v.b * u);
    const float t = v.f0 + (v.occ ? (float)rounds * (v.f1 + step) : u * v.f1 + step);
    if (t < bt) {
      bt = t;
      best = i;
    }
  }
  return best;
}

template <int KIND, int ACT, bool GATED, bool AGAIN = false>
void launch(int variant, const PlaneParams& p, hipStream_t st) {
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n));
  // the waves a tile's K is split over and the register ring, as measured per weight kind: float32
  // steps hold three planes of both operands, so fewer fit
  constexpr bool F = KIND == W_F32, B = fold_steps(KIND) > 0;
  constexpr int NST = F ? 3 : 4;
#define CV3_REG(RM, RN, WK, PF) \
  hipLaunchKernelGGL((k_pg_reg<KIND, ACT, GATED, AGAIN, RM, RN, WK, PF>), grid, dim3(64 * (WK)), 0, st, p)
#define CV3_LDS(WM, WN, RM, RN) \
  hipLaunchKernelGGL((k_pg_lds<KIND, ACT, GATED, AGAIN, WM, WN, RM, RN, NST>), grid, dim3(64 * (WM) * (WN)), 0, st, p)
  switch (variant) {
    case V_R11: CV3_REG(1, 1, (F ? 4 : 8), 4); break;
    case V_R12: CV3_REG(1, 2, (F ? 4 : 8), (F ? 3 : 4)); break;
    case V_R22: CV3_REG(2, 2, (B ? 4 : 8), (F ? 2 : B ? 4 : 3)); break;
    case V_L12: CV3_LDS(2, 2, 1, 2); break;
    case V_L22: CV3_LDS((F ? 4 : 2), 2, (F ? 1 : 2), 2); break;
    default: CV3_LDS(4, 1, 1, 3); break;
  }
#undef CV3_REG
#undef CV3_LDS
}

template <int KIND>
int launch_act(int act, int variant, const PlaneParams& p, hipStream_t st) {
  const bool gated = p.epi.gate || p.epi.residual;
  CV3_REQUIRE(!gated || act == CV3_ACT_NONE, CV3_EUNSUPPORTED,
              "plane linear: a gate or residual comes without an activation here");
  const bool again = p.fx != nullptr;
  if (act == CV3_ACT_NONE) {
    if (gated && again)
      launch<KIND, CV3_ACT_NONE, true, true>(variant, p, st);
    else if (gated)
      launch<KIND, CV3_ACT_NONE, true>(variant, p, st);
    else if (again)
      launch<KIND, CV3_ACT_NONE, false, true>(variant, p, st);
    else
      launch<KIND, CV3_ACT_NONE, false>(variant, p, st);
    return CV3_OK;
  }
  if constexpr (KIND != W_B32) {
    if (act == CV3_ACT_GELU_TANH) {
      if (again)
        launch<KIND, CV3_ACT_GELU_TANH, false, true>(variant, p, st);
      else
        launch<KIND, CV3_ACT_GELU_TANH, false>(variant, p, st);
      return CV3_OK;
    }
  }
  if constexpr (KIND != W_F32) {
    if (act == A_SWIGLU) {
      launch<KIND, A_SWIGLU, false>(variant, p, st);
      return CV3_OK;
    }
    if (act == A_QKV) {
      launch<KIND, A_QKV, false>(variant, p, st);
      return CV3_OK;
    }
  }
  return fail(CV3_EUNSUPPORTED, "plane linear: activation %d has no epilogue here", act);
}

// Fills the shape, tile and operands of p (its epilogue set) and launches it.
int plane_launch(int kind, int act, PlaneParams& p, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w,
                 const float* scales, int64_t n, const float* bias, int64_t plan_rows, hipStream_t st) {
  auto a16 = [](const void* q) { return (uintptr_t)q % 16 == 0; };
  CV3_REQUIRE(k % 64 == 0 && k >= (fold_steps(kind) ? 256 : 128) && n % 4 == 0, CV3_EUNSUPPORTED,
              "plane linear needs K %% 64 == 0, K >= 128 (block scales: 256), N %% 4 == 0 (K = %lld, N = %lld)",
              (long long)k, (long long)n);
  CV3_REQUIRE(a16(x) && a16(w) && a16(scales) && a16(bias) && a16(p.c) && a16(p.yp) && p.ldc % 4 == 0, CV3_EINVAL,
              "plane linear operands must be 16-byte aligned rows");
  CV3_REQUIRE(m < (1ll << 30) && plan_rows < (1ll << 30) && n < (1ll << 30) && k < (1ll << 30), CV3_EINVAL,
              "plane linear too large");
  p.S = (int)(k / 16);
  p.nbw = (int)ceil_div(n, 32);
  p.nbx = (int)ceil_div(m, 32);
  p.w = reinterpret_cast<const uint4*>(w);
  p.wpl = (int64_t)p.nbw * p.S * 64;
  p.x = reinterpret_cast<const uint4*>(x);
  p.xpl = (int64_t)p.nbx * p.S * 64;
  p.scales = scales;
  p.m = (int)m;
  p.n = (int)n;
  p.bias = bias;
  const int v = plane_variant(kind, (int)ceil_div(plan_rows > 0 ? plan_rows : m, 32), p.nbw, p.S);
  const Variant& t = kVariants[std::min(kind, (int)W_B64)][v];
  p.tiles_m = (int)ceil_div(p.nbx, t.tm);
  p.tiles_n = (int)ceil_div(p.nbw, t.tn);
  CV3_REQUIRE((int64_t)p.tiles_m * p.tiles_n < (1ll << 31), CV3_EINVAL, "plane linear too large");
  // an XCD's run of tiles as near to the fewest bytes of both operands as whole rows of tiles allow
  const double per = (double)p.tiles_m * p.tiles_n / 8, wb = (kind == W_F32 ? 3.0 : 1.0) * t.tn, xb = 3.0 * t.tm;
  int gm = 1;
  while (gm < p.tiles_m && (double)gm * gm * xb < per * wb) ++gm;
  p.gm = gm;
  const int rc = kind == W_F32   ? launch_act<W_F32>(act, v, p, st)
                 : kind == W_ROW ? launch_act<W_ROW>(act, v, p, st)
                 : kind == W_B64 ? launch_act<W_B64>(act, v, p, st)
                                 : launch_act<W_B32>(act, v, p, st);
  if (rc) return rc;
  CV3_LAUNCHED();
  return CV3_OK;
}

int plane_linear(int kind, const uint16_t* x, int64_t m, int64_t k, const uint16_t* w, const float* scales, int64_t n,
                 const float* bias, float* y, int64_t ldy, uint16_t* y_planes, const cv3_epilogue* epi,
                 int64_t plan_rows, hipStream_t st, const float* fx = nullptr, int64_t ldfx = 0) {
  CV3_REQUIRE(!y_planes || n % 16 == 0, CV3_EUNSUPPORTED, "a result in planes needs N %% 16 == 0 (N = %lld)", (long long)n);
  auto a16 = [](const void* q) { return (uintptr_t)q % 16 == 0; };
  PlaneParams p{};
  p.epi = epi ? *epi : cv3_epilogue{};
  const cv3_epilogue& e = p.epi;
  CV3_REQUIRE(a16(e.residual) && e.ld_res % 4 == 0 && a16(e.gate) && e.gate_stride % 4 == 0 && a16(e.rope_cos) &&
                  a16(e.rope_sin) && e.rows_per_gate < (1ll << 31),
              CV3_EINVAL, "plane linear operands must be 16-byte aligned rows");
  CV3_REQUIRE(!e.rope_cos || (e.rope_sin && e.rope_rows > 0 && e.rope_period > 0 && e.rope_period % 4 == 0 &&
                              e.rope_width % 4 == 0 && e.rope_rows * e.rope_width < (1ll << 31)),
              CV3_EINVAL, "plane linear: rotary widths must be multiples of four, the table within 32 bits");
  p.c = y;
  p.ldc = ldy;
  p.yp = reinterpret_cast<uint2*>(y_planes);
  p.ypl = ceil_div(m, 32) * (n / 16) * 128;
  p.fx = fx;
  p.ldfx = ldfx;
  return plane_launch(kind, e.act, p, x, m, k, w, scales, n, bias, plan_rows, st);
}

// One wave per row of at most 1024 columns (a multiple of 16): lane l holds the 8-column chunks l and
// l + 64, which are its fragments' 16 bytes.  RMS: y = (x * 1 / sqrt(mean x^2 + eps)) * w; else
// LayerNorm with the AdaLN shift and scale rows (elementwise.hip has both as float32 kernels, with
// the same operations in the same order).
__device__ __forceinline__ float lane_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <bool RMS>
__global__ __launch_bounds__(256) void k_norm_planes(const float* __restrict__ x, uint4* __restrict__ out, int64_t rows,
                                                     int cols, float eps, const float* __restrict__ w,
                                                     const float* __restrict__ shift, const float* __restrict__ scale,
                                                     int64_t opl) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int chunks = cols / 8;
  const float* xr = x + row * cols;
  float v[2][8], a[2][8], b[2][8];
  auto load8 = [](const float* s, float (&d)[8]) {
    const float4 lo = *reinterpret_cast<const float4*>(s), hi = *reinterpret_cast<const float4*>(s + 4);
    d[0] = lo.x; d[1] = lo.y; d[2] = lo.z; d[3] = lo.w;
    d[4] = hi.x; d[5] = hi.y; d[6] = hi.z; d[7] = hi.w;
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = min(lane + 64 * i, chunks - 1) * 8;
    load8(xr + c, v[i]);
    if constexpr (RMS) {
      load8(w + c, a[i]);
    } else {
      load8(scale + c, a[i]);
      load8(shift + c, b[i]);
    }
  }
  float s = 0.f;
  float mu = 0.f;
  if constexpr (!RMS) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (lane + 64 * i < chunks) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[i][e];
      }
    mu = lane_sum(s) / (float)cols;
  }
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (lane + 64 * i < chunks) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[i][e] - mu;
        q = fmaf(d, d, q);
      }
    }
  const float den = sqrtf(lane_sum(q) / (float)cols + eps);
  const float inv = 1.0f / den;
  const int S = cols / 16;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = lane + 64 * i;
    if (c >= chunks) continue;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      o[e] = RMS ? (v[i][e] * inv) * a[i][e] : (v[i][e] - mu) / den * (1.0f + a[i][e]) + b[i][e];
    uint4 hi, mid, lo;
    split_x3(make_float4(o[0], o[1], o[2], o[3]), make_float4(o[4], o[5], o[6], o[7]), hi, mid, lo);
    const int64_t at = ((row >> 5) * S + (c >> 1)) * 64 + (row & 31) + 32 * (c & 1);
    out[at] = hi;
    out[at + opl] = mid;
    out[at + 2 * opl] = lo;
  }
}

int norm_planes(bool rms, const float* x, uint16_t* planes, int64_t rows, int64_t cols, float eps, const float* w,
                const float* shift, const float* scale, hipStream_t st) {
  auto a16 = [](const void* q) { return (uintptr_t)q % 16 == 0; };
  CV3_REQUIRE(cols % 16 == 0 && cols >= 16 && cols <= 1024, CV3_EUNSUPPORTED,
              "a norm into planes takes 16 .. 1024 columns, a multiple of 16 (cols = %lld)", (long long)cols);
  CV3_REQUIRE(a16(x) && a16(planes) && a16(w) && a16(shift) && a16(scale), CV3_EINVAL,
              "a norm into planes needs 16-byte aligned operands");
  if (rows <= 0) return CV3_OK;
  const dim3 grid((unsigned)ceil_div(rows, 4));
  const int64_t opl = ceil_div(rows, 32) * (cols / 16) * 64;
  if (rms)
    hipLaunchKernelGGL(k_norm_planes<true>, grid, dim3(256), 0, st, x, reinterpret_cast<uint4*>(planes), rows, (int)cols,
                       eps, w, shift, scale, opl);
  else
    hipLaunchKernelGGL(k_norm_planes<false>, grid, dim3(256), 0, st, x, reinterpret_cast<uint4*>(planes), rows,
                       (int)cols, eps, w, shift, scale, opl);
  CV3_LAUNCHED();
  return CV3_OK;
}

// ---- the vocoder's causal convolutions on planes ----
// y[t] = bias + sum_tap W_tap x[t - (taps - 1 - tap) dil] over channels-last rows: a plane linear of
// K = taps C whose activation fragment of a step is the channel step's, read some rows up.  The producer
// has already applied Snake and split, once per element instead of once per tap and column tile.  Then,
// in the order of the reference: bias, residual, the float rows, and Snake of them as the next conv's
// planes.
// K is split over eight waves as in k_pg_reg.  The tile's rows and their halo go to LDS once (by passes over
// the channels where they exceed it) and every tap reads them there, so only the weight's fragments stream
// from L2: 3 KB against 6 RM products a step.  Few registers (two workgroups to a CU) beat a deep ring:
// 32-row tiles with four stages 9.6 us, with twelve 11.0.  What bounds it at a second of mel is latency: 5 to
// 6 us of a launch of 7 (k = 3) to 13 us (k = 11) go to the first fetch, the sum over waves and the launch.
// A resblock step of the 256-channel stage over 440 rows, k = 7: 41 us in five launches before, 21 in two.
struct ConvPlaneParams {
  const uint4 *x, *w;
  int64_t xpl, wpl;   // 16-byte fragments per plane
  uint32_t xbytes;
  int S, SC, SP, taps, dil;  // 16-k steps in all, per tap, and per tap and pass (SC / SP passes over channels)
  int m, n, nbx, nbw;
  const float *bias, *res, *alpha;
  float eps;
  float* y;
  uint2* yp;
  int64_t ypl;
  int tiles_m, tiles_n, cx, rows_x, cols_x;  // XCD x: cols_x columns from x % cx, rows_x rows from x / cx
};

__device__ __forceinline__ float snake(float v, float a, float eps) {
  const float s = sinf(a * v);
  return v + (1.0f / (a + eps)) * (s * s);
}

// 16 bytes per lane, global -> LDS, zeros past the descriptor's bound
__device__ __forceinline__ void buffer_dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint4* l) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 16, (int)voff, 0, 0, 0);
}

template <int RM, int PF, int XB>
__global__ __launch_bounds__(512, 4) void k_conv_planes(ConvPlaneParams p) {
  constexpr int WK = 8, RN = 1;
  static_assert(PF % XB == 0, "the x registers alternate within a turn of the weight ring");
  // x of the tile and pass, [plane][channel step][half][row], 16 bytes each; then the waves' partial sums
  extern __shared__ uint4 xs[];
  float4(*red)[RM * RN * 4 * 64] = reinterpret_cast<float4(*)[RM * RN * 4 * 64]>(xs);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
  const int xcd = blockIdx.x & 7, at_x = blockIdx.x >> 3;
  const int tm = xcd / p.cx * p.rows_x + at_x / p.cols_x, tn = xcd % p.cx * p.cols_x + at_x % p.cols_x;
  if (tm >= p.tiles_m || tn >= p.tiles_n) return;
  const int steps = p.taps * p.SP, s0 = steps * wave / WK, s1 = steps * (wave + 1) / WK;  // of each pass
  const int start = max(min(s0, s1 - 1), 0), tap0 = start / p.SP, cs0 = start - tap0 * p.SP;
  const uint4* wp = p.w + (int64_t)tn * p.S * 64 + lane;
  f32x16 big[RM][RN], small[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i) big[i][0] = small[i][0] = f32x16{0.f};
  uint4 bx[XB][RM][3], bw[PF][RN][3];
  // rows first .. first + R - 1 of x; those before 0 and past the tensor's blocks are zeros by the bound
  const int halo = (p.taps - 1) * p.dil, R = 32 * RM + halo, first = tm * RM * 32 - halo;
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(p.x), (short)0, (int)p.xbytes, 0x00027000);
  const int cols = 2 * p.SP, total = 3 * cols * R, dcol = 512 / R, drow = 512 - dcol * R;
  for (int c0 = 0; c0 < p.SC; c0 += p.SP) {
    // the weight's next step: past the wave's last it stays there (an empty range: at one before it)
    int sn = start, wtap = tap0, wcs = cs0;
    auto load = [&](int buf) {
      const int64_t at = (int64_t)(wtap * p.SC + c0 + wcs) * 64;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) bw[buf][0][pl] = wp[pl * p.wpl + at];
      if (sn + 1 < s1) {
        ++sn;
        if (++wcs == p.SP) {
          wcs = 0;
          ++wtap;
        }
      }
    };
#pragma unroll
    for (int j = 0; j < PF - 1; ++j) load(j);
    if (c0) __syncthreads();  // every wave has read the pass before
    int col = threadIdx.x / R, r = threadIdx.x - col * R;
    for (int i = threadIdx.x; i < total; i += 512) {
      const int g = first + r, pl = col / cols, ch = col - pl * cols;
      const uint32_t at = (uint32_t)(pl * p.xpl + (int64_t)((g >> 5) * p.SC + c0 + (ch >> 1)) * 64 + 32 * (ch & 1) +
                                     (g & 31)) * 16u;
      buffer_dma16(xr, g < 0 || g >= 32 * p.nbx ? 0x80000000u : at, xs + i - lane);
      col += dcol;
      r += drow;
      if (r >= R) {
        r -= R;
        ++col;
      }
    }
    __builtin_amdgcn_s_waitcnt(CV3_VM(0));
    __syncthreads();
    int tap = tap0, cs = cs0;  // the next step of x
    auto read = [&](int buf) {
      const uint4* from = xs + (cs * 2 + h) * R + (lane & 31) + tap * p.dil;
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
#pragma unroll
        for (int i = 0; i < RM; ++i) bx[buf][i][pl] = from[pl * cols * R + 32 * i];
      if (++cs == p.SP) {
        cs = 0;
        tap = min(tap + 1, p.taps - 1);
      }
    };
    if constexpr (XB == 2) read(0);
    __builtin_amdgcn_sched_barrier(0);
    for (int s = s0; s < s1; s += PF) {
#pragma unroll
      for (int j = 0; j < PF; ++j) {
        if (s + j < s1) {
          load((j + PF - 1) % PF);
          read((j + 1) % XB);
          mma_step<W_F32, RM, RN, false>(big, small, bx[j % XB], bw[j]);
          if constexpr (XB == 2) {
            interleave<0x100, 1, 0x8, 1, 3 * RM>();
            interleave<0x20, 1, 0x8, 1, 3>();
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  __syncthreads();  // every wave has read its x
  // the waves' partial sums meet in LDS, in wave order; each wave finishes its share of the groups
  constexpr int GROUPS = RM * RN * 4, G = GROUPS > WK ? GROUPS / WK : 1;
  int m[G], n[G];
  float4 bias[G], res[G], alpha[G];
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int id = min(wave * G + q, GROUPS - 1), blk = id >> 2;
    m[q] = (tm * RM + blk / RN) * 32 + (lane & 31);
    n[q] = (tn * RN + blk % RN) * 32 + 8 * (id & 3) + 4 * h;
    const int mm = min(m[q], p.m - 1), nn = min(n[q], p.n - 4);
    bias[q] = *reinterpret_cast<const float4*>(p.bias + nn);
    if (p.res) res[q] = *reinterpret_cast<const float4*>(p.res + (int64_t)mm * p.n + nn);
    if (p.yp) alpha[q] = *reinterpret_cast<const float4*>(p.alpha + nn);
  }
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = big[i][j][4 * g + e] + small[i][j][4 * g + e];
        red[wave][((i * RN + j) * 4 + g) * 64 + lane] = make_float4(o[0], o[1], o[2], o[3]);
      }
  __syncthreads();
  if (wave * G >= GROUPS) return;  // more waves than groups: the first ones finish
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int id = wave * G + q;
    float4 v = red[0][id * 64 + lane];
#pragma unroll
    for (int u = 1; u < WK; ++u) {
      const float4 t = red[u][id * 64 + lane];
      v = make_float4(v.x + t.x, v.y + t.y, v.z + t.z, v.w + t.w);
    }
    if (m[q] >= p.m || n[q] >= p.n) continue;
    v = make_float4(v.x + bias[q].x, v.y + bias[q].y, v.z + bias[q].z, v.w + bias[q].w);
    if (p.res) v = make_float4(res[q].x + v.x, res[q].y + v.y, res[q].z + v.z, res[q].w + v.w);
    if (p.y) *reinterpret_cast<float4*>(p.y + (int64_t)m[q] * p.n + n[q]) = v;
    if (p.yp) {
      uint2 hi, mid, lo;
      split_x3(snake(v.x, alpha[q].x, p.eps), snake(v.y, alpha[q].y, p.eps), hi.x, mid.x, lo.x);
      split_x3(snake(v.z, alpha[q].z, p.eps), snake(v.w, alpha[q].w, p.eps), hi.y, mid.y, lo.y);
      const int64_t at =
          (((int64_t)(m[q] >> 5) * (p.n >> 4) + (n[q] >> 4)) * 64 + (m[q] & 31) + 32 * ((n[q] >> 3) & 1)) * 2 +
          ((n[q] >> 2) & 1);
      p.yp[at] = hi;
      p.yp[at + p.ypl] = mid;
      p.yp[at + 2 * p.ypl] = lo;
    }
  }
}

// Snake of x (+ add, kept in sum) with up to three alphas, each as planes: one pass where a resblock
// group forks.  A thread owns eight channels of a row, the 16 bytes of each plane.
struct SnakePlanes {
  const float* alpha[3];
  uint4* planes[3];
};

__global__ __launch_bounds__(256) void k_snake_planes(const float* x, const float* add, float* sum, int64_t t, int c,
                                                      float eps, int count, SnakePlanes o, int64_t per_plane) {
  const int SC = c / 16;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < per_plane;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(i & 63);
    const int64_t b = (i >> 6) / SC;
    const int k0 = 16 * (int)((i >> 6) - b * SC) + 8 * (l >> 5);
    const int64_t row = b * 32 + (l & 31);
    float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
    if (row < t) {
      const int64_t at = row * c + k0;
      u = *reinterpret_cast<const float4*>(x + at);
      v = *reinterpret_cast<const float4*>(x + at + 4);
      if (add) {
        const float4 a = *reinterpret_cast<const float4*>(add + at), d = *reinterpret_cast<const float4*>(add + at + 4);
        u = make_float4(u.x + a.x, u.y + a.y, u.z + a.z, u.w + a.w);
        v = make_float4(v.x + d.x, v.y + d.y, v.z + d.z, v.w + d.w);
      }
      if (sum) {
        *reinterpret_cast<float4*>(sum + at) = u;
        *reinterpret_cast<float4*>(sum + at + 4) = v;
      }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      if (j >= count) break;
      const float4 a = *reinterpret_cast<const float4*>(o.alpha[j] + k0);
      const float4 d = *reinterpret_cast<const float4*>(o.alpha[j] + k0 + 4);
      uint4 hi, mid, lo;
      split_x3(make_float4(snake(u.x, a.x, eps), snake(u.y, a.y, eps), snake(u.z, a.z, eps), snake(u.w, a.w, eps)),
               make_float4(snake(v.x, d.x, eps), snake(v.y, d.y, eps), snake(v.z, d.z, eps), snake(v.w, d.w, eps)), hi,
               mid, lo);
      o.planes[j][i] = hi;
      o.planes[j][i + per_plane] = mid;
      o.planes[j][i + 2 * per_plane] = lo;
    }
  }
}

// leaky((((x0 + x1) + x2) ..) / count): the resblocks' mean and the activation its one reader applies
struct MeanInputs {
  const float* x[4];
};

__global__ __launch_bounds__(256) void k_mean_leaky(MeanInputs in, int count, float* y, int64_t n4, float slope) {
  const float by = (float)count;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    float4 v = reinterpret_cast<const float4*>(in.x[0])[i];
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      if (j >= count) break;
      const float4 a = reinterpret_cast<const float4*>(in.x[j])[i];
      v = make_float4(v.x + a.x, v.y + a.y, v.z + a.z, v.w + a.w);
    }
    v = make_float4(v.x / by, v.y / by, v.z / by, v.w / by);
    reinterpret_cast<float4*>(y)[i] = make_float4(v.x >= 0.f ? v.x : slope * v.x, v.y >= 0.f ? v.y : slope * v.y,
                                                  v.z >= 0.f ? v.z : slope * v.z, v.w >= 0.f ? v.w : slope * v.w);
  }
}

}  // namespace

extern "C" {

int cv3_plane_linear_tile(int kind, int64_t block, int64_t rows, int64_t k, int64_t n, int* tile, int* count,
                          int* row_blocks, int* col_blocks, int* ring) {
  CV3_REQUIRE(tile && count && row_blocks && col_blocks && ring && rows > 0 && k > 0 && n > 0 && rows < (1ll << 30) &&
                  k < (1ll << 30) && n < (1ll << 30) && block > 0,
              CV3_EINVAL, "bad plane linear shape");
  const int wk = kind == CV3_KIND_F32 ? W_F32 : block >= k ? W_ROW : block == 64 ? W_B64 : W_B32;
  const int v = plane_variant(wk, (int)ceil_div(rows, 32), (int)ceil_div(n, 32), (int)(k / 16));
  const Variant& t = kVariants[std::min(wk, (int)W_B64)][v];
  *tile = v;
  *count = V_COUNT;
  *row_blocks = t.tm;
  *col_blocks = t.tn;
  *ring = t.occ > 0;
  return CV3_OK;
}

int cv3_linear_x3_planes(const uint16_t* x, int64_t m, int64_t k, const uint16_t* frag, int64_t n, const float* bias,
                         float* y, int64_t ldy, uint16_t* y_planes, const cv3_epilogue* epi, int64_t plan_rows,
                         cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(m >= 0 && k > 0 && n >= 0 && (!y || ldy >= n) && (y || y_planes), CV3_EINVAL,
              "bad plane linear shape m=%lld k=%lld n=%lld", (long long)m, (long long)k, (long long)n);
  if (!m || !n) return CV3_OK;
  return plane_linear(W_F32, x, m, k, frag, nullptr, n, bias, y, ldy, y_planes, epi, plan_rows, stream_of(s));
}

int cv3_code_planes_elems(int64_t n, int64_t k, int64_t block, int64_t* codes, int64_t* scales) {
  CV3_REQUIRE(n >= 0 && k > 0 && block > 0 && codes && scales, CV3_EINVAL, "bad shape or null output");
  const int64_t npad = ceil_div(n, 32) * 32;
  *codes = npad * k;
  *scales = npad * (block >= k ? 1 : ceil_div(k, block));
  return CV3_OK;
}

int cv3_pack_code_planes(int kind, const void* q, int64_t n, int64_t k, const void* scales, int scale_dtype, int64_t kp,
                         int64_t block, int64_t span, int64_t limit, uint16_t* frag, float* scales_t, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(kind == CV3_KIND_Q8 || kind == CV3_KIND_Q4, CV3_EINVAL, "unknown quant kind %d", kind);
  CV3_REQUIRE(n >= 0 && k > 0 && k % 64 == 0 && block > 0 && kp >= k && kp % block == 0 && kp % 16 == 0, CV3_EINVAL,
              "bad code pack shape n=%lld k=%lld block=%lld", (long long)n, (long long)k, (long long)block);
  CV3_REQUIRE(span >= 0 && span % 2 == 0 && (span ? limit >= 0 && limit <= n && limit % span == 0 : limit == 0),
              CV3_EINVAL, "bad row interleave span=%lld limit=%lld", (long long)span, (long long)limit);
  CV3_REQUIRE(block == 64 || block == 32 || block >= k, CV3_EUNSUPPORTED,
              "plane codes take 32- or 64-code blocks or one scale a row");
  CV3_REQUIRE(kind == CV3_KIND_Q8 || (block == 32 && scale_dtype == CV3_F16), CV3_EUNSUPPORTED,
              "q4 codes come in 32-code blocks with float16 scales");
  CV3_REQUIRE((uintptr_t)q % 8 == 0 && (uintptr_t)frag % 16 == 0 && (uintptr_t)scales_t % 16 == 0, CV3_EINVAL,
              "plane codes need aligned rows");
  const int64_t npad = ceil_div(n, 32) * 32, total = npad * k / 8, use = block >= k ? 1 : k / block;
  if (!total) return CV3_OK;
  hipStream_t st = stream_of(s);
  const bool q4 = kind == CV3_KIND_Q4;
  hipLaunchKernelGGL(k_pack_codes, dim3((unsigned)(ceil_div(total, 256) < 65536 ? ceil_div(total, 256) : 65536)),
                     dim3(256), 0, st, reinterpret_cast<const uint8_t*>(q), q4, n, k, q4 ? kp / 2 : kp, span, limit,
                     reinterpret_cast<uint4*>(frag), total);
  hipLaunchKernelGGL(k_scales_t, dim3((unsigned)ceil_div(use * npad, 256)), dim3(256), 0, st, scales,
                     scale_dtype == CV3_F16 ? 1 : 0, n, npad, kp / block, use, span, limit, scales_t);
  CV3_LAUNCHED();
  return CV3_OK;
}

int cv3_linear_code_planes(const uint16_t* x, int64_t m, int64_t k, const uint16_t* frag, const float* scales_t,
                         int64_t block, int64_t n, const float* bias, float* y, int64_t ldy, uint16_t* y_planes,
                         const cv3_epilogue* epi, int64_t plan_rows, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(m >= 0 && k > 0 && n >= 0 && (!y || ldy >= n) && (y || y_planes) && scales_t, CV3_EINVAL,
              "bad plane linear shape m=%lld k=%lld n=%lld", (long long)m, (long long)k, (long long)n);
  CV3_REQUIRE(block == 64 || block == 32 || block >= k, CV3_EUNSUPPORTED,
              "plane codes take 32- or 64-code blocks or one scale a row");
  if (!m || !n) return CV3_OK;
  return plane_linear(block >= k ? W_ROW : block == 64 ? W_B64 : W_B32, x, m, k, frag, scales_t, n, bias, y, ldy, y_planes, epi,
                      plan_rows, stream_of(s));
}

// ops.linear on float32 rows: x split into planes in a workspace of the library's allocator, then the plane
// linear.
int cv3_linear_rows_planes(int kind, const float* x, int64_t m, int64_t k, int64_t ldx, const uint16_t* frag,
                           const float* scales_t, int64_t block, int64_t n, const float* bias, float* y, int64_t ldy,
                           const cv3_epilogue* epi, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(kind == CV3_KIND_F32 || kind == CV3_KIND_Q8 || kind == CV3_KIND_Q4, CV3_EINVAL, "unknown weight kind %d", kind);
  CV3_REQUIRE(m >= 0 && k > 0 && n >= 0 && ldx >= k && ldy >= n && y && (kind == CV3_KIND_F32 || (scales_t && block > 0)),
              CV3_EINVAL, "bad linear shape m=%lld k=%lld n=%lld", (long long)m, (long long)k, (long long)n);
  CV3_REQUIRE(kind == CV3_KIND_F32 || block == 64 || block == 32 || block >= k, CV3_EUNSUPPORTED,
              "plane codes take 32- or 64-code blocks or one scale a row");
  CV3_REQUIRE(k % 64 == 0 && (uintptr_t)x % 16 == 0 && ldx % 4 == 0, CV3_EUNSUPPORTED,
              "rows split into planes need K %% 64 == 0 and 16-byte alignment");
  if (!m || !n) return CV3_OK;
  hipStream_t st = stream_of(s);
  CV3_REQUIRE(st, CV3_EHIP, "no stream");
  void* ws = nullptr;
  int rc = scratch_alloc(&ws, (size_t)(6 * ceil_div(m, 32) * 32 * k), st);
  if (rc) return rc;
  uint16_t* planes = reinterpret_cast<uint16_t*>(ws);
  rc = split_x3_frag(x, m, k, ldx, planes, st);
  if (!rc) {
    const int wk = kind == CV3_KIND_F32 ? W_F32 : block >= k ? W_ROW : block == 64 ? W_B64 : W_B32;
    rc = plane_linear(wk, planes, m, k, frag, scales_t, n, bias, y, ldy, nullptr, epi, 0, st, x, ldx);
  }
  const int rf = scratch_free(ws, st);
  return rc ? rc : rf;
}

int cv3_layer_norm_planes(const float* x, uint16_t* planes, int64_t rows, int64_t cols, float eps, const float* shift,
                          const float* scale, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(shift && scale, CV3_EINVAL, "a layer norm into planes needs its shift and scale rows");
  return norm_planes(false, x, planes, rows, cols, eps, nullptr, shift, scale, stream_of(s));
}

int cv3_rms_norm_planes(const float* x, const float* w, uint16_t* planes, int64_t rows, int64_t cols, float eps,
                        cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(w, CV3_EINVAL, "an RMS norm needs its weight");
  return norm_planes(true, x, planes, rows, cols, eps, w, nullptr, nullptr, stream_of(s));
}

// Qwen2Model.forward over t prompt rows at positions pos0 .. (qwen2.py:139-179), then the last position's
// head logits: seven launches a layer.
namespace {
__global__ void k_set_pos(int64_t* pos, int64_t v) { *pos = v; }
}  // namespace

int cv3_qwen2_prefill(const cv3_qwen2_model* m, const cv3_qwen2_state* st, const cv3_qwen2_planes* w, const float* x,
                      int64_t t, int64_t pos0, float* h, float* q, uint16_t* planes, uint16_t* inter_planes,
                      cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(m && st && w && x && h && q && planes && inter_planes, CV3_EINVAL, "null prefill operand");
  const int64_t D = m->hidden, I = m->inter, H = m->heads, Hk = m->kv_heads, L = m->layers, cap = st->cap;
  const int64_t R = (H + 2 * Hk) * 64;
  CV3_REQUIRE(m->head_dim == 64 && H > 0 && Hk > 0 && H % Hk == 0 && H * 64 == D && D % 64 == 0 && D <= 1024 && D >= 256 &&
                  I % 64 == 0 && I >= 256,
              CV3_EUNSUPPORTED, "prompt planes take head dim 64, hidden 256 .. 1024 and multiples of 64");
  CV3_REQUIRE(t > 0 && pos0 >= 0 && pos0 + t <= cap && cap < (1ll << 30), CV3_EINVAL, "the prompt does not fit the KV cache");
  hipStream_t stream = stream_of(s);
  auto kind_of = [](int64_t block, int64_t k) { return block >= k ? W_ROW : block == 64 ? W_B64 : W_B32; };
  // a projection's fragments and scales per layer
  auto at = [&](const cv3_code_planes& c, int64_t l, int64_t rows, int64_t k, const uint16_t*& f, const float*& sc) {
    f = c.frag + l * rows * k;
    sc = c.scales + l * rows * (c.block >= k ? 1 : k / c.block);
  };
  const uint16_t* f;
  const float* sc;
  int rc;
  for (int64_t l = 0; l < L; ++l) {
    const float* in = l ? h : x;
    if ((rc = norm_planes(true, in, planes, t, D, m->eps, m->ln1 + l * D, nullptr, nullptr, stream))) return rc;
    at(w->qkv, l, R, D, f, sc);
    PlaneParams p{};
    p.c = q;
    p.ldc = H * 64;
    p.kc = st->k_cache + (l * Hk * cap + pos0) * 64;
    p.vc = st->v_cache + (l * Hk * cap + pos0) * 64;
    p.heads = (int)H;
    p.kv_heads = (int)Hk;
    p.cap = (int)cap;
    p.pos0 = (int)pos0;
    p.cos = m->rope_cos;
    p.sin = m->rope_sin;
    if ((rc = plane_launch(kind_of(w->qkv.block, D), A_QKV, p, planes, t, D, f, sc, R, w->qkv_bias + l * R, 0, stream)))
      return rc;
    const int64_t qs[3] = {0, 64, H * 64}, ks[3] = {0, cap * 64, 64};
    if ((rc = cv3_attention_x3_planes(q, st->k_cache + l * Hk * cap * 64, st->v_cache + l * Hk * cap * 64, planes, 1, (int)H,
                                      (int)Hk, t, pos0 + t, 64, qs, ks, ks, 0.125f, t > 1 ? 1 : 0, pos0, 0, s)))
      return rc;
    at(w->o, l, D, D, f, sc);
    cv3_epilogue e{};
    e.residual = in;
    e.ld_res = D;
    if ((rc = plane_linear(kind_of(w->o.block, D), planes, t, D, f, sc, D, nullptr, h, D, nullptr, &e, 0, stream))) return rc;
    if ((rc = norm_planes(true, h, planes, t, D, m->eps, m->ln2 + l * D, nullptr, nullptr, stream))) return rc;
    at(w->gate_up, l, 2 * I, D, f, sc);
    PlaneParams g{};
    g.yp = reinterpret_cast<uint2*>(inter_planes);
    g.ypl = ceil_div(t, 32) * (I / 16) * 128;
    if ((rc = plane_launch(kind_of(w->gate_up.block, D), A_SWIGLU, g, planes, t, D, f, sc, 2 * I, nullptr, 0, stream)))
      return rc;
    at(w->down, l, D, I, f, sc);
    e.residual = h;
    if ((rc = plane_linear(kind_of(w->down.block, I), inter_planes, t, I, f, sc, D, nullptr, h, D, nullptr, &e, 0, stream)))
      return rc;
  }
  // the last position: final norm, head, and its position for the decode
  if ((rc = cv3_rms_norm(h + (t - 1) * D, m->norm, q, 1, D, m->eps, s))) return rc;
  const cv3_qweight& hd = m->head;
  if ((rc = cv3_linear_q(hd.kind, q, 1, D, D, hd.q, hd.scales, hd.scale_dtype, hd.kp, hd.block, hd.rows, m->head_bias,
                         st->logits, hd.rows, nullptr, s)))
    return rc;
  hipLaunchKernelGGL(k_set_pos, dim3(1), dim3(1), 0, stream, st->pos, pos0 + t - 1);
  CV3_LAUNCHED();
  return CV3_OK;
}

// ---- vocoder ----
int cv3_conv_planes(const uint16_t* x, int64_t t, int64_t cin, const uint16_t* w_frag, int64_t cout, int64_t k,
                    int64_t dilation, const float* bias, const float* residual, float* y, const float* alpha,
                    float eps, uint16_t* y_planes, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(x && w_frag && bias && (y || y_planes) && t >= 0 && cin > 0 && cout > 0 && k > 0 && dilation > 0,
              CV3_EINVAL, "bad plane convolution");
  CV3_REQUIRE(cin % 16 == 0 && k * cin % 64 == 0 && cout % 16 == 0, CV3_EUNSUPPORTED,
              "plane convolution needs C %% 16 == 0 and K %% 64 == 0");
  CV3_REQUIRE(!y_planes || alpha, CV3_EINVAL, "planes out need an alpha");
  CV3_REQUIRE(((uintptr_t)x | (uintptr_t)w_frag | (uintptr_t)bias | (uintptr_t)residual | (uintptr_t)y | (uintptr_t)alpha |
               (uintptr_t)y_planes) % 16 == 0, CV3_EUNSUPPORTED, "plane convolution needs 16-byte alignment");
  const int64_t rows = ceil_div(t, 32) * 32, bytes = 6 * rows * cin;
  CV3_REQUIRE(bytes < (1ll << 31) && 6 * rows * cout < (1ll << 34) && (k - 1) * dilation < (1 << 24) && k * cin < (1 << 24),
              CV3_EUNSUPPORTED, "plane convolution over 2^31 bytes or more");
  if (!t) return CV3_OK;
  ConvPlaneParams p{};
  p.x = reinterpret_cast<const uint4*>(x);
  p.w = reinterpret_cast<const uint4*>(w_frag);
  p.xpl = rows * cin / 8;
  p.wpl = ceil_div(cout, 32) * 32 * k * cin / 8;
  p.xbytes = (uint32_t)bytes;
  p.S = (int)(k * cin / 16);
  p.SC = (int)(cin / 16);
  p.taps = (int)k;
  p.dil = (int)dilation;
  p.m = (int)t;
  p.n = (int)cout;
  p.nbx = (int)(rows / 32);
  p.nbw = (int)ceil_div(cout, 32);
  p.bias = bias;
  p.res = residual;
  p.alpha = alpha;
  p.eps = eps;
  p.y = y;
  p.yp = reinterpret_cast<uint2*>(y_planes);
  p.ypl = rows / 32 * (cout / 16) * 128;
  // 256 workgroups at a time, shared with two more launches (a stage's resblocks, or windows, run side by
  // side; 1 to 8 of them change a decode by 3 %), each as long as its products and its weight's fetch; ties to
  // the larger tile
  auto tiles = [&](int rm) { return 3. * (double)(ceil_div(p.nbx, rm) * p.nbw); };
  auto cost = [&](int rm) { return std::max(1., tiles(rm) / 256) * (rm + 1); };
  const int rm = cost(2) <= cost(1) ? 2 : 1;
  // x of one pass in LDS: all channels while a CU has one workgroup anyway, else at most half of the LDS, so that
  // a second workgroup's products run under this one's fetch (10 s whole: one workgroup to a CU 3.4 ms, two 2.75)
  const int64_t most = (tiles(rm) <= 256 ? 160 : 80) << 10, per_step = (32 * rm + (k - 1) * dilation) * 96;
  p.SP = p.SC;
  while (p.SP > 1 && p.SP * per_step > most) p.SP = p.SP % 2 ? 1 : p.SP / 2;
  const int64_t lds = std::max<int64_t>(p.SP * per_step, 8 * rm * 4096);
  CV3_REQUIRE(lds <= 160 << 10, CV3_EUNSUPPORTED, "plane convolution: a tile with its halo needs %lld bytes of LDS",
              (long long)lds);
  p.tiles_m = (int)ceil_div(p.nbx, rm);
  p.tiles_n = p.nbw;
  // each XCD's L2 fetches its own columns of the weight and rows of x: the split of the eight that fetches least
  // (440 rows of 256 channels, K = 2816: 4.4 MB each in row runs, 1.2 in columns)
  double least = 0.;
  for (int cx = 1; cx <= 8 && cx <= p.tiles_n; cx *= 2) {
    const double fetch = (double)p.wpl / cx + (double)p.xpl / std::min(8 / cx, p.tiles_m);
    if (cx > 1 && fetch >= least) continue;
    least = fetch;
    p.cx = cx;
  }
  p.rows_x = (int)ceil_div(p.tiles_m, 8 / p.cx);
  p.cols_x = (int)ceil_div(p.tiles_n, p.cx);
  const dim3 grid((unsigned)(8 * p.rows_x * p.cols_x));
  hipStream_t st = stream_of(s);
  if (rm == 2)
    hipLaunchKernelGGL((k_conv_planes<2, 2, 1>), grid, dim3(512), (uint32_t)lds, st, p);
  else
    hipLaunchKernelGGL((k_conv_planes<1, 4, 2>), grid, dim3(512), (uint32_t)lds, st, p);
  CV3_LAUNCHED();
  return CV3_OK;
}

int cv3_snake_planes(const float* x, const float* add, float* sum, int64_t t, int64_t c, float eps, int count,
                     const float* const* alphas, uint16_t* const* planes, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(x && t >= 0 && c > 0 && c < (1 << 24) && count >= 1 && count <= 3 && alphas && planes, CV3_EINVAL,
              "bad snake planes");
  CV3_REQUIRE(c % 16 == 0 && ((uintptr_t)x | (uintptr_t)add | (uintptr_t)sum) % 16 == 0, CV3_EUNSUPPORTED,
              "snake planes need C %% 16 == 0 and 16-byte alignment");
  SnakePlanes o{};
  for (int j = 0; j < count; ++j) {
    CV3_REQUIRE(alphas[j] && planes[j] && ((uintptr_t)alphas[j] | (uintptr_t)planes[j]) % 16 == 0, CV3_EINVAL,
                "bad snake planes output %d", j);
    o.alpha[j] = alphas[j];
    o.planes[j] = reinterpret_cast<uint4*>(planes[j]);
  }
  const int64_t per_plane = ceil_div(t, 32) * 32 * c / 8;
  if (!per_plane) return CV3_OK;
  const int64_t blocks = std::min<int64_t>(ceil_div(per_plane, 256), 65536);
  hipLaunchKernelGGL(k_snake_planes, dim3((unsigned)blocks), dim3(256), 0, stream_of(s), x, add, sum, t, (int)c, eps,
                     count, o, per_plane);
  CV3_LAUNCHED();
  return CV3_OK;
}

int cv3_mean_leaky(int count, const float* const* x, float* y, int64_t n, float slope, cv3_stream_t s) {
  CV3_ALIVE();
  CV3_REQUIRE(count >= 1 && count <= 4 && x && y && n >= 0, CV3_EINVAL, "bad mean");
  MeanInputs in{};
  uintptr_t all = (uintptr_t)y;
  for (int j = 0; j < count; ++j) {
    CV3_REQUIRE(x[j], CV3_EINVAL, "null input %d of a mean", j);
    in.x[j] = x[j];
    all |= (uintptr_t)x[j];
  }
  CV3_REQUIRE(n % 4 == 0 && all % 16 == 0, CV3_EUNSUPPORTED, "mean needs multiples of 16 bytes");
  if (!n) return CV3_OK;
  hipLaunchKernelGGL(k_mean_leaky, dim3((unsigned)std::min<int64_t>(ceil_div(n / 4, 256), 65536)), dim3(256), 0,
                     stream_of(s), in, count, y, n / 4, slope);
  CV3_LAUNCHED();
  return CV3_OK;
}

}  // extern "C"
