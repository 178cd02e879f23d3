// Split-KV attention of a multi-position step on the f32 matrix cores, bit for bit equal to the decode kernels
// (k_attn_tiles, kernels.hip).
//
// The f32 MFMAs are fused multiply-add chains: v_mfma_f32_16x16x1 adds one product to every element of its four
// 16x16 blocks, and v_mfma_f32_16x16x4 adds its four products in the order of k, each step rounded as fmaf rounds it
// (subnormals included; tests/test_gpu_prefill.py compares whole steps with the decode kernels' chains). So the
// scores' chain over the 64 dims and p.v's chain over the 64 positions of a tile run on them unchanged.
//
// A workgroup serves 16 units (a unit is one query head at one position of the step) of one KV head and one split,
// each of its waves one of the split's tiles of 64 positions, as k_attn_tiles does (a split of more than 4 tiles in
// rounds of 4). Per tile:
//   scores  64 MFMAs 16x16x1: rows = the tile's 64 positions (4 blocks), columns = units. A lane holds one K row and
//           its unit's query.
//   p       element (b, r) of a lane of group G = lane / 16 is position 16 b + 4 r + G of unit lane % 16: the K rows
//           are dealt to the lanes so that it is. That is the k = G operand of the p.v MFMA over positions
//           4 (4 b + r) .. +3, so p goes from one product into the next without leaving its register.
//   p.v     64 MFMAs 16x16x4: 16 steps of 4 positions, 4 blocks of 16 dims (lane i: dims 4 i .. 4 i + 3, one 8-byte
//           load of a V row)
// Neither K, V nor p passes through LDS; it carries the tile maxima, alphas and sums, and the p.v of each tile into
// the in-order combine, which the waves share by dims.
// Bound: the matrix cores (128 MFMAs of 32 cycles per tile and wave, against about 600 vector instructions, half of
// them the 16 exps of a lane) once every SIMD has waves to overlap the two; with few positions the latency of a wave.
// A tile per wave and not a split per wave: the three tiles of a split one after the other left one wave on a SIMD
// and took 29 us where this took 21, both measured before the one-sided exp (3B shape, 32 positions after 4096
// cached, 3 tiles per split; one FMA chain per lane on the vector unit took 38 us). Now 19.6 in a kernel trace.
#include "attn_dev.h"
#include "kernels.h"
#include "launch.h"

namespace moert {

typedef float mm_f4 __attribute__((ext_vector_type(4)));
typedef float mm_f16 __attribute__((ext_vector_type(16)));

constexpr int kMmUnits = 16;  // units of a workgroup

__device__ __forceinline__ float half_of(uint32_t w, int hi) { return h2f((uint16_t)(hi ? w >> 16 : w & 0xffffu)); }

// Nonzero when one of the two halves of w is an inf or NaN (exponent bits all ones: adding one carries into the sign).
__device__ __forceinline__ uint32_t nonfinite2(uint32_t w) { return ((w & 0x7c007c00u) + 0x04000400u) & 0x80008000u; }

template <int G, int T>
__global__ __launch_bounds__(T * 64, 4) void k_attn_mm(const float* __restrict__ q, const uint16_t* __restrict__ kc,
                                                   const uint16_t* __restrict__ vc, const int* __restrict__ lenp,
                                                   int len_add, int max_len, float scale, int tps, int kvh, int splits,
                                                   int ny, float* __restrict__ part) {
  constexpr int NR = (4 + T - 1) / T;  // quads of dims of a wave in the combine: w, w + T, ... of a lane's four
  __shared__ __align__(16) mm_f4 Pv[T][4][64];
  __shared__ __align__(16) float Qs[kMmUnits][68];  // rows 4 banks apart: a lane group's 16-byte reads do not collide
  __shared__ float Tm[T][16], Al[T][16], Ts[T][16];
  // the KV head is the fastest index: with 8 of them each XCD reads the rows of one head only
  const int g = blockIdx.x % kvh, s = blockIdx.x / kvh % splits, u0 = blockIdx.x / (kvh * splits) * kMmUnits;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, gq = lane >> 4;
  const int units = ny * G, u = u0 + i, uc = min(u, units - 1);
  const int y = uc / G, nh = kvh * G;
  const int y_lo = u0 / G, y_hi = min(units - 1, u0 + kMmUnits - 1) / G;
  const float NEG_INF = __int_as_float(0xff800000);
  const size_t head = (size_t)y * nh + g * G + uc % G;
  const int len0 = *lenp + len_add;  // length seen by position 0 of the step; position y sees len0 + y
  const int t0 = s * tps, t1 = min(t0 + tps, (len0 + y_hi + 63) / 64);
  if (t0 >= t1) return;  // no unit reaches this split
#pragma unroll
  for (int e = 0; e < (256 + T * 64 - 1) / (T * 64); e++) {  // the units' queries, 16 float4 each
    const int f = min((int)threadIdx.x + e * T * 64, 255), fu = min(u0 + f / 16, units - 1);
    *reinterpret_cast<float4*>(&Qs[f / 16][4 * (f & 15)]) =
        gload_f4(q + ((size_t)(fu / G) * nh + g * G + fu % G) * 64 + 4 * (f & 15));
  }
  float m = NEG_INF, l = 0.0f;
  mm_f4 acc[NR];
#pragma unroll
  for (int a = 0; a < NR; a++) acc[a] = mm_f4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int tr = t0; tr < t1; tr += T) {
    // a wave past the split's tiles goes through its last tile with no row valid and nothing of it is used: a branch
    // around the loads would keep their registers live through the whole loop (129 spilled at 128 registers)
    const int tw = tr + w, t = min(tw, t1 - 1);
    const int nv = tw < t1 ? len0 + y - t * 64 : 0;  // rows of the tile that the lane's unit sees (<= 0: none)
    float p[16];
    uint4 kr[8];
    uint2 vr[16];
    // this lane's K row, and its dims of every fourth V row
    const uint16_t* kp = kc + (((size_t)g * max_len + t * 64) + 16 * gq + 4 * (i & 3) + (i >> 2)) * 64;
    const uint16_t* vp = vc + (((size_t)g * max_len + t * 64) + gq) * 64 + 4 * i;
#pragma unroll
    for (int e = 0; e < 8; e++) kr[e] = gload_u4(kp + 8 * e);
    if (tr == t0) __syncthreads();  // queries
    mm_f16 sa = {};
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t wv[4] = {kr[e].x, kr[e].y, kr[e].z, kr[e].w};
      const float4 qa = *reinterpret_cast<const float4*>(&Qs[i][8 * e]);
      const float4 qb = *reinterpret_cast<const float4*>(&Qs[i][8 * e + 4]);
      const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
      for (int c = 0; c < 8; c++)
        sa = __builtin_amdgcn_mfma_f32_16x16x1f32(half_of(wv[c >> 1], c & 1), qv[c], sa, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);  // not all conversions first: they would not fit the registers
    }
    // V is requested once the K rows' registers are free, and arrives behind the exps
#pragma unroll
    for (int e = 0; e < 16; e++) vr[e] = gload_u2(vp + 4 * 64 * e);
    __builtin_amdgcn_sched_barrier(0);
    // lo, hi: rows of the tile that the first and the last position see; whole tiles are not masked
    const int lo = tw < t1 ? len0 + y_lo - t * 64 : 0, hi = len0 + y_hi - t * 64;
#pragma unroll
    for (int v = 0; v < 16; v++) p[v] = sa[v] * scale;
    if (lo < 64) {
#pragma unroll
      for (int v = 0; v < 16; v++) p[v] = 4 * v < nv - gq ? p[v] : NEG_INF;
    }
    float tm;
    {
      float x[8];
#pragma unroll
      for (int v = 0; v < 8; v++) x[v] = __builtin_fmaxf(p[v], p[v + 8]);
#pragma unroll
      for (int v = 0; v < 4; v++) x[v] = __builtin_fmaxf(x[v], x[v + 4]);
      tm = __builtin_fmaxf(__builtin_fmaxf(x[0], x[2]), __builtin_fmaxf(x[1], x[3]));
    }
    tm = max_stage<16>(tm);
    tm = max_stage<32>(tm);
    if constexpr (T > 1) {
      if (gq == 0) Tm[w][i] = tm;
      __syncthreads();  // tile maxima
    }
    float mprev = m;
    if constexpr (T > 1) {
#pragma unroll
      for (int v = 0; v < T - 1; v++)
        if (v < w) mprev = mprev > Tm[v][i] ? mprev : Tm[v][i];
    }
    const float mn = mprev > tm ? mprev : tm;
    const float alpha = dexp_neg(mprev - mn);
    float ts;
    mm_f4 pv[4];
#pragma unroll
    for (int v = 0; v < 16; v++) {
      p[v] = dexp_neg(p[v] - mn);
      if ((v & 3) == 3) __builtin_amdgcn_sched_barrier(0);  // four exps side by side
    }
    // the pairwise tree over the 64 positions: bits 0, 1 of a position are the lane group, bits 2, 3 the element
    // inside a block, bits 4, 5 the block
    float b[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
      float x[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        x[r] = p[4 * a + r] + partner<16>(p[4 * a + r]);
        x[r] = x[r] + partner<32>(x[r]);
      }
      b[a] = (x[0] + x[1]) + (x[2] + x[3]);
      __builtin_amdgcn_sched_barrier(0);
    }
    ts = (b[0] + b[1]) + (b[2] + b[3]);
    asm volatile("" : "+v"(ts));  // summed here: left until its use it would keep 12 partial sums through p.v
    // Rows past a unit's length have p = 0 and must not reach its sum. Rows that no unit sees enter as +0. A row
    // that only the later positions see stays (fma(0, v, c) is c for a finite v), unless it holds an inf or NaN:
    // then the tile is taken once per position, each with its own rows.
    bool apart = false;
    if (lo < 64) {
      uint32_t bad = 0u;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const uint32_t b2 = nonfinite2(vr[e].x) | nonfinite2(vr[e].y);
        bad |= 4 * e >= lo - gq && 4 * e < hi - gq ? b2 : 0u;
      }
      apart = __ballot(bad != 0u) != 0;
    }
    const int rows = (apart ? lo : hi) - gq;
    if (lo < 64) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const bool in = 4 * e < rows;
        vr[e].x = in ? vr[e].x : 0u;
        vr[e].y = in ? vr[e].y : 0u;
      }
    }
#pragma unroll
    for (int a = 0; a < 4; a++) pv[a] = mm_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < 16; e++) {
      pv[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(half_of(vr[e].x, 0), p[e], pv[0], 0, 0, 0);
      pv[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(half_of(vr[e].x, 1), p[e], pv[1], 0, 0, 0);
      pv[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(half_of(vr[e].y, 0), p[e], pv[2], 0, 0, 0);
      pv[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(half_of(vr[e].y, 1), p[e], pv[3], 0, 0, 0);
      if (e & 1) __builtin_amdgcn_sched_barrier(0);
    }
    if (apart) {
#pragma unroll
      for (int e = 0; e < 16; e++) vr[e] = gload_u2(vp + 4 * 64 * e);  // unmasked again
      for (int yy = y_lo + 1; yy <= y_hi; yy++) {
        const int rows_y = len0 + yy - t * 64 - gq;
#pragma unroll
        for (int a = 0; a < 4; a++) {  // one block of dims at a time: few registers
          mm_f4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int e = 0; e < 16; e++) {
            uint32_t x = 4 * e < rows_y ? (a < 2 ? vr[e].x : vr[e].y) : 0u;
            asm("" : "+v"(x));  // converted here: not shared with the first product, at 64 registers more
            o = __builtin_amdgcn_mfma_f32_16x16x4f32(half_of(x, a & 1), p[e], o, 0, 0, 0);
            if (e & 1) __builtin_amdgcn_sched_barrier(0);
          }
          pv[a] = y == yy ? o : pv[a];
        }
      }
    }
    // quad r of the lane: dims 16 gq + 4 r .. +3 of its unit, element r of the four dim blocks
    if constexpr (T == 1) {
      if (nv > 0) {
        l = __builtin_fmaf(l, alpha, ts);
        m = mn;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int a = 0; a < 4; a++) acc[r][a] = __builtin_fmaf(acc[r][a], alpha, pv[a][r]);
      }
    } else {
      if (gq == 0) {
        Al[w][i] = alpha;
        Ts[w][i] = ts;
      }
#pragma unroll
      for (int r = 0; r < 4; r++) Pv[w][r][lane] = mm_f4{pv[0][r], pv[1][r], pv[2][r], pv[3][r]};
      __syncthreads();  // p.v, alpha and sums of every tile of the round
#pragma unroll
      for (int v = 0; v < T; v++) {
        if (len0 + y - (tr + v) * 64 > 0 && tr + v < t1) {
          const float a1 = Al[v][i];
          l = __builtin_fmaf(l, a1, Ts[v][i]);
          m = m > Tm[v][i] ? m : Tm[v][i];
#pragma unroll
          for (int r = 0; r < NR; r++) {
            if (w + T * r < 4) {
              const mm_f4 x = Pv[v][w + T * r][lane];
#pragma unroll
              for (int a = 0; a < 4; a++) acc[r][a] = __builtin_fmaf(acc[r][a], a1, x[a]);
            }
          }
        }
      }
      if (tr + T < t1) __syncthreads();  // the round's entries are read
    }
  }
  if (u >= units || t0 * 64 >= len0 + y) return;
  float* pp = part + (head * splits + s) * 66;
  if (w == 0 && gq == 0) *reinterpret_cast<float2*>(pp) = make_float2(m, l);
  // 8-byte stores of consecutive dims (one dword at a time, 16 lines to a store, took 62 us where this takes 42: 300
  // positions after 1000, 3B shape, one tile per split)
  float2* po = reinterpret_cast<float2*>(pp + 2 + 16 * gq);
#pragma unroll
  for (int r = 0; r < NR; r++)
    if (w + T * r < 4) {
      po[2 * (w + T * r)] = make_float2(acc[r][0], acc[r][1]);
      po[2 * (w + T * r) + 1] = make_float2(acc[r][2], acc[r][3]);
    }
}

hipError_t launch_attn_mm(hipStream_t s, int G, int kvh, int tps, const float* q, const uint16_t* kc,
                          const uint16_t* vc, const int* lenp, int len_add, int max_len, float scale, int ny,
                          float* part) {
  const int splits = attn_splits_for(max_len, tps);
  if (splits > 64 || max_len % 64 || ny < 1) return hipErrorInvalidValue;
  const int grid = kvh * splits * ((ny * G + kMmUnits - 1) / kMmUnits), T = tps < 4 ? tps : 4;
#define MM_CASE(GG, TT)                                                                                             \
  if (G == GG && T == TT) {                                                                                         \
    klaunch(k_attn_mm<GG, TT>, grid, TT * 64, 0, s, q, kc, vc, lenp, len_add, max_len, scale, tps, kvh, splits, ny, \
            part);                                                                                                  \
    return hipGetLastError();                                                                                       \
  }
  MM_CASE(1, 1) MM_CASE(2, 1) MM_CASE(3, 1) MM_CASE(4, 1)
  MM_CASE(1, 2) MM_CASE(2, 2) MM_CASE(3, 2) MM_CASE(4, 2)
  MM_CASE(1, 3) MM_CASE(2, 3) MM_CASE(3, 3) MM_CASE(4, 3)
  MM_CASE(1, 4) MM_CASE(2, 4) MM_CASE(3, 4) MM_CASE(4, 4)
#undef MM_CASE
  return hipErrorInvalidValue;
}

}  // namespace moert
