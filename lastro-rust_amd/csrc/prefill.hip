// Multi-position step of the whole model: consecutive positions in one pass per layer (the block prefill `le_ids`,
// rust/moe-rt/src/motor/leitura.rs:79-85, through begin_step_tokens and the per-position loops of the model step,
// cuda_backend.rs:499-516, 751-917). Every weight row is read once per block of positions and applied to each
// position's activation with the decode kernels' per-row chain (chunk j of a row accumulated by lane j % 64 as an
// fmaf chain, then the pairwise lane tree), so the step equals single-position decode steps bit for bit: the KV rows
// it appends, every hidden state and the last position's logits.
//
// A step of few positions runs the kernels of few.hip instead.
//
// Kernels per layer (one stream, in order; xn holds the normalised input of the layer on entry):
//   k_qkv_x        [q; k; v] of every position, RoPE, q to qb[v], k and v to row pos0 + v of the KV cache
//   attention      attn_mm.hip over the positions, position v attending to pos0 + v + 1, and the decode combine
//   k_oproj_x      output projection, h[v] += res * (Wo att[v])
//   k_route_x      per position: the MoE norm and router in moe_norm.h's order, top-k and weights; xn[v] for the
//                  experts; the position enters its experts' member lists
//   k_moe_up_x     per expert and tile of its members: gate/up rows, SwiGLU into act[slot] (slot = v * k + rank)
//   k_moe_down_x   per expert and tile of its members: o[slot] = down . act[slot]
//   k_moe_comb_x   h[v] += res * sum over j in top-k order of w[v][j] * o[v][j], and the next layer's xn[v]
#include <algorithm>

#include "cache.h"
#include "dev_rows.h"
#include "grouped.h"
#include "launch.h"
#include "moe_norm.h"
#include "prefill.h"

namespace moert {

// ------------------------------------------------------------------------------------------------------------
// The row products on the f32 matrix cores. v_mfma_f32_16x16x1 is one fmaf on every element of four 16x16 blocks, so
// the chain of decode lane c of a row is a run of MFMAs over its elements in index order, block b of the instruction
// being lane 4G + b: A = element i of chunk 4G + b of 16 rows (a lane dequantises its row's chunk from one 16-byte
// load, as a decode lane does), B = element i of that chunk of 16 positions' activations. The pairwise lane tree then
// adds blocks (0 + 1) + (2 + 3) inside a lane, groups of four lanes after that.
//
// A workgroup holds MT x NT tiles of 16 rows x 16 positions. Its waves share the groups of four chains: wave w takes
// the runs of SUB adjacent groups w, w + KW, ... (so that the chunks past the row's 64th, which only the first groups
// have, spread over all waves), one tree node per run goes to LDS, and every thread adds the NN nodes of its outputs.
// Bound: instruction issue. f32 MFMAs (32 cycles for 1024 products, 127 TFLOP/s on 256 CUs) do not overlap with vector
// instructions, so that a row's dequantisation, two of them an element and row tile, counts in full and serves NT
// position tiles. 512 positions of the 3B shape: gate/up 183 us under the trace, 75 TFLOP/s, 77% of its issue bound; down 104, q/k/v
// 59, output projection 37. 32 positions: 31, 18.5, 10, 10 us, where one vector fma chain per lane with the activations
// in LDS took 60, 47, 32, 28. Measured and not taken, all within 3%: activations laid out so that a B load takes 64
// consecutive bytes per position, three waves to a SIMD without the register prefetch, K over two waves.
typedef float xg_f16 __attribute__((ext_vector_type(16)));

template <int DT, int K>
struct XGeo {
  using G = Geo<DT, K>;
  static constexpr int SE = G::CE < 16 ? G::CE : 16;  // elements of a step (Q4_0: two steps per chunk)
  static constexpr int HPC = G::CE / SE;              // steps per chunk
  static constexpr int NG = G::LPR / 4;               // groups of four chains
  static constexpr int KW = NG < 4 ? NG : 4;          // waves
  static constexpr int NT_ = KW * 64;                 // threads
  // Every wave of a round has the chunks 4G + b + LPR * jj of its run, or none has.
  static constexpr bool even(int sub) {
    for (int r = 0; r < NG / (KW * sub); r++)
      for (int jj = 0; jj < G::NJ; jj++) {
        const int lo = 4 * r * KW * sub + G::LPR * jj, hi = 4 * (r + 1) * KW * sub + G::LPR * jj;
        if (lo < G::NCH && hi > G::NCH) return false;
      }
    return true;
  }
  static constexpr int SUB = NG >= 2 * KW && even(2) ? 2 : 1;
  static constexpr int ROUNDS = NG / (KW * SUB);
  static constexpr int NN = NG / SUB;  // tree nodes of an output
  static_assert(even(SUB), "a round's waves must have the same chunks");
  static constexpr bool valid(int r, int jj) { return 4 * r * KW * SUB + G::LPR * jj < G::NCH; }
  struct Step {
    int r, u, jj, half;
  };
  static constexpr int steps() {
    int n = 0;
    for (int r = 0; r < ROUNDS; r++)
      for (int jj = 0; jj < G::NJ; jj++) n += valid(r, jj) ? SUB * HPC : 0;
    return n;
  }
  static constexpr int N = steps();
  static constexpr Step step(int s) {
    int n = 0;
    for (int r = 0; r < ROUNDS; r++)
      for (int u = 0; u < SUB; u++)
        for (int jj = 0; jj < G::NJ; jj++)
          for (int h = 0; h < HPC; h++)
            if (valid(r, jj) && n++ == s) return Step{r, u, jj, h};
    return Step{-1, -1, -1, -1};
  }
};

// Element i of a chunk whose payload words and scale are in registers: q * d, exact, as fma_chunk forms it.
template <int DT>
__device__ __forceinline__ float xg_elem(const uint4& v, float d, int i) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  if (DT == DT_Q8_0) return (float)(int8_t)(w[i >> 2] >> (8 * (i & 3))) * d;
  if (DT == DT_Q4_0) {
    const int b = i & 15;
    return (float)((int)((w[b >> 2] >> (8 * (b & 3) + (i >= 16 ? 4 : 0))) & 15u) - 8) * d;
  }
  return __uint_as_float(w[i]);
}

template <int DT, int K, int MT, int NT>
struct XgRegs {
  RawChunk a[2][MT];
  float4 b[2][NT][XGeo<DT, K>::SE / 4];
  xg_f16 acc[MT][NT];
  float node[MT][NT][4];
};

template <int DT, int K, int MT, int NT, int S>
__device__ __forceinline__ void xg_load(XgRegs<DT, K, MT, NT>& x, const DMat& m, const size_t (&row)[MT],
                                        const float* const (&xp)[NT], int w, int gq) {
  using X = XGeo<DT, K>;
  using G = Geo<DT, K>;
  constexpr typename X::Step st = X::step(S);
  const int j = 4 * ((st.r * X::KW + w) * X::SUB + st.u) + gq + G::LPR * st.jj;
  if constexpr (st.half == 0) {
#pragma unroll
    for (int t = 0; t < MT; t++) x.a[S / X::HPC & 1][t] = load_chunk<DT>(m, row[t], j);
  }
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int e = 0; e < X::SE / 4; e++) x.b[S & 1][t][e] = gload_f4(xp[t] + j * G::CE + st.half * X::SE + 4 * e);
}

template <int DT, int K, int MT, int NT, int S>
__device__ __forceinline__ void xg_steps(XgRegs<DT, K, MT, NT>& x, const DMat& m, const size_t (&row)[MT],
                                         const float* const (&xp)[NT], float* nodes, int lane, int w) {
  using X = XGeo<DT, K>;
  if constexpr (S < X::N) {
    constexpr typename X::Step st = X::step(S), nx = X::step(S + 1);
    constexpr bool first = st.jj == 0 && st.half == 0;                          // of its group
    constexpr bool last = S + 1 == X::N || nx.r != st.r || nx.u != st.u;        // of its group
    if constexpr (S + 1 < X::N) {
      xg_load<DT, K, MT, NT, S + 1>(x, m, row, xp, w, lane >> 4);
      __builtin_amdgcn_sched_barrier(0);  // the next step's loads ahead of this step's products
    }
    if constexpr (first) {
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) x.acc[t][n] = xg_f16{};
    }
    float d[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) d[t] = chunk_scale(x.a[S / X::HPC & 1][t]);
#pragma unroll
    for (int i = 0; i < X::SE; i++) {
      float av[MT];
#pragma unroll
      for (int t = 0; t < MT; t++) av[t] = xg_elem<DT>(x.a[S / X::HPC & 1][t].v, d[t], st.half * X::SE + i);
#pragma unroll
      for (int n = 0; n < NT; n++) {
        const float4 q = x.b[S & 1][n][i >> 2];
        const float bv = (i & 3) == 0 ? q.x : (i & 3) == 1 ? q.y : (i & 3) == 2 ? q.z : q.w;
#pragma unroll
        for (int t = 0; t < MT; t++)
          x.acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x1f32(av[t], bv, x.acc[t][n], 0, 0, 0);
      }
    }
    if constexpr (last) {
#pragma unroll
      for (int t = 0; t < MT; t++)
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const xg_f16& c = x.acc[t][n];
            const float f = (c[r] + c[4 + r]) + (c[8 + r] + c[12 + r]);
            x.node[t][n][r] = st.u == 0 ? f : x.node[t][n][r] + f;
            if (st.u == X::SUB - 1) nodes[(((st.r * X::KW + w) * MT + t) * NT + n) * 256 + 64 * r + lane] = x.node[t][n][r];
          }
    }
    xg_steps<DT, K, MT, NT, S + 1>(x, m, row, xp, nodes, lane, w);
  }
}

// The balanced pairwise tree over n nodes `stride` floats apart.
template <int N>
__device__ __forceinline__ float xg_tree(const float* p, int stride) {
  if constexpr (N == 1) {
    return p[0];
  } else {
    return xg_tree<N / 2>(p, stride) + xg_tree<N / 2>(p + N / 2 * stride, stride);
  }
}

// Floats of LDS for the nodes of MT x NT tiles.
template <int DT, int K, int MT, int NT>
__host__ __device__ constexpr int xg_lds() {
  return XGeo<DT, K>::NN * MT * NT * 256;
}

// MT x NT tiles: lane i = lane % 16 supplies rows row[t] (one of the 16 of tile t) and the activations at xp[n] (one
// of the 16 positions of tile n). done(n, r, v) is called for every output of this thread: v[t] is row 4 (lane / 16)
// + r of tile t against position lane % 16 of tile n.
template <int DT, int K, int MT, int NT, class F>
__device__ __forceinline__ void xg_run(const DMat& m, const size_t (&row)[MT], const float* const (&xp)[NT],
                                       float* nodes, int lane, int w, const F& done) {
  using X = XGeo<DT, K>;
  XgRegs<DT, K, MT, NT> x;
  xg_load<DT, K, MT, NT, 0>(x, m, row, xp, w, lane >> 4);
  xg_steps<DT, K, MT, NT, 0>(x, m, row, xp, nodes, lane, w);
  // runs without a chunk (a row that does not reach all 64 lanes) add +0
#pragma unroll
  for (int r = 0; r < X::ROUNDS; r++)
    if constexpr (!X::valid(X::ROUNDS - 1, 0)) {
      if (!X::valid(r, 0))
#pragma unroll
        for (int t = 0; t < MT * NT * 4; t++) nodes[(r * X::KW + w) * MT * NT * 256 + 64 * t + lane] = 0.0f;
    }
  __syncthreads();
  constexpr int RPT = NT * 4 / X::KW;  // outputs of a thread: (n, r) = its RPT consecutive of NT x 4
#pragma unroll
  for (int e = 0; e < RPT; e++) {
    const int it = w * RPT + e;
    float v[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) v[t] = xg_tree<X::NN>(nodes + t * NT * 256 + it * 64 + lane, MT * NT * 256);
    done(it >> 2, it & 3, v);
  }
}

// ------------------------------------------------------------------------------------------------------------
// [q; k; v] rows (j, j + 32) of a head (tile pair 16 a .. +16 and 32 + 16 a .. +16) for NT tiles of positions, RoPE,
// q and the KV rows (k_qkv's arithmetic per position). The first workgroup also empties the experts' member lists.
template <int DT, int K, int NT>
__global__ __launch_bounds__((XGeo<DT, K>::NT_), 2) void k_qkv_x(DMat m, const float* __restrict__ xn, int pos0, int nv,
                                                               const float* __restrict__ rope, int heads, int kvh,
                                                               int max_len, float* __restrict__ q,
                                                               uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
                                                               int* __restrict__ cnt) {
  __shared__ float nodes[xg_lds<DT, K, 2, NT>()];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15;
  const int head = blockIdx.x >> 1, a16 = 16 * (blockIdx.x & 1), p0 = blockIdx.y * 16 * NT;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 64) cnt[threadIdx.x] = 0;
  const size_t row[2] = {(size_t)head * 64 + a16 + i, (size_t)head * 64 + a16 + i + 32};
  const float* xp[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) xp[n] = xn + (size_t)min(p0 + 16 * n + i, nv - 1) * K;
  xg_run<DT, K, 2, NT>(m, row, xp, nodes, lane, w, [&](int n, int r, const float (&v)[2]) {
    const int p = p0 + 16 * n + i, jp = a16 + 4 * (lane >> 4) + r;
    if (p >= nv) return;
    const int pos = pos0 + p;
    const float x1 = v[0], x2 = v[1], c = rope[(size_t)pos * 64 + jp], sn = rope[(size_t)pos * 64 + 32 + jp];
    if (head < heads) {
      float* qv = q + ((size_t)p * heads + head) * 64;
      qv[jp] = x1 * c - x2 * sn;
      qv[jp + 32] = x2 * c + x1 * sn;
    } else if (head < heads + kvh) {
      uint16_t* kp = kc + ((size_t)(head - heads) * max_len + pos) * 64;
      kp[jp] = f2h(x1 * c - x2 * sn);
      kp[jp + 32] = f2h(x2 * c + x1 * sn);
    } else {
      uint16_t* vp = vc + ((size_t)(head - heads - kvh) * max_len + pos) * 64;
      vp[jp] = f2h(x1);
      vp[jp + 32] = f2h(x2);
    }
  });
}

// h[v][r] = h[v][r] + res * (Wo att[v])[r] for 32 rows and NT tiles of positions (k_oproj's arithmetic per position).
template <int DT, int K, int NT>
__global__ __launch_bounds__((XGeo<DT, K>::NT_), 2) void k_oproj_x(DMat m, const float* __restrict__ att, int nv,
                                                                 float res, float* __restrict__ h) {
  __shared__ float nodes[xg_lds<DT, K, 2, NT>()];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15;
  const int r0 = blockIdx.x * 32, p0 = blockIdx.y * 16 * NT, H = m.rows;
  const size_t row[2] = {(size_t)r0 + i, (size_t)r0 + 16 + i};
  const float* xp[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) xp[n] = att + (size_t)min(p0 + 16 * n + i, nv - 1) * K;
  xg_run<DT, K, 2, NT>(m, row, xp, nodes, lane, w, [&](int n, int r, const float (&v)[2]) {
    const int p = p0 + 16 * n + i;
    if (p >= nv) return;
    float* hv = h + (size_t)p * H + r0 + 4 * (lane >> 4) + r;
    const float h0 = hv[0], h1 = hv[16];
    hv[0] = h0 + res * v[0];
    hv[16] = h1 + res * v[1];
  });
}

// ------------------------------------------------------------------------------------------------------------
// Position v = blockIdx.x: the MoE norm and the router in moe_norm.h's order. A wave takes whole experts (the last
// item is the sum of squares): lane l forms the 8-column chains of blocks l, l + 64, .. itself and adds them in that
// order, so no partials pass through memory (8.8 us for 70 positions, 16.6 for 512, 3B shape; with the partials written
// by the output projection's epilogue the router took 4.8 us for 32 and the epilogue 8). Then ranks, ids and weights in top-k order (the decode router), xn for
// the experts, and slot v * k + rank into the member list of each expert chosen (the order of a list does not enter
// any result: every member is a column of its own).
// 16 waves, 8 for f32 rows (whose registers would not fit 16), as k_route_up
__host__ __device__ constexpr int route_x_waves(int dt) { return dt == DT_F32 ? 8 : 16; }

template <int DT, int K>
__global__ __launch_bounds__(route_x_waves(DT) * 64) void k_route_x(DMat router, const float* __restrict__ bias,
                                                                  const float* __restrict__ h,
                                                                  const float* __restrict__ lnw, float eps, int k,
                                                                  int cap, float* __restrict__ xn,
                                                                  float* __restrict__ wts, int* __restrict__ cnt,
                                                                  int* __restrict__ list) {
  constexpr int NW = route_x_waves(DT), NT = NW * 64;
  constexpr int NB = K / kNormBlk, NQ = (NB + 63) / 64;  // column blocks, and those of a lane
  constexpr int IPW = (65 + NW - 1) / NW;                // items of a wave
  constexpr int XP = (K + NT - 1) / NT;                  // elements of xn per thread
  __shared__ __align__(16) float lg[64];
  __shared__ int part[NW][64];
  __shared__ float rs;
  __shared__ int sid[8];
  const int v = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int E = router.rows;
  const float* hv = h + (size_t)v * K;
  float hb[NQ][8], ub[NQ][8];
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int c0 = kNormBlk * min(lane + 64 * q, NB - 1);
    const float4 a = gload_f4(hv + c0), b = gload_f4(hv + c0 + 4), la = gload_f4(lnw + c0), lb = gload_f4(lnw + c0 + 4);
    const float ha[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}, lw[8] = {la.x, la.y, la.z, la.w, lb.x, lb.y, lb.z, lb.w};
#pragma unroll
    for (int t = 0; t < 8; t++) {
      hb[q][t] = ha[t];
      ub[q][t] = lw[t] * ha[t];
    }
  }
  // item E (the sum of squares) is wave 0's first, so that r is known when the experts' sums are
  float z[IPW];
#pragma unroll
  for (int it = 0; it < IPW; it++) {
    const int item = wave + NW * it, e = item == 0 ? E : item - 1;
    float acc = 0.0f;
    if (e < E) {
      Col8 c[NQ];
#pragma unroll
      for (int q = 0; q < NQ; q++) c[q] = load_col8<DT>(router, e, kNormBlk * min(lane + 64 * q, NB - 1));
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        const int c0 = kNormBlk * min(lane + 64 * q, NB - 1);
        float a = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; t++) a = __builtin_fmaf(col8_elem<DT>(c[q], t, c0), ub[q][t], a);
        if (lane + 64 * q < NB) acc = acc + a;
      }
    } else if (item == 0) {
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        float a = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; t++) a = __builtin_fmaf(hb[q][t], hb[q][t], a);
        if (lane + 64 * q < NB) acc = acc + a;
      }
    }
    z[it] = group_sum<64>(acc);
  }
  if (threadIdx.x == 0) rs = 1.0f / sqrtf(z[0] / (float)K + eps);
  __syncthreads();
  const float r = rs;
#pragma unroll
  for (int it = 0; it < IPW; it++) {
    const int item = wave + NW * it, e = item - 1;
    if (item > 0 && e < E && lane == 0) lg[e] = bias ? z[it] * r + bias[e] : z[it] * r;
  }
#pragma unroll
  for (int e = 0; e < XP; e++) {
    const int i = threadIdx.x + e * NT;
    if (i < K) xn[(size_t)v * K + i] = lnw[i] * (hv[i] * r);
  }
  __syncthreads();
  int eid[8];
  const int rank = wg_rank<NW>(lg, E, lane, wave, part);
  const bool sel = lane < E && rank < k;
  ids_by_rank(sel, rank, k, eid);
  if (wave == 0) {
    route_weights(lg, sel, rank, k, lane, eid, sid, wts + (size_t)v * k);
    if (sel) list[(size_t)lane * cap + atomicAdd(&cnt[lane], 1)] = v * k + rank;
  }
}

// ------------------------------------------------------------------------------------------------------------
// Gate/up rows (16 of each) of one expert for a tile of its members: act[slot][r] = silu(gate_r . xn) * (up_r . xn)
// (k_route_up's expert arithmetic per position). A last tile of at most 16 members runs as one position tile.
template <int DT, int K, int NT>
__global__ __launch_bounds__((XGeo<DT, K>::NT_), 2) void k_moe_up_x(DMat gu, const float* __restrict__ xn,
                                                                  const int* __restrict__ cnt,
                                                                  const int* __restrict__ list, int cap, int k,
                                                                  int inter, float* __restrict__ act) {
  __shared__ float nodes[xg_lds<DT, K, 2, NT>()];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15;
  int first = 0, members = 0;
  const int e = member_tile<16 * NT>(cnt, blockIdx.y, lane, &first, &members);
  if (e < 0) return;
  const int r0 = blockIdx.x * 16;
  const size_t row[2] = {(size_t)e * 2 * inter + r0 + i, (size_t)e * 2 * inter + inter + r0 + i};
  const float* xp[NT];
  int slot[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) {
    slot[n] = list[(size_t)e * cap + min(first + 16 * n + i, members - 1)];
    xp[n] = xn + (size_t)(slot[n] / k) * K;
  }
  auto done = [&](int n, int r, const float (&v)[2]) {
    if (first + 16 * n + i >= members) return;
    const int sl = NT == 1 || n == 0 ? slot[0] : slot[NT - 1];
    act[(size_t)sl * inter + r0 + 4 * (lane >> 4) + r] = silu_mul(v[0], v[1]);
  };
  if (NT == 2 && first + 16 >= members) {
    const float* const x1[1] = {xp[0]};
    xg_run<DT, K, 2, 1>(gu, row, x1, nodes, lane, w, done);
  } else {
    xg_run<DT, K, 2, NT>(gu, row, xp, nodes, lane, w, done);
  }
}

// 32 down rows of one expert for a tile of its members: o[slot][r] = down_r . act[slot] (k_expert_down's dot).
template <int DT, int K, int NT>
__global__ __launch_bounds__((XGeo<DT, K>::NT_), 2) void k_moe_down_x(DMat dn, const float* __restrict__ act,
                                                                    const int* __restrict__ cnt,
                                                                    const int* __restrict__ list, int cap, int hidden,
                                                                    float* __restrict__ o) {
  __shared__ float nodes[xg_lds<DT, K, 2, NT>()];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lane & 15;
  int first = 0, members = 0;
  const int e = member_tile<16 * NT>(cnt, blockIdx.y, lane, &first, &members);
  if (e < 0) return;
  const int r0 = blockIdx.x * 32;
  const size_t row[2] = {(size_t)e * hidden + r0 + i, (size_t)e * hidden + r0 + 16 + i};
  const float* xp[NT];
  int slot[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) {
    slot[n] = list[(size_t)e * cap + min(first + 16 * n + i, members - 1)];
    xp[n] = act + (size_t)slot[n] * K;
  }
  auto done = [&](int n, int r, const float (&v)[2]) {
    if (first + 16 * n + i >= members) return;
    const int sl = NT == 1 || n == 0 ? slot[0] : slot[NT - 1];
    float* ov = o + (size_t)sl * hidden + r0 + 4 * (lane >> 4) + r;
    ov[0] = v[0];
    ov[16] = v[1];
  };
  if (NT == 2 && first + 16 >= members) {
    const float* const x1[1] = {xp[0]};
    xg_run<DT, K, 2, 1>(dn, row, x1, nodes, lane, w, done);
  } else {
    xg_run<DT, K, 2, NT>(dn, row, xp, nodes, lane, w, done);
  }
}

// ------------------------------------------------------------------------------------------------------------
// Position blockIdx.x: h[r] = h[r] + res * y, y = sum over j = 0 .. k-1 in order of w[j] * o[j][r] (k_expert_down's
// combine; k = 0: h stays), then with lnw the next layer's input xn = lnw * (h * rms scale) in the canonical order: one
// pass over h where the q/k/v kernel normalised every position in every workgroup. Bound: latency (7 us for 70 positions,
// 8.8 for 512: 27 MB of expert outputs at 3 TB/s).
template <int K>
__global__ __launch_bounds__(256) void k_moe_comb_x(const float* __restrict__ o, const float* __restrict__ wts, int k,
                                                    float res, float* __restrict__ h, const float* __restrict__ lnw,
                                                    float eps, float* __restrict__ xn) {
  constexpr int Q = K / 4, PER = (Q + 255) / 256;
  __shared__ __align__(16) float hs[K];
  __shared__ float rs;
  const int v = blockIdx.x;
  float4* hv = reinterpret_cast<float4*>(h + (size_t)v * K);
  float4 hq[PER];
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const int q = threadIdx.x + 256 * e, qc = min(q, Q - 1);
    float4 t = hv[qc];
    if (k > 0) {
      float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      for (int j = 0; j < k; j++) {
        const float wj = wts[v * k + j];
        const float4 x = reinterpret_cast<const float4*>(o + ((size_t)v * k + j) * K)[qc];
        y.x = y.x + wj * x.x;
        y.y = y.y + wj * x.y;
        y.z = y.z + wj * x.z;
        y.w = y.w + wj * x.w;
      }
      t.x = t.x + res * y.x;
      t.y = t.y + res * y.y;
      t.z = t.z + res * y.z;
      t.w = t.w + res * y.w;
      if (q < Q) hv[q] = t;
    }
    hq[e] = t;
    if (q < Q) reinterpret_cast<float4*>(hs)[q] = t;
  }
  if (!lnw) return;
  __syncthreads();
  if (threadIdx.x < 64) {
    const float r = rms_scale<K>(hs, eps, threadIdx.x);
    if (threadIdx.x == 0) rs = r;
  }
  __syncthreads();
  const float r = rs;
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const int q = threadIdx.x + 256 * e;
    if (q >= Q) continue;
    const float4 lw = reinterpret_cast<const float4*>(lnw)[q], t = hq[e];
    reinterpret_cast<float4*>(xn + (size_t)v * K)[q] =
        make_float4(lw.x * (t.x * r), lw.y * (t.y * r), lw.z * (t.z * r), lw.w * (t.w * r));
  }
}

// Embedding rows of the nv tokens (k_embed per position).
template <int DT>
__global__ __launch_bounds__(256) void k_embed_b(DMat e, const int* __restrict__ toks, float mult,
                                                 float* __restrict__ h, int* __restrict__ state, int last) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    state[ST_POS] = last;
    state[ST_FIXED] = last + 1;
  }
  const int v = blockIdx.y, tok = toks[v];
  const int H = e.cols;
  float* hv = h + (size_t)v * H;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < H; i += gridDim.x * 256) {
    float x;
    if (DT == DT_Q8_0) {
      x = (float)(int8_t)e.q[(size_t)tok * H + i] * h2f(e.d[(size_t)tok * (H / 32) + i / 32]);
    } else if (DT == DT_Q4_0) {
      const int b = i / 32, w = i % 32;
      const uint8_t byte = e.q[(size_t)tok * (H / 2) + b * 16 + (w & 15)];
      x = (float)((int)(w < 16 ? (byte & 15) : (byte >> 4)) - 8) * h2f(e.d[(size_t)tok * (H / 32) + b]);
    } else {
      x = reinterpret_cast<const float*>(e.q)[(size_t)tok * H + i];
    }
    hv[i] = x * mult;
  }
}

// ------------------------------------------------------------------------------------------------------------
// Launchers.
static inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

hipError_t launch_embed_b(hipStream_t s, const DMat& emb, const Dims& d, const PfBufs& p, const int* toks, int nv,
                          int* state, int last) {
  const dim3 grid((d.hidden + 255) / 256, nv);
  switch (emb.dtype) {
    case DT_Q8_0: klaunch(k_embed_b<DT_Q8_0>, grid, 256, 0, s, emb, toks, d.emb_mult, p.h, state, last); break;
    case DT_Q4_0: klaunch(k_embed_b<DT_Q4_0>, grid, 256, 0, s, emb, toks, d.emb_mult, p.h, state, last); break;
    case DT_F32: klaunch(k_embed_b<DT_F32>, grid, 256, 0, s, emb, toks, d.emb_mult, p.h, state, last); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// One or two position tiles per workgroup of the dense products: two share a row's reads and dequantisation, one makes
// twice the workgroups. With c workgroups on the fullest of the device's `cus` compute units one tile takes about 10.4 +
// 5.65 (c - 1) us and two 14.4 + 9.6 (c - 1) (rows of 1536): two where 17 c2 < 10 c1. One / two, Q8_0, 256 compute units:
//   3B q/k/v  48 10.5 / 14.2   64 15.8 / 14.2  128 21.5 / 23.2  192 27.4 / 23.9  256 33.2 / 32.6  512 60.6 / 52.1
//      output 64 9.8 / 13.0   128 15.3 / 12.9  256 21.2 / 22.1  512 38.4 / 32.6
//   1B q/k/v  64 7.8 / 10.9   128 11.1 / 10.6  192 15.5 / 17.4  256 19.6 / 18.0  384 27.4 / 25.9  512 35.0 / 31.7
//      output 128 7.4 / 9.7   192 11.0 / 9.9   256 11.1 / 10.0  384 15.2 / 17.0  512 19.2 / 17.1
// It takes the faster one at each of these but 3B q/k/v at 256, where the two are 2% apart.
static bool two_tiles(int row_groups, int nv, int cus) {
  const int c1 = cdiv((long)row_groups * cdiv(nv, 16), cus), c2 = cdiv((long)row_groups * cdiv(nv, 32), cus);
  return 17 * c2 < 10 * c1;
}

static hipError_t comb_dispatch(hipStream_t s, const Dims& d, const PfBufs& p, int nv, int k, const float* lnw) {
#define COMB(KK)                                                                                                 \
  case KK: klaunch(k_moe_comb_x<KK>, nv, 256, 0, s, p.o, p.w, k, d.res_mult, p.h, lnw, d.eps, p.xn); break;
  switch (d.hidden) {
    MOERT_K_CASES(COMB)
    default: return hipErrorInvalidValue;
  }
#undef COMB
  return hipGetLastError();
}

hipError_t launch_norm_b(hipStream_t s, const Dims& d, const PfBufs& p, int nv, const float* lnw) {
  return comb_dispatch(s, d, p, nv, 0, lnw);
}

hipError_t launch_layer_b(hipStream_t s, const LayerDev& L, const Dims& d, const PfBufs& p, const int* state, int pos0,
                          int nv, const float* rope, const float* next_lnw, int cus) {
  if (nv < 1 || nv > p.cap || cus < 1 || d.top_k > 8 || d.experts > 64 || d.head_dim != 64) return hipErrorInvalidValue;
  if (L.qkv.rows != (d.heads + 2 * d.kv_heads) * 64 || d.hidden % 32 || d.inter % 16) return hipErrorInvalidValue;
#define QKV(KK, NN)                                                                                                 \
  klaunch(k_qkv_x<DTC, KK, NN>, dim3(L.qkv.rows / 32, cdiv(nv, 16 * NN)), XGeo<DTC, KK>::NT_, 0, s, L.qkv, p.xn, pos0, \
          nv, rope, d.heads, d.kv_heads, d.max_len, p.q, L.k_cache, L.v_cache, p.cnt)
#define BODY(KK)                                        \
  case KK: {                                            \
    if (two_tiles(L.qkv.rows / 32, nv, cus)) QKV(KK, 2);     \
    else QKV(KK, 1);                                    \
  } break;
  MOERT_DISPATCH(L.qkv.dtype, L.qkv.cols, BODY)
#undef BODY
#undef QKV
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // position v attends to pos0 + v + 1 positions: the length is counted from the last position on the device
  if ((e = launch_attn_batched(s, L, d, state + ST_POS, 2 - nv, nv, p.q, p.part, p.att)) != hipSuccess) return e;
#define OPROJ(KK, NN)                                                                                              \
  klaunch(k_oproj_x<DTC, KK, NN>, dim3(L.o.rows / 32, cdiv(nv, 16 * NN)), XGeo<DTC, KK>::NT_, 0, s, L.o, p.att, nv, \
          d.res_mult, p.h)
#define BODY(KK)                                        \
  case KK: {                                            \
    if (two_tiles(L.o.rows / 32, nv, cus)) OPROJ(KK, 2);     \
    else OPROJ(KK, 1);                                  \
  } break;
  MOERT_DISPATCH(L.o.dtype, L.o.cols, BODY)
#undef BODY
#undef OPROJ
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (L.router.dtype != L.gate_up.dtype || L.router.cols != L.gate_up.cols) return hipErrorInvalidValue;
#define BODY(KK)                                                                                                    \
  case KK: {                                                                                                        \
    klaunch(k_route_x<DTC, KK>, nv, route_x_waves(DTC) * 64, 0, s, L.router, L.router_bias, p.h, L.ln_moe, d.eps,   \
            d.top_k, p.cap, p.xn, p.w, p.cnt, p.list);                                                              \
  } break;
  MOERT_DISPATCH(L.router.dtype, L.router.cols, BODY)
#undef BODY
  if ((e = hipGetLastError()) != hipSuccess) return e;
  // One position tile per workgroup while an expert has at most 16 members on average (gate/up with one / two, uniform
  // tokens: 3B 64 positions, 13 members, 39.0 / 42.6 us; 96, 19 members, 51.9 / 50.6; 512 187 / 163. 1B 64, 16 members,
  // 27.8 / 29.6; 96 34.8 / 32.7; 128 40.9 / 41.5; 512 126 / 115). The tiles of all experts are
  // at most the members' over a tile and one more per expert used; a workgroup past the last ends at once.
  const bool two = (long)nv * d.top_k > 16L * d.experts;
  const int slots = nv * d.top_k, tiles = slots / (two ? 32 : 16) + std::min(slots, d.experts);
#define UP(KK, NN)                                                                                                 \
  klaunch(k_moe_up_x<DTC, KK, NN>, dim3(d.inter / 16, tiles), XGeo<DTC, KK>::NT_, 0, s, L.gate_up, p.xn, p.cnt, p.list, \
          p.cap, d.top_k, d.inter, p.act)
#define BODY(KK)               \
  case KK: {                   \
    if (two) UP(KK, 2);        \
    else UP(KK, 1);            \
  } break;
  MOERT_DISPATCH(L.gate_up.dtype, L.gate_up.cols, BODY)
#undef BODY
#undef UP
  if ((e = hipGetLastError()) != hipSuccess) return e;
#define DOWN(KK, NN)                                                                                              \
  klaunch(k_moe_down_x<DTC, KK, NN>, dim3(d.hidden / 32, tiles), XGeo<DTC, KK>::NT_, 0, s, L.down, p.act, p.cnt, p.list, \
          p.cap, d.hidden, p.o)
#define BODY(KK)               \
  case KK: {                   \
    if (two) DOWN(KK, 2);      \
    else DOWN(KK, 1);          \
  } break;
  switch (L.down.dtype) {
    case DT_Q8_0: {
      constexpr int DTC = DT_Q8_0;
      switch (L.down.cols) { MOERT_KDOWN_CASES(BODY) default: return hipErrorInvalidValue; }
    } break;
    case DT_Q4_0: {
      constexpr int DTC = DT_Q4_0;
      switch (L.down.cols) { MOERT_KDOWN_CASES(BODY) default: return hipErrorInvalidValue; }
    } break;
    case DT_F32: {
      constexpr int DTC = DT_F32;
      switch (L.down.cols) { MOERT_KDOWN_CASES(BODY) default: return hipErrorInvalidValue; }
    } break;
    default: return hipErrorInvalidValue;
  }
#undef BODY
#undef DOWN
  if ((e = hipGetLastError()) != hipSuccess) return e;
  return comb_dispatch(s, d, p, nv, d.top_k, next_lnw);
}

hipError_t launch_layer_grouped(hipStream_t s, const LayerDev& L, const Dims& d, const PfBufs& p, const int* state,
                                int pos0, int nv, const float* rope, const GroupBufs& g, const float* next_lnw) {
  if (nv < 1 || nv > p.cap || nv > g.cap || d.top_k > 8 || d.experts > 64 || d.head_dim != 64) return hipErrorInvalidValue;
  GroupBufs gg = g;
  gg.ids = p.ids;
  gg.w = p.w;
  hipError_t e;
  if ((e = launch_gd_qkv(s, d, nv, pos0, rope, p.q, L.k_cache, L.v_cache, gg)) != hipSuccess) return e;
  // position v attends to pos0 + v + 1 positions: the length is counted from the last position on the device
  if ((e = launch_attn_batched(s, L, d, state + ST_POS, 2 - nv, nv, p.q, p.part, p.att)) != hipSuccess) return e;
  if ((e = launch_grp_codes(s, d.heads * 64, nv, p.att, gg)) != hipSuccess) return e;
  if ((e = launch_gd_oproj(s, nv, d.res_mult, p.h, gg)) != hipSuccess) return e;
  if ((e = launch_grp_route_norm(s, L, nv, d.top_k, p.h, L.ln_moe, d.eps, gg)) != hipSuccess) return e;
  if ((e = launch_grp_experts(s, d.hidden, d.experts, nv, d.top_k, d.inter, gg)) != hipSuccess) return e;
  return launch_gd_combine(s, d.hidden, nv, d.top_k, d.res_mult, p.h, next_lnw, d.eps, gg);
}

}  // namespace moert
