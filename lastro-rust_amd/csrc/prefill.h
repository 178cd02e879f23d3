// Multi-position step of the whole model (prefill.hip): device buffers and launchers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "grouped.h"
#include "kernels.h"

namespace moert {

constexpr int kPfMaxPos = 32;  // positions of one step call (the reference's block limit, cuda_backend.rs:272-274)
// Positions per pass over the layers of a longer prompt. A pass reads every weight once, and its row products work on
// tiles of 16 or 32 positions per expert: more positions fill more of a tile and hide more of the reads. 512 tokens
// of the 3B shape, 4 layers: passes of 32 positions 7915 us, 128: 3015, 256: 2375, 512: 2000 (of which gate/up
// 4 x 183); the buffers of a pass grow with it (512 positions: 0.25 GB at 64 splits). Passes of 1024 were measured
// too: 1024 tokens 3182 us against 3507 in two of 512, 4096 tokens 14.4 ms against 15.7, with twice the buffers.
constexpr int kPfBlock = 512;
// Positions of a pass that goes through few.hip instead (its buffers hold kFewPos). A tile of 16 positions on the matrix
// cores costs the same for one as for 16; few.hip's time grows with the positions. A whole call, 16 layers, us, few.hip
// / tiles, at 0 cached positions:
//   Q8_0  1B  1: 664 / 859   4: 855 / 1017   8: 1065 / 1099   9: 1113 / 1103   16: 1422 / 1150
//         3B  1: 724 / 1052  4: 1053 / 1255  8: 1362 / 1368   9: 1454 / 1379   16: 1943 / 1505
//   Q4_0  1B  1: 660 / 812   4: 833 / 982    8: 1013 / 1055   9: 1063 / 1061
//         3B  1: 708 / 1042  4: 985 / 1235   8: 1284 / 1333   9: 1375 / 1335
//   f32   1B  1: 724 / 987   8: 1273 / 1463  14: 1575 / 1586  16: 1657 / 1593
//         3B  1: 843 / 1247  8: 1666 / 1983  14: 2098 / 2231  16: 2239 / 2326
// (f32 rows need no dequantisation, and the tiles read them in shorter steps; 4000 cached positions move no line.)
constexpr int kFewPos = 14;
constexpr int few_positions(int dtype) { return dtype == DT_F32 ? kFewPos : 8; }

// Device buffers of one multi-position step, sized for `cap` positions.
struct PfBufs {
  int cap;       // positions
  float* h;      // [m, H] residual streams
  float* q;      // [m, heads*d] queries
  float* att;    // [m, heads*d] attention outputs
  float* part;   // [m, heads, splits, 2 + d] split-KV partials
  float* xn;     // [m, H] normalised input: of the layer until q/k/v, of the experts from the router on
  float* w;      // [m, k] routing weights
  int* cnt;      // [64] members of each expert
  int* list;     // [64, cap] their slots: position * k + top-k rank
  float* act;    // [m, k, I] SwiGLU activations
  float* o;      // [m, k, H] expert outputs
  int* ids;      // [m, k] routed experts, top-k order (grouped mode, few positions)
  float* zpart;  // [kFewPos, kNormItems] MoE-norm partials of each position (few positions)
};

// Embedding rows of the nv tokens at `toks` (device) into h; the step state becomes position `last` and first free
// position last + 1.
hipError_t launch_embed_b(hipStream_t s, const DMat& emb, const Dims& d, const PfBufs& p, const int* toks, int nv,
                          int* state, int last);
// xn = rmsnorm(h, lnw) of every position: the first layer's input.
hipError_t launch_norm_b(hipStream_t s, const Dims& d, const PfBufs& p, int nv, const float* lnw);
// One layer for positions pos0 .. pos0 + nv - 1 (state[ST_POS] == pos0 + nv - 1 on the device), rope: the [max_len, 64] table; the
// decode kernels' chains, so that the results equal nv decode steps bit for bit. On entry xn = rmsnorm(h, L.ln_attn);
// with next_lnw the layer leaves rmsnorm(h, next_lnw) there for the next one. cus: the device's compute units.
hipError_t launch_layer_b(hipStream_t s, const LayerDev& L, const Dims& d, const PfBufs& p, const int* state, int pos0,
                          int nv, const float* rope, const float* next_lnw, int cus);
// The same layer for at most kFewPos positions (few.hip), which normalises its input h itself: nothing is expected in xn
// and nothing left there.
hipError_t launch_layer_few(hipStream_t s, const LayerDev& L, const Dims& d, const PfBufs& p, const int* state, int pos0,
                            int nv, const float* rope);
// The same layer in grouped mode: q/k/v, output projection and experts through the int8 MFMA kernels of grouped.h,
// g holding the layer's tiled matrices. On entry g's codes are those of rmsnorm(h, L.ln_attn) (launch_norm_codes or
// the previous layer's combine); with next_lnw the layer leaves the codes of rmsnorm(h, next_lnw) for the next one.
hipError_t launch_layer_grouped(hipStream_t s, const LayerDev& L, const Dims& d, const PfBufs& p, const int* state,
                                int pos0, int nv, const float* rope, const GroupBufs& g, const float* next_lnw);

}  // namespace moert
