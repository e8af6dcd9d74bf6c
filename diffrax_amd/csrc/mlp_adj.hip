// mlp_adj.hip -- discrete adjoint of the neural-ODE solve (erk_mlp.hip): gradients of a
// loss on the saved states with respect to y0 and all MLP weights and biases.
//
// Semantics (RecursiveCheckpointAdjoint, _adjoint.py:264-312): reverse mode through the
// accepted step sequence with the step sizes held fixed -- the controller's factor is
// stop_gradient (_step_size_controller/pid.py:498-530) and rejected steps leave y and the
// FSAL state unchanged (_integrate.py:422-426), so they carry no gradient.  The forward
// pass (gradient mode) recorded the accepted (t_n, t_{n+1}) and the state at every C-th
// accepted step.  The backward walks segments of C steps from the last one; for each
// segment and each tile of 32 trajectories this kernel
//   1. recomputes the segment forward from its checkpoint (the three-piece form's
//      arithmetic), keeping every stage's f(z_i) in scratch and its layer inputs
//      (z_i, h1, h2) in blocked row buffers;
//   2. runs the exact reverse sweep: cotangents of the SaveAt(ts) values enter through the
//      Tsit5 interpolant (k_i gets b_i(theta) ybar_s), the SSAL output y_{n+1} = z_6, and
//      each stage k_i = dt f(z_i) is pulled back through the MLP on MFMA
//      (tanh' = 1 - f^2 from the kept f, softplus' = 1 - exp(-h) from the kept h), with no
//      forward re-evaluation;
//   3. stages the deltas of every stage in blocked row buffers beside the layer inputs.
// A split-K MFMA GEMM then forms dW_l = sum_rows delta_l^T input_l for the segment, and a
// fixed-order reduction adds it to the float32 accumulators (deterministic result).
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>
#include <type_traits>

#include "../../include/diffrax_amd.h"
#include "erk_small.hpp"
#include "mlp_tile.hpp"

namespace dfx {

// Six row buffers: D1 (width 256), Z (64), D2 (256), H1 (256), D3 (64), H2 (256).
constexpr int kRowWidths[6] = {MLP_H, MLP_D, MLP_H, MLP_H, MLP_D, MLP_H};
constexpr int kRowFloats = 4 * MLP_H + 2 * MLP_D;

struct RowBufs {  // float32 blocks of 32 rows, in the order of rows_frag
  float* b[6];
};

struct AdjArgs {
  const double* grid;
  const float* ckpt;
  const int32_t* stats;
  const double* ts;
  const float* ys_bar;
  float* ybar;
  float* zs;
  int32_t* evals;  // out [tiles]: evaluations (row blocks) of each tile, negative where some
                   // value is outside the range of its three-piece products (SplitRange)
  const int32_t* wflags;  // float32 form: nonzero where a weight or bias is outside
                          // (kWeightFlags), and marked tiles are left to the float32 kernel;
                          // else null
  int64_t B, ts_stride;
  int32_t max_steps, n_ckpt, C, Cs, seg, n_ts, n_out, save_t0;
  double t0, t1;
};

// The float32 form's LDS: the forward's with partials of their own (h1 is read again after
// layer 3) and the deltas of layers 3 and 2.
struct MlpLdsBack : MlpLds<PolicyF32> {
  float d[MLP_TILE * LDH];
  float d3[MLP_TILE * LDX];
  float part_[4 * MLP_TILE * LDP];
  __device__ __forceinline__ float* part() { return part_; }
};
static_assert(sizeof(MlpLdsBack) <= 160 * 1024, "one workgroup per CU");

// The tile's rows of an LDS buffer (columns at PolicyF32::pos) to a block of a row buffer, and
// back.
template <int Wd>
__device__ __forceinline__ void rows_out(const float* lds, int ld, float* dst, int64_t block) {
  for (int e = threadIdx.x; e < MLP_TILE * Wd / 4; e += blockDim.x) {
    const int l = e & 63, i = (e >> 6) & 3, t = e >> 8;
    const float* p = lds + (8 * i + 4 * (l >> 5)) * ld + PolicyF32::pos(32 * t + (l & 31));
    *reinterpret_cast<float4*>(dst + rows_frag(block, Wd, t, i, l)) =
        make_float4(p[0], p[ld], p[2 * ld], p[3 * ld]);
  }
}
template <int Wd>
__device__ __forceinline__ void rows_in(float* lds, int ld, const float* src, int64_t block) {
  for (int e = threadIdx.x; e < MLP_TILE * Wd / 4; e += blockDim.x) {
    const int l = e & 63, i = (e >> 6) & 3, t = e >> 8;
    float* p = lds + (8 * i + 4 * (l >> 5)) * ld + PolicyF32::pos(32 * t + (l & 31));
    const float4 v = *reinterpret_cast<const float4*>(src + rows_frag(block, Wd, t, i, l));
    p[0] = v.x; p[ld] = v.y; p[2 * ld] = v.z; p[3 * ld] = v.w;
  }
}

// The vector-Jacobian product of one evaluation on float32 MFMA: from delta3 (L.d3) and the
// activations (L.h1, L.h2), just stored, to the owners' zb; the deltas to their row block.
// Leaves delta1 in L.h2.
template <int NW>
__device__ __forceinline__ void pull_back_f32(const MlpWeights<PolicyF32>& W, MlpLdsBack& L,
                                              const RowBufs& R, int64_t block, int wave, int lane,
                                              int orow, int c0, float (&zb)[MlpWaves<NW>::CPT]) {
  using P = PolicyF32;
  using WV = MlpWaves<NW>;
  constexpr int NT = WV::NT12, NT3 = WV::NT3, F1 = MLP_D / P::KSTEP, F2 = MLP_H / P::KSTEP;
  const int half = lane >> 5, row = lane & 31;
  // delta = acc softplus'(h) of the layer whose activations h are given, into dst
  auto put_delta = [&](const floatx16_t (&acc)[NT], const float* hbuf, float* dst) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int o = row * L.LDH + P::pos(32 * (NT * wave + t) + 8 * i + 4 * half);
        const float2 he = *reinterpret_cast<const float2*>(hbuf + o);
        const float2 ho = *reinterpret_cast<const float2*>(hbuf + o + 4);
        *reinterpret_cast<float2*>(dst + o) =
            make_float2(acc[t][4 * i] * dsoftplus_from_value(he.x),
                        acc[t][4 * i + 2] * dsoftplus_from_value(he.y));
        *reinterpret_cast<float2*>(dst + o + 4) =
            make_float2(acc[t][4 * i + 1] * dsoftplus_from_value(ho.x),
                        acc[t][4 * i + 3] * dsoftplus_from_value(ho.y));
      }
    }
  };
  __syncthreads();
  rows_out<MLP_D>(L.d3, L.LDX, R.b[4], block);
  // delta2 = (delta3 . W3) softplus'(h2)
  floatx16_t acc[NT];
  GemmF32<F1, NT> g3t;
  g3t.preload(W.w3t, NT * wave, 0, lane);
  g3t.template run<F1>(L.d3, L.LDX, 0, acc, lane);
  put_delta(acc, L.h2, L.d);
  __syncthreads();
  // delta1 = (delta2 . W2) softplus'(h1), into the h2 buffer (h2 is in its row buffer)
  GemmF32<F2, NT> g2t;
  g2t.preload(W.w2t, NT * wave, 0, lane);
  g2t.template run<F2>(L.d, L.LDH, 0, acc, lane);
  put_delta(acc, L.h1, L.h2);
  __syncthreads();
  rows_out<MLP_H>(L.d, L.LDH, R.b[2], block);
  rows_out<MLP_H>(L.h2, L.LDH, R.b[0], block);
  // zb = delta1 . W1 (split-K over the 256 hidden units)
  const int qk = WV::quarter(wave), n3 = WV::nt3(wave);
  floatx16_t acc3[NT3];
  GemmF32<F2, NT3> g1t;
  g1t.preload(W.w1t, n3, qk * (F2 / 4), lane);
  g1t.template run<F2 / 4>(L.h2, L.LDH, qk * (F2 / 4), acc3, lane);
  float* part = L.part();
  put_partials<NT3>(acc3, part, L.LDP, qk, n3, lane);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < WV::CPT; ++j) {
    const int c = c0 + j;
    float sv = part[(0 * MLP_TILE + orow) * L.LDP + c];
    sv += part[(1 * MLP_TILE + orow) * L.LDP + c];
    sv += part[(2 * MLP_TILE + orow) * L.LDP + c];
    sv += part[(3 * MLP_TILE + orow) * L.LDP + c];
    zb[j] = sv;
  }
}

// ---- recompute and reverse sweep of one segment ---------------------------------------------
// P = PolicyBF16x3: every product runs on the six-pass three-piece MFMA (Gemm3) for both matmul
// forms: the deltas are split like the activations, so the gradients are those of the
// float32-weight model that both forwards evaluate, and the six bf16 passes take 3/8 of
// the MFMA time of one float32 pass.  Float32 MFMA throughout took 1.97 ms for the
// float32 form's segment of 8,192 trajectories and 4 steps.
// P = PolicyF32, launched behind it by the float32 form: the tiles that the first pass marked,
// because some weight, layer input or delta of theirs is outside the pieces' range
// (SplitRange), from their start again on float32 MFMA; every other workgroup ends at once.
// The first pass looks at what enters a product from outside (weights, biases, states, delta3)
// and at what a pull-back gives, zb.  Their limits bound all the rest:
//   above: h1 <= 64 2^10 2^24 = 2^40, h2 <= 256 2^10 2^40 = 2^58, delta2 <= 64 2^10 2^50 =
//     2^66, delta1 <= 256 2^10 2^66 = 2^84, zb <= 2^102, and 4,096 rows of dW <= 2^120 (biases
//     add little);
//   below: a delta's pieces are off by 2^-134 at most, so a sum for delta1 by 256 2^10 2^-134 =
//     2^-116 and one for zb by 2^-98, a quarter of 2^-24 of the least zb that passes.
// Looking at every delta instead took 15 of 700 us; this is within the launch's spread (8,192
// trajectories 709 us, without any test 721; 3,001 537 and 537).  In the bf16 form, which
// evaluates in pieces anyway, nothing reads the marks.
// The row
// buffers hold float32 values (layer inputs and deltas written before their split into
// pieces) for the weight-gradient GEMM.  LDS: the forward planes;
// in the sweep the x planes take delta3, the h1 planes delta2 and then the split-K partials,
// the h2 planes delta1 (the activations come back from the row buffers).  NW waves per tile
// share the products as in the forward (MlpWaves); the arithmetic of every element does not
// depend on NW.

// Evaluations of a tile: its first state (slot 0), then six per step (slot 1 + 6q + i - 1 for
// stage i of step q).  A step's last stage is the next one's first (FSAL: f at the same
// point), so the sweep adds the two cotangents of f there and pulls them back once, and the
// weight-gradient GEMM sees one row block for both.  A tile runs as many steps as its
// longest trajectory has; evals[tile] tells the GEMM how many of its E = 1 + 6 Cs slots
// (block tile * E + slot) hold rows.
// One segment of 8,192 trajectories and up to 4 steps: 0.70 ms (and 5 us for the float32
// launch that finds no tile marked); 0.92 ms with seven
// pull-backs a step, idle steps run, and the products' loads waited for in the K loop (and
// the GEMM 0.26 against 0.31 ms for the rows that went).  15 us per evaluation: MFMA, the
// splits and the LDS stores of one column at a time, one after the other, bound it, not the
// 1.3 GB of rows.
constexpr float SPLIT_WEIGHT_END = 1024.0f, SPLIT_STATE_END = 16777216.0f,
                SPLIT_DELTA_END = 1125899906842624.0f;  // 2^10, 2^24 (also of biases), 2^50
// Flags of the weights, one per 256, then of the biases.
constexpr int kMatrixFlags = MLP_H * (2 * MLP_D + MLP_H) / 256;
constexpr int kWeightFlags = kMatrixFlags + (2 * MLP_H + MLP_D + 255) / 256;
template <class P>
using AdjLds = std::conditional_t<P::PIECES == 3, MlpLds<P>, MlpLdsBack>;

template <class P, int NW>
__global__ void __launch_bounds__(64 * NW, 1)
mlp_adj_segment_kernel(const AdjArgs a, const MlpWeights<P> W, const RowBufs R) {
  constexpr bool Pieces = P::PIECES == 3;
  static_assert(kWeightFlags <= 64 * NW, "a thread per flag");
  extern __shared__ __align__(16) unsigned char smem[];
  AdjLds<P>& L = *reinterpret_cast<AdjLds<P>*>(smem);
  using Tab = Tsit5Tab;
  constexpr int S = Tab::S;
  using WV = MlpWaves<NW>;
  constexpr int CPT = WV::CPT, GRP = MLP_D / CPT, NT = WV::NT12, NT3 = WV::NT3;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int orow = tid / GRP, c0 = (tid % GRP) * CPT, gbase = lane & ~(GRP - 1);
  const int tile = blockIdx.x;
  const int64_t traj = (int64_t)tile * MLP_TILE + orow;
  const bool valid = traj < a.B;
  const int nacc = valid ? a.stats[traj * 3 + 1] : 0;
  const int n0 = a.seg * a.C;
  const int steps_here = min(max(nacc - n0, 0), a.Cs);
  if (!Pieces && a.evals[tile] >= 0) return;
  int tile_steps = 0;
  while (__syncthreads_or(tile_steps < steps_here)) ++tile_steps;
  int evals = tile_steps > 0 ? 1 + 6 * tile_steps : 0;
  int32_t* mark = a.evals + tile;
  int redo = a.wflags != nullptr;
  if (Pieces) {
    const bool out = __syncthreads_or(redo && tid < kWeightFlags && a.wflags[tid] != 0);
    if (tid == 0) *mark = out ? -evals : evals;
    if (tile_steps == 0 || out) return;
    // kept for the end in vector registers: scalar ones spill
    asm("" : "+v"(evals), "+v"(mark), "+v"(redo));
  }
  SplitRange rng;
  const int dir = (a.t0 < a.t1) ? 1 : -1;
  const double* ts_row = a.ts ? a.ts + (valid ? traj : 0) * a.ts_stride : nullptr;
  using TL = TabLit<Tab, float>;
  const int64_t slot0 = (int64_t)tile * (1 + 6 * a.Cs);
  auto slot_of = [&](int q, int i) { return slot0 + 6 * q + i; };  // stage i >= 1, or (0, 0)
  auto fslot = [&](int64_t slot) { return a.zs + (slot * MLP_TILE + orow) * MLP_D + c0; };
  // The layer inputs of an evaluation go to its row block as they are formed: the stage value
  // by its owner threads, the activations from the forward's epilogues.
  auto put_cols = [&](float* rows, int64_t slot, const float (&v)[CPT]) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) rows[rows_index(slot, MLP_D, orow, c0 + j)] = v[j];
  };
  auto step_times = [&](int q, double& ta, double& tb) {
    const bool act = q < steps_here;
    const double* g = a.grid + (traj * a.max_steps + n0 + q) * 2;
    ta = act ? g[0] : 0.0;
    tb = act ? g[1] : 0.0;
    return act;
  };
  mlp_begin<P>(W, L);

  // ---- 1. recompute the segment: keep every evaluation's f (scratch) and its layer inputs
  //      (row buffers), so that the reverse sweep needs no forward re-evaluation ----
  auto forward = [&](int64_t slot, const float (&z)[CPT],
                     float (&f)[CPT]) __attribute__((always_inline)) {
    put_cols(R.b[1], slot, z);
    store_inputs(L, orow, c0, z);
    if constexpr (Pieces) {
#pragma unroll
      for (int j = 0; j < CPT; j += 4) rng.see(z[j], z[j + 1], z[j + 2], z[j + 3]);
    }
    __syncthreads();
    if constexpr (Pieces) {
      mlp_forward_rows<NW>(W, L, wave, lane, orow, c0, f, R.b[3], R.b[5], slot);
    } else {
      mlp_forward<P, NW>(W, L, wave, lane, orow, c0, f);
      rows_out<MLP_H>(L.h1, L.LDH, R.b[3], slot);
      rows_out<MLP_H>(L.h2, L.LDH, R.b[5], slot);
    }
    float* fp = fslot(slot);
#pragma unroll
    for (int j = 0; j < CPT; ++j) fp[j] = f[j];
  };
  float y[CPT], f[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) y[j] = (steps_here > 0) ? a.ckpt[(traj * a.n_ckpt + a.seg) * MLP_D + c0 + j] : 0.0f;
  forward(slot0, y, f);
  for (int q = 0; q < tile_steps; ++q) {
    double ta, tb;
    const bool act = step_times(q, ta, tb);
    const float control = (float)((double)dir * (tb - ta));
    float k[S][CPT], z[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) k[0][j] = control * f[j];
    static_for<1, S>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        float kc[S];
#pragma unroll
        for (int m = 0; m < S; ++m) kc[m] = (m < i) ? k[m][j] : 0.0f;
        z[j] = y[j] + comb<Tab, 0, i, 0, i, false>(TL::v.a[i], kc, 0.0f);
      }
      forward(slot_of(q, i), z, f);
#pragma unroll
      for (int j = 0; j < CPT; ++j) k[i][j] = control * f[j];
    });
    if (act) {
#pragma unroll
      for (int j = 0; j < CPT; ++j) y[j] = z[j];
    }
  }

  // ---- 2. reverse sweep ----
  // Pull the cotangent fb of an evaluation's f back to its input: delta3 = fb (1 - f^2),
  // delta2 = (delta3 . W3) softplus'(h2), delta1 = (delta2 . W2) softplus'(h1), zb = delta1 .
  // W1, the deltas to their row blocks.  LDS: delta3 in the x planes, delta2 in h1, delta1 in
  // h2, then the split-K partials in h1; every buffer's last readers are behind a barrier
  // when it is written.
  auto pull_back = [&](int64_t slot, const float (&fb)[CPT],
                       float (&zb)[CPT]) __attribute__((always_inline)) {
    const float* fp = fslot(slot);
    float d3[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) d3[j] = fb[j] * (1.0f - fp[j] * fp[j]);
    if constexpr (!Pieces) {
      __syncthreads();  // the save weights of other rows lie in the h2 buffer
#pragma unroll
      for (int j = 0; j < CPT; ++j) L.d3[orow * L.LDX + P::pos(c0 + j)] = d3[j];
      rows_in<MLP_H>(L.h1, L.LDH, R.b[3], slot);
      rows_in<MLP_H>(L.h2, L.LDH, R.b[5], slot);
      pull_back_f32<NW>(W, L, R, slot, wave, lane, orow, c0, zb);
    } else {
      constexpr int KS1 = MLP_D / 16, KS2 = MLP_H / 16, HP = MLP_TILE * MlpLds<P>::LDH;
      float4 h[NT][4];
      auto load_h = [&](const float* rows) {  // ahead of the product it follows
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            h[t][i] = *reinterpret_cast<const float4*>(rows + rows_frag(slot, MLP_H, NT * wave + t, i, lane));
        }
      };
      floatx16_t acc[NT];
      auto delta = [&](int t, int i) {
        return make_float4(acc[t][4 * i] * dsoftplus_from_value(h[t][i].x),
                           acc[t][4 * i + 1] * dsoftplus_from_value(h[t][i].y),
                           acc[t][4 * i + 2] * dsoftplus_from_value(h[t][i].z),
                           acc[t][4 * i + 3] * dsoftplus_from_value(h[t][i].w));
      };
      Gemm3<KS1, NT, false> g3;
      Gemm3<KS2, NT, false> g2;
      Gemm3<KS2, NT3> g1;
      g3.preload(W.w3t, W.plane3, NT * wave, 0, lane);
      load_h(R.b[5]);
      __builtin_amdgcn_sched_barrier(0);
      put_cols(R.b[4], slot, d3);
      store_inputs(L, orow, c0, d3);
#pragma unroll
      for (int j = 0; j < CPT; j += 4) {
        constexpr float s = SPLIT_STATE_END / SPLIT_DELTA_END;
        rng.most(s * d3[j], s * d3[j + 1], s * d3[j + 2], s * d3[j + 3]);
        rng.least(d3[j], d3[j + 1], d3[j + 2], d3[j + 3]);
      }
      __syncthreads();
      g3.template run<KS1>(L.x[0], MLP_TILE * MlpLds<P>::LDX, L.LDX, 0, acc, lane);
      g2.preload(W.w2t, W.plane2, NT * wave, 0, lane);
      __builtin_amdgcn_sched_barrier(0);
      put_rows<NW>(L, L.h1[0], R.b[2], slot, wave, lane, delta);
      load_h(R.b[3]);
      __syncthreads();
      g2.template run<KS2>(L.h1[0], HP, L.LDH, 0, acc, lane);
      const int qk = WV::quarter(wave), n3 = WV::nt3(wave);
      g1.preload(W.w1t, W.plane1, n3, qk * (KS2 / 4), lane);
      __builtin_amdgcn_sched_barrier(0);
      put_rows<NW>(L, L.h2[0], R.b[0], slot, wave, lane, delta);
      __syncthreads();
      floatx16_t acc3[NT3];
      g1.template run<KS2 / 4>(L.h2[0], HP, L.LDH, qk * (KS2 / 4), acc3, lane);
      float* part = L.part();
      put_partials<NT3>(acc3, part, L.LDP, qk, n3, lane);
      __syncthreads();
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        const int c = c0 + j;
        float s = part[(0 * MLP_TILE + orow) * L.LDP + c];
        s += part[(1 * MLP_TILE + orow) * L.LDP + c];
        s += part[(2 * MLP_TILE + orow) * L.LDP + c];
        s += part[(3 * MLP_TILE + orow) * L.LDP + c];
        zb[j] = s;
      }
#pragma unroll
      for (int j = 0; j < CPT; j += 4) rng.least(zb[j], zb[j + 1], zb[j + 2], zb[j + 3]);
    }
  };
  // yb: cotangent of the state at the end of step q; fb: of f there, from the next step's
  // first stage.
  float yb[CPT], fb[CPT], zb[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    yb[j] = valid ? a.ybar[traj * MLP_D + c0 + j] : 0.0f;
    fb[j] = 0.0f;
  }
  for (int q = tile_steps - 1; q >= 0; --q) {
    double ta, tb;
    const bool act = step_times(q, ta, tb);
    const int n = n0 + q;
    const float control = (float)((double)dir * (tb - ta));
    float kb[S][CPT], ybn[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      ybn[j] = yb[j];
#pragma unroll
      for (int m = 0; m < S; ++m) kb[m][j] = (act && m < S - 1) ? TL::v.a[S - 1][m] * yb[j] : 0.0f;
    }
    if (act && a.n_ts > 0) {
      // SaveAt(ts) rows interpolated inside this step, (ta, tb] (from the start for the
      // solve's first step): counted and weighted by the owner group, one time per owner
      // (the weights pass through the h2 planes, idle here)
      const int qo = lane & (GRP - 1);
      int jlo = 0, jhi = 0;
      for (int s0 = 0; s0 < a.n_ts; s0 += GRP) {
        const double t = s0 + qo < a.n_ts ? ts_row[s0 + qo] * dir : __builtin_inf();
        const unsigned grp = (unsigned)((1ull << GRP) - 1);
        jlo += __builtin_popcount((unsigned)(__ballot(n > 0 && t <= ta) >> gbase) & grp);
        jhi += __builtin_popcount((unsigned)(__ballot(t <= tb) >> gbase) & grp);
      }
      float* wts = reinterpret_cast<float*>(&L.h2[0]) + orow * GRP * 8;
      for (int s0 = jlo; s0 < jhi; s0 += GRP) {
        const int cnt = min(GRP, jhi - s0);
        {
          double bb[7];
          tsit5_weights(linear_rescale(ta, ts_row[min(s0 + qo, jhi - 1)] * dir, tb), bb);
          float4* o = reinterpret_cast<float4*>(wts + 8 * qo);
          o[0] = make_float4((float)bb[0], (float)bb[1], (float)bb[2], (float)bb[3]);
          o[1] = make_float4((float)bb[4], (float)bb[5], (float)bb[6], 0.0f);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const float* g = a.ys_bar + (traj * a.n_out + (a.save_t0 ? 1 : 0) + s0) * MLP_D + c0;
        for (int e = 0; e < cnt; ++e) {
          const float4 w0 = reinterpret_cast<const float4*>(wts)[2 * e];
          const float4 w1 = reinterpret_cast<const float4*>(wts)[2 * e + 1];
          const float bb[7] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z};
#pragma unroll
          for (int j = 0; j < CPT; ++j) {
            const float gv = g[e * MLP_D + j];
            ybn[j] += gv;
#pragma unroll
            for (int m = 0; m < 7; ++m) kb[m][j] += bb[m] * gv;
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
    }
    // stages 6 .. 1: z_i = y_n + sum_{m<i} a_im k_m
    static_for<0, S - 1>([&](auto ic) {
      constexpr int i = S - 1 - decltype(ic)::value;
      float fbi[CPT];
#pragma unroll
      for (int j = 0; j < CPT; ++j)
        fbi[j] = (act ? control * kb[i][j] : 0.0f) + (i == S - 1 ? fb[j] : 0.0f);
      pull_back(slot_of(q, i), fbi, zb);
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        const float z = act ? zb[j] : 0.0f;
        ybn[j] += z;
#pragma unroll
        for (int m = 0; m < i; ++m) kb[m][j] += TL::v.a[i][m] * z;
      }
    });
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      fb[j] = act ? control * kb[0][j] : 0.0f;
      yb[j] = act ? ybn[j] : yb[j];
    }
  }
  pull_back(slot0, fb, zb);
  if constexpr (Pieces) {
    if (__syncthreads_or(rng.outside(SPLIT_STATE_END))) {
      if (tid == 0) *mark = -evals;
      if (redo) return;  // left to the float32 kernel
    }
  }
  if (valid) {
#pragma unroll
    for (int j = 0; j < CPT; ++j)
      a.ybar[traj * MLP_D + c0 + j] = steps_here > 0 ? yb[j] + zb[j] : yb[j];
  }
}

// Three-piece planes (mlp_pack_layout(3)) of a float32 packed buffer (mlp_pack_layout(1)), and
// the flags of the weights (by the workgroups of the first three matrices) and biases (by
// those that follow).
__global__ void __launch_bounds__(256) mlp_split_packed_kernel(const float* __restrict__ packed,
                                                               const float* __restrict__ b1,
                                                               const float* __restrict__ b2,
                                                               const float* __restrict__ b3,
                                                               __bf16* __restrict__ out,
                                                               int32_t* __restrict__ wflags) {
  int e = blockIdx.x * 256 + threadIdx.x, m, before;
  mlp_pack_find(e, m, before);
  if (m == 6) return;
  const MlpPackShape sh = mlp_pack_shape(m);
  int n, k;
  mlp_frag_nk<PolicyBF16x3>(e, sh.k, n, k);
  const float v = packed[before + mlp_frag_index<PolicyF32>(n, k, sh.k)];
  __bf16* o = out + 3 * before + e;
  split3(v, o[0], o[sh.n * sh.k], o[2 * sh.n * sh.k]);
  if (blockIdx.x < kWeightFlags) {
    SplitRange rng;
    float end = SPLIT_WEIGHT_END;
    if (m < 3) {  // (whole workgroups: the matrices are multiples of 256)
      rng.see(v, v, v, v);
    } else {
      const int i = (int)(blockIdx.x - kMatrixFlags) * 256 + (int)threadIdx.x;
      if (i < 2 * MLP_H + MLP_D) {
        const float b = i < MLP_H ? b1[i] : (i < 2 * MLP_H ? b2[i - MLP_H] : b3[i - 2 * MLP_H]);
        rng.most(b, b, b, b);
      }
      end = SPLIT_STATE_END;
    }
    const int outside = __syncthreads_or(rng.outside(end));
    if (threadIdx.x == 0) wflags[blockIdx.x] = outside;
  }
}

// ---- weight gradients of one segment ---------------------------------------------------
// Output tiles: matrix 0 = dW1 [256 x 64] (D1, Z), 1 = dW2 [256 x 256] (D2, H1),
// 2 = dW3 [64 x 256] (D3, H2); 32x32 tiles numbered matrix by matrix, row-major.
struct DwLayout {
  int n1[3], n2[3], first[4];
};
__host__ __device__ inline DwLayout dw_layout() {
  DwLayout l{{MLP_H, MLP_H, MLP_D}, {MLP_D, MLP_H, MLP_H}, {0, 0, 0, 0}};
  for (int m = 0; m < 3; ++m) l.first[m + 1] = l.first[m] + (l.n1[m] / 32) * (l.n2[m] / 32);
  return l;
}

// Launch order is XCD-aware: workgroups are dealt to the 8 XCDs round-robin by linear id,
// so workgroup b runs on XCD b % 8; XCD x takes chunks x, x + 8, ... and runs the workgroups
// of a chunk back to back, which then read the chunk's rows through one L2 instead of eight.
constexpr int kXcds = 8;

// Chunks of row blocks the GEMM splits K into: 24 one-wave workgroups (64 x 64 output
// pieces) each, two per SIMD of the chip resident at once, so 80 chunks (1,920 waves), but no
// more than there are four-block chunks, and as many times 80 as it takes that none has more
// than 128 blocks: the float32 accumulators' rounding grows with their 4,096 rows (8,192
// trajectories and 64 steps, 98,560 blocks: 800 chunks; with 80 the sums were off by 6e-6 of
// the largest, now by 1.4e-6).
__host__ __device__ inline int dw_chunks(int64_t blocks) {
  const int64_t few = (blocks + 3) / 4, rounds = (blocks + 80 * 128 - 1) / (80 * 128);
  const int64_t n = few < 80 ? few : 80 * rounds;
  return (int)(n < 1 ? 1 : n);
}

// partial[chunk][tile] = A^T B over one chunk of row blocks (A = deltas, B = layer inputs)
// for every 32 x 32 output tile, each wave on a 2 x 2 block of tiles (a 64 x 64 piece of one
// matrix: dW1 4 x 1, dW2 4 x 4, dW3 1 x 4 pieces).  A lane's sixteen values of a block piece
// are the rows of its two k halves (rows_frag), so fragments go from memory through the
// split straight to the MFMAs: six bf16 products per pair of fragments, as in Gemm3,
// with float32 accumulation.  The next block's values load while this one's are split.
// Waves in the first piece column of a matrix also produce the chunk's column sums of A (the
// bias gradient partials, partial_db: [chunk][db1 | db2 | db3]).
// evals: of every `slots` blocks (a tile) only the first |evals[tile]| hold rows (null: all do).
// SC: the rows of A are multiplied by rscale[row] (the backsolve's per-row weights dt * b_i,
// zero for rejected steps and idle rows; a row of zero weight is dropped from both operands,
// so a non-finite value in it contributes nothing).
// Bound: the rows' HBM reads, 4.6 KB a row: 0.31 ms for the 229,376 rows of 8,192
// trajectories and 4 steps (3.4 TB/s, 290 TFLOP/s of 6 bf16 passes each), where float32 MFMA
// with a 4-byte load per operand and MFMA took 0.72 ms (and 0.58 ms for 105,000 rows, now
// 0.115).  Against float64 the gradients are closer than before (5.6e-7 to 8e-7 of the
// largest, 1.3e-6 to 1.8e-6 with float32 MFMA).
__host__ __device__ inline int dw_pieces_of(int m) {
  const DwLayout l = dw_layout();
  return (l.n1[m] / 64) * (l.n2[m] / 64);
}

template <bool SC>
__global__ void __launch_bounds__(64, 2)
mlp_dw_gemm_kernel(const RowBufs R, float* __restrict__ partial, float* __restrict__ partial_db,
                   int64_t blocks, int nch, const int32_t* __restrict__ evals, int slots,
                   const float* __restrict__ rscale) {
  const DwLayout lay = dw_layout();
  const int npc = dw_pieces_of(0) + dw_pieces_of(1) + dw_pieces_of(2);
  const int xcd = (int)(blockIdx.x % kXcds), slot = (int)(blockIdx.x / kXcds);
  const int chunk = (slot / npc) * kXcds + xcd;
  int pg = slot - (slot / npc) * npc;
  if (chunk >= nch) return;
  int m = 0;
  while (pg >= dw_pieces_of(m)) { pg -= dw_pieces_of(m); ++m; }
  const int W1 = m == 2 ? MLP_D : MLP_H, W2 = m == 0 ? MLP_D : MLP_H;  // columns of A and B
  const int npj = W2 / 64;
  const int pi = pg / npj, pj = pg - pi * npj;
  const float* A = m == 0 ? R.b[0] : m == 1 ? R.b[2] : R.b[4];
  const float* Bm = m == 0 ? R.b[1] : m == 1 ? R.b[3] : R.b[5];
  const int lane = threadIdx.x, half = lane >> 5;
  const bool col_sums = (pj == 0);
  const int64_t b0 = blocks * chunk / nch, b1 = blocks * (chunk + 1) / nch;
  using P = PolicyBF16x3;
  using frag_t = P::frag_t;
  floatx16_t acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x) { acc[x][0] = floatx16_t{}; acc[x][1] = floatx16_t{}; }
  float csum[2] = {0.0f, 0.0f};
  float4 va[2][4], vb[2][4];
  auto load = [&](int64_t blk) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        va[x][i] = *reinterpret_cast<const float4*>(A + rows_frag(blk, W1, 2 * pi + x, i, lane));
        vb[x][i] = *reinterpret_cast<const float4*>(Bm + rows_frag(blk, W2, 2 * pj + x, i, lane));
      }
    }
  };
  // the first block with rows at or after blk (b1: none); lim: the end of its tile's
  int64_t lim = evals ? b0 : b1;
  auto next = [&](int64_t blk) {
    while (blk >= lim && blk < b1) {
      const int64_t tile = blk / slots;
      lim = min(tile * slots + abs(evals[tile]), b1);
      if (blk >= lim) {
        blk = min((tile + 1) * slots, b1);
        lim = blk;
      }
    }
    return blk;
  };
  // the loaded block's rows times their weights (SC)
  auto scale = [&](int64_t blk) {
    float4 ws[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ws[i] = *reinterpret_cast<const float4*>(rscale + blk * 32 + 8 * i + 4 * half);
    __builtin_amdgcn_sched_barrier(0);  // one wait for the four loads
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 w = ws[i];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        auto sc = [](float wt, float& da, float& db) {
          da = (wt != 0.0f) ? da * wt : 0.0f;
          db = (wt != 0.0f) ? db : 0.0f;
        };
        sc(w.x, va[x][i].x, vb[x][i].x);
        sc(w.y, va[x][i].y, vb[x][i].y);
        sc(w.z, va[x][i].z, vb[x][i].z);
        sc(w.w, va[x][i].w, vb[x][i].w);
      }
    }
  };
  auto add_columns = [&]() {
    if (col_sums) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          csum[x] += (va[x][i].x + va[x][i].y) + (va[x][i].z + va[x][i].w);
      }
    }
  };
  int64_t nxt = next(b0);
  if (nxt < b1) load(nxt);
  while (nxt < b1) {
    const int64_t blk = nxt;
    nxt = next(blk + 1);
    if constexpr (SC) scale(blk);
    add_columns();
    // k half s: the rows 16 s .. 16 s + 15 of the block, in the same order for both operands
    frag_t fa[2][2][3], fb[2][2][3];  // [s][x][piece]
    auto split = [&](const float4& u, const float4& v, frag_t (&f)[3]) {
      const Split4 s0 = split3x4(u.x, u.y, u.z, u.w), s1 = split3x4(v.x, v.y, v.z, v.w);
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) {
        const uint4 q = make_uint4(s0.p[pc].x, s0.p[pc].y, s1.p[pc].x, s1.p[pc].y);
        f[pc] = __builtin_bit_cast(frag_t, q);
      }
    };
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        split(va[x][2 * s], va[x][2 * s + 1], fa[s][x]);
        split(vb[x][2 * s], vb[x][2 * s + 1], fb[s][x]);
      }
    }
    if (nxt < b1) load(nxt);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int pq = 0; pq < 6; ++pq) {  // p0q0, p0q1, p1q0, p0q2, p1q1, p2q0
        constexpr int pa[6] = {0, 0, 1, 0, 1, 2}, pb[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int y = 0; y < 2; ++y)
            acc[x][y] = P::mfma(fa[s][x][pa[pq]], fb[s][y][pb[pq]], acc[x][y]);
        }
      }
    }
  }
  // The sums tell whether the pieces could be trusted (SplitRange).  A value that has none, or a
  // sum of theirs that overflows, leaves an accumulator that is not finite.  Pieces are off by
  // 2^-134 at most, 4,096 products by 2^-112 for activations up to 2^10: less than 2^-24 of
  // sums whose largest is SPLIT_MIN or more.  Else the chunk runs once more on float32 MFMA, its
  // rows as the k of v_mfma_f32_32x32x2 (row 8i + j from lane half 0, 8i + 4 + j from half 1),
  // in a loop of its own (beside the pieces' registers it would spill).
  bool finite = true;
  float most = 0.0f;
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int y = 0; y < 2; ++y) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        finite = finite && fabsf(acc[x][y][v]) < __builtin_inff();
        most = fmaxf(most, fabsf(acc[x][y][v]));
      }
    }
  }
  if (__any(!finite) || (__any(most > 0.0f) && !__any(most >= SPLIT_MIN))) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      acc[x][0] = floatx16_t{};
      acc[x][1] = floatx16_t{};
      csum[x] = 0.0f;
    }
    lim = evals ? b0 : b1;
    for (int64_t blk = next(b0); blk < b1; blk = next(blk + 1)) {
      load(blk);
      if constexpr (SC) scale(blk);
      add_columns();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            auto mm = [&](float p, float q) {
              acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(p, q, acc[x][y], 0, 0, 0);
            };
            mm(va[x][i].x, vb[y][i].x);
            mm(va[x][i].y, vb[y][i].y);
            mm(va[x][i].z, vb[y][i].z);
            mm(va[x][i].w, vb[y][i].w);
          }
        }
      }
    }
  }
  const int ntj = W2 / 32;
  const int first = m == 0 ? lay.first[0] : m == 1 ? lay.first[1] : lay.first[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int tg = first + (2 * pi + x) * ntj + (2 * pj + y);
      float4* o = reinterpret_cast<float4*>(partial + ((int64_t)chunk * lay.first[3] + tg) * 1024);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i * 64 + lane] = make_float4(acc[x][y][4 * i], acc[x][y][4 * i + 1], acc[x][y][4 * i + 2],
                                       acc[x][y][4 * i + 3]);
    }
  }
  if (col_sums) {
    const int off = (m == 0) ? 0 : (m == 1 ? MLP_H : 2 * MLP_H);
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const float c = csum[x] + __shfl_xor(csum[x], 32);
      if (lane < 32)
        partial_db[(int64_t)chunk * (2 * MLP_H + MLP_D) + off + pi * 64 + 32 * x + lane] = c;
    }
  }
}

// dw_acc (dW1 | dW2 | dW3 | db1 | db2 | db3, row-major) += partials over the chunks.  A
// workgroup takes 64 float4 of the partials; its four waves sum every fourth chunk each and
// the four sums are added in order.  (One thread per output over all chunks, its loads one
// behind the other and 64 bytes apart: 34 us.)
__global__ void __launch_bounds__(256) mlp_dw_reduce_kernel(const float* __restrict__ partial,
                                                            const float* __restrict__ partial_db,
                                                            int nchunks,
                                                            float* __restrict__ dw_acc) {
  __shared__ float4 sum[4][64];
  const DwLayout lay = dw_layout();
  const int ntile = lay.first[3], nb = (2 * MLP_H + MLP_D) / 4;
  const int col = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int blk = blockIdx.x;
  const bool weights = blk < ntile * 4;  // then the bias partials, 144 float4
  const int e = weights ? blk * 64 + col : (blk - ntile * 4) * 64 + col;
  const bool live = weights || e < nb;
  const int64_t stride = weights ? (int64_t)ntile * 256 : nb;
  const float4* src = reinterpret_cast<const float4*>(weights ? partial : partial_db) + e;
  float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (live) {
#pragma unroll 4
    for (int ch = part; ch < nchunks; ch += 4) {
      const float4 v = src[ch * stride];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
  }
  sum[part][col] = s;
  __syncthreads();
  if (part != 0 || !live) return;
#pragma unroll
  for (int q = 1; q < 4; ++q) {
    const float4 v = sum[q][col];
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  const int nW = MLP_H * MLP_D + MLP_H * MLP_H + MLP_D * MLP_H;
  const float sv[4] = {s.x, s.y, s.z, s.w};
  if (!weights) {
#pragma unroll
    for (int j = 0; j < 4; ++j) dw_acc[nW + 4 * e + j] += sv[j];
    return;
  }
  // float4 i of tile tg, lane col: rows 8i + 4(col/32) + j, column col%32
  const int tg = blk >> 2, i = blk & 3;
  int m = 0;
  while (tg >= lay.first[m + 1]) ++m;
  const int W2 = m == 0 ? MLP_D : MLP_H, ntj = W2 / 32;
  const int off = m == 0 ? 0 : m == 1 ? MLP_H * MLP_D : MLP_H * MLP_D + MLP_H * MLP_H;
  const int ti = (tg - lay.first[m]) / ntj, tj = (tg - lay.first[m]) % ntj;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = 32 * ti + 8 * i + 4 * (col >> 5) + j;
    dw_acc[off + r * W2 + 32 * tj + (col & 31)] += sv[j];
  }
}

// ---- BacksolveAdjoint of the neural ODE ---------------------------------------------
// The continuous adjoint (_adjoint.py:539-873) with the adjoint seminorm
// (_misc.py:85-116): between consecutive save times, from the last one back to t0, the
// augmented state (y, a_y, a_theta) is integrated backwards by Tsit5 with the integral PID
// controller, after a_y takes that save's cotangent and y restarts from the forward's saved
// state, under the adjoint vector field (AdjointTerm, _term.py:767-917):
//   dy/dt = f(y),  da_y/dt = vjp(f, y)(-a_y),  da_theta/dt = vjp(f, theta)(-a_y).
// The seminorm leaves a_theta out of the error norm (RMS over the 128 components of y and
// a_y), so a_theta only accumulates: a_theta(t0) = sum over accepted steps and stages of
// dt b_i vjp_theta(z_i).  Each stage's vjp_theta is the set of outer products delta_l x
// input_l; the kernel writes those rows (unscaled) to the row buffers and their weights
// dt b_i (0 for rejected steps and idle rows) to rscale, and the split-K GEMM above forms
// the sum over all rows (trajectories, steps and stages) for the launch.
// One workgroup per tile of 32 rows; each launch runs at most Q lock-step iterations (one
// attempted step of every row) and leaves unfinished rows' state in BsRow / ya for the
// next launch.  Each iteration evaluates stage 0 afresh: f(y) at an unchanged y gives the
// same value as the FSAL stage, and fresh evaluation also covers the first step after
// each save (made_jump).
struct BsRow {
  double tprev, tnext, T1, floor_t1, inv, pinv;
  int32_t at_dtmin, s, nsteps, dir, result, res_total, done, pad_;
};

struct BsArgs {
  const float* ys;       // [B, n_out, 64] forward saved states
  const double* ts_out;  // [B, n_out] their times
  const float* ys_bar;   // [B, n_out, 64] cotangents
  float* ya;             // [B_pad, 128] y then a_y of each row between launches
  BsRow* rows;           // [B_pad]
  float* rscale;         // [Q * 7 * B_pad] weights of the weight-gradient rows
  float* ybar;           // out [B, 64] cotangent of y0
  int32_t* result;       // out [B]
  int32_t* counters;     // [2]: rows unfinished after the launch, iterations run (max)
  int64_t B, B_pad;
  int32_t n_out, save_t0, max_steps, Q, first;
  double t0, dt0;        // the forward t0; dt0 of the backward solves
  PidParams pid;         // the backward controller
};

template <int NW>
__global__ void __launch_bounds__(64 * NW, 1)
mlp_backsolve_kernel(const BsArgs a, const MlpWeights<PolicyF32> W, const RowBufs R) {
  using P = PolicyF32;
  extern __shared__ __align__(16) unsigned char smem[];
  MlpLdsBack& L = *reinterpret_cast<MlpLdsBack*>(smem);
  using Tab = Tsit5Tab;
  constexpr int S = Tab::S;
  using TL = TabLit<Tab, float>;
  using WV = MlpWaves<NW>;
  constexpr int CPT = WV::CPT, GRP = MLP_D / CPT;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int orow = tid / GRP, c0 = (tid % GRP) * CPT, gbase = lane & ~(GRP - 1);
  const bool lead = (tid % GRP) == 0;
  const int tile = blockIdx.x;
  const int64_t traj = (int64_t)tile * MLP_TILE + orow;
  const bool valid = traj < a.B;
  const int s_end = a.save_t0 ? 1 : 0;

  float y[CPT], av[CPT];
  BsRow st;
  // Start the backward solve over save interval s: y from the forward's row s, a_y plus
  // that row's cotangent, span [ts_out[s], ts_out[s - 1] or t0] (_scan_fun).
  auto begin = [&](int s) {
    const float* ysr = a.ys + (traj * a.n_out + s) * MLP_D + c0;
    const float* gr = a.ys_bar + (traj * a.n_out + s) * MLP_D + c0;
#pragma unroll
    for (int j = 0; j < CPT; ++j) { y[j] = ysr[j]; av[j] = av[j] + gr[j]; }
    const double t0r = a.ts_out[traj * a.n_out + s];
    const double t1r = s > 0 ? a.ts_out[traj * a.n_out + s - 1] : a.t0;
    st.s = s;
    st.dir = (t0r < t1r) ? 1 : -1;
    const double T0 = t0r * st.dir;
    st.T1 = t1r * st.dir;
    double fl = st.T1;
    for (int r = 0; r < 100; ++r) fl = prevbefore(fl);
    st.floor_t1 = fl;
    double dt0v = a.dt0 * st.dir;
    if (a.pid.has_dtmax) dt0v = jmin(dt0v, a.pid.dtmax);
    if (a.pid.has_dtmin) dt0v = jmax(dt0v, a.pid.dtmin);
    st.tprev = T0;
    st.tnext = jmin(T0 + dt0v, st.T1);
    st.inv = 1.0; st.pinv = 1.0; st.at_dtmin = 0;
    st.nsteps = 0;
    st.result = DFX_SUCCESSFUL;
  };
  // Move past finished intervals; after the last one the row's a_y (plus the t0 row's
  // cotangent when t0 was saved) is dL/dy0.
  auto settle = [&]() {
    while (!st.done) {
      if (st.tprev < st.T1 && st.result == DFX_SUCCESSFUL && st.nsteps < a.max_steps) return;
      if (st.tprev < st.T1 && st.result == DFX_SUCCESSFUL) st.result = DFX_MAX_STEPS_REACHED;
      if (st.res_total == DFX_SUCCESSFUL) st.res_total = st.result;
      if (st.s - 1 >= s_end) {
        begin(st.s - 1);
      } else {
        if (a.save_t0 && a.n_out > 0) {
          const float* g0 = a.ys_bar + traj * a.n_out * MLP_D + c0;
#pragma unroll
          for (int j = 0; j < CPT; ++j) av[j] = av[j] + g0[j];
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) a.ybar[traj * MLP_D + c0 + j] = av[j];
        if (lead) a.result[traj] = st.res_total;
        st.done = 1;
      }
    }
  };

  if (!valid) {
    st.done = 1;
  } else if (a.first) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) av[j] = 0.0f;
    st.res_total = DFX_SUCCESSFUL;
    st.done = 0;
    if (a.n_out - 1 >= s_end) {
      begin(a.n_out - 1);
    } else {
      st.tprev = st.T1 = 0.0;  // nothing saved after t0: no interval
      st.s = s_end;
      st.result = DFX_SUCCESSFUL;
    }
    settle();
  } else {
    st = a.rows[traj];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      y[j] = a.ya[traj * 128 + c0 + j];
      av[j] = a.ya[traj * 128 + 64 + c0 + j];
    }
  }

  mlp_begin<P>(W, L);  // the first iteration's barriers come before its first use
  const int64_t rb0 = (int64_t)tile * MLP_TILE + orow;
  const int64_t ntiles = a.B_pad / MLP_TILE;
  int q = 0;
  for (; q < a.Q; ++q) {
    const bool run = !st.done;
    if (!__syncthreads_or(run)) break;
    const double ts0 = st.tprev, ts1 = st.tnext;
    const float control = run ? (float)((double)st.dir * (ts1 - ts0)) : 0.0f;
    float ky[S][CPT], ka[S][CPT], zy[CPT], za[CPT];
    static_for<0, S>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        if constexpr (i == 0) {
          zy[j] = y[j];
          za[j] = av[j];
        } else {
          float cy[S], ca[S];
#pragma unroll
          for (int m = 0; m < S; ++m) {
            cy[m] = (m < i) ? ky[m][j] : 0.0f;
            ca[m] = (m < i) ? ka[m][j] : 0.0f;
          }
          zy[j] = y[j] + comb<Tab, 0, i, 0, i, false>(TL::v.a[i], cy, 0.0f);
          za[j] = av[j] + comb<Tab, 0, i, 0, i, false>(TL::v.a[i], ca, 0.0f);
        }
        if (!run) { zy[j] = 0.0f; za[j] = 0.0f; }  // idle rows: zero deltas
      }
      store_inputs(L, orow, c0, zy);
      __syncthreads();
      float f[CPT];
      mlp_forward<P, NW>(W, L, wave, lane, orow, c0, f);
      const int64_t block = ((int64_t)q * S + i) * ntiles + tile;
      rows_out<MLP_D>(L.x, L.LDX, R.b[1], block);
      rows_out<MLP_H>(L.h1, L.LDH, R.b[3], block);
      rows_out<MLP_H>(L.h2, L.LDH, R.b[5], block);
      // vjp with cotangent w = -a_y of the stage: delta3 = w (1 - f^2)
#pragma unroll
      for (int j = 0; j < CPT; ++j)
        L.d3[orow * L.LDX + P::pos(c0 + j)] = -za[j] * (1.0f - f[j] * f[j]);
      float sv[CPT];
      pull_back_f32<NW>(W, L, R, block, wave, lane, orow, c0, sv);
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        ky[i][j] = control * f[j];
        ka[i][j] = control * sv[j];
      }
      __syncthreads();
    });
    // y1, a1 = the last stage (SSAL); embedded error over the 128 components of (y, a_y)
    bool anynan = false;
    float ey[CPT], ea[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      float cy[S], ca[S];
#pragma unroll
      for (int m = 0; m < S; ++m) { cy[m] = ky[m][j]; ca[m] = ka[m][j]; }
      ey[j] = comb<Tab, 2, 0, 0, S, false>(TL::v.berr, cy, 0.0f);
      ea[j] = comb<Tab, 2, 0, 0, S, false>(TL::v.berr, ca, 0.0f);
      anynan = anynan || (zy[j] != zy[j]) || (za[j] != za[j]);
    }
    const unsigned long long nanmask = __ballot(anynan);
    const bool group_nan = ((nanmask >> gbase) & ((1ull << GRP) - 1)) != 0;
    auto sq_err = [&](float e0, float v0, float v1) {
      const double v1c = group_nan ? (double)v0 : (double)v1;
      const double yy = jmax(fabs((double)v0), fabs(v1c));
      double e = (double)e0;
      if (e != e) e = __builtin_inf();
      e = e / (a.pid.atol + yy * a.pid.rtol);
      return e * e;
    };
    double ty[CPT], ta[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      ty[j] = sq_err(ey[j], y[j], zy[j]);
      ta[j] = sq_err(ea[j], av[j], za[j]);
    }
    // Eight partials, one per eight-component block: the block's y terms then its a_y
    // terms, in component order; then the partials in order.  With four components per
    // owner, the pair's sums pass between its two owners so that the order is the same.
    double part = 0.0;
    int stride = 1, first = 0;
    if constexpr (CPT == 8) {
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ty[j];
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ta[j];
    } else {
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ty[j];      // even: its y terms
      part = __shfl(part, lane & ~1);
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ty[j];      // odd: + its y terms
      part = __shfl(part, lane | 1);
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ta[j];      // even: + its a_y terms
      part = __shfl(part, lane & ~1);
#pragma unroll
      for (int j = 0; j < CPT; ++j) part += ta[j];      // odd: + its a_y terms
      stride = 2;
      first = 1;
    }
    double ssum = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) ssum += __shfl(part, gbase + stride * k + first);
    const double scaled = sqrt(ssum / 128.0);
    PidState npid;
    npid.inv = st.inv; npid.pinv = st.pinv; npid.at_dtmin = st.at_dtmin;
    double ntprev, ntnext;
    int code = 0;
    const bool keep = pid_adapt<PID_INTEGRAL>(a.pid, scaled, ts0, ts1, npid, ntprev, ntnext, code);
    ntprev = jmin(ntprev, st.T1);
    if (ntnext > st.floor_t1) ntnext = keep ? st.T1 : ntprev + 0.5 * (st.T1 - ntprev);
    // weights of this iteration's weight-gradient rows: dt b_i for an accepted step
    if (lead) {
#pragma unroll
      for (int i = 0; i < S; ++i)
        a.rscale[((int64_t)q * S + i) * a.B_pad + rb0] = (run && keep) ? control * TL::v.b[i] : 0.0f;
    }
    if (run) {
      st.inv = npid.inv; st.pinv = npid.pinv; st.at_dtmin = npid.at_dtmin;
      ++st.nsteps;
      if (st.result == DFX_SUCCESSFUL) st.result = code;
      if (keep) {
#pragma unroll
        for (int j = 0; j < CPT; ++j) { y[j] = zy[j]; av[j] = za[j]; }
      }
      st.tprev = ntprev;
      st.tnext = ntnext;
      settle();
    }
  }
  // rows of the iterations this tile did not run carry no weight
  if (lead) {
    for (int qq = q; qq < a.Q; ++qq) {
#pragma unroll
      for (int i = 0; i < S; ++i) a.rscale[((int64_t)qq * S + i) * a.B_pad + rb0] = 0.0f;
    }
  }
  if (tid == 0 && q > 0) atomicMax(&a.counters[1], q);
  // Every row's state goes back, finished rows included: the next launch must see their
  // done flag (or it would run their intervals again from an older state).
  if (valid) {
    if (!st.done) {
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        a.ya[traj * 128 + c0 + j] = y[j];
        a.ya[traj * 128 + 64 + c0 + j] = av[j];
      }
    }
    if (lead) {
      a.rows[traj] = st;
      if (!st.done) atomicAdd(&a.counters[0], 1);
    }
  }
}

}  // namespace dfx

using namespace dfx;

namespace {

int64_t padded_batch(int64_t B) { return (B + MLP_TILE - 1) / MLP_TILE * MLP_TILE; }

// Rows that the row buffers are sized for: seven evaluations of every trajectory per step of a
// segment (which writes 1 + 6 per step) or per iteration of a backsolve launch, in whole
// blocks of 4,096, the sizes that callers of dfx_mlp_*_workspace know.
int64_t step_rows(int64_t B, int32_t steps) { return padded_batch(B) * 7 * (int64_t)steps; }
int64_t alloc_rows(int64_t B, int32_t steps) { return (step_rows(B, steps) + 4095) / 4096 * 4096; }

RowBufs row_bufs(void* rows, int64_t nrow) {
  RowBufs R;
  float* base = reinterpret_cast<float*>(rows);
  for (int i = 0; i < 6; base += nrow * kRowWidths[i], ++i) R.b[i] = base;
  return R;
}

// The backsolve's state buffer: ya [B_pad, 128] floats, rows [B_pad] BsRow, rscale [nrow]
// floats (every row of the row buffers), counters [2] int32; 256-byte aligned.
struct BsStateLayout {
  size_t ya, rows, rscale, counters, total;
};
BsStateLayout bs_state_layout(int64_t Bp, int64_t nrow) {
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  BsStateLayout l;
  l.ya = 0;
  l.rows = up(l.ya + (size_t)Bp * 128 * sizeof(float));
  l.rscale = up(l.rows + (size_t)Bp * sizeof(BsRow));
  l.counters = up(l.rscale + (size_t)nrow * sizeof(float));
  l.total = up(l.counters + 2 * sizeof(int32_t));
  return l;
}

// Zero the launch counters.
__global__ void bs_reset_kernel(int32_t* counters) {
  if (threadIdx.x < 2) counters[threadIdx.x] = 0;
}

// The weight gradients of `blocks` row blocks (SC: per-row weights rscale) added to dw.
template <bool SC>
void launch_dw(const RowBufs& R, float* partial, int64_t blocks, const int32_t* evals, int slots,
               const float* rscale, float* dw, hipStream_t s) {
  const int nch = dw_chunks(blocks);
  const DwLayout lay = dw_layout();
  float* partial_db = partial + (int64_t)nch * lay.first[3] * 1024;
  const int groups = (nch + kXcds - 1) / kXcds;
  const int npc = dw_pieces_of(0) + dw_pieces_of(1) + dw_pieces_of(2);
  hipLaunchKernelGGL((mlp_dw_gemm_kernel<SC>), dim3(kXcds * npc * groups), dim3(64), 0, s, R,
                     partial, partial_db, blocks, nch, evals, slots, rscale);
  const int nblk = lay.first[3] * 4 + ((2 * MLP_H + MLP_D) / 4 + 63) / 64;
  hipLaunchKernelGGL(mlp_dw_reduce_kernel, dim3(nblk), dim3(256), 0, s, partial, partial_db, nch,
                     dw);
}

// Floats of the weight-gradient partials of `blocks` row blocks; behind them, for a segment,
// come its tiles' evaluation counts and (float32 form) the weights' flags and three-piece planes.
int64_t partial_floats(int64_t blocks) {
  return (dw_chunks(blocks) * ((int64_t)dw_layout().first[3] * 1024 + 2 * MLP_H + MLP_D) + 63) / 64 * 64;
}

// One segment: the recompute + sweep kernel on three-piece weights (a bf16 buffer as it is;
// a float32 one split into the tail of io->partial first), the same on float32 MFMA for the
// tiles that it marked (float32 form), then the weight-gradient GEMM over the float32 row
// buffers and the fixed-order reduction.
int run_segment(const dfx_mlp_problem* p, const void* packed, const float* b1, const float* b2,
                const float* b3, const dfx_mlp_adj_io* io, int32_t seg, int32_t seg_steps,
                hipStream_t s) {
  using P = PolicyBF16x3;
  constexpr int NW = 8;  // two waves per SIMD; four (one per SIMD) took a sixth longer
  AdjArgs a;
  memset(&a, 0, sizeof(a));
  a.grid = io->grid; a.ckpt = io->ckpt; a.stats = io->stats; a.ts = io->ts; a.ys_bar = io->ys_bar;
  a.ybar = io->ybar; a.zs = io->zs;
  a.B = p->batch;
  a.max_steps = p->max_steps; a.n_ckpt = dfx_mlp_n_ckpt(p); a.C = p->ckpt_every;
  a.Cs = seg_steps; a.seg = seg; a.n_ts = p->n_ts; a.ts_stride = p->ts_stride;
  a.n_out = (p->save_t0 ? 1 : 0) + p->n_ts + (p->save_t1 ? 1 : 0);
  a.save_t0 = p->save_t0; a.t0 = p->t0; a.t1 = p->t1;
  const int slots = 1 + 6 * seg_steps;
  const int64_t ntiles64 = padded_batch(p->batch) / MLP_TILE, blocks = ntiles64 * slots;
  a.evals = reinterpret_cast<int32_t*>(io->partial + partial_floats(blocks));
  const bool f32 = p->precision == DFX_F32;
  const void* pieces = packed;
  if (f32) {
    int32_t* wflags = a.evals + (ntiles64 + 63) / 64 * 64;
    __bf16* planes = reinterpret_cast<__bf16*>(wflags + (kWeightFlags + 63) / 64 * 64);
    const unsigned nb = (unsigned)(mlp_pack_layout(1).total / 256);
    hipLaunchKernelGGL(mlp_split_packed_kernel, dim3(nb), dim3(256), 0, s,
                       reinterpret_cast<const float*>(packed), b1, b2, b3, planes, wflags);
    pieces = planes;
    a.wflags = wflags;
  }
  const MlpWeights<P> W = mlp_weights_from<P>(pieces, P::PIECES, b1, b2, b3);
  const RowBufs R = row_bufs(io->rows, alloc_rows(p->batch, seg_steps));
  const unsigned ntiles = (unsigned)ntiles64;
  auto sweep = [&](auto policy, auto&& w) {
    using Q = decltype(policy);
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_adj_segment_kernel<Q, NW>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(AdjLds<Q>));
    hipLaunchKernelGGL((mlp_adj_segment_kernel<Q, NW>), dim3(ntiles), dim3(64 * NW),
                       sizeof(AdjLds<Q>), s, a, w, R);
  };
  sweep(P{}, W);
  if (f32) sweep(PolicyF32{}, mlp_weights_from<PolicyF32>(packed, 1, b1, b2, b3));
  launch_dw<false>(R, io->partial, blocks, a.evals, slots, nullptr, io->dw, s);
  return hipGetLastError() == hipSuccess ? DFX_OK : DFX_E_HIP;
}

}  // namespace

extern "C" {

int dfx_mlp_adj_workspace(const dfx_mlp_problem* p, int32_t seg_steps, size_t* zs_bytes,
                          size_t* rows_bytes, size_t* partial_bytes) {
  if (!p || seg_steps <= 0 || !zs_bytes || !rows_bytes || !partial_bytes) return DFX_E_ARG;
  const int64_t Bp = padded_batch(p->batch);
  const int64_t ntiles = Bp / MLP_TILE;
  *zs_bytes = (size_t)(step_rows(p->batch, seg_steps) * MLP_D) * sizeof(float);
  *rows_bytes = (size_t)(alloc_rows(p->batch, seg_steps) * kRowFloats) * sizeof(float);
  *partial_bytes = (size_t)(partial_floats(ntiles * (1 + 6 * (int64_t)seg_steps)) +
                            (ntiles + 63) / 64 * 64) * sizeof(float);
  if (p->precision == DFX_F32)
    *partial_bytes += (kWeightFlags + 63) / 64 * 64 * sizeof(int32_t) +
                      (size_t)mlp_pack_layout(3).total * sizeof(__bf16);
  return DFX_OK;
}

int dfx_mlp_backsolve_workspace(const dfx_mlp_problem* p, int32_t chunk_iters,
                                size_t* state_bytes, size_t* rows_bytes, size_t* partial_bytes) {
  if (!p || chunk_iters <= 0 || !state_bytes || !rows_bytes || !partial_bytes) return DFX_E_ARG;
  const int64_t Bp = padded_batch(p->batch);
  const int64_t nrow = alloc_rows(p->batch, chunk_iters);
  *state_bytes = bs_state_layout(Bp, nrow).total;
  *rows_bytes = (size_t)(nrow * kRowFloats) * sizeof(float);
  *partial_bytes = (size_t)partial_floats(step_rows(p->batch, chunk_iters) / MLP_TILE) * sizeof(float);
  return DFX_OK;
}

int dfx_mlp_backsolve(const dfx_mlp_problem* back, const void* packed, const float* b1,
                      const float* b2, const float* b3, const dfx_mlp_backsolve_io* io,
                      int32_t chunk_iters, int32_t first, void* stream) {
  if (!back || !packed || !b1 || !b2 || !b3 || !io) return DFX_E_ARG;
  if (back->d != MLP_D || back->hidden != MLP_H || back->solver != DFX_TSIT5) return DFX_E_ARG;
  if (back->precision != DFX_F32) return DFX_E_ARG;  // float32 products on a float32 packing
  if (chunk_iters <= 0 || isnan(back->dt0) || back->max_steps <= 0) return DFX_E_ARG;
  const int32_t n_out = (back->save_t0 ? 1 : 0) + back->n_ts + (back->save_t1 ? 1 : 0);
  if (!io->ys || !io->ts_out || !io->ys_bar || !io->state || !io->rows || !io->partial ||
      !io->dw || !io->ybar || !io->result)
    return DFX_E_ARG;
  if (back->batch == 0) return DFX_OK;
  BsArgs a;
  memset(&a, 0, sizeof(a));
  if (!mlp_pid_params(back, a.pid)) return DFX_E_ARG;
  const int64_t Bp = padded_batch(back->batch);
  const int64_t nrow = alloc_rows(back->batch, chunk_iters);
  const BsStateLayout sl = bs_state_layout(Bp, nrow);
  unsigned char* sb = reinterpret_cast<unsigned char*>(io->state);
  a.ys = io->ys; a.ts_out = io->ts_out; a.ys_bar = io->ys_bar;
  a.ya = reinterpret_cast<float*>(sb + sl.ya);
  a.rows = reinterpret_cast<BsRow*>(sb + sl.rows);
  a.rscale = reinterpret_cast<float*>(sb + sl.rscale);
  a.counters = reinterpret_cast<int32_t*>(sb + sl.counters);
  a.ybar = io->ybar; a.result = io->result;
  a.B = back->batch; a.B_pad = Bp;
  a.n_out = n_out; a.save_t0 = back->save_t0; a.max_steps = back->max_steps;
  a.Q = chunk_iters; a.first = first ? 1 : 0;
  a.t0 = back->t0; a.dt0 = back->dt0;
  // The backward solves run on float32 MFMA for both matmul forms (the caller packs the
  // weights for DFX_F32): the bfloat16 form's forward evaluates the float32-weight model too.
  using P = PolicyF32;
  const MlpWeights<P> W = mlp_weights_from<P>(packed, 1, b1, b2, b3);
  const RowBufs R = row_bufs(io->rows, nrow);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(bs_reset_kernel, dim3(1), dim3(64), 0, s, a.counters);
  const unsigned ntiles = (unsigned)(Bp / MLP_TILE);
  // four waves per tile: 256 VGPRs without spills (eight spill 2 per lane; calls with 8,192
  // trajectories take 12.4 ms at four and 11.9 at eight, the same bits)
  constexpr int NWB = 4;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_backsolve_kernel<NWB>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(MlpLdsBack));
  hipLaunchKernelGGL((mlp_backsolve_kernel<NWB>), dim3(ntiles), dim3(64 * NWB),
                     sizeof(MlpLdsBack), s, a, W, R);
  launch_dw<true>(R, io->partial, step_rows(back->batch, chunk_iters) / MLP_TILE, nullptr, 0,
                  a.rscale, io->dw, s);
  return hipGetLastError() == hipSuccess ? DFX_OK : DFX_E_HIP;
}

int dfx_mlp_backsolve_status(const dfx_mlp_problem* back, int32_t chunk_iters,
                             const void* state, const int32_t** counters) {
  if (!back || chunk_iters <= 0 || !state || !counters) return DFX_E_ARG;
  const int64_t Bp = padded_batch(back->batch);
  const BsStateLayout sl = bs_state_layout(Bp, alloc_rows(back->batch, chunk_iters));
  *counters = reinterpret_cast<const int32_t*>(reinterpret_cast<const unsigned char*>(state) +
                                               sl.counters);
  return DFX_OK;
}

int dfx_mlp_adj_segment(const dfx_mlp_problem* p, const void* packed, const float* b1,
                        const float* b2, const float* b3, const dfx_mlp_adj_io* io,
                        int32_t segment, int32_t seg_steps, void* stream) {
  if (!p || !packed || !b1 || !b2 || !b3 || !io) return DFX_E_ARG;
  if (p->d != MLP_D || p->hidden != MLP_H || p->solver != DFX_TSIT5) return DFX_E_ARG;
  if (p->precision != DFX_F32 && p->precision != DFX_BF16_F32) return DFX_E_ARG;
  if (p->ckpt_every <= 0 || seg_steps <= 0 || seg_steps > p->ckpt_every || segment < 0 ||
      segment >= dfx_mlp_n_ckpt(p))
    return DFX_E_ARG;
  if (!io->grid || !io->ckpt || !io->stats || !io->ys_bar || !io->ybar || !io->zs || !io->rows ||
      !io->partial || !io->dw)
    return DFX_E_ARG;
  if (p->n_ts > 0 && !io->ts) return DFX_E_ARG;
  if (p->ts_stride != 0 && p->ts_stride != p->n_ts) return DFX_E_ARG;
  if (p->batch == 0) return DFX_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return run_segment(p, packed, b1, b2, b3, io, segment, seg_steps, s);
}

}  // extern "C"
