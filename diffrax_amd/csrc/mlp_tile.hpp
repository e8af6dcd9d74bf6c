// mlp_tile.hpp -- the registered neural vector field f(y) = tanh(W3 sp(W2 sp(W1 y + b1) + b2) + b3)
// (sp = softplus; d = 64 -> 256 -> 256 -> 64) evaluated for a tile of 32 trajectories by one
// workgroup of NW = 4 or 8 waves on MFMA, plus its vector-Jacobian product.
//
// Layout of one tile:
//  - owner threads: 2 NW adjacent lanes of one wave own a trajectory, 32 / NW consecutive
//    state components each;
//  - activations live in LDS, row-major [32 rows][K + padding] (float32 with the columns of a
//    fragment reordered, PolicyF32::pos); every MFMA reads its fragment (32 rows x KSTEP)
//    straight from there;
//  - weights come as MFMA fragments from a packed copy (dfx_mlp_pack; fragment (n_tile,
//    k_step) is 64 lanes x KA contiguous elements, one coalesced load per lane).  In the
//    solve's products they are the A operand and the activations B, so a lane's accumulators
//    are runs of four outputs of one trajectory; where the adjoint writes row buffers it is
//    the other way round (Gemm3's WA);
//  - layers 1 and 2: each wave produces 256 / NW output columns; layer 3 (64 outputs, K = 256)
//    is split over K in quarters, whose four partial sums meet in LDS, where the owner
//    threads add them in order (MlpWaves).
// Precision policies: three-piece BF16 operands with f32 accumulate
// (v_mfma_f32_32x32x16_bf16), or f32 throughout (v_mfma_f32_32x32x2f32).  Activation
// functions are evaluated in f32.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/diffrax_amd.h"
#include "erk_common.hpp"

namespace dfx {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));

constexpr int MLP_D = 64;
constexpr int MLP_H = 256;
constexpr int MLP_TILE = 32;
constexpr int MLP_THREADS = 256;

// Float32 MFMA.  One fragment is four consecutive k steps of v_mfma_f32_32x32x2_f32 (k = 8g
// .. 8g + 7 of the sum): a lane holds its four k values together, one 16-byte load from the
// packed weights and one from LDS for four MFMAs, where a fragment per MFMA (4-byte loads)
// left the matrix cores waiting on L2 for half of the time (8,192 trajectories: 0.52 ms).
struct PolicyF32 {
  using act_t = float;
  typedef float frag_t __attribute__((ext_vector_type(4)));
  static constexpr int KSTEP = 8;  // k per fragment
  static constexpr int KA = 4;     // elements per lane per fragment
  static constexpr int PIECES = 1;
  // The k of element j of a lane in half h (lanes 0-31, 32-63) within the fragment: MFMA j
  // takes k = 2j from half 0 and 2j + 1 from half 1.
  __host__ __device__ static constexpr int k_of(int h, int j) { return 2 * j + h; }
  // Where column k of an activation row is stored, so that a lane's four lie together.
  __host__ __device__ static constexpr int pos(int k) {
    return (k & ~7) | ((k & 1) << 2) | ((k >> 1) & 3);
  }
  __device__ __forceinline__ static floatx16_t mfma(frag_t a, frag_t b, floatx16_t c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
};

// BF16 MFMA (float32 accumulate) with every operand carried as three bfloat16 pieces,
// v = p0 + p1 + p2 exactly for a float32 v (split3).  The six products p_i q_j with
// i + j <= 2 give each layer sum to ~2^-24 relative, float32 MFMA accuracy, from six bf16
// MFMA passes: the float32-weight model itself is evaluated (the weights are split, not
// rounded), and the products of the leading pieces accumulate apart from the five
// correction products.  bf16 MFMA has 16x the float32 MFMA rate on gfx950.  A single
// bfloat16 operand (8 bits) would turn f into a step function at the scale of the O(dt f)
// differences between stages, and the embedded error estimate would measure rounding noise.
struct PolicyBF16x3 {
  using act_t = __bf16;
  using frag_t = bf16x8_t;
  static constexpr int KSTEP = 16;  // K per MFMA
  static constexpr int KA = 8;      // elements per lane per fragment
  static constexpr int PAD = 8;     // LDS row padding (elements); keeps 16-byte alignment
  static constexpr int PIECES = 3;
  __host__ __device__ static constexpr int k_of(int h, int j) { return 8 * h + j; }
  __device__ __forceinline__ static frag_t load_a(const act_t* p) {
    return *reinterpret_cast<const frag_t*>(p);
  }
  __device__ __forceinline__ static floatx16_t mfma(frag_t a, frag_t b, floatx16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

// v = p0 + p1 + p2 with bfloat16 pieces: each residual is exact in float32 and the last
// one has at most 8 significant bits.
__device__ __forceinline__ void split3(float v, __bf16& p0, __bf16& p1, __bf16& p2) {
  p0 = (__bf16)v;
  const float r1 = v - (float)p0;
  p1 = (__bf16)r1;
  p2 = (__bf16)(r1 - (float)p1);
}

// split3 of four values, the pieces packed for 8-byte LDS stores.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
struct Split4 {
  uint2 p[3];
};
__device__ __forceinline__ Split4 split3x4(float a, float b, float c, float d) {
  Split4 s;
  floatx2_t lo = {a, b}, hi = {c, d};
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2_t ql = __builtin_convertvector(lo, bf16x2_t);
    const bf16x2_t qh = __builtin_convertvector(hi, bf16x2_t);
    s.p[i] = make_uint2(__builtin_bit_cast(unsigned, ql), __builtin_bit_cast(unsigned, qh));
    if (i < 2) {
      lo = lo - __builtin_convertvector(ql, floatx2_t);
      hi = hi - __builtin_convertvector(qh, floatx2_t);
    }
  }
  return s;
}

// Whether every value seen may be carried in three pieces in place of float32: zero, or of a
// magnitude from SPLIT_MIN up to a limit.  Down to 2^-110 the pieces hold all 24 bits (a
// bfloat16 ends at 2^-133, so below that a piece sum is off by at most 2^-134; products and
// sums below 2^-126 are kept, the MFMA does not flush them); an infinity has no pieces (inf -
// inf), and a number near the largest rounds up to one.  A caller that finds a value outside
// takes float32 MFMA: gradients of cotangents scaled by 2^-112 and 2^-116 were off by 5e-6 and
// 7e-5 in pieces and by 5e-7 and 8e-7 that way.
constexpr float SPLIT_MIN = 2.1175823681357508e-22f;   // 2^-72
struct SplitRange {
  float hi = 0.0f;            // the largest magnitude
  unsigned lo = 0xffffffffu;  // the least 2 bits - 1 of the magnitudes (of zero: the most)
  __device__ __forceinline__ void most(float a, float b, float c, float d) {
    hi = fmaxf(fmaxf(hi, fmaxf(fabsf(a), fabsf(b))), fmaxf(fabsf(c), fabsf(d)));
    asm("" : "+v"(hi));
  }
  __device__ __forceinline__ void least(float a, float b, float c, float d) {
    auto key = [](float v) { return (__builtin_bit_cast(unsigned, v) << 1) - 1u; };
    lo = min(min(lo, min(key(a), key(b))), min(key(c), key(d)));
    asm("" : "+v"(lo));  // (not split into comparisons whose masks fill the scalar registers)
  }
  __device__ __forceinline__ void see(float a, float b, float c, float d) {
    most(a, b, c, d);
    least(a, b, c, d);
  }
  __device__ __forceinline__ bool outside(float limit) const {
    return !(hi < limit) || lo < (__builtin_bit_cast(unsigned, SPLIT_MIN) << 1) - 1u;
  }
};

// Packed weight buffer: six matrices (w1, w2, w3 forward; w1t, w2t, w3t transposed), each
// `pieces` planes of its fragment array (bf16: the three split3 pieces, plane 0 the
// rounded weight; float32: one plane).  Element offsets of plane 0 and plane sizes.
struct MlpPackLayout {
  int64_t off[6], size[6], total;
};
__host__ __device__ inline MlpPackLayout mlp_pack_layout(int pieces) {
  const int64_t D = MLP_D, H = MLP_H;
  const int64_t sz[6] = {H * D, H * H, D * H, D * H, H * H, H * D};
  MlpPackLayout l;
  int64_t o = 0;
  for (int i = 0; i < 6; ++i) {
    l.off[i] = o;
    l.size[i] = sz[i];
    o += sz[i] * pieces;
  }
  l.total = o;
  return l;
}

// The packed matrices' input columns K (MFMA reduction lengths), and whether B[k][n] =
// W[n][k] (forward) or W[k][n] (transposed).
struct MlpPackShape {
  int n, k, forward;
};
__host__ __device__ constexpr MlpPackShape mlp_pack_shape(int m) {
  return m == 0   ? MlpPackShape{MLP_H, MLP_D, 1}
         : m == 1 ? MlpPackShape{MLP_H, MLP_H, 1}
         : m == 2 ? MlpPackShape{MLP_D, MLP_H, 1}
         : m == 3 ? MlpPackShape{MLP_D, MLP_H, 0}
         : m == 4 ? MlpPackShape{MLP_H, MLP_H, 0}
                  : MlpPackShape{MLP_H, MLP_D, 0};
}

// The matrix m and element e within it of element `e` of all six, and the number of elements
// before it (times the pieces: its offset).  m = 6 past the end.
__host__ __device__ inline void mlp_pack_find(int& e, int& m, int& before) {
  m = before = 0;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const int size = mlp_pack_shape(i).n * mlp_pack_shape(i).k;
    if (m == i && e >= size) { e -= size; before += size; ++m; }
  }
}

// Element e of a packed matrix with K input columns <-> its (n, k): fragments (n tile,
// k step) of 64 lanes x KA elements.
template <class P>
__host__ __device__ inline void mlp_frag_nk(int e, int K, int& n, int& k) {
  const int j = e % P::KA, lane = e / P::KA % 64;
  const int f = e / P::KA / 64;
  const int nks = K / P::KSTEP;  // 4, 8, 16 or 32
  const int nt = f / nks;
  n = nt * 32 + (lane & 31);
  k = (f - nt * nks) * P::KSTEP + P::k_of(lane >> 5, j);
}
template <class P>
__host__ __device__ inline int mlp_frag_index(int n, int k, int K) {
  const int kk = k % P::KSTEP;
  int h = 0, j = 0;
  while (P::k_of(h, j) != kk) {
    if (++j == P::KA) { j = 0; ++h; }
  }
  return ((n / 32 * (K / P::KSTEP) + k / P::KSTEP) * 64 + (n & 31) + 32 * h) * P::KA + j;
}

// Packed weights of one solve.  Forward fragments: B[k][n] = W[n][k].  Backward fragments
// (transposed products): B[k][n] = W[k][n].
template <class P>
struct MlpWeights {
  const typename P::act_t* w1;   // layer 1 forward fragments (N = 256, K = 64)
  const typename P::act_t* w2;   // layer 2 forward (N = 256, K = 256)
  const typename P::act_t* w3;   // layer 3 forward (N = 64, K = 256)
  const typename P::act_t* w1t;  // z-bar = d1 . W1   (N = 64, K = 256)
  const typename P::act_t* w2t;  // h1-bar = d2 . W2  (N = 256, K = 256)
  const typename P::act_t* w3t;  // h2-bar = d3 . W3  (N = 256, K = 64)
  const float* b1;
  const float* b2;
  const float* b3;
  int64_t plane1, plane2, plane3;  // elements between the pieces of w1, w2, w3 (PIECES > 1)
};

// The weights of a packed buffer (mlp_pack_layout) for a policy; a one-piece policy on a
// three-piece buffer reads plane 0.
template <class P>
__host__ __device__ inline MlpWeights<P> mlp_weights_from(const void* packed, int pieces,
                                                          const float* b1, const float* b2,
                                                          const float* b3) {
  const MlpPackLayout l = mlp_pack_layout(pieces);
  const typename P::act_t* base = reinterpret_cast<const typename P::act_t*>(packed);
  MlpWeights<P> W;
  W.w1 = base + l.off[0]; W.w2 = base + l.off[1]; W.w3 = base + l.off[2];
  W.w1t = base + l.off[3]; W.w2t = base + l.off[4]; W.w3t = base + l.off[5];
  W.b1 = b1; W.b2 = b2; W.b3 = b3;
  W.plane1 = l.size[0]; W.plane2 = l.size[1]; W.plane3 = l.size[2];
  return W;
}

template <class P>
struct MlpLds;

// Float32: columns of x, h1 and h2 at P::pos.  The row strides (17 and 65 16-byte units) are
// odd, so the 16-byte reads of 32 rows are free of bank conflicts.  The split-K partials of
// layer 3 take the h1 buffer, which nobody reads after layer 2.  79,104 bytes: two
// workgroups per CU.
template <>
struct MlpLds<PolicyF32> {
  static constexpr int LDX = MLP_D + 4;
  static constexpr int LDH = MLP_H + 4;
  static constexpr int LDP = MLP_D + 4;
  float x[MLP_TILE * LDX];      // layer-1 input (stage value)
  float h1[4 * MLP_TILE * LDP]; // softplus(layer 1) [32][LDH], then the partials [4][32][LDP]
  float h2[MLP_TILE * LDH];     // softplus(layer 2)
  float bias[2 * MLP_H + MLP_D];
  __device__ __forceinline__ float* part() { return h1; }
};
static_assert(4 * MlpLds<PolicyF32>::LDP >= MlpLds<PolicyF32>::LDH, "h1 fits");
static_assert(2 * sizeof(MlpLds<PolicyF32>) <= 160 * 1024, "two workgroups per CU");

// ---- activations ------------------------------------------------------------------------
// Softplus / tanh through the hardware exp2, log2 and reciprocal (about 1 ulp each): the
// vector field stays within 8.4e-7 of a float64 evaluation (the libm forms gave 8e-7)
// and the forward runs 2x faster, its VALU work having been the larger part of a step.
__device__ __forceinline__ float softplus_f(float x) {
  // jax.nn.softplus(x) = logaddexp(x, 0) = max(x, 0) + log1p(exp(-|x|))
  const float e = __builtin_amdgcn_exp2f(-fabsf(x) * 1.4426950408889634f);
  return fmaxf(x, 0.0f) + 0.6931471805599453f * __builtin_amdgcn_logf(1.0f + e);
}
__device__ __forceinline__ float tanh_f(float x) {
  // tanh(x) = sign(x) (1 - 2 / (exp(2|x|) + 1))
  const float e = __builtin_amdgcn_exp2f(fminf(2.0f * fabsf(x), 60.0f) * 1.4426950408889634f);
  const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
  return copysignf(t, x);
}
// derivative of softplus from its value h = softplus(s): sigmoid(s) = 1 - exp(-h)
__device__ __forceinline__ float dsoftplus_from_value(float h) {
  return 1.0f - __builtin_amdgcn_exp2f(-h * 1.4426950408889634f);
}

// C layout: accumulator element v (= 4i + j) of lane l sits at row 8i + (l/32)*4 + j, column
// l%32 of the 32x32 tile.

// ---- the float32 form ------------------------------------------------------------------
// One wave's share of a layer: acc[t] = sum over fragments [g0, g0 + G) of W . x, the weights
// of output tile nt0 + t as the A operand and the activation rows (LDS) as B, so that a
// lane's accumulators are four runs of four consecutive outputs of one trajectory (wide
// LDS stores).  NG: fragments along K of the matrix.  Weights come from L2, whose latency
// is longer than a fragment's MFMAs: PF fragments are in flight, the first of them loaded
// by preload() ahead of the barrier that the activations wait for.
template <int NG, int NT, int PF = 4>
struct GemmF32 {
  using P = PolicyF32;
  using frag_t = P::frag_t;
  frag_t b[PF][NT];
  const frag_t* wp;
  __device__ __forceinline__ void preload(const float* w, int nt0, int g0, int lane) {
    wp = reinterpret_cast<const frag_t*>(w) + ((int64_t)nt0 * NG + g0) * 64 + lane;
#pragma unroll
    for (int p = 0; p < PF; ++p) {
#pragma unroll
      for (int t = 0; t < NT; ++t) b[p][t] = wp[(t * NG + p) * 64];
    }
  }
  // A ring slot is refilled right after its MFMAs (the load may write the registers they
  // read), so the loop carries no copies that would wait for the loads it just issued.
  template <int G>
  __device__ __forceinline__ void run(const float* act, int ld, int g0, floatx16_t (&acc)[NT],
                                      int lane) {
    static_assert(G % PF == 0 && G >= PF && PF % 2 == 0, "whole rings");
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = floatx16_t{};
    const float* ap = act + (lane & 31) * ld + 8 * g0 + 4 * (lane >> 5);
    auto load_a = [&](int g) { return *reinterpret_cast<const frag_t*>(ap + 8 * g); };
    frag_t a[2] = {load_a(0), load_a(1)};
    auto ring = [&](int g, auto last) {
#pragma unroll
      for (int p = 0; p < PF; ++p) {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = P::mfma(b[p][t], a[p & 1], acc[t]);
        if (!decltype(last)::value) {
#pragma unroll
          for (int t = 0; t < NT; ++t) b[p][t] = wp[(t * NG + g + p + PF) * 64];
        }
        if (!decltype(last)::value || p + 2 < PF) a[p & 1] = load_a(g + p + 2);
        __builtin_amdgcn_sched_barrier(0);  // the loads stay here, ahead of the next MFMAs
      }
    };
#pragma unroll 1
    for (int g = 0; g < G - PF; g += PF) ring(g, std::false_type{});
    ring(G - PF, std::true_type{});
  }
};

// ---- the three-piece bf16 form --------------------------------------------------------
// LDS: the three pieces of the layer-1 input and of both hidden activations (115 KB).  The
// split-K partials of layer 3 reuse the h1 planes, which nobody reads after layer 2.
template <>
struct MlpLds<PolicyBF16x3> {
  static constexpr int LDX = MLP_D + PolicyBF16x3::PAD;
  static constexpr int LDH = MLP_H + PolicyBF16x3::PAD;
  static constexpr int LDP = MLP_D + 4;
  __bf16 x[3][MLP_TILE * LDX];
  __bf16 h1[3][MLP_TILE * LDH];
  __bf16 h2[3][MLP_TILE * LDH];
  float bias[2 * MLP_H + MLP_D];
  __device__ __forceinline__ float* part() { return reinterpret_cast<float*>(&h1[0][0]); }
};
static_assert(4 * MLP_TILE * MlpLds<PolicyBF16x3>::LDP * sizeof(float) <=
                  sizeof(MlpLds<PolicyBF16x3>::h1),
              "layer-3 partials fit in the h1 planes");

// Store N consecutive values (4 or 8, from a multiple of N) of the layer-1 input's row r.
template <int N>
__device__ __forceinline__ void store_inputs(MlpLds<PolicyBF16x3>& L, int r, int c0,
                                             const float (&v)[N]) {
#pragma unroll
  for (int j = 0; j < N; j += 4) {
    const Split4 s = split3x4(v[j], v[j + 1], v[j + 2], v[j + 3]);
#pragma unroll
    for (int pc = 0; pc < 3; ++pc)
      *reinterpret_cast<uint2*>(&L.x[pc][r * L.LDX + c0 + j]) = s.p[pc];
  }
}
template <int N>
__device__ __forceinline__ void store_inputs(MlpLds<PolicyF32>& L, int r, int c0,
                                             const float (&v)[N]) {
#pragma unroll
  for (int j = 0; j < N; j += 4) {
    float* o = L.x + r * L.LDX + PolicyF32::pos(c0 + j);
    *reinterpret_cast<float2*>(o) = make_float2(v[j], v[j + 2]);
    *reinterpret_cast<float2*>(o + 4) = make_float2(v[j + 1], v[j + 3]);
  }
}

// Kernels call this once before their first evaluation (a barrier follows it there).
template <class P>
__device__ __forceinline__ void mlp_begin(const MlpWeights<P>& W, MlpLds<P>& L) {
  for (int i = threadIdx.x; i < 2 * MLP_H + MLP_D; i += blockDim.x)
    L.bias[i] = i < MLP_H ? W.b1[i] : (i < 2 * MLP_H ? W.b2[i - MLP_H] : W.b3[i - 2 * MLP_H]);
}

// The three-piece product of one wave: acc[t] (32x32 f32) = sum over k steps of W . x, both
// operands in three pieces: the activation rows from LDS planes, the weights of output tile
// nt0 + t from L2.  The leading products w0 x0 accumulate in acc, the five corrections (w1
// x0, w0 x1, w2 x0, w1 x1, w0 x2) apart, added at the end.
// WA: the weights are the A operand, so that a lane's accumulators are four runs of four
// consecutive outputs of one trajectory; else the activations are, and the runs are four
// consecutive trajectories of one output.  Either way the same bits.
// PF k steps of weights are in flight, the first loaded by preload() ahead of the barrier
// that the activations wait for; a ring slot is refilled right after its MFMAs, and the
// loads are pinned there.  One evaluation of a 32-trajectory tile by eight waves takes 23,000
// cycles, 9,200 of them MFMA on every SIMD and 6,700 VALU (softplus and the splits, between
// the barriers, so that little of it overlaps); with a ring that was copied (and so waited
// for), 2-byte LDS stores and a split per value it took 26,400 and 10,100 VALU (8,192
// trajectories: 0.33-0.35 against 0.30 ms; 33: 0.266 against 0.234).
template <int NKS, int NT, bool WA = true, int PF = 2>
struct Gemm3 {
  using P = PolicyBF16x3;
  using frag_t = P::frag_t;
  frag_t b[PF][3][NT];
  const frag_t* wp;
  int plane;
  __device__ __forceinline__ static floatx16_t mm(frag_t w, frag_t x, floatx16_t c) {
    return WA ? P::mfma(w, x, c) : P::mfma(x, w, c);
  }
  __device__ __forceinline__ void load(int p, int k) {
#pragma unroll
    for (int pc = 0; pc < 3; ++pc) {
#pragma unroll
      for (int t = 0; t < NT; ++t) b[p][pc][t] = wp[pc * plane + (t * NKS + k) * 64];
    }
  }
  __device__ __forceinline__ void preload(const __bf16* w, int64_t pl, int nt0, int k0, int lane) {
    wp = reinterpret_cast<const frag_t*>(w) + ((int64_t)nt0 * NKS + k0) * 64 + lane;
    plane = (int)(pl / P::KA);
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p, p);
  }
  template <int G>
  __device__ __forceinline__ void run(const __bf16* act, int aplane, int ld, int k0,
                                      floatx16_t (&acc)[NT], int lane) {
    static_assert(G % PF == 0 && G >= PF, "whole rings");
    floatx16_t sml[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) { acc[t] = floatx16_t{}; sml[t] = floatx16_t{}; }
    const __bf16* ap = act + (lane & 31) * ld + P::KSTEP * k0 + P::KA * (lane >> 5);
    frag_t x[2][3];
    auto load_x = [&](int q, int k) {
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) x[q][pc] = P::load_a(ap + pc * aplane + P::KSTEP * k);
    };
    load_x(0, 0);
    load_x(1, 1);
    auto ring = [&](int g, auto last) {
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const int q = p & 1;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          acc[t] = mm(b[p][0][t], x[q][0], acc[t]);
          sml[t] = mm(b[p][1][t], x[q][0], sml[t]);
          sml[t] = mm(b[p][0][t], x[q][1], sml[t]);
          sml[t] = mm(b[p][2][t], x[q][0], sml[t]);
          sml[t] = mm(b[p][1][t], x[q][1], sml[t]);
          sml[t] = mm(b[p][0][t], x[q][2], sml[t]);
        }
        if (!decltype(last)::value) load(p, g + p + PF);
        if (!decltype(last)::value || p + 2 < PF) load_x(q, g + p + 2);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll 1
    for (int g = 0; g < G - PF; g += PF) ring(g, std::false_type{});
    ring(G - PF, std::true_type{});
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = acc[t] + sml[t];
  }
};

// The adjoint's row buffers hold float32 rows in blocks of 32 (one tile's rows of one stage),
// each 32-column piece of a block in the accumulator order of its MFMA tile: the four rows
// 8i + 4(l/32) + j, j = 0..3, of column l%32 are one float4 of lane l.  The epilogues that
// produce a block store it in whole lines, and a lane's sixteen values are the k values of
// two MFMA operands of the weight-gradient product (whose k are the rows).
__host__ __device__ inline int64_t rows_frag(int64_t block, int width, int t, int i, int lane) {
  return (((block * (width / 32) + t) * 4 + i) * 64 + lane) * 4;
}
__host__ __device__ inline int64_t rows_index(int64_t block, int width, int row, int col) {
  return rows_frag(block, width, col / 32, row / 8, col % 32 + 32 * (row % 8 / 4)) + row % 4;
}

// Store four rows r .. r + 3 of one column in the three planes of an LDS buffer.
__device__ __forceinline__ void store_col4(__bf16* buf, int plane, int ld, int r, int col,
                                           const float4 v) {
  const Split4 s = split3x4(v.x, v.y, v.z, v.w);
#pragma unroll
  for (int pc = 0; pc < 3; ++pc) {
    unsigned short* o = reinterpret_cast<unsigned short*>(buf + pc * plane + r * ld + col);
    o[0] = (unsigned short)s.p[pc].x;
    o[ld] = (unsigned short)(s.p[pc].x >> 16);
    o[2 * ld] = (unsigned short)s.p[pc].y;
    o[3 * ld] = (unsigned short)(s.p[pc].y >> 16);
  }
}

// The tile's waves split the work: layers 1 and 2 by output columns (NT12 tiles of 32 per
// wave), layer 3 by K quarters (four waves: both 32-column tiles of one quarter; eight
// waves: one tile of one quarter), into the same four partial slabs.  The owners of a row
// hold 32 / NW of its components.
template <int NW>
struct MlpWaves {
  static_assert(NW == 4 || NW == 8, "four or eight waves per tile");
  static constexpr int NT12 = 8 / NW;
  static constexpr int NT3 = NW == 4 ? 2 : 1;
  static constexpr int CPT = 32 / NW;
  __device__ static int nt3(int wave) { return NW == 4 ? 0 : (wave & 1); }
  __device__ static int quarter(int wave) { return NW == 4 ? wave : (wave >> 1); }
};

// Layer 3's split-K partials (accumulators with the outputs along a lane's runs), which take
// the h1 buffer (layer 2, its last reader, is behind a barrier), and the output from them.
template <int NT3>
__device__ __forceinline__ void put_partials(const floatx16_t (&acc)[NT3], float* part, int ldp,
                                             int qk, int n3, int lane) {
#pragma unroll
  for (int t = 0; t < NT3; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<float4*>(part + (qk * MLP_TILE + (lane & 31)) * ldp + 32 * (n3 + t) + 8 * i +
                                 4 * (lane >> 5)) =
          make_float4(acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]);
  }
}
template <int CPT>
__device__ __forceinline__ void sum_partials(const float* part, int ldp, const float* b3,
                                             int owner_row, int owner_c0, float (&fout)[CPT]) {
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int c = owner_c0 + j;
    float s = part[(0 * MLP_TILE + owner_row) * ldp + c];
    s += part[(1 * MLP_TILE + owner_row) * ldp + c];
    s += part[(2 * MLP_TILE + owner_row) * ldp + c];
    s += part[(3 * MLP_TILE + owner_row) * ldp + c];
    fout[j] = tanh_f(s + b3[c]);
  }
}

// A row-buffered layer's values (unsplit accumulator runs: four trajectories of one output):
// to the block's pieces in `rows`, and split to the three planes of `buf`.
template <int NW, class F>
__device__ __forceinline__ void put_rows(MlpLds<PolicyBF16x3>& L, __bf16* buf, float* rows,
                                         int64_t block, int wave, int lane, F&& value) {
  constexpr int NT = MlpWaves<NW>::NT12;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tn = NT * wave + t;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 v = value(t, i);
      *reinterpret_cast<float4*>(rows + rows_frag(block, MLP_H, tn, i, lane)) = v;
      store_col4(buf, MLP_TILE * L.LDH, L.LDH, 8 * i + 4 * (lane >> 5), 32 * tn + (lane & 31), v);
    }
  }
}

// The forward of the three-piece form with its hidden activations kept in row buffers as well
// (the adjoint's recompute): mlp_forward's bits.
template <int NW>
__device__ __forceinline__ void mlp_forward_rows(const MlpWeights<PolicyBF16x3>& W,
                                                 MlpLds<PolicyBF16x3>& L, int wave, int lane,
                                                 int owner_row, int owner_c0,
                                                 float (&fout)[MlpWaves<NW>::CPT], float* h1_rows,
                                                 float* h2_rows, int64_t block) {
  using WV = MlpWaves<NW>;
  using LD = MlpLds<PolicyBF16x3>;
  constexpr int NT = WV::NT12, NT3 = WV::NT3, KS1 = MLP_D / 16, KS2 = MLP_H / 16;
  constexpr int HP = MLP_TILE * LD::LDH;
  floatx16_t acc[NT];
  auto hidden = [&](const float* bias) {
    return [&, bias](int t, int i) {
      const float b = bias[32 * (NT * wave + t) + (lane & 31)];
      return make_float4(softplus_f(acc[t][4 * i] + b), softplus_f(acc[t][4 * i + 1] + b),
                         softplus_f(acc[t][4 * i + 2] + b), softplus_f(acc[t][4 * i + 3] + b));
    };
  };
  Gemm3<KS1, NT, false> g1;
  Gemm3<KS2, NT, false> g2;
  Gemm3<KS2, NT3> g3;
  g1.preload(W.w1, W.plane1, NT * wave, 0, lane);
  g1.template run<KS1>(L.x[0], MLP_TILE * LD::LDX, L.LDX, 0, acc, lane);
  g2.preload(W.w2, W.plane2, NT * wave, 0, lane);
  __builtin_amdgcn_sched_barrier(0);  // issued here, ahead of the epilogue
  put_rows<NW>(L, L.h1[0], h1_rows, block, wave, lane, hidden(L.bias));
  __syncthreads();
  g2.template run<KS2>(L.h1[0], HP, L.LDH, 0, acc, lane);
  const int qk = WV::quarter(wave), n3 = WV::nt3(wave);
  g3.preload(W.w3, W.plane3, n3, qk * (KS2 / 4), lane);
  __builtin_amdgcn_sched_barrier(0);
  put_rows<NW>(L, L.h2[0], h2_rows, block, wave, lane, hidden(L.bias + MLP_H));
  __syncthreads();
  floatx16_t acc3[NT3];
  g3.template run<KS2 / 4>(L.h2[0], HP, L.LDH, qk * (KS2 / 4), acc3, lane);
  put_partials<NT3>(acc3, L.part(), L.LDP, qk, n3, lane);
  __syncthreads();
  sum_partials<WV::CPT>(L.part(), L.LDP, L.bias + 2 * MLP_H, owner_row, owner_c0, fout);
}

// Forward of the MLP on the tile: reads L.x (stage values), leaves softplus activations in
// L.h1 / L.h2 and returns f for the owner's 32 / NW components in fout (NW waves per tile;
// MlpWaves).  The three-piece form takes its first branch.
template <class P, int NW = 4, class Lds = MlpLds<P>>
__device__ __forceinline__ void mlp_forward(const MlpWeights<P>& W, Lds& L, int wave,
                                            int lane, int owner_row, int owner_c0,
                                            float (&fout)[MlpWaves<NW>::CPT]) {
  if constexpr (P::PIECES == 3) {
    using WV = MlpWaves<NW>;
    constexpr int NT = WV::NT12, NT3 = WV::NT3, KS1 = MLP_D / 16, KS2 = MLP_H / 16;
    constexpr int HP = MLP_TILE * Lds::LDH;
    const int half = lane >> 5, row = lane & 31;
    auto put_hidden = [&](const floatx16_t (&acc)[NT], const float* bias, __bf16* buf) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = 32 * (NT * wave + t) + 8 * i + 4 * half;
          const float4 bv = *reinterpret_cast<const float4*>(bias + n);
          const Split4 s = split3x4(softplus_f(acc[t][4 * i] + bv.x), softplus_f(acc[t][4 * i + 1] + bv.y),
                                    softplus_f(acc[t][4 * i + 2] + bv.z), softplus_f(acc[t][4 * i + 3] + bv.w));
#pragma unroll
          for (int pc = 0; pc < 3; ++pc)
            *reinterpret_cast<uint2*>(buf + pc * HP + row * L.LDH + n) = s.p[pc];
        }
      }
    };
    floatx16_t acc[NT];
    Gemm3<KS1, NT> g1;
    Gemm3<KS2, NT> g2;
    Gemm3<KS2, NT3> g3;
    g1.preload(W.w1, W.plane1, NT * wave, 0, lane);
    g1.template run<KS1>(L.x[0], MLP_TILE * Lds::LDX, L.LDX, 0, acc, lane);
    g2.preload(W.w2, W.plane2, NT * wave, 0, lane);
    __builtin_amdgcn_sched_barrier(0);  // issued here, ahead of the epilogue
    put_hidden(acc, L.bias, L.h1[0]);
    __syncthreads();
    g2.template run<KS2>(L.h1[0], HP, L.LDH, 0, acc, lane);
    const int qk = WV::quarter(wave), n3 = WV::nt3(wave);
    g3.preload(W.w3, W.plane3, n3, qk * (KS2 / 4), lane);
    __builtin_amdgcn_sched_barrier(0);
    put_hidden(acc, L.bias + MLP_H, L.h2[0]);
    __syncthreads();
    floatx16_t acc3[NT3];
    g3.template run<KS2 / 4>(L.h2[0], HP, L.LDH, qk * (KS2 / 4), acc3, lane);
    put_partials<NT3>(acc3, L.part(), L.LDP, qk, n3, lane);
    __syncthreads();
    sum_partials<WV::CPT>(L.part(), L.LDP, L.bias + 2 * MLP_H, owner_row, owner_c0, fout);
  } else {
    using WV = MlpWaves<NW>;
    constexpr int NT = WV::NT12, NT3 = WV::NT3;
    const int half = lane >> 5, row = lane & 31;
    // softplus of a layer's accumulators into buf: per run of four outputs n .. n + 3, the
    // even and the odd ones lie together (P::pos)
    auto put_hidden = [&](const floatx16_t (&acc)[NT], const float* bias, float* buf) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = 32 * (NT * wave + t) + 8 * i + 4 * half;
          const float4 bv = *reinterpret_cast<const float4*>(bias + n);
          const float h0 = softplus_f(acc[t][4 * i] + bv.x), h1 = softplus_f(acc[t][4 * i + 1] + bv.y);
          const float h2 = softplus_f(acc[t][4 * i + 2] + bv.z), h3 = softplus_f(acc[t][4 * i + 3] + bv.w);
          float* o = buf + row * L.LDH + P::pos(n);
          *reinterpret_cast<float2*>(o) = make_float2(h0, h2);
          *reinterpret_cast<float2*>(o + 4) = make_float2(h1, h3);
        }
      }
    };
    floatx16_t acc[NT];
    GemmF32<MLP_D / P::KSTEP, NT> g1;
    GemmF32<MLP_H / P::KSTEP, NT> g2;
    GemmF32<MLP_H / P::KSTEP, NT3> g3;
    g1.preload(W.w1, NT * wave, 0, lane);
    g1.template run<MLP_D / P::KSTEP>(L.x, L.LDX, 0, acc, lane);
    g2.preload(W.w2, NT * wave, 0, lane);
    __builtin_amdgcn_sched_barrier(0);  // issued here, ahead of the epilogue
    put_hidden(acc, L.bias, L.h1);
    __syncthreads();
    g2.template run<MLP_H / P::KSTEP>(L.h1, L.LDH, 0, acc, lane);
    // layer 3 (split-K): wave w sums a quarter of K
    constexpr int G3 = MLP_H / P::KSTEP / 4;
    const int qk = WV::quarter(wave), n3 = WV::nt3(wave);
    g3.preload(W.w3, n3, qk * G3, lane);
    __builtin_amdgcn_sched_barrier(0);
    put_hidden(acc, L.bias + MLP_H, L.h2);
    __syncthreads();
    floatx16_t acc3[NT3];
    g3.template run<G3>(L.h2, L.LDH, qk * G3, acc3, lane);
    put_partials<NT3>(acc3, L.part(), L.LDP, qk, n3, lane);
    __syncthreads();
    sum_partials<WV::CPT>(L.part(), L.LDP, L.bias + 2 * MLP_H, owner_row, owner_c0, fout);
  }
}

// The PID parameters of a neural-ODE problem (PIDController.__init__, pid.py:299-311, with
// its coefficients divided by the error order); false unless the controller is the integral
// one the neural-ODE kernels implement.
inline bool mlp_pid_params(const dfx_mlp_problem* p, PidParams& q) {
  const double error_order = isnan(p->error_order) ? 5.0 : p->error_order;
  q.rtol = p->rtol; q.atol = p->atol;
  q.coeff1 = (p->icoeff + p->pcoeff + p->dcoeff) / error_order;
  q.coeff2 = -(p->pcoeff + 2.0 * p->dcoeff) / error_order;
  q.coeff3 = p->dcoeff / error_order;
  q.dtmin = p->dtmin; q.dtmax = p->dtmax;
  q.has_dtmin = !isnan(p->dtmin); q.has_dtmax = !isnan(p->dtmax);
  q.force_dtmin = p->force_dtmin; q.factormin = p->factormin; q.factormax = p->factormax;
  q.safety = p->safety;
  q.pad_ = 0;
  return pid_is_integral(q);
}

}  // namespace dfx
