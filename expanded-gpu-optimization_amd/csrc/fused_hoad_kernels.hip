// gfx950 (MI355X) kernels for the forward-Laplacian jet of the fixed 2 -> 64x4 -> 1 tanh MLP
// and its adjoint-jet backward, plus the C ABI declared in include/fused_hoad.h.
//
// Math (same as /root/reference/csrc/fused_residual.cu:16-23 and
// /root/reference/src/fused_hoad/backends/forward_laplacian.py:1-17): every point carries a
// jet (v, J0, J1, L) = (value, d/dx, d/dy, Laplacian) through the network.
//   linear:  z_v = W v + b,  z_J = W J,  z_L = W L
//   tanh:    a = tanh(z_v), s = 1 - a^2
//            v = a,  J = s z_J,  L = s z_L - 2 a s (z_J0^2 + z_J1^2)
//   output:  u = w_out . v + b_out,  lap = w_out . L
//
// Register layout. A wave owns a tile of 16 points. Each hidden layer is the product
// Z[64 x 64] = W[64 x 64] * H[64 x (4 components x 16 points)], done on the bf16 matrix cores with
// operands split into three bf16 parts (float32 precision: see split_pair). With m = lane % 16
// and g = lane / 16, the MFMA accumulator of output block mb and component c holds, in register r,
//     Z[o = 16 mb + 4 g + r][c][point m].
// The contraction order is free, so half t of it (32 neurons, one v_mfma_f32_16x16x32_bf16 per
// product of parts) assigns lane group g the input neurons i = 32 t + 16 (e / 4) + 4 g + e % 4,
// e = 0..7. Then the B operand a lane must supply, H[i][c][point m], is the previous layer's
// accumulators of blocks 2 t and 2 t + 1 in the same lane: a layer's output, split, is already in
// the operand layout of the next layer, and the tanh-jet update (which needs the 4 components of one
// (neuron, point)) is local to a lane. Only the weights come from LDS.
//
// Scaled jet. With c = -2 log2(e) and lambda = log2(e), kernels carry the layer outputs as
//   (v', J0', J1', L') = (c v / 4, J0 / 2, J1 / 2, lambda L / 4)
// and stage the hidden weights as 4 W and the value biases as c b (exact power-of-two factors
// aside from c). The pre-activations then come out of the MFMAs as
//   z'_v = 4 W (c v / 4) + c b = c z_v,   z'_J = 4 W (J / 2) = 2 z_J,   z'_L = lambda z_L,
// and with s' = s / 4 and q' = |z'_J|^2 = 4 q the tanh jet keeps its form:
//   v' = (c / 4) tanh z_v,   J' = s' z'_J,   L' = s' (z'_L + v' q') = lambda L / 4
// (because c = -2 lambda), with the same scales at every layer. exp(-2 z_v) is exp2(z'_v) with
// no multiply, and (v', s') take 3 VALU + 2 transcendental instructions (tanh_scaled). Layer 0
// uses z'_J = 2 W0 columns; w_out is staged as 4 w_out / c and 4 w_out / lambda for u and lap.
// The backward is backpropagation through this scaled network (weights 4 W): its dW sums are
// of d/d(4 W), so the partial rows take a factor 4; bias gradients take c; layer-0 weight
// gradients c for the x terms and 2 for the z_J terms.
//
// What bounds the kernels: instruction issue and power. A wave's VALU instruction takes 4.4 clocks
// of its SIMD (exp and rcp 8.5), a bf16 MFMA 8.5 clocks of issue and 16 (16 x 16 x 32) or 32
// (32 x 32 x 16) of the matrix core, whose rest the VALU can use (v_dot2 instructions cannot). With
// random data in all the matrix cores the shader clock falls from 2.4 to about 2.1 GHz.
//
// LDS weight layout: every kernel but forward_split_kernel (which keeps a wave's 16 rows in
// registers) holds one copy of the split hidden weights in operand order (stage_operand_weights);
// the backward kernels read W^T operands from the same copy with transposed LDS reads.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "fused_hoad.h"
#include "mlp_abi.h"

namespace fhoad {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;
constexpr int kTile = 16;     // points per wave tile (the MFMA N dimension)

// Scale factors of the carried jet (see the header comment).
constexpr float kC = -2.8853900817779268f;       // c = -2 log2(e)
constexpr float kLambda = 1.4426950408889634f;   // lambda = log2(e)
constexpr float kKappa = -0.96090602783640284f;  // -8 / c^2 (tanh_jet_adjoint_layer0)
constexpr float kHalfC = 0.5f * kC;              // c / 2 (layer-0 weight gradients)

// Small parameter blocks in LDS (float offsets inside s_small), each [64] over neurons.
constexpr int kSmallCwx = 0;                       // c W0[:, 0]
constexpr int kSmallCwy = kSmallCwx + kHidden;     // c W0[:, 1]
constexpr int kSmallCb0 = kSmallCwy + kHidden;     // c b0
constexpr int kSmallWx = kSmallCb0 + kHidden;      // 2 W0[:, 0] (layer 0's z'_J0)
constexpr int kSmallWy = kSmallWx + kHidden;       // 2 W0[:, 1]
constexpr int kSmallQ0 = kSmallWy + kHidden;       // 4 (W0[:, 0]^2 + W0[:, 1]^2) = |z'_J|^2
constexpr int kSmallBh = kSmallQ0 + kHidden;       // c b1..b3, [3][64]
constexpr int kSmallWoutV = kSmallBh + 3 * kHidden;  // 4 w_out / c
constexpr int kSmallWoutL = kSmallWoutV + kHidden;   // 4 w_out / lambda
constexpr int kSmallBout = kSmallWoutL + kHidden;    // b_out
constexpr int kSmallFloats = kSmallBout + 4;

__device__ __forceinline__ f4 lds4(const float* p) { return *reinterpret_cast<const f4*>(p); }

// ---------------------------------------------------------------------------------------------
// Hidden products on the bf16 matrix cores at float32 precision. A float32 value is the exact
// sum of three bf16 values, x = hi + mid + lo (round to nearest even each time: 8 + 8 + 8
// significant bits and the signs of the remainders), so a product of two values is the sum of
// nine bf16 products, each exact in float32. Six of them are formed on v_mfma_f32_16x16x32_bf16,
// which accumulates in float32: 16 clocks for a 16 x 16 x 32 product against 256 for
// v_mfma_f32_16x16x4f32 (32 clocks, K = 4), so the six cost 3/8 of the float32 product. Left out are
// lo lo, lo mid and mid lo: |mid| is at most 2^-8 and |lo| 2^-17 of the value (over all significands),
// so together they are at most 2^-24 of the product, half a unit in its last place, and 2^-27.5 root
// mean square. Against float64, a 64-term product of random values is off by 0.9e-7 of its norm this
// way and by 1.45e-7 with v_mfma_f32_16x16x4f32 (fewer roundings along the accumulation).
// Values down to 1e-32 keep their 24 bits; below, the low parts are subnormal bf16 values, which the
// matrix cores take as zero (gradients of upstream gradients of size 2^-110: 3e-6 off, 2^-118: 7e-4).
// An infinite value, or one that rounds to an infinite bf16 (above 3.39e38), has an infinite hi
// and a NaN remainder: what follows from it is NaN. The forward kernels therefore form a NaN result
// again from float32 products (float32_outputs). The gradient kernels do not: a hidden weight's
// gradient is NaN where float32 products could give an infinity.
typedef unsigned u4 __attribute__((ext_vector_type(4)));  // 8 bf16 values, two to a register
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int kParts = 3;  // hi, mid, lo

// Two values rounded to bf16, a in the low half.
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f2{a, b}), bf2));
}

// The three parts of two values, each part packed as bf16_pair packs them.
__device__ __forceinline__ void split_pair(float a, float b, unsigned& hi, unsigned& mid,
                                           unsigned& lo) {
#pragma clang fp contract(off)  // x - hi of the float32 x, also where x is a product just formed
  hi = bf16_pair(a, b);
  a -= __builtin_bit_cast(float, hi << 16);
  b -= __builtin_bit_cast(float, hi & 0xffff0000u);
  mid = bf16_pair(a, b);
  a -= __builtin_bit_cast(float, mid << 16);
  b -= __builtin_bit_cast(float, mid & 0xffff0000u);
  lo = bf16_pair(a, b);
}

// The parts of four values as the halves (two registers each) of operands.
__device__ __forceinline__ void split4(const f4 x, u2 (&part)[kParts]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    unsigned hi, mid, lo;
    split_pair(x[2 * i], x[2 * i + 1], hi, mid, lo);
    part[0][i] = hi;
    part[1][i] = mid;
    part[2][i] = lo;
  }
}

__device__ __forceinline__ f4 mfma_bf16(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a),
                                                 __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// The six products in the order they accumulate, smallest first: parts of A and of B.
constexpr int kProducts = 6;
__device__ __forceinline__ constexpr int part_a(int k) { return k == 0 ? 2 : k == 1 || k == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int part_b(int k) { return k == 2 ? 2 : k == 1 || k == 4 ? 1 : 0; }

// A layer's output as the next product's B operand: half t (32 neurons) of the contraction, jet
// component c, part s. The 32 k of a step are free to order, so lane group g's 8 are rows
// 16 (2 t + e / 4) + 4 g + e % 4: the 4 values that the lane holds of output blocks 2 t and
// 2 t + 1.
struct JetOperand {
  u4 part[2][4][kParts];
};

// -I as the A operand of v_mfma_f32_16x16x16_bf16 (lane (m, g) holds k = 4 g .. 4 g + 3 of row m).
__device__ __forceinline__ u2 minus_identity(int m, int g) {
  const int e = m - 4 * g;
  return u2{e == 0 ? 0x0000bf80u : e == 1 ? 0xbf800000u : 0u,
            e == 2 ? 0x0000bf80u : e == 3 ? 0xbf800000u : 0u};
}

// x - part for an output block's component in accumulator layout: its part, packed, is also the
// B operand of a K = 16 product whose k are the block's rows. Exact, like the subtraction (one
// nonzero product per row, and the difference is a float32 value).
__device__ __forceinline__ f4 remainder_mfma(u2 minus_one, u2 part, f4 x) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, minus_one),
                                                   __builtin_bit_cast(s4, part), x, 0, 0, 0);
}

// The parts of an output block (16 rows x 4 components, accumulator layout). The kernels here
// are bound by instruction issue (a VALU instruction takes 4.4 clocks of a SIMD's issue, an MFMA
// 8.5 of its 16), so the two remainders of each value are formed on the matrix cores: 6 VALU
// and 2 MFMA instructions per 4 values against 22 VALU (split4).
__device__ __forceinline__ void split_block(u2 minus_one, const f4 (&x)[4], u2 (&part)[4][kParts]) {
  f4 rest[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) rest[c] = x[c];
#pragma unroll
  for (int s = 0; s < kParts; ++s) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      part[c][s] = u2{bf16_pair(rest[c][0], rest[c][1]), bf16_pair(rest[c][2], rest[c][3])};
      if (s + 1 < kParts) rest[c] = remainder_mfma(minus_one, part[c][s], rest[c]);
    }
  }
}

// Output block mb of a layer into its half of the next operand.
__device__ __forceinline__ void put_block(u2 minus_one, JetOperand& h, int mb, const f4 (&x)[4]) {
  u2 part[4][kParts];
  split_block(minus_one, x, part);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
      h.part[mb >> 1][c][s][2 * (mb & 1)] = part[c][s][0];
      h.part[mb >> 1][c][s][2 * (mb & 1) + 1] = part[c][s][1];
    }
  }
}

// The weights' A operands of one output block: [half][part].
struct WeightOperand {
  u4 part[2][kParts];
};

// The products of a block in the order they accumulate: the five small ones of the contraction's
// half 0, those of half 1, then hi hi of both: every addition to an accumulator rounds at its size,
// so it takes its large terms last and few of them.
template <int t>
__device__ __forceinline__ void small_products(const WeightOperand& w, const JetOperand& h, f4 (&z)[4]) {
#pragma unroll
  for (int k = 0; k < kProducts - 1; ++k) {
#pragma unroll
    for (int c = 0; c < 4; ++c) z[c] = mfma_bf16(w.part[t][part_a(k)], h.part[t][c][part_b(k)], z[c]);
  }
}

__device__ __forceinline__ void large_products(const WeightOperand& w, const JetOperand& h, f4 (&z)[4]) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int c = 0; c < 4; ++c) z[c] = mfma_bf16(w.part[t][0], h.part[t][c][0], z[c]);
  }
}

// One output block: z[c] = W[16 mb + ., :] h_c, plus the bias for the value component.
__device__ __forceinline__ void block_product(const WeightOperand& w, const JetOperand& h,
                                              const f4 bias, f4 (&z)[4]) {
  z[0] = bias;
#pragma unroll
  for (int c = 1; c < 4; ++c) z[c] = f4{0.f, 0.f, 0.f, 0.f};
  small_products<0>(w, h, z);
  small_products<1>(w, h, z);
  large_products(w, h, z);
}

// tanh in the scaled jet, four values at a time. Input zv = c z_v; outputs v = (c / 4) tanh(z_v)
// and s = (1 - tanh^2 z_v) / 4. With t = exp(-2 z_v) = exp2(zv) and u = 1 / (1 + t):
//   tanh z_v = 2 u - 1,   1 - tanh^2 z_v = 4 u (1 - u),
// so v = fma(u, c / 2, -c / 4) and s = fma(-u, u, u): 3 VALU + 2 transcendental instructions
// (v_exp_f32, v_rcp_f32) per value (tanh_value, tanh_slope). t overflows to +inf for z_v < -44 (u = 0: tanh = -1,
// s = 0) and flushes to 0 for z_v > 44 (u = 1: tanh = 1, s = 0). Near tanh = +1, s carries the
// absolute rounding of u (about 6e-8), as 1 - a^2 does.
// The four values go in stages: the four exp2, then the four rcp, then the rest (each value's
// chain is serial).
__device__ __forceinline__ float tanh_value(float u) { return __builtin_fmaf(u, 0.5f * kC, -0.25f * kC); }
__device__ __forceinline__ float tanh_slope(float u) { return __builtin_fmaf(-u, u, u); }

__device__ __forceinline__ void tanh_scaled4(const f4 zv, f4& u, f4& v, f4& s) {
#pragma unroll
  for (int r = 0; r < 4; ++r) u[r] = __builtin_amdgcn_exp2f(zv[r]);
#pragma unroll
  for (int r = 0; r < 4; ++r) u[r] = __builtin_amdgcn_rcpf(u[r] + 1.0f);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    v[r] = tanh_value(u[r]);
    s[r] = tanh_slope(u[r]);
  }
}

// tanh_jet of four values (component vectors z[c][r] of one accumulator row block), the tanh
// four at a time (tanh_scaled4): out[c][r] is the scaled output jet, u[r] tanh_scaled4's.
__device__ __forceinline__ void tanh_jet4(const f4 (&z)[4], f4 (&out)[4], f4& u) {
  f4 v, sl;
  tanh_scaled4(z[0], u, v, sl);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float q = __builtin_fmaf(z[1][r], z[1][r], z[2][r] * z[2][r]);
    out[0][r] = v[r];
    out[1][r] = sl[r] * z[1][r];
    out[2][r] = sl[r] * z[2][r];
    out[3][r] = sl[r] * __builtin_fmaf(v[r], q, z[3][r]);
  }
}

__device__ __forceinline__ void tanh_jet4(const f4 (&z)[4], f4 (&out)[4]) {
  f4 u;
  tanh_jet4(z, out, u);
}

// Adjoint of the tanh jet (tanh_jet4, per value) in the scaled variables (the adjoint of a
// scaled quantity is the unscaled adjoint divided by the scale). With v' = (c / 4) tanh z_v,
// s' = s / 4, z'_J = 2 z_J, q' = |z'_J|^2, P = z'_L + v' q' and kappa = -8 / c^2 (so
// d s' / d(c z_v) = kappa v' s'):
//   zbar_v' = s' [vbar' + kappa v' (Jbar' . z'_J) + Lbar' (kappa v' P + s' q')]
//   zbar_Jd' = s' (Jbar_d' + 2 Lbar' v' z'_Jd)
//   zbar_L' = s' Lbar'
// the unscaled formulas with every quantity replaced by its scaled form (the factors cancel).
// This is the reference's tanh_backward (/root/reference/csrc/fused_backward.cu:29-33, 75-89)
// rewritten for the scaled jet. The adjoint (vbar', J0bar', J1bar', Lbar') is replaced in
// place. Evaluated as
//   zbar_L' = s' Lbar',   zbar_v' = s' [vbar' + kappa v' (Jbar' . z'_J + Lbar' P) + zbar_L' q'],
//   zbar_Jd' = s' Jbar_d' + 2 zbar_L' v' z'_Jd
//
// Here for layer 0, whose z_J are the W0 columns and z_L = 0 (tanh_jet_adjoint_h is the hidden
// layers' form): q = |z_J|^2 is
// the per-neuron constant staged in kSmallQ0 (the same fma), and p = v q.
__device__ __forceinline__ void tanh_jet_adjoint_layer0(float v, float s, float zj0, float zj1,
                                                        float q, float& bv, float& bj0,
                                                        float& bj1, float& bl) {
  const float dot = __builtin_fmaf(bj0, zj0, bj1 * zj1);
  const float p = v * q;
  const float kv = kKappa * v;
  const float bls = bl * s;
  const float t = __builtin_fmaf(kv, __builtin_fmaf(bl, p, dot), bv);
  const float nv = s * __builtin_fmaf(bls, q, t);
  const float m2 = 2.0f * (bls * v);
  bj0 = __builtin_fmaf(m2, zj0, s * bj0);
  bj1 = __builtin_fmaf(m2, zj1, s * bj1);
  bv = nv;
  bl = bls;
}

// An opaque copy of a value: the compiler cannot see that it equals the input, so it cannot
// hoist arithmetic on it (addresses, lane masks) out of the enclosing loop and keep the results
// live, where at full register use they would be spilled; and a loaded value passed through it
// is waited for there, not where the compiler would first use it.
template <typename T>
__device__ __forceinline__ T opaque(T x) {
  __asm__ volatile("" : "+v"(x));
  return x;
}

// Keep a value in an accumulation register (AGPR) from here on: for state that a full register
// file has to hold through phases that do not use it. VALU instructions reach only the 256
// architectural registers, and left alone the allocator spilled to memory instead.
__device__ __forceinline__ void park(float& x) { __asm__ volatile("" : "+a"(x)); }
__device__ __forceinline__ void park_block(f4 (&x)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float y = x[c][r];
      park(y);
      x[c][r] = y;
    }
  }
}

// Small-parameter staging shared by all kernels, in the scaled forms listed at kSmallCwx (the
// factors 2 and 4 are exact), split into its global loads (load_small) and its LDS writes
// (store_small), so that a kernel can issue these loads together with its other staging loads
// and wait for global memory once: written as one function, each group of loads waited for the
// previous group's LDS writes, and the forward's prologue made four round trips.
// Thread tid < 64 holds neuron tid's W0 row, b0 and w_out, thread tid < 192 one hidden bias,
// and every thread b_out (a uniform load).
struct SmallLoads {
  float wx, wy, b0, wo, bh, bout;
};

template <int kThreads>
__device__ __forceinline__ SmallLoads load_small(const float* __restrict__ params, int tid) {
  static_assert(kThreads >= 3 * kHidden, "one thread per hidden bias");
  SmallLoads s{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (tid < kHidden) {
    s.wx = params[kInputs * tid];
    s.wy = params[kInputs * tid + 1];
    s.b0 = params[kLayer0Bias + tid];
    s.wo = params[kOutputBase + tid];
  }
  if (tid < 3 * kHidden) {
    s.bh = params[kHiddenBase + (tid >> 6) * kHiddenStride + kHidden * kHidden + (tid & 63)];
  }
  s.bout = params[kOutputBase + kHidden];
  return s;
}

// Called after the caller's other staging loads are issued. The values are waited for here: the
// opaque copies keep the compiler from moving the scaling up into load_small's branches, where
// it would wait for the loads at once.
__device__ __forceinline__ void store_small(float* s_small, int tid, SmallLoads s) {
  s.wx = opaque(s.wx);
  s.wy = opaque(s.wy);
  s.b0 = opaque(s.b0);
  s.wo = opaque(s.wo);
  s.bh = opaque(s.bh);
  s.bout = opaque(s.bout);
  if (tid < kHidden) {
    s_small[kSmallCwx + tid] = kC * s.wx;
    s_small[kSmallCwy + tid] = kC * s.wy;
    s_small[kSmallCb0 + tid] = kC * s.b0;
    s_small[kSmallWx + tid] = 2.0f * s.wx;
    s_small[kSmallWy + tid] = 2.0f * s.wy;
    s_small[kSmallQ0 + tid] = 4.0f * __builtin_fmaf(s.wx, s.wx, s.wy * s.wy);
    s_small[kSmallWoutV + tid] = 4.0f * (s.wo * (1.0f / kC));
    s_small[kSmallWoutL + tid] = 4.0f * (s.wo * (1.0f / kLambda));
  }
  if (tid < 3 * kHidden) s_small[kSmallBh + tid] = kC * s.bh;
  if (tid == 0) s_small[kSmallBout] = s.bout;
}

// Operands in LDS: one operand of a wave is 64 entries of 16 bytes, lane (m, g)'s at operand_entry.
// The rotation of the 16 entries of each g by 4 g (as an xor) spreads the transposed reads
// (lds_transposed), whose 16 lanes take 8 bytes at 4 m and all four g, over all banks. A wave's plain
// reads of its entries pay for it: each ds_read_b128 has 4 cycles of conflicts (SQ_LDS_BANK_CONFLICT,
// forward at 65,536 points: 36 % of the LDS cycles).
__device__ __forceinline__ int operand_entry(int m, int g) { return 16 * g + (m ^ (4 * g)); }

// LDS layout of the hidden weights, in MFMA operand order and split into bf16 parts: for hidden
// layer l, output block mb, contraction half t, part s and lane (m, g), the 16 bytes at u4 index
// (24 l + (2 mb + t) 3 + s) * 64 + operand_entry(m, g) hold part s of 4 W[16 mb + m][32 t +
// 16 (e / 4) + 4 g + e % 4], e = 0..7 (the scaled jet's weights, in JetOperand's order). The offsets
// within a layer are immediates. 72 KB.
constexpr int kBlockU4 = 2 * kParts * kWave;  // u4 entries of one output block
constexpr int kLayerU4 = 4 * kBlockU4;        // of one layer (24 KB)

// One lane's operand of (layer, mb, t): 8 weights, loaded as two runs of four of a row and split.
template <bool kAligned>
__device__ __forceinline__ void load_weights8(const float* __restrict__ params, int layer, int mb, int t,
                                              int lane, f4 (&w)[2]) {
  const float* p = params + kHiddenBase + layer * kHiddenStride + (16 * mb + (lane & 15)) * kHidden +
                   32 * t + 4 * (lane >> 4);
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const float* q = p + 16 * half;
    w[half] = kAligned ? *reinterpret_cast<const f4*>(q) : f4{q[0], q[1], q[2], q[3]};
  }
}

__device__ __forceinline__ void split_weights8(const f4 (&w)[2], u4 (&part)[kParts]) {
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    u2 parts[kParts];
    split4(4.0f * w[half], parts);
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
      part[s][2 * half] = parts[s][0];
      part[s][2 * half + 1] = parts[s][1];
    }
  }
}

// Staging: work item (l, mb, t, lane). A thread issues the loads of all its items before its
// first LDS write; one branch on the parameters' alignment holds them all (with a branch at each
// load, each waited for the one before: 2.9 us of a gradient kernel's start).
template <int kThreads>
__device__ __forceinline__ void stage_operand_weights(const float* __restrict__ params, u4* s_wa,
                                                      int tid) {
  constexpr int kItems = 3 * 4 * 2 * kWave;  // (layer, mb, t, lane)
  constexpr int kPerThread = (kItems + kThreads - 1) / kThreads;
  static_assert(kItems % kThreads == 0, "whole items per thread");
  f4 rows[kPerThread][2];
  if ((reinterpret_cast<uintptr_t>(params) & 15) == 0) {
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
      const int item = tid + n * kThreads;
      load_weights8<true>(params, item >> 9, (item >> 7) & 3, (item >> 6) & 1, item & 63, rows[n]);
    }
  } else {
#pragma unroll
    for (int n = 0; n < kPerThread; ++n) {
      const int item = tid + n * kThreads;
      load_weights8<false>(params, item >> 9, (item >> 7) & 3, (item >> 6) & 1, item & 63, rows[n]);
    }
  }
#pragma unroll
  for (int n = 0; n < kPerThread; ++n) {
    const int item = tid + n * kThreads;
    u4 parts[kParts];
    split_weights8(rows[n], parts);
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
      s_wa[((item >> 6) * kParts + s) * kWave + operand_entry(item & 15, (item >> 4) & 3)] = parts[s];
    }
  }
}

// One output block's operands from LDS; w is this lane's entry of the layer's first operand.
__device__ __forceinline__ WeightOperand lds_weights(const u4* w, int mb) {
  WeightOperand o;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int s = 0; s < kParts; ++s) o.part[t][s] = w[mb * kBlockU4 + (t * kParts + s) * kWave];
  }
  return o;
}

// Layer-0 data of the 4 neurons o = 16 mb + 4 g + r (r = 0..3) held by this lane.
struct Layer0Weights {
  f4 cwx, cwy, cb;  // scaled, for the pre-activation c z_v = c (W0 x + b0)
  f4 wx, wy, q;     // z'_J0, z'_J1 of layer 0 (2 x the W0 columns) and their squared norm
};

__device__ __forceinline__ Layer0Weights layer0_weights(const float* s_small, int mb, int g) {
  const int o = 16 * mb + 4 * g;
  Layer0Weights w;
  w.cwx = lds4(s_small + kSmallCwx + o);
  w.cwy = lds4(s_small + kSmallCwy + o);
  w.cb = lds4(s_small + kSmallCb0 + o);
  w.wx = lds4(s_small + kSmallWx + o);
  w.wy = lds4(s_small + kSmallWy + o);
  w.q = lds4(s_small + kSmallQ0 + o);
  return w;
}

__device__ __forceinline__ float layer0_zv(const Layer0Weights& w, int r, float x0, float x1) {
  return __builtin_fmaf(w.cwx[r], x0, __builtin_fmaf(w.cwy[r], x1, w.cb[r]));
}

// Layer 0 in closed form: the input jet is (x, I, 0), so z_J = W0 columns and z_L = 0, and
// the tanh jet's q = |z_J|^2 is a per-neuron constant.
// One block: the jet of neurons 16 mb + 4 g + r, r = 0..3, in h[c][r].
__device__ __forceinline__ void layer0_block(const float* s_small, int mb, int g, float x0,
                                             float x1, f4 (&h)[4]) {
  const Layer0Weights w = layer0_weights(s_small, mb, g);
  f4 zv, u, v, s;
#pragma unroll
  for (int r = 0; r < 4; ++r) zv[r] = layer0_zv(w, r, x0, x1);
  tanh_scaled4(zv, u, v, s);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    h[0][r] = v[r];
    h[1][r] = s[r] * w.wx[r];
    h[2][r] = s[r] * w.wy[r];
    h[3][r] = s[r] * (v[r] * w.q[r]);
  }
}

// The small LDS parameters read per tile have loop-invariant addresses; left alone, the
// compiler hoists those reads out of the tile loop and keeps ~100 values live in registers for
// the whole kernel. An empty asm statement with a memory clobber at the top of each tile keeps
// them as per-tile LDS reads.
__device__ __forceinline__ void keep_lds_reads_in_loop() { __asm__ volatile("" ::: "memory"); }

// Value of lane l ^ 32 (permlane32) or l ^ 16 (permlane16) in every lane, with gfx950's
// v_permlane32_swap / v_permlane16_swap (VALU, no LDS round trip). swap(u, 0) leaves the
// partner in .second of the low half, swap(0, u) in .first of the high half, and the other
// halves are zero. (Swapping a register with a copy of itself would need one swap, but the
// compiler folds that form to the wrong result.)
__device__ __forceinline__ float partner32(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto a = __builtin_amdgcn_permlane32_swap(u, 0u, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(0u, u, false, false);
  return __builtin_bit_cast(float, a[1] | b[0]);
}

__device__ __forceinline__ float partner16(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, 0u, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(0u, u, false, false);
  return __builtin_bit_cast(float, a[1] | b[0]);
}

// x[l] + x[l ^ 32] + x[l ^ 16] + x[l ^ 48] in every lane, bitwise identical across the four
// lanes (each pairwise sum adds the same two operands).
__device__ __forceinline__ float sum_lane_groups(float x) {
  const float y = x + partner32(x);
  return y + partner16(y);
}

// Sum over the 16 lanes of a row (lanes 16 g .. 16 g + 15), identical in all 16 lanes: DPP
// butterflies xor 1 and xor 2 (quad_perm), then the 8- and 16-lane mirrors.
__device__ __forceinline__ float sum_row16(float x) {
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, true));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x4E, 0xF, 0xF, true));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x141, 0xF, 0xF, true));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x140, 0xF, 0xF, true));
  return x;
}

template <int kCtrl>
__device__ __forceinline__ float dpp_read(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), kCtrl, 0xF, 0xF, true));
}

// Reduce-scatter over the 16 lanes of a row: lane m of the row (m = lane % 16) returns the sum
// of v[m] over the row's lanes. Four butterfly stages, with partners given by DPP: the row
// mirror (lane 15 - m), the half-row mirror (7 - m within each 8), then quad xor 2 and xor 1.
// At each stage a lane keeps the half of its partial sums whose indices it or its remaining
// partners will own and adds the partner's copy of that half, so the work halves per stage:
// 45 VALU instructions, against 80 for 16 full row sums and picks.
__device__ __forceinline__ float row_reduce_scatter16(const float (&v)[16], int m) {
  const bool b3 = (m & 8) != 0, b2 = (m & 4) != 0, b1 = (m & 2) != 0, b0 = (m & 1) != 0;
  float s8[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float keep = b3 ? v[j + 8] : v[j];
    const float send = b3 ? v[j] : v[j + 8];
    s8[j] = keep + dpp_read<0x140>(send);
  }
  float s4[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float keep = b2 ? s8[k + 4] : s8[k];
    const float send = b2 ? s8[k] : s8[k + 4];
    s4[k] = keep + dpp_read<0x141>(send);
  }
  float s2[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float keep = b1 ? s4[k + 2] : s4[k];
    const float send = b1 ? s4[k] : s4[k + 2];
    s2[k] = keep + dpp_read<0x4E>(send);
  }
  const float keep = b0 ? s2[1] : s2[0];
  const float send = b0 ? s2[0] : s2[1];
  return keep + dpp_read<0xB1>(send);
}

// ---------------------------------------------------------------------------------------------
// Forward kernel (replaces fused_forward_laplacian_tiled_kernel<2>,
// /root/reference/csrc/fused_residual.cu:157-295). A grid of at most one workgroup per CU
// stages the weights once, then its 8 waves (two per SIMD, 256 registers each) run 16-point tiles:
// tiles blockIdx.x + k grid below `whole`, k from a counter in LDS.
//
// `whole` is a multiple of 4 x grid (one tile per SIMD per round). The tiles past the last whole
// round (`split` tiles, fewer than one per SIMD) would each add a whole tile's time to the SIMD that
// got it; instead, the last four waves of each workgroup (one per SIMD) run them with a
// 16-point tile's rows split between them, forward_split_kernel's decomposition: wave q
// computes rows 16 q .. 16 q + 15 of every layer (a quarter of the MFMAs) and the
// layer outputs go to the other three through LDS (20,011 points: 15.6 us with whole tiles alone,
// 12.3 with split ones). The four meet at an LDS counter
// (quad_sync), not at s_barrier, which would wait for the workgroup's waves still on whole
// tiles. A split tile's chains are a whole tile's accumulators (mb = q, c) with the same
// operands in the same order, so both paths give bitwise the same results.
//
// A tile is 672 MFMAs (10.8K clocks of the matrix core) and 1,070 VALU instructions; with both
// waves of a SIMD on tiles it takes about 13.6K clocks, issue-bound, at a shader clock that power
// holds at 2.1 GHz (zero data runs at 2.4 GHz, 18 % faster). 1,000,003 points 738 -> 400 us against
// the same kernel on v_mfma_f32_16x16x4f32, 65,536 points 51.0 -> 29.0.
constexpr int kQuadSpinLimit = 1 << 24;  // about 0.5 s of s_sleep(1); never reached by a whole quad

// Device status word, one per GPU: bit kStatusQuadTimeout is set when a quad meeting gave up
// (quad_sync below). fhoad_check_device reads and clears it.
constexpr unsigned kStatusQuadTimeout = 1u;
__device__ unsigned g_device_status = 0;

// The four waves of a quad each add 1 to `flag` per meeting and wait until it reaches `target`
// (4 x the meetings so far), polling at most `spin_limit` times. The release fence completes the
// wave's LDS writes before its arrival; the acquire fence orders its later reads after the
// others' arrivals. Every quad wave takes the same split tiles and meetings, so the wait ends;
// the limit only bounds it. Returns false when the wave gave up: it then sets
// kStatusQuadTimeout in the device status word (a global atomic OR) and goes on, and the caller
// writes NaN for that tile's u and Laplacian.
__device__ __forceinline__ bool quad_sync(unsigned* flag, unsigned target, int spin_limit) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if ((threadIdx.x & (kWave - 1)) == 0) {
    __hip_atomic_fetch_add(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  bool met = false;
  for (int spin = 0; spin < spin_limit; ++spin) {
    if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) {
      met = true;
      break;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  if (!met && (threadIdx.x & (kWave - 1)) == 0) {
    __hip_atomic_fetch_or(&g_device_status, kStatusQuadTimeout, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
  }
  return met;
}

// Layer 0's output as the first hidden product's operand.
__device__ __forceinline__ void layer0_operand(const float* s_small, u2 minus_one, int g, float x0,
                                               float x1, JetOperand& h) {
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    f4 x[4];
    layer0_block(s_small, mb, g, x0, x1, x);
    put_block(minus_one, h, mb, x);
  }
}

// One output block's terms of u = w_out . v + b_out and lap = w_out . L, from the scaled jet.
// Every path adds the four blocks' terms in block order.
__device__ __forceinline__ f2 output_terms(const float* s_small, int mb, int g, const f4 (&h)[4]) {
  const f4 wv = lds4(s_small + kSmallWoutV + 16 * mb + 4 * g);
  const f4 wl = lds4(s_small + kSmallWoutL + 16 * mb + 4 * g);
  f2 out{0.0f, 0.0f};
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    out[0] = __builtin_fmaf(wv[r], h[0][r], out[0]);
    out[1] = __builtin_fmaf(wl[r], h[3][r], out[1]);
  }
  return out;
}

// Exchange of a 16-point tile whose rows are split over four waves: wave q's block of a layer's
// output goes, split into parts, into its half of the next operand's entries, so that each wave
// reads the whole operand 16 bytes at a time (1 KB contiguous per wave).
struct Exchange {
  u4 part[2][4][kParts][kWave];  // [half t][component][part][operand_entry], 24 KB
};

__device__ __forceinline__ void put_exchange(Exchange& x, u2 minus_one, int q, int entry,
                                             const f4 (&mine)[4]) {
  u2 part[4][kParts];
  split_block(minus_one, mine, part);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
      reinterpret_cast<u2*>(&x.part[q >> 1][c][s][entry])[q & 1] = part[c][s];
    }
  }
}

__device__ __forceinline__ void get_exchange(const Exchange& x, int entry, JetOperand& h) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) h.part[t][c][s] = x.part[t][c][s][entry];
    }
  }
}

// (u - b_out, lap) of a tile's points from float32 products (v_mfma_f32_16x16x4f32, k-step 16 ib + j
// taking inputs 16 ib + 4 g + j from the lane groups), the weights read from global memory. For
// results that split products cannot give: with an infinite hidden weight the tanh saturates and u is
// finite, and a Laplacian can be infinite rather than NaN.
__device__ __forceinline__ f2 float32_outputs(const float* __restrict__ params, const float* s_small, int m,
                                              int g, float x0, float x1) {
  f4 h[4][4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) layer0_block(s_small, mb, g, x0, x1, h[mb]);
  f2 out{0.0f, 0.0f};
#pragma unroll 1
  for (int layer = 0; layer < 3; ++layer) {
    const float* row = params + kHiddenBase + layer * kHiddenStride + m * kHidden + 4 * g;
    f4 next[4][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      f4 z[4];
      z[0] = lds4(s_small + kSmallBh + layer * kHidden + 16 * mb + 4 * g);
      z[1] = z[2] = z[3] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float w = 4.0f * row[16 * mb * kHidden + 16 * ib + j];
#pragma unroll
          for (int c = 0; c < 4; ++c) z[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, h[ib][c][j], z[c], 0, 0, 0);
        }
      }
      tanh_jet4(z, next[mb]);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
      for (int c = 0; c < 4; ++c) h[mb][c] = next[mb][c];
    }
  }
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    const f2 terms = output_terms(s_small, mb, g, h[mb]);
    out[0] = mb ? out[0] + terms[0] : terms[0];
    out[1] = mb ? out[1] + terms[1] : terms[1];
  }
  return f2{sum_lane_groups(out[0]), sum_lane_groups(out[1])};
}

__device__ __forceinline__ bool is_nan(float a, float b) { return a != a || b != b; }

// At a forward kernel's end, after some tile of the workgroup (blockIdx.x + k gridDim.x) came out
// NaN: its waves read the tiles' results back and write the NaN ones, and only those, again from
// float32_outputs. Here nothing else is live (the lane's indexes are formed anew and the wave's is a
// scalar); inside the tile loops the same work cost registers. A NaN parameter makes every result NaN
// whatever the products, so then nothing is tried (s_nan = 2): 1,000,003 points of a network that has
// diverged take 380 us, 1,194 without that look at the parameters.
template <int kWaves>
__device__ __forceinline__ void retry_nan_tiles(const float* __restrict__ coordinates, const float* __restrict__ params,
                                                const float* s_small, float* __restrict__ output,
                                                float* __restrict__ laplacian, int64_t batch, int64_t tiles,
                                                int wave, unsigned& s_nan) {
  bool hopeless = false;
  for (int k = threadIdx.x; k < kOutputBase + kHidden; k += kWaves * kWave) hopeless |= params[k] != params[k];
  if (hopeless) s_nan = 2;
  __syncthreads();
  if (s_nan == 2) return;
  const int lane = opaque(__lane_id());
  const int m = lane & 15, g = lane >> 4;
  for (int64_t tile = blockIdx.x + static_cast<int64_t>(wave) * gridDim.x; tile < tiles;
       tile += static_cast<int64_t>(kWaves) * gridDim.x) {
    const int64_t point = tile * kTile + m;
    const bool active = point < batch;
    const float u = active ? output[point] : 0.0f, lap = active ? laplacian[point] : 0.0f;
    if (!__any(is_nan(u, lap))) continue;
    const float x0 = active ? coordinates[2 * point] : 0.0f, x1 = active ? coordinates[2 * point + 1] : 0.0f;
    const f2 again = float32_outputs(params, s_small, m, g, x0, x1);
    if (g == 0 && active) {
      if (u != u) output[point] = again[0] + s_small[kSmallBout];
      if (lap != lap) laplacian[point] = again[1];
    }
  }
}

template <int kWaves>
__global__ void __launch_bounds__(kWaves * kWave)
forward_kernel(const float* __restrict__ coordinates, const float* __restrict__ params,
               float* __restrict__ output, float* __restrict__ laplacian, int64_t batch,
               int64_t whole, int64_t tiles, int spin_limit) {
  __shared__ u4 s_wa[3 * kLayerU4];
  __shared__ __attribute__((aligned(16))) float s_small[kSmallFloats];
  __shared__ Exchange s_x[2];  // split tiles
  __shared__ unsigned s_quad;  // split tiles: quad_sync counter
  __shared__ unsigned s_next;  // the next k to take
  __shared__ unsigned s_nan;   // some result is NaN
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int g = lane >> 4;
  const int m = lane & 15;
  // A workgroup's tiles are blockIdx.x + k gridDim.x; its waves take k from a counter in LDS as
  // they go. A SIMD issues from its older wave first, so with equal shares the younger one of
  // each pair was left to run the last 40 % of the time alone.
  // Coordinates are read one tile ahead (the first tile's during the staging), so no tile
  // waits for global memory; a wave that runs alone on its SIMD would expose that latency.
  int64_t tile = blockIdx.x + static_cast<int64_t>(wave) * gridDim.x;
  float next_x0 = 0.0f, next_x1 = 0.0f;
  if (tile < whole && tile * kTile + m < batch) {
    next_x0 = coordinates[2 * (tile * kTile + m)];
    next_x1 = coordinates[2 * (tile * kTile + m) + 1];
  }
  if (threadIdx.x == 0) {
    s_quad = 0;
    s_next = kWaves;
    s_nan = 0;
  }
  bool nan = false;
  const int wave_index = __builtin_amdgcn_readfirstlane(wave);
  const SmallLoads small = load_small<kWaves * kWave>(params, threadIdx.x);
  stage_operand_weights<kWaves * kWave>(params, s_wa, threadIdx.x);
  store_small(s_small, threadIdx.x, small);
  __syncthreads();
  next_x0 = opaque(next_x0);  // delivered before the loop, for the same reason as below
  next_x1 = opaque(next_x1);
  const int entry = operand_entry(m, g);
  const u4* wa_lane = s_wa + entry;
  const u2 minus_one = minus_identity(m, g);

  // ---- split tiles first: the last four waves, one 16-point tile at a time, rows split ----
  // (first, so their quarter tiles interleave with the other waves' whole tiles on each SIMD)
  const int q = wave - (kWaves - 4);
  if (q >= 0 && whole < tiles) {
    // Raised wave priority while on split tiles: the four waves of a quad meet three times a
    // tile, each meeting waits for the slowest of them, and each shares its SIMD with waves
    // on whole tiles.
    __builtin_amdgcn_s_setprio(2);
    unsigned meetings = 0;
    int phase = 0;  // alternates the exchange buffers across layers and tiles
    for (int64_t t = whole + blockIdx.x; t < tiles; t += gridDim.x) {
      keep_lds_reads_in_loop();
      const int64_t point = t * kTile + m;
      const bool active = point < batch;
      float x0 = 0.0f, x1 = 0.0f;
      if (active) {
        x0 = coordinates[2 * point];
        x1 = coordinates[2 * point + 1];
      }
      JetOperand h;
      layer0_operand(s_small, minus_one, g, x0, x1, h);
      bool met = true;  // every quad meeting of this tile completed
#pragma unroll
      for (int layer = 0; layer < 3; ++layer) {
        const f4 bias = lds4(s_small + kSmallBh + layer * kHidden + 16 * q + 4 * g);
        f4 z[4], mine[4];
        block_product(lds_weights(wa_lane + layer * kLayerU4, q), h, bias, z);
        tanh_jet4(z, mine);
        Exchange& buf = s_x[phase];
        phase ^= 1;
        meetings += 4;
        if (layer < 2) {
          put_exchange(buf, minus_one, q, entry, mine);
          met = quad_sync(&s_quad, meetings, spin_limit) && met;
          get_exchange(buf, entry, h);
        } else {
          f2* terms = reinterpret_cast<f2*>(&buf);
          terms[q * kWave + lane] = output_terms(s_small, q, g, mine);
          met = quad_sync(&s_quad, meetings, spin_limit) && met;
          if (q == 0) {
            f2 out = terms[lane];
#pragma unroll
            for (int mb = 1; mb < 4; ++mb) {
              const f2 more = terms[mb * kWave + lane];
              out[0] += more[0];
              out[1] += more[1];
            }
            const float u = sum_lane_groups(out[0]), lap = sum_lane_groups(out[1]);
            if (met) nan |= active && is_nan(u, lap);
            if (g == 0 && active) {
              // A tile whose meetings gave up read stale rows: its outputs are NaN (and the
              // device status word says why).
              output[point] = met ? u + s_small[kSmallBout] : __builtin_nanf("");
              laplacian[point] = met ? lap : __builtin_nanf("");
            }
          }
        }
      }
    }
  }

  __builtin_amdgcn_s_setprio(0);
  while (tile < whole) {
    keep_lds_reads_in_loop();
    const int64_t point = tile * kTile + m;
    const bool active = point < batch;
    const float x0 = next_x0, x1 = next_x1;
    unsigned k = 0;
    if (lane == 0) k = __hip_atomic_fetch_add(&s_next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    k = __builtin_amdgcn_readfirstlane(k);
    tile = blockIdx.x + static_cast<int64_t>(k) * gridDim.x;
    const int64_t next_point = tile * kTile + m;
    if (tile < whole && next_point < batch) {
      next_x0 = coordinates[2 * next_point];
      next_x1 = coordinates[2 * next_point + 1];
    }
    JetOperand h;
    layer0_operand(s_small, minus_one, g, x0, x1, h);
    f2 out{0.0f, 0.0f};
#pragma unroll
    for (int layer = 0; layer < 3; ++layer) {
      JetOperand next;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        f4 z[4], mine[4];
        block_product(lds_weights(wa_lane + layer * kLayerU4, mb), h,
                      lds4(s_small + kSmallBh + layer * kHidden + 16 * mb + 4 * g), z);
        tanh_jet4(z, mine);
        if (layer < 2) {
          put_block(minus_one, next, mb, mine);
        } else {
          const f2 terms = output_terms(s_small, mb, g, mine);
          out[0] = mb ? out[0] + terms[0] : terms[0];
          out[1] = mb ? out[1] + terms[1] : terms[1];
        }
      }
      if (layer < 2) h = next;
    }
    // Take delivery of the next coordinates here, before this tile's stores: a wait at the
    // top of the next tile would also wait for those stores (they sit behind a branch, so the
    // compiler cannot count them), and a store takes far longer than a tile's head.
    next_x0 = opaque(next_x0);
    next_x1 = opaque(next_x1);
    const float u = sum_lane_groups(out[0]), lap = sum_lane_groups(out[1]);
    nan |= active && is_nan(u, lap);
    if (g == 0 && active) {
      output[point] = u + s_small[kSmallBout];
      laplacian[point] = lap;
    }
  }
  if (nan) s_nan = 1;
  __syncthreads();  // also: the workgroup's results are written
  if (s_nan) {
    retry_nan_tiles<kWaves>(coordinates, params, s_small, output, laplacian, batch, tiles, wave_index, s_nan);
  }
}

// ---------------------------------------------------------------------------------------------
// Small-batch forward. With fewer tiles than SIMDs, forward_kernel's call time is one tile's
// latency. Here a workgroup of 4 waves (one per SIMD) runs one 16-point tile at a time, and wave
// w computes output rows 16 w .. 16 w + 15 of every layer (a quarter of the MFMAs). The tanh-jet
// outputs go through LDS to the other waves, which need all 64 rows as the next layer's operand
// (Exchange). Two LDS buffers alternate, so one barrier per layer suffices.
//
// Wave w's chains are forward_kernel's accumulators (mb = w, c) with the same operands in the
// same order, layer 0 is the same closed form, and wave 0 adds the blocks' output terms in
// forward_kernel's order, so both kernels give bitwise the same results.
constexpr int kSplitWaves = 4;

__global__ void __launch_bounds__(kSplitWaves * kWave)
forward_split_kernel(const float* __restrict__ coordinates, const float* __restrict__ params,
                     float* __restrict__ output, float* __restrict__ laplacian, int64_t batch,
                     int64_t tiles) {
  __shared__ Exchange s_x[2];
  __shared__ __attribute__((aligned(16))) float s_small[kSmallFloats];
  __shared__ unsigned s_nan;  // some result is NaN
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int m = lane & 15;
  const int g = lane >> 4;
  if (threadIdx.x == 0) s_nan = 0;
  bool nan = false;
  const int wave_index = __builtin_amdgcn_readfirstlane(w);
  // The small parameters are staged first and this wave's operands loaded after (they are needed
  // only after the barrier and the first tile's coordinates): issued together, the operand loads
  // were waited for before the barrier and a 1K-point call took 0.4 us longer.
  store_small(s_small, threadIdx.x, load_small<kSplitWaves * kWave>(params, threadIdx.x));
  // This wave's operands (output block w of every layer), loaded once (global memory,
  // L2-resident) instead of staging the whole matrix in LDS.
  WeightOperand wa[3];
  {
    f4 rows[3][2][2];
    if ((reinterpret_cast<uintptr_t>(params) & 15) == 0) {
#pragma unroll
      for (int l = 0; l < 3; ++l) {
#pragma unroll
        for (int t = 0; t < 2; ++t) load_weights8<true>(params, l, w, t, lane, rows[l][t]);
      }
    } else {
#pragma unroll
      for (int l = 0; l < 3; ++l) {
#pragma unroll
        for (int t = 0; t < 2; ++t) load_weights8<false>(params, l, w, t, lane, rows[l][t]);
      }
    }
#pragma unroll
    for (int l = 0; l < 3; ++l) {
#pragma unroll
      for (int t = 0; t < 2; ++t) split_weights8(rows[l][t], wa[l].part[t]);
    }
  }
  __syncthreads();  // s_small

  const u2 minus_one = minus_identity(m, g);
  const int entry = operand_entry(m, g);
  int phase = 0;  // alternates the exchange buffers across layers and tiles
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    keep_lds_reads_in_loop();
    const int64_t point = tile * kTile + m;
    const bool active = point < batch;
    float x0 = 0.0f, x1 = 0.0f;
    if (active) {
      x0 = coordinates[2 * point];
      x1 = coordinates[2 * point + 1];
    }
    JetOperand h;
    layer0_operand(s_small, minus_one, g, x0, x1, h);
#pragma unroll
    for (int layer = 0; layer < 3; ++layer) {
      const f4 bias = lds4(s_small + kSmallBh + layer * kHidden + 16 * w + 4 * g);
      f4 z[4], mine[4];
      block_product(wa[layer], h, bias, z);
      tanh_jet4(z, mine);
      Exchange& buf = s_x[phase];
      phase ^= 1;
      if (layer < 2) {
        put_exchange(buf, minus_one, w, entry, mine);
        __syncthreads();
        get_exchange(buf, entry, h);
      } else {
        f2* terms = reinterpret_cast<f2*>(&buf);
        terms[w * kWave + lane] = output_terms(s_small, w, g, mine);
        __syncthreads();
        if (w == 0) {
          f2 out = terms[lane];
#pragma unroll
          for (int mb = 1; mb < 4; ++mb) {
            const f2 more = terms[mb * kWave + lane];
            out[0] += more[0];
            out[1] += more[1];
          }
          const float u = sum_lane_groups(out[0]), lap = sum_lane_groups(out[1]);
          nan |= active && is_nan(u, lap);
          if (g == 0 && active) {
            output[point] = u + s_small[kSmallBout];
            laplacian[point] = lap;
          }
        }
      }
    }
  }
  if (nan) s_nan = 1;
  __syncthreads();  // also: the workgroup's results are written
  if (s_nan) {
    retry_nan_tiles<kSplitWaves>(coordinates, params, s_small, output, laplacian, batch, tiles, wave_index, s_nan);
  }
}

// ---------------------------------------------------------------------------------------------
// Backward (replaces fused_backward_occupancy_kernel<false,true,false,true> and the host-side
// partials.sum(0), /root/reference/csrc/fused_backward.cu:424-850, 859-934).
//
// One workgroup per CU, 4 waves (one per SIMD, up to 512 registers each), 64-point workgroup
// tiles (16 points per wave). Per tile:
//   1. every wave re-runs the forward for its 16 points, keeping each hidden layer's tanh-jet
//      output h in registers;
//   2. the adjoint is seeded from the linear output layer and walked back through layers 3..1
//      (backward_layer): hbar = W^T zbar one 16-row input block at a time, each block's hbar
//      feeding that block's tanh-jet adjoint at once (tanh_jet_adjoint_h, from h, no tanh
//      re-evaluated), and dW += zbar h_prev^T; finally layer 0 in closed form;
//   3. dW contracts over the points of all 4 waves: zbar and h_prev go through LDS one jet
//      component at a time, split into bf16 parts, and wave w owns the 32 x 32 block
//      (w >> 1, w & 1) of every dW (with it the waves read 96 KB of operands per layer each; a
//      wave's 16 rows would take 120). Bias, W0, b0 and w_out gradients are summed over each wave's
//      points in registers (row_reduce_scatter16) and over the 4 waves once per slot.
// Every hidden product runs on the bf16 matrix cores with split operands (see split_pair).
// Weight gradients accumulate across the tiles of a "slot": slot s takes the
// workgroup tiles s, s + slots, s + 2 slots, ... in that order and writes one partial row.
// A second kernel sums the rows in a fixed tree. The slot count depends only on the batch,
// so the result does not depend on the grid size. No float atomics anywhere.
//
// A tile is 1,656 MFMAs (31K clocks of a SIMD's matrix core) and about 4,700 VALU instructions and
// takes 55K clocks: one wave per SIMD, bound by its instruction issue and the stalls between
// dependent instructions. Registers (512, all used) leave no room for a second wave. Backward call
// at 65,536 points 166.8 -> 107.6 us against v_mfma_f32_16x16x4f32, 262,144 points 638 -> 384.
constexpr int kBwdWaves = 4;
constexpr int kBwdTile = kBwdWaves * kTile;  // 64 points
constexpr int kMaxSlots = 256;
constexpr int kRowStride = 12800;            // floats per partial row (>= 12737)
constexpr int kReduceGroups = 16;            // fixed reduction tree: 16 groups of 16 slots
static_assert(kMaxSlots % kReduceGroups == 0, "reduction tree must tile the slots");

typedef float f16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f4 zero4() { return f4{0.f, 0.f, 0.f, 0.f}; }

// Transposed read of bf16 values in LDS (ds_read_b64_tr_b16): within each 16 lanes, lanes
// 4 j .. 4 j + 3 point at the 16 values of row j, 8 bytes each, and lane l gets column l of the
// four rows.
__device__ __forceinline__ u2 lds_transposed(const u2* p) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4 lds_s4;
  return __builtin_bit_cast(u2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p));
}

// W^T operands from the same LDS copy as the forward's (stage_operand_weights): for hbar of input
// block ib, lane (m, g) supplies W[32 t + 16 (e / 4) + 4 g + e % 4][16 ib + m], e = 0..7: two
// transposed reads of rows 4 g .. 4 g + 3 of output blocks 2 t and 2 t + 1. w is this lane's entry
// (transposed_entry) of the layer.
__device__ __forceinline__ int transposed_entry(int m, int g) { return operand_entry(4 * g + (m >> 2), m & 3); }

__device__ __forceinline__ void lds_transposed_half(const u4* w, int ib, int t, u4 (&part)[kParts]) {
#pragma unroll
  for (int s = 0; s < kParts; ++s) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const u4* entry = w + (2 * t + i) * kBlockU4 + ((ib >> 1) * kParts + s) * kWave;
      const u2 v = lds_transposed(reinterpret_cast<const u2*>(entry) + (ib & 1));
      part[s][2 * i] = v[0];
      part[s][2 * i + 1] = v[1];
    }
  }
}

__device__ __forceinline__ WeightOperand lds_transposed_weights(const u4* w, int ib) {
  WeightOperand o;
  lds_transposed_half(w, ib, 0, o.part[0]);
  lds_transposed_half(w, ib, 1, o.part[1]);
  return o;
}

// dW operands. A 16-point set's values of one tensor and component, split, lie in LDS as they are
// the hidden products' B operand: entry (t, s, lane (m, g)) holds part s of rows 32 t + 16 (e / 4) +
// 4 g + e % 4 at point m. For v_mfma_f32_32x32x16_bf16 (A or B: lane (n, h) = (lane % 32, lane / 32)
// supplies row n at points 8 h .. 8 h + 7), two transposed reads give 4 points each of row n of
// half t, points 8 h .. 8 h + 3 from `lo` and 8 h + 4 .. 8 h + 7 from `hi` (this lane's 8 bytes of
// part 0: dw_lane_offset, and half t's entries).
struct DwOperand {
  u4 part[kParts];
};
struct DwPointers {
  const u2 *lo, *hi;
};

__device__ __forceinline__ int dw_lane_offset(int m, int g, int i) {  // in u2 (8 bytes)
  return 2 * operand_entry(8 * (g >> 1) + 4 * i + (m >> 2), m & 3) + (g & 1);
}

__device__ __forceinline__ DwPointers dw_pointers(const u4* entries, int m, int g) {
  const u2* p = reinterpret_cast<const u2*>(entries);
  return {p + dw_lane_offset(m, g, 0), p + dw_lane_offset(m, g, 1)};
}

// `at`: u4 offset of the set from the pointers'.
__device__ __forceinline__ DwOperand lds_dw_operand(const DwPointers& p, int at) {
  DwOperand o;
#pragma unroll
  for (int s = 0; s < kParts; ++s) {
    const u2 lo = lds_transposed(p.lo + 2 * (at + s * kWave)), hi = lds_transposed(p.hi + 2 * (at + s * kWave));
    o.part[s] = u4{lo[0], lo[1], hi[0], hi[1]};
  }
  return o;
}

__device__ __forceinline__ f16 mfma_dw(u4 a, u4 b, f16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// sum[0] + sum[1] += A B^T over the operands' 16 points, the products smallest first in each. Two
// accumulators in turn: a 32 x 32 product takes the matrix core 32 clocks but gives its result
// after 64, so one chain of them runs at half rate (64K points: 123.1 -> 121.1 us per backward call).
//
// The matrix cores drop low bits as they align the addends of a step, an error whose mean is not
// zero, so the errors of many additions do not cancel: adjoints and weight-gradient sums formed there
// without more care were up to 4 times further from float64 than with float32 products (gradients
// of 262,144 points whose contributions cancel). So every other tile of a slot, and every other
// slot's first, runs its whole walk back on the negated upstream gradients (walk_sign) and its
// sums are subtracted: the mean errors of both halves cancel. And an accumulator holds one tile (64
// points); the slot's sums are formed in float32, rounded to nearest (add_sums). The forward's chains
// (12 steps) need no such care: the mean error of u over 262,144 points is the float32 products' (3.5e-8
// against 3.4e-8 of u's rms between the network as it is and with every odd quantity negated), and so
// are the gradients of steps whose residual is 1 % of the Laplacian (0.94 to 1.02 of their errors).
__device__ __forceinline__ void add_products(const DwOperand& a, const DwOperand& b, f16 (&sum)[2]) {
#pragma unroll
  for (int k = 0; k < kProducts; ++k) sum[k & 1] = mfma_dw(a.part[part_a(k)], b.part[part_b(k)], sum[k & 1]);
}

__device__ __forceinline__ void add_sums(f16& dw, float sign, const f16 (&sum)[2]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) dw[r] = __builtin_fmaf(sign, sum[0][r] + sum[1][r], dw[r]);
}

__device__ __forceinline__ float walk_sign(int slot, int round) { return ((slot ^ round) & 1) ? -1.0f : 1.0f; }

__device__ __forceinline__ f16 zero16() { return f16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}; }

// Per-neuron sums over a wave's 16 points without LDS: lane (m, g) holds x for neuron
// 16 mb + 4 g + r at point m, so summing value k = 4 mb + r over the 16 lanes of row g gives
// that neuron's total; row_reduce_scatter16 leaves the total of k = m in lane m. Lane (m, g)
// thus keeps the total of neuron owned_neuron(m, g) = 16 (m >> 2) + 4 g + (m & 3): the 64 lanes
// own the 64 neurons once each.
__device__ __forceinline__ int owned_neuron(int m, int g) { return 16 * (m >> 2) + 4 * g + (m & 3); }

// ---- the interior tiles of backward_kernel: the walk back from each layer's tanh-jet output ----
//
// The adjoint of the tanh jet (tanh_jet_adjoint_layer0) needs s', z'_J and P = z'_L + v' q' only
// in the products the jet's output already holds: h' = (v', s' z'_J0, s' z'_J1, s' P), so
// s' z'_J = h'_J, s' P = h'_L and s'^2 q' = |h'_J|^2. The adjoint is
//   zbar_L' = s' Lbar',   zbar_Jd' = s' Jbar_d' + 2 Lbar' v' h'_Jd,
//   zbar_v' = s' vbar' + kappa v' (Jbar' . h'_J + Lbar' h'_L) + Lbar' |h'_J|^2
// (18 instructions per value). A tile therefore keeps each hidden layer's output h (which the
// forward re-run produces anyway, and which the weight gradient of the layer above needs) and
// evaluates no tanh in the walk back. Of the value component it keeps tanh_scaled4's u instead of v':
// each of v' and s' is one fma of u (tanh_value, tanh_slope), and s' = u - u^2 is relatively exact
// where tanh nears -1, while s' from v' (1/4 + (kappa / 2) v'^2) carries an absolute rounding of 3e-8
// there, 4 % of s' at z = -7.
__device__ __forceinline__ void tanh_jet_adjoint_h(float u, float hj0, float hj1, float hl,
                                                   float& bv, float& bj0, float& bj1, float& bl) {
  const float v = tanh_value(u), s = tanh_slope(u);
  const float kv = kKappa * v;
  const float lv2 = bl * (v + v);
  const float dot = __builtin_fmaf(bj0, hj0, bj1 * hj1);
  const float q = __builtin_fmaf(hj0, hj0, hj1 * hj1);
  const float t = __builtin_fmaf(bl, hl, dot);
  const float nv = __builtin_fmaf(bl, q, __builtin_fmaf(kv, t, s * bv));
  bj0 = __builtin_fmaf(lv2, hj0, s * bj0);
  bj1 = __builtin_fmaf(lv2, hj1, s * bj1);
  bv = nv;
  bl = s * bl;
}

// tanh_jet_adjoint_h for the output layer's seed: Jbar' = 0 and, with kZeroV (interior points
// of the fused step), vbar' = 0; only operations on those zeros are dropped.
template <bool kZeroV>
__device__ __forceinline__ void tanh_jet_adjoint_h_seed(float u, float hj0, float hj1, float hl,
                                                        float& bv, float& bj0, float& bj1,
                                                        float& bl) {
  const float v = tanh_value(u), s = tanh_slope(u);
  const float kv = kKappa * v;
  const float lv2 = bl * (v + v);
  const float q = __builtin_fmaf(hj0, hj0, hj1 * hj1);
  const float t = bl * hl;
  const float w = kZeroV ? kv * t : __builtin_fmaf(kv, t, s * bv);
  bv = __builtin_fmaf(bl, q, w);
  bj0 = lv2 * hj0;
  bj1 = lv2 * hj1;
  bl = s * bl;
}

// A wave of backward_kernel is alone on its SIMD, so its MFMAs and VALU work must alternate in its
// own instruction stream: an MFMA takes 16 clocks (32 for the 32 x 32 form) of which its issue
// takes 8.5, and the VALU can work in the rest. The tile is cut into scheduling regions
// (region_end), each holding the MFMAs of one block and independent VALU work of the block before,
// and interleave<n, v, r, w>() asks for n groups of one MFMA, r LDS reads, w LDS writes and v VALU
// instructions in the region (issued in one run, LDS instructions stall the wave behind the
// workgroup's other three: 10 % of the time).
__device__ __forceinline__ void region_end() { __builtin_amdgcn_sched_barrier(0); }

template <int kMfmas, int kValu, int kReads = 0, int kWrites = 0>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < kMfmas; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (kReads > 0) __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
    if (kWrites > 0) __builtin_amdgcn_sched_group_barrier(0x200, kWrites, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
  }
}

// Step j (0..11) of a block's product: one product of the four components, in block_product's
// order (half 0's small products, half 1's, then hi hi of both).
__device__ __forceinline__ void product_step(int j, const WeightOperand& w, const JetOperand& h, f4 (&z)[4]) {
  const int t = j < 5 ? 0 : j < 10 ? 1 : j - 10, k = j < 5 ? j : j < 10 ? j - 5 : kProducts - 1;
#pragma unroll
  for (int c = 0; c < 4; ++c) z[c] = mfma_bf16(w.part[t][part_a(k)], h.part[t][c][part_b(k)], z[c]);
}

// The same for hbar, in the order S0, hi hi 0, S1, hi hi 1: half 0's operands are free after six.
__device__ __forceinline__ void hbar_step(int j, const WeightOperand& w, const JetOperand& h, f4 (&z)[4]) {
  const int t = j / kProducts, k = j % kProducts;
#pragma unroll
  for (int c = 0; c < 4; ++c) z[c] = mfma_bf16(w.part[t][part_a(k)], h.part[t][c][part_b(k)], z[c]);
}

// The work on an output block after its product, in twelve stages to run one per step of the next
// block's: the tanh jet (tanh_jet4; out[0] keeps u, see tanh_jet_adjoint_h) and, with kOperand, the
// split into the next operand (split_block), whose remainders have a step or two to come out of the
// matrix cores.
template <bool kOperand>
struct BlockWork {
  f4 z[4], v, s, q;
  u2 part[4][kParts];
  __device__ __forceinline__ void stage(int j, u2 minus_one, f4 (&out)[4]) {
    if (j == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = __builtin_amdgcn_exp2f(z[0][r]);
        q[r] = __builtin_fmaf(z[1][r], z[1][r], z[2][r] * z[2][r]);
      }
    } else if (j == 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = __builtin_amdgcn_rcpf(v[r] + 1.0f);
    } else if (j == 2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s[r] = tanh_slope(v[r]);
        z[0][r] = tanh_value(v[r]);
      }
      out[0] = v;
    } else if (j == 3) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        out[1][r] = s[r] * z[1][r];
        out[2][r] = s[r] * z[2][r];
      }
    } else if (j == 4) {
#pragma unroll
      for (int r = 0; r < 4; ++r) out[3][r] = s[r] * __builtin_fmaf(z[0][r], q[r], z[3][r]);
#pragma unroll
      for (int c = 1; c < 4; ++c) z[c] = out[c];
    } else if (kOperand && (j == 5 || j == 8 || j == 11)) {
      const int p = (j - 5) / 3;
#pragma unroll
      for (int c = 0; c < 4; ++c) part[c][p] = u2{bf16_pair(z[c][0], z[c][1]), bf16_pair(z[c][2], z[c][3])};
    } else if (kOperand && (j == 6 || j == 9)) {
      const int p = (j - 6) / 3;
#pragma unroll
      for (int c = 0; c < 4; ++c) z[c] = remainder_mfma(minus_one, part[c][p], z[c]);
    }
  }
  __device__ __forceinline__ void put(JetOperand& h, int mb) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int p = 0; p < kParts; ++p) {
        h.part[mb >> 1][c][p][2 * (mb & 1)] = part[c][p][0];
        h.part[mb >> 1][c][p][2 * (mb & 1) + 1] = part[c][p][1];
      }
    }
  }
};

// One hidden layer of the forward re-run (forward_kernel's chains): h_out in registers and, with
// kOperand, as the next product's operand. Each block's work runs between the MFMAs of the next
// block, block 3's between the next layer's first ones: before(j), j = 0..4, does the previous
// layer's, and `work` leaves this layer's block 3. w and bias hold block 0's operands on entry and
// the next layer's (w_after) on exit.
template <bool kOperand, typename Before>
__device__ __forceinline__ void forward_layer(const float* s_small, const u4* w_layer, const u4* w_after,
                                              u2 minus_one, int layer, int g, const JetOperand& in,
                                              f4 (&hout)[4][4], JetOperand& next, WeightOperand& w, f4& bias,
                                              BlockWork<kOperand>& work, Before before) {
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    const WeightOperand cur = w;
    f4 z[4];
    z[0] = bias;
#pragma unroll
    for (int c = 1; c < 4; ++c) z[c] = zero4();
    w = lds_weights(mb < 3 ? w_layer : w_after, (mb + 1) & 3);
    if (mb < 3 || kOperand) bias = lds4(s_small + kSmallBh + layer * kHidden + 16 * (mb + 1) + 4 * g);
#pragma unroll
    for (int j = 0; j < 12; ++j) {
      product_step(j, cur, in, z);
      if (mb == 0 && j < 5) before(j);
      if (mb > 0) work.stage(j, minus_one, hout[mb - 1]);
      if (j == 0) {
        interleave<4, 2, 2>();
      } else {
        interleave<4, 2>();
      }
      region_end();
    }
    if (mb > 0 && kOperand) {
      work.put(next, mb - 1);
      park_block(hout[mb - 1]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) work.z[c] = z[c];
  }
}

// dW staging of a 64-point tile: one jet component of zbar and of h_prev, each wave's 16 points
// as a set of entries (see DwOperand): 24 KB each.
constexpr int kSetU4 = 2 * kParts * kWave;
//
// The slot's sums of hidden layers 2 and 3 lie beside it (16 KB each), each lane's 16 in four
// 16-byte entries; those of layer 1 stay in registers (all three do during split tiles, whose
// scratch overlays this one). In registers they were 32 of the ones that spilled to memory.
constexpr int kLdsDw = 2;
struct DwStage {
  u4 z[kBwdWaves][kSetU4];
  u4 h[kBwdWaves][kSetU4];
  f4 dw[kLdsDw][4][kBwdWaves * kWave];
};

__device__ __forceinline__ void load_dw(const f4* p, f16& dw) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f4 x = p[i * kBwdWaves * kWave];
#pragma unroll
    for (int r = 0; r < 4; ++r) dw[4 * i + r] = x[r];
  }
}

__device__ __forceinline__ void keep_dw(f4* p, const f16& dw) {
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i * kBwdWaves * kWave] = f4{dw[4 * i], dw[4 * i + 1], dw[4 * i + 2], dw[4 * i + 3]};
}

// One lane's pointers into the staging: its entries of its wave's sets, and its wave's operands
// (half w >> 1 of zbar, half w & 1 of h_prev) in wave 0's set.
struct StagePointers {
  u4 *wz, *wh;
  DwPointers ra, rb;
};

// Output block mb's parts of one component into the entries of its half.
__device__ __forceinline__ void put_component(const u2 (&p)[kParts], int mb, u4 (&part)[2][kParts]) {
#pragma unroll
  for (int s = 0; s < kParts; ++s) {
    part[mb >> 1][s][2 * (mb & 1)] = p[s][0];
    part[mb >> 1][s][2 * (mb & 1) + 1] = p[s][1];
  }
}

// One hidden layer of the walk back: dW += zbar h^T, and hbar = W^T zbar given to
// adjoint(ib, r, hb) per input block and register. The two are interleaved, one component of dW
// with one block of hbar, so that hbar's MFMAs cover the staging's writes, barriers and first
// reads: stage component c; block c's products, with the adjoint of block c - 1 between them and
// the barrier and dW's first reads halfway; dW over the four waves' points, each set's operands
// read behind the previous set's MFMAs, with the next component's split between them; the second
// barrier (every wave has read component c) before the last set's MFMAs. w holds block 0's operands
// on entry and w_after's on exit.
template <typename Adjoint>
__device__ __forceinline__ void backward_layer(const u4* w_t, const u4* w_after, const StagePointers& sp, u2 minus_one,
                                               const JetOperand& zb, const f4 (&h)[4][4], f16 (&sum)[2],
                                               WeightOperand& w, Adjoint adjoint) {
  sum[0] = sum[1] = zero16();
  u4 part[2][kParts];  // of the component to stage next
  {
    f4 x[4];  // v' from the kept u
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
      for (int r = 0; r < 4; ++r) x[mb][r] = tanh_value(h[mb][0][r]);
    }
    u2 p[4][kParts];
    split_block(minus_one, x, p);
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) put_component(p[mb], mb, part);
  }
  auto stage = [&](int c) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) {
        sp.wz[(t * kParts + s) * kWave] = zb.part[t][c][s];
        sp.wh[(t * kParts + s) * kWave] = part[t][s];
      }
    }
  };
  stage(0);
  region_end();
  f4 done[4];  // the previous block's hbar
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    f4 hb[4] = {zero4(), zero4(), zero4(), zero4()};
    DwOperand a, b;
    u4 next0[kParts];  // half 0 of the next block's weights
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i == 2) {
        __syncthreads();  // component c is staged
        a = lds_dw_operand(sp.ra, 0);
        b = lds_dw_operand(sp.rb, 0);
      }
      if (i == 3) lds_transposed_half(c < 3 ? w_t : w_after, (c + 1) & 3, 0, next0);
#pragma unroll
      for (int j = 0; j < 3; ++j) hbar_step(3 * i + j, w, zb, hb);
      if (c > 0) adjoint(c - 1, i, done);
      if (i < 2) {
        interleave<12, 2>();
      } else {
        interleave<12, 2, 1>();
      }
      region_end();
    }
#pragma unroll
    for (int set = 0; set < kBwdWaves; ++set) {
      const DwOperand ca = a, cb = b;
      if (set + 1 < kBwdWaves) {
        a = lds_dw_operand(sp.ra, (set + 1) * kSetU4);
        b = lds_dw_operand(sp.rb, (set + 1) * kSetU4);
      } else {
        __syncthreads();  // every wave has read component c
        lds_transposed_half(c < 3 ? w_t : w_after, (c + 1) & 3, 1, w.part[1]);
      }
      add_products(ca, cb, sum);
      if (c < 3) {
        // The next component's split (VALU only: these MFMAs leave it 24 of their 32 clocks) between
        // the first three sets' MFMAs, its staging behind the last set's.
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          if ((mb ? mb - 1 : 0) != set) continue;
          u2 p[kParts];
          split4(h[mb][c + 1], p);
          put_component(p, mb, part);
        }
        if (set == 3) stage(c + 1);
      } else {
        adjoint(3, set, hb);
      }
      if (set < 3) {
        interleave<6, 4, 2>();
      } else {
        interleave<6, 4, 1, 2>();
      }
      region_end();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) done[i] = hb[i];
#pragma unroll
    for (int s = 0; s < kParts; ++s) w.part[0][s] = next0[s];
  }
}

// All blocks of a layer's adjoint into an operand, 16 independent chains of conversions and
// remainders (split_block of one block would wait for each of its MFMAs).
__device__ __forceinline__ void put_all(u2 minus_one, JetOperand& h, f4 (&x)[4][4]) {
#pragma unroll
  for (int s = 0; s < kParts; ++s) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const u2 part = {bf16_pair(x[mb][c][0], x[mb][c][1]), bf16_pair(x[mb][c][2], x[mb][c][3])};
        h.part[mb >> 1][c][s][2 * (mb & 1)] = part[0];
        h.part[mb >> 1][c][s][2 * (mb & 1) + 1] = part[1];
        if (s + 1 < kParts) x[mb][c] = remainder_mfma(minus_one, part, x[mb][c]);
      }
    }
  }
}

// Seed of the fused Poisson training step (kLoss). The loss is the PINN loss
//   mean_interior (lap - f)^2 + w mean_boundary u^2
// (/root/reference/src/fused_hoad/training.py:66-88; with no boundary points, the loss of
// /root/reference/benchmarks/benchmark_training.py:46-48). The kernel already re-runs the
// forward, so it forms the upstream gradients autograd would form for that loss itself:
//   interior points: grad_u = 0, grad_lap = fl(1 / B) (2 r) with r = lap - f;
//   boundary points: grad_u = fl(w / B_b) (2 u), grad_lap = 0.
// Tiles [0, interior_tiles) hold interior points and the rest boundary points, 16 per tile in
// both gradient kernels (split_tile<1>). sum r^2 and
// sum u^2 go into columns kLossColumn and kLossColumn + 1 of the slot's partial row. `step` is
// the Adam step counter, advanced here (one lane of workgroup 0) so that the update kernel that
// follows reads a settled value.
struct LossSeed {
  const float* source;     // f[batch]
  const float* boundary;   // boundary coordinates [boundary_count][2]
  int64_t interior_tiles;  // ceil(batch / 64) (backward_kernel) or ceil(batch / 16) (split)
  int64_t boundary_count;
  float inv_batch;         // fl(1 / B)
  float boundary_scale;    // fl(fl(w) / B_b)
  float* step;             // Adam step counter (one float)
};

constexpr int kLossColumn = kParameterCount;  // partial-row columns of sum r^2, sum u_b^2
static_assert(kLossColumn + 1 < kRowStride, "the loss columns must fit in a partial row");

// Per-point inputs of one gradient-kernel tile for this lane: coordinates and, for interior
// points, the upstream gradients (gu, gl) or, with kLoss, the source f (in a). Boundary tiles
// (kLoss, tile >= seed.interior_tiles) take boundary coordinates. Inactive lanes get zeros.
struct TileInputs {
  float x0, x1, a, b;
};

template <bool kLoss, bool kRest = false>
__device__ __forceinline__ TileInputs load_tile_inputs(const float* __restrict__ coordinates,
                                                       const float* __restrict__ grad_output,
                                                       const float* __restrict__ grad_laplacian,
                                                       int64_t batch, int64_t whole,
                                                       const LossSeed& seed, int64_t tile, int w,
                                                       int m) {
  TileInputs in{0.f, 0.f, 0.f, 0.f};
  if (kLoss && tile >= seed.interior_tiles) {  // 16-point boundary tile, shared by the waves
    const int64_t point = (tile - seed.interior_tiles) * kTile + m;
    if (point < seed.boundary_count) {
      in.x0 = seed.boundary[2 * point];
      in.x1 = seed.boundary[2 * point + 1];
    }
    return in;
  }
  // 64-point tiles below `whole`, then (kRest) 16-point tiles shared by the waves (split_tile).
  const int64_t point = !kRest || tile < whole ? tile * kBwdTile + kTile * w + m
                                               : whole * kBwdTile + (tile - whole) * kTile + m;
  if (point < batch) {
    in.x0 = coordinates[2 * point];
    in.x1 = coordinates[2 * point + 1];
    if (kLoss) {
      in.a = seed.source[point];
    } else {
      in.a = grad_output ? grad_output[point] : 0.0f;  // a null upstream gradient is zero
      in.b = grad_laplacian ? grad_laplacian[point] : 0.0f;
    }
  }
  return in;
}

// Force delivery of prefetched inputs at this point (an opaque use of each register).
__device__ __forceinline__ void deliver(TileInputs& in) {
  in.x0 = opaque(in.x0);
  in.x1 = opaque(in.x1);
  in.a = opaque(in.a);
  in.b = opaque(in.b);
}

// backward_split_kernel up to this many 16-point tiles, two per CU: its time goes up by a tile's with
// every 256, backward_kernel's is one 64-point tile's up to 16,384 points. Fused step, split against
// tiled: 4,096 points 23.9 against 32.7 us, 6,000 32.7 against 33.2, 8,192 34.1 against 33.7, 9,000
// 41.9 against 34.2, 12,288 44.4 against 35.7.
constexpr int kSplitBwdMaxTiles = 512;

// Scratch of one 16-point tile whose rows are split over the workgroup's 4 waves: the layer
// outputs h1, h2 and the adjoint as operands of all 64 rows (Exchange, 24 KB each; dW reads
// them transposed), and the partial coordinate gradients.
struct SplitScratch {
  Exchange h1, h2, z;
  float gx[kSplitWaves][2][kTile];
};

// Per-lane point sums of split_tile, of row 16 w + 4 g + (m & 3) (bh, w0x, w0y, b0, wout), or the
// same in every lane of a wave (bout, loss, bloss).
struct SplitSums {
  float bh[3], w0x, w0y, b0, wout, bout, loss, bloss;
};

// This lane's share of the point sums of rows 16 w + 4 g + r: sum over the 16 lanes of row g of
// x[r], r = m & 3.
__device__ __forceinline__ float row_total(const f4 x, int m) {
  f4 t;
#pragma unroll
  for (int r = 0; r < 4; ++r) t[r] = sum_row16(x[r]);
  const float lo = (m & 1) ? t[1] : t[0];
  const float hi = (m & 1) ? t[3] : t[2];
  return (m & 2) ? hi : lo;
}

// The operand entries of the components in use: JetOperand's and Exchange's first C.
template <int C>
__device__ __forceinline__ void get_components(const Exchange& x, int entry, JetOperand& h) {
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) h.part[t][c][s] = x.part[t][c][s][entry];
    }
  }
}

// One 16-point tile, all 4 waves: wave w owns rows 16 w .. 16 w + 15 of every layer for the
// forward re-run and W^T zbar (48 MFMAs per layer each with 4 components) and the 32 x 32 block
// (w >> 1, w & 1) of every dW. Layer outputs and adjoints go to the other waves through LDS
// (Exchange), where dW also reads them, transposed, so dW contracts over the tile's points one
// component at a time. dW accumulates into `dw` (the layout of backward_kernel's);
// grad_coordinates of interior points are written here. w_lane and w_t are this lane's entries of
// the staged weights (forward and transposed).
//
// kComponents = 1: a boundary tile of the fused step. Boundary points enter the loss through u
// alone (grad_lap = 0), so the output seed is (vbar', Jbar', Lbar') = (4 gu w_out / c, 0, 0), and
// the tanh-jet adjoint maps (vbar', 0, 0, 0) to (s' vbar', 0, 0, 0): every adjoint component but
// the value one is exactly zero at every layer. The weight-gradient terms reduce to
// zbar_v h_v^T, and the forward's J and L components feed nothing. A boundary tile therefore
// runs the value channel only; the terms it skips are exact zeros.
template <int kComponents, bool kLoss>
__device__ __forceinline__ void split_tile(const u4* w_lane, const u4* w_t, const float* s_small,
                                           SplitScratch& sc, u2 minus_one, int w, int g, int m,
                                           float x0, float x1, float gu, float gl, float f,
                                           bool active, float sign, int64_t point,
                                           float* __restrict__ grad_coordinates,
                                           const LossSeed& seed, f16 (&dw)[3], SplitSums& sums) {
  constexpr int C = kComponents;
  constexpr bool kBoundary = C == 1;
  const int lane = 16 * g + m;
  const int entry = operand_entry(m, g);
  // The jet's output rows, and what the walk back keeps of them: u for v' (tanh_jet_adjoint_h).
  auto tanh_rows = [&](const f4 (&z)[4], f4 (&out)[4], f4 (&keep)[4]) {
    if (kBoundary) {
      f4 unused;
      tanh_scaled4(z[0], keep[0], out[0], unused);
    } else {
      tanh_jet4(z, out, keep[0]);
#pragma unroll
      for (int c = 1; c < 4; ++c) keep[c] = out[c];
    }
  };
  auto split_rows = [&](const f4 (&x)[4], u2 (&part)[4][kParts]) {
    f4 rest[4];
#pragma unroll
    for (int c = 0; c < C; ++c) rest[c] = x[c];
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        part[c][s] = u2{bf16_pair(rest[c][0], rest[c][1]), bf16_pair(rest[c][2], rest[c][3])};
        if (s + 1 < kParts) rest[c] = remainder_mfma(minus_one, part[c][s], rest[c]);
      }
    }
  };
  auto put_rows = [&](Exchange& x, const f4 (&mine)[4]) {
    u2 part[4][kParts];
    split_rows(mine, part);
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) {
        reinterpret_cast<u2*>(&x.part[w >> 1][c][s][entry])[w & 1] = part[c][s];
      }
    }
  };
  auto product = [&](const WeightOperand& a, const JetOperand& b, const f4 start, f4 (&z)[4]) {
    z[0] = start;
#pragma unroll
    for (int c = 1; c < C; ++c) z[c] = zero4();
#pragma unroll
    for (int i = 0; i < 2 * kProducts; ++i) {  // the order of block_product
      const int t = i < 2 * (kProducts - 1) ? i / (kProducts - 1) : i - 2 * (kProducts - 1);
      const int k = i < 2 * (kProducts - 1) ? i % (kProducts - 1) : kProducts - 1;
#pragma unroll
      for (int c = 0; c < C; ++c) z[c] = mfma_bf16(a.part[t][part_a(k)], b.part[t][c][part_b(k)], z[c]);
    }
  };

  // ---- forward re-run: all 64 rows of layer 0, then this wave's rows of layers 1..3 ----
  JetOperand op;
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    f4 x[4];
    layer0_block(s_small, mb, g, x0, x1, x);
    u2 part[4][kParts];
    split_rows(x, part);
#pragma unroll
    for (int c = 0; c < C; ++c) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) {
        op.part[mb >> 1][c][s][2 * (mb & 1)] = part[c][s][0];
        op.part[mb >> 1][c][s][2 * (mb & 1) + 1] = part[c][s][1];
      }
    }
  }
  f4 h[3][4], out[4];  // this wave's rows of the hidden layers' outputs: as kept, and the last one's
#pragma unroll
  for (int layer = 0; layer < 3; ++layer) {
    const f4 bias = lds4(s_small + kSmallBh + layer * kHidden + 16 * w + 4 * g);
    f4 z[4];
    product(lds_weights(w_lane + layer * kLayerU4, w), op, bias, z);
    tanh_rows(z, out, h[layer]);
    if (layer < 2) {
      Exchange& x = layer ? sc.h2 : sc.h1;
      put_rows(x, out);
      __syncthreads();
      get_components<C>(x, entry, op);
    }
  }

  if (kLoss) {
    // u (boundary) or lap (interior) over all 64 rows, in forward_kernel's order.
    float* terms = reinterpret_cast<float*>(&sc.z);
    {
      const f4 wo = lds4(s_small + (kBoundary ? kSmallWoutV : kSmallWoutL) + 16 * w + 4 * g);
      float t = 0.0f;
#pragma unroll
      for (int r = 0; r < 4; ++r) t = __builtin_fmaf(wo[r], out[kBoundary ? 0 : 3][r], t);
      terms[w * kWave + lane] = t;
    }
    __syncthreads();
    float total = terms[lane];
#pragma unroll
    for (int mb = 1; mb < 4; ++mb) total += terms[mb * kWave + lane];
    total = sum_lane_groups(total);
    __syncthreads();  // sc.z is free again
    // u (boundary) or the residual lap - f (interior).
    const float e = active ? (kBoundary ? total + s_small[kSmallBout] : total - f) : 0.0f;
    const float sq = sum_row16(e * e);
    if (kBoundary) {
      gu = sign * (seed.boundary_scale * (2.0f * e));
      sums.bloss += sq;
    } else {
      gl = sign * (seed.inv_batch * (2.0f * e));
      sums.loss += sq;
    }
  } else {
    gu *= sign;
    gl *= sign;
  }

  // ---- output layer: this wave's rows of the seed and of dw_out ----
  f4 hb[4];
  {
    const float gu_c = gu * (4.0f / kC);
    const float gl_l = gl * (4.0f / kLambda);
    const f4 wv = lds4(s_small + kSmallWoutV + 16 * w + 4 * g);
    const f4 wl = lds4(s_small + kSmallWoutL + 16 * w + 4 * g);
    f4 terms;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      terms[r] = kBoundary ? gu_c * out[0][r] : __builtin_fmaf(gu_c, out[0][r], gl_l * out[3][r]);
      hb[0][r] = gu * wv[r];
      if (!kBoundary) {
        hb[1][r] = 0.0f;
        hb[2][r] = 0.0f;
        hb[3][r] = gl * wl[r];
      }
    }
    sums.wout += sign * row_total(terms, m);
    sums.bout += sign * sum_row16(gu);
  }

  // ---- hidden layers 3, 2, 1 ----
#pragma unroll
  for (int layer = 2; layer >= 0; --layer) {
    // zbar of this wave's rows (tanh-jet adjoint, lane-local)
    f4 zb[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (kBoundary) {
        zb[0][r] = tanh_slope(h[layer][0][r]) * hb[0][r];
      } else {
        float bv = hb[0][r], bj0 = hb[1][r], bj1 = hb[2][r], bl = hb[3][r];
        tanh_jet_adjoint_h(h[layer][0][r], h[layer][1][r], h[layer][2][r], h[layer][3][r], bv, bj0, bj1, bl);
        zb[0][r] = bv;
        zb[1][r] = bj0;
        zb[2][r] = bj1;
        zb[3][r] = bl;
      }
    }
    sums.bh[layer] += sign * row_total(zb[0], m);
    if (layer < 2) __syncthreads();  // every wave has read the layer above's adjoint and h
    put_rows(sc.z, zb);
    if (layer == 0) {  // layer 0's output, this wave's rows, in place of h2
      f4 own[4];
      layer0_block(s_small, w, g, x0, x1, own);
      put_rows(sc.h2, own);
    }
    __syncthreads();
    // hbar of this wave's rows of the layer below, before dW: the next adjoint waits for it alone, and
    // its VALU work runs behind dW's MFMAs (the region's end holds the compiler to it). Backward call at
    // 1,000 points 18.2 -> 17.1 us; with a rest of split tiles, 30,000 points 74.5 -> 70.4, 70,001
    // 127.4 -> 122.6.
    get_components<C>(sc.z, entry, op);
    const u4* wt = w_t + layer * kLayerU4 + (w >> 1) * kParts * kWave;
    WeightOperand a;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int s = 0; s < kParts; ++s) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const u2 v = lds_transposed(reinterpret_cast<const u2*>(wt + (2 * t + i) * kBlockU4 + s * kWave) + (w & 1));
          a.part[t][s][2 * i] = v[0];
          a.part[t][s][2 * i + 1] = v[1];
        }
      }
    }
    product(a, op, zero4(), hb);
    region_end();
    // dW += sum over (c, points) of zbar h_prev^T.
    {
      const Exchange& hx = layer == 1 ? sc.h1 : sc.h2;
      const DwPointers a = dw_pointers(&sc.z.part[w >> 1][0][0][0], m, g);
      const DwPointers b = dw_pointers(&hx.part[w & 1][0][0][0], m, g);
      f16 sum[2] = {zero16(), zero16()};
#pragma unroll
      for (int c = 0; c < C; ++c) {
        add_products(lds_dw_operand(a, c * kParts * kWave), lds_dw_operand(b, c * kParts * kWave), sum);
      }
      add_sums(dw[layer], sign, sum);
    }
  }

  // ---- layer 0 for this wave's rows: dW0, db0 and this wave's part of grad_x ----
  {
    const Layer0Weights w0 = layer0_weights(s_small, w, g);
    const float cx0 = kHalfC * x0, cx1 = kHalfC * x1;
    float gx0 = 0.f, gx1 = 0.f;
    f4 zv4, unused, v4, s4, tx, ty, tb;
#pragma unroll
    for (int r = 0; r < 4; ++r) zv4[r] = layer0_zv(w0, r, x0, x1);
    tanh_scaled4(zv4, unused, v4, s4);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float bv = hb[0][r];
      if (kBoundary) {
        bv *= s4[r];
        tx[r] = bv * cx0;
        ty[r] = bv * cx1;
      } else {
        float bj0 = hb[1][r], bj1 = hb[2][r], bl = hb[3][r];
        tanh_jet_adjoint_layer0(v4[r], s4[r], w0.wx[r], w0.wy[r], w0.q[r], bv, bj0, bj1, bl);
        gx0 = __builtin_fmaf(w0.cwx[r], bv, gx0);
        gx1 = __builtin_fmaf(w0.cwy[r], bv, gx1);
        tx[r] = __builtin_fmaf(bv, cx0, bj0);
        ty[r] = __builtin_fmaf(bv, cx1, bj1);
      }
      tb[r] = bv;
    }
    sums.w0x += sign * row_total(tx, m);
    sums.w0y += sign * row_total(ty, m);
    sums.b0 += sign * row_total(tb, m);
    if (!kBoundary) {
      gx0 = sum_lane_groups(gx0);
      gx1 = sum_lane_groups(gx1);
      if (g == 0) {
        sc.gx[w][0][m] = gx0;
        sc.gx[w][1][m] = gx1;
      }
    }
    __syncthreads();  // also: every wave is done with the exchanges
    if (!kBoundary && w == 0 && g == 0 && active && grad_coordinates != nullptr) {
      grad_coordinates[2 * point] = sign * (((sc.gx[0][0][m] + sc.gx[1][0][m]) + sc.gx[2][0][m]) + sc.gx[3][0][m]);
      grad_coordinates[2 * point + 1] = sign * (((sc.gx[0][1][m] + sc.gx[1][1][m]) + sc.gx[2][1][m]) + sc.gx[3][1][m]);
    }
  }
}

// A wave's 32 x 32 block (w >> 1, w & 1) of each hidden dW into the partial row: register r of
// lane (n, h) holds row 8 (r / 4) + 4 h + r % 4, column n of the block. The sums are of d/d(4 W).
// Non-temporal stores: the row is read once, by the reduction kernel, so it is streamed out
// at once instead of waiting dirty in L2 for the write-back at the kernel's end (with every
// workgroup's row dirty there, that write-back took about 3 us of a short call's tail).
__device__ __forceinline__ void store_dw(float* row, int w, int lane, const f16 (&dw)[3]) {
  const int at = opaque((32 * (w >> 1) + 4 * (lane >> 5)) * kHidden + 32 * (w & 1) + (lane & 31));
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    float* block = row + kHiddenBase + l * kHiddenStride;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      __builtin_nontemporal_store(4.0f * dw[l][r], &block[at + (8 * (r >> 2) + (r & 3)) * kHidden]);
    }
  }
}

// Phase clock of backward_kernel, compiled only into a measurement build (-DFHOAD_PHASE_CLOCK;
// the library build reads no clock and every mark below compiles to nothing). Each wave adds
// the shader-clock cycles (s_memtime) it spends in each phase of its tiles to its row of
// g_phase_clock and counts its tiles; fhoad_phase_clock_read copies the table out. A clock
// read waits for the wave's outstanding LDS and scalar loads, so the measured kernel runs
// somewhat slower than the library's.
enum ClockField : int {
  kClockStage,          // kernel start to the end of the parameter staging
  kClockForward,        // a tile's start: layer 0 and hidden layers 1..3 (the forward re-run)
  kClockSeed,           // the loss and output seed, zbar3 split
  kClockLayer3,         // dW3 and W3^T zbar3 into layer 2's adjoint
  kClockLayer2,         // dW2 and W2^T zbar2 into layer 1's adjoint
  kClockLayer1,         // layer 0 rebuilt, dW1, W1^T zbar1, layer 0's adjoint, coordinate gradients
  kClockRest,           // 16-point split tiles past the last whole round
  kClockBoundary,       // boundary tiles of the fused step
  kClockPartials,       // the slot's partial row
  kClockTiles,          // count of 64-point tiles
  kClockBoundaryTiles,  // count of boundary tiles
  kClockWallStart,      // s_memrealtime (100 MHz) at the kernel's start
  kClockWallEnd,        // s_memrealtime after the partial row's stores are issued
  kClockFields
};
constexpr int kClockWorkgroups = 1024;  // rows kept: workgroups 0 .. 1023

#ifdef FHOAD_PHASE_CLOCK
__device__ unsigned long long g_phase_clock[kClockWorkgroups][kBwdWaves][kClockFields];

struct PhaseClock {
  unsigned long long last, fields[kClockFields];
  __device__ __forceinline__ PhaseClock() {
#pragma unroll
    for (int i = 0; i < kClockFields; ++i) fields[i] = 0;
    fields[kClockWallStart] = wall_clock64();
    last = clock64();
  }
  __device__ __forceinline__ void mark(ClockField field) {
    const unsigned long long now = clock64();
    fields[field] += now - last;
    last = now;
  }
  __device__ __forceinline__ void count(ClockField field) { fields[field] += 1; }
  __device__ __forceinline__ void store(int w) {
    fields[kClockWallEnd] = wall_clock64();
    if ((threadIdx.x & (kWave - 1)) == 0 && blockIdx.x < kClockWorkgroups) {
#pragma unroll
      for (int i = 0; i < kClockFields; ++i) g_phase_clock[blockIdx.x][w][i] = fields[i];
    }
  }
};
#else
struct PhaseClock {
  __device__ __forceinline__ void mark(ClockField) {}
  __device__ __forceinline__ void count(ClockField) {}
  __device__ __forceinline__ void store(int) {}
};
#endif

// The outputs h1, h2, h3 of the hidden layers stay in registers through the walk back (a layer's
// zbar replaces h3, then is built beside the h that dW still reads).
//
// kLoss: grad_output and grad_laplacian are unused and the seed comes from `seed` (above);
// grad_coordinates may be null.
//
// kBoundary: with boundary tiles in it, the fused step's kernel spills more registers in its 64-point
// tiles, so a step of whole rounds without boundary points runs a form without them (262,144 points
// 396.5 -> 389.3 us). With a rest of split tiles the two forms are within 2 % either way (30,000 points
// 74.1 against 72.6 without, 250,001 386 against 387.5), so that one always has them.
template <bool kLoss, bool kRest, bool kBoundary>
__global__ void __launch_bounds__(kBwdWaves * kWave, 1)
backward_kernel(const float* __restrict__ coordinates, const float* __restrict__ params,
                const float* __restrict__ grad_output, const float* __restrict__ grad_laplacian,
                float* __restrict__ grad_coordinates, float* __restrict__ partials,
                int64_t batch, int64_t whole, int64_t tiles, int slots, LossSeed seed) {
  static_assert(kLoss || !kBoundary, "boundary points belong to the fused step's loss");
  constexpr int kCombined = 7;  // point sums combined over the waves: w0x, w0y, b0, wout, bh[3]
  union Scratch {
    DwStage stage;
    SplitScratch split;
    float comb[kCombined][kBwdWaves][kHidden];
  };
  __shared__ u4 s_w[3 * kLayerU4];
  __shared__ __attribute__((aligned(16))) float s_small[kSmallFloats];
  __shared__ Scratch s_x;
  __shared__ float s_red[3][kBwdWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int m = lane & 15;
  const int g = lane >> 4;
  PhaseClock clock;
  // The first slot's first tile inputs are read before the staging, which hides their latency.
  TileInputs next{0.f, 0.f, 0.f, 0.f};
  if (static_cast<int>(blockIdx.x) < slots) {
    next = load_tile_inputs<kLoss, kRest>(coordinates, grad_output, grad_laplacian, batch, whole, seed,
                                   blockIdx.x, w, m);
  }
  // kLoss: the Adam step count is read with the staging loads and advanced after the barrier
  // (an increment in place waited for its load before wave 0 issued any staging load).
  const float step_count = kLoss ? seed.step[0] : 0.0f;
  const SmallLoads small = load_small<kBwdWaves * kWave>(params, threadIdx.x);
  stage_operand_weights<kBwdWaves * kWave>(params, s_w, threadIdx.x);
  store_small(s_small, threadIdx.x, small);
  __syncthreads();
  if (kLoss && blockIdx.x == 0 && threadIdx.x == 0) seed.step[0] = step_count + 1.0f;
  clock.mark(kClockStage);

  const u2 minus_one = minus_identity(m, g);
  const int entry = operand_entry(m, g);
  const u4* w_lane = s_w + entry;
  const u4* w_t = s_w + transposed_entry(m, g);
  StagePointers sp;
  sp.wz = s_x.stage.z[w] + entry;
  sp.wh = s_x.stage.h[w] + entry;
  sp.ra = dw_pointers(s_x.stage.z[0] + (w >> 1) * kParts * kWave, m, g);
  sp.rb = dw_pointers(s_x.stage.h[0] + (w & 1) * kParts * kWave, m, g);

  f4* dw_lane = &s_x.stage.dw[0][0][threadIdx.x];  // this lane's sums of layers 2 and 3

  for (int slot = blockIdx.x; slot < slots; slot += gridDim.x) {
    f16 dw[3] = {zero16(), zero16(), zero16()};
    keep_dw(dw_lane, dw[1]);
    keep_dw(dw_lane + 4 * kBwdWaves * kWave, dw[2]);
    // Point sums of this wave (lane = owned neuron), and of r^2 and u_b^2 (kLoss).
    float sum[kCombined] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float sum_bout = 0.f, sum_loss = 0.f, sum_bloss = 0.f;

    // Per-point inputs are read one tile ahead and delivered mid-tile (deliver), so no tile
    // starts with a wait on global memory: with one wave per SIMD nothing would hide it. The
    // delivery sits before the tile's own stores, which a wait at the next tile's head would
    // also have to wait for (they are behind branches, so the compiler cannot count them).
    if (slot != static_cast<int>(blockIdx.x)) {
      next = load_tile_inputs<kLoss, kRest>(coordinates, grad_output, grad_laplacian, batch, whole, seed, slot,
                                     w, m);
    }
    deliver(next);
    // A slot's interior tiles come before its boundary tiles (kLoss), so two loops run them in
    // the same order as one would. One loop with both kinds of tile cost about 100 register
    // copies a tile, where the two paths' accumulators met at the loop's back edge.
    int64_t tile = slot;
    int round = 0;  // tiles of this slot so far (walk_sign)
    const int64_t interior_end = kLoss ? std::min<int64_t>(tiles, seed.interior_tiles) : tiles;
    const int64_t loop_end = kRest ? whole : interior_end;
    f4 h1[4][4], h2[4][4], h3[4][4];  // hidden-layer outputs of the current tile
    for (; tile < loop_end; tile += slots, ++round) {
      keep_lds_reads_in_loop();
      const int m_pick = opaque(m);  // row_reduce_scatter16's lane masks stay inside the tile
      const TileInputs in = next;
      if (tile + slots < tiles) {
        next = load_tile_inputs<kLoss, kRest>(coordinates, grad_output, grad_laplacian, batch, whole, seed,
                                       tile + slots, w, m);
      }
      const float x0 = in.x0, x1 = in.x1;
      const int64_t point = tile * kBwdTile + kTile * w + m;
      const bool active = point < batch;
      const float sign = walk_sign(slot, round);
      const float gu = kLoss ? 0.f : sign * in.a;
      float gl = kLoss ? 0.f : sign * in.b;

      // ---- 1. forward re-run ----
      {
        JetOperand a, b;
        WeightOperand wf = lds_weights(w_lane, 0);
        f4 bias = lds4(s_small + kSmallBh + 4 * g);
        layer0_operand(s_small, minus_one, g, x0, x1, a);
        BlockWork<true> work;
        BlockWork<false> last;
        // The previous layer's block 3 in the five steps before its operand is needed.
        auto finish = [&](int j, f4 (&out)[4], JetOperand& op) {
          const int from = j == 0 ? 0 : 2 * j + 2, to = j == 0 ? 4 : 2 * j + 4;
#pragma unroll
          for (int i = 0; i < 12; ++i) {
            if (i >= from && i < to) work.stage(i, minus_one, out);
          }
          if (j == 4) {
            work.put(op, 3);
            park_block(out);
          }
        };
        forward_layer<true>(s_small, w_lane, w_lane + kLayerU4, minus_one, 0, g, a, h1, b, wf, bias, work,
                            [](int) {});
        forward_layer<true>(s_small, w_lane + kLayerU4, w_lane + 2 * kLayerU4, minus_one, 1, g, b, h2, a, wf,
                            bias, work, [&](int j) { finish(j, h1[3], b); });
        forward_layer<false>(s_small, w_lane + 2 * kLayerU4, w_lane, minus_one, 2, g, a, h3, b, wf, bias, last,
                             [&](int j) { finish(j, h2[3], a); });
#pragma unroll
        for (int j = 0; j < 5; ++j) last.stage(j, minus_one, h3[3]);
        region_end();
      }
      clock.mark(kClockForward);

      // ---- 2. output layer: w_out / b_out gradients, and hidden layer 3's adjoint ----
      // In the scaled jet u = (4 w_out / c) . v' + b_out and lap = (4 w_out / lambda) . L', so
      // dw_out = sum_p (4 gu / c) v' + (4 gl / lambda) L' and the seeds are
      // vbar' = 4 gu w_out / c, Lbar' = 4 gl w_out / lambda, Jbar' = 0. The point sums stay in
      // registers (row_reduce_scatter16). With kLoss, gu = 0 on interior points: the value seed
      // and the u terms are dropped (their products with zero).
      if (kLoss) {
        // lap = w_out . L in the forward kernel's order, then the seed.
        float out = 0.0f;
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          const f4 wo = lds4(s_small + kSmallWoutL + 16 * mb + 4 * g);
          float t = 0.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) t = __builtin_fmaf(wo[r], h3[mb][3][r], t);
          out = mb ? out + t : t;
        }
        out = sum_lane_groups(out);
        const float res = active ? out - in.a : 0.0f;
        gl = sign * (seed.inv_batch * (2.0f * res));
        sum_loss += sum_row16(res * res);
      }
      JetOperand zb;
      {
        const float gu_c = gu * (4.0f / kC);
        const float gl_l = gl * (4.0f / kLambda);
        float wout_terms[16], bias_terms[16];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          const f4 wv = lds4(s_small + kSmallWoutV + 16 * mb + 4 * g);
          const f4 wl = lds4(s_small + kSmallWoutL + 16 * mb + 4 * g);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            wout_terms[4 * mb + r] = kLoss ? gl_l * h3[mb][3][r]
                                           : __builtin_fmaf(gu_c, tanh_value(h3[mb][0][r]), gl_l * h3[mb][3][r]);
            float bv = kLoss ? 0.0f : gu * wv[r], bj0, bj1, bl = gl * wl[r];
            tanh_jet_adjoint_h_seed<kLoss>(h3[mb][0][r], h3[mb][1][r], h3[mb][2][r], h3[mb][3][r],
                                           bv, bj0, bj1, bl);
            h3[mb][0][r] = bv;
            h3[mb][1][r] = bj0;
            h3[mb][2][r] = bj1;
            h3[mb][3][r] = bl;
            bias_terms[4 * mb + r] = bv;
          }
        }
        put_all(minus_one, zb, h3);
        sum[3] += sign * row_reduce_scatter16(wout_terms, m_pick);
        sum[6] += sign * row_reduce_scatter16(bias_terms, m_pick);
        if (!kLoss) sum_bout += sign * sum_row16(gu);
      }
      clock.mark(kClockSeed);

      // ---- 3. hidden layers 3 and 2: dW from (zbar, h_prev), W^T zbar into the adjoint of the
      // layer below, which is the next zbar ----
      WeightOperand wt = lds_transposed_weights(w_t + 2 * kLayerU4, 0);
      auto walk = [&](int layer, const f4 (&h)[4][4], float& bias) {
        f4 z[4][4];
        f16 sums[2];
        backward_layer(w_t + layer * kLayerU4, w_t + (layer - 1) * kLayerU4, sp, minus_one, zb, h, sums, wt,
                       [&](int ib, int r, const f4 (&hb)[4]) {
                         float bv = hb[0][r], bj0 = hb[1][r], bj1 = hb[2][r], bl = hb[3][r];
                         tanh_jet_adjoint_h(h[ib][0][r], h[ib][1][r], h[ib][2][r], h[ib][3][r], bv, bj0,
                                            bj1, bl);
                         z[ib][0][r] = bv;
                         z[ib][1][r] = bj0;
                         z[ib][2][r] = bj1;
                         z[ib][3][r] = bl;
                       });
        f16 kept;
        load_dw(dw_lane + (layer - 1) * 4 * kBwdWaves * kWave, kept);
        add_sums(kept, sign, sums);
        keep_dw(dw_lane + (layer - 1) * 4 * kBwdWaves * kWave, kept);
        float terms[16];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
#pragma unroll
          for (int r = 0; r < 4; ++r) terms[4 * mb + r] = z[mb][0][r];
        }
        put_all(minus_one, zb, z);
        bias += sign * row_reduce_scatter16(terms, m_pick);
      };
      walk(2, h2, sum[5]);
      clock.mark(kClockLayer3);
      walk(1, h1, sum[4]);
      clock.mark(kClockLayer2);
      deliver(next);  // the next tile's inputs, before this tile's stores

      // ---- 4. hidden layer 1, whose h_prev is layer 0's output, rebuilt from its closed form
      // z' = (c (W0 x + b0), 2 W0[:,0], 2 W0[:,1], 0), and layer 0 in closed form ----
      // bv is the adjoint of z'_v = c z_v and bj_d that of z'_Jd = 2 W0[:, d], so
      // grad_x = (c W0)^T bv, dW0[o][d] = sum_p bv (c x_d) + 2 bj_d = 2 sum_p (bv (c x_d / 2) + bj_d)
      // (the row takes the 2), db0 = c sum_p bv.
      {
        f4 h0[4][4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          const Layer0Weights w0 = layer0_weights(s_small, mb, g);
          f4 zv, v, s;
#pragma unroll
          for (int r = 0; r < 4; ++r) zv[r] = layer0_zv(w0, r, x0, x1);
          tanh_scaled4(zv, h0[mb][0], v, s);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            h0[mb][1][r] = s[r] * w0.wx[r];
            h0[mb][2][r] = s[r] * w0.wy[r];
            h0[mb][3][r] = s[r] * (v[r] * w0.q[r]);
          }
        }
        float gx0 = 0.f, gx1 = 0.f, tx[16], ty[16], tb[16];
        const float cx0 = kHalfC * x0, cx1 = kHalfC * x1;
        f16 sums[2];
        Layer0Weights lw = layer0_weights(s_small, 0, g);  // of the block at hand, read a block ahead
        backward_layer(w_t, w_t, sp, minus_one, zb, h0, sums, wt, [&](int ib, int r, const f4 (&hb)[4]) {
          float bv = hb[0][r], bj0 = hb[1][r], bj1 = hb[2][r], bl = hb[3][r];
          const float u = h0[ib][0][r];
          tanh_jet_adjoint_layer0(tanh_value(u), tanh_slope(u), lw.wx[r], lw.wy[r], lw.q[r], bv, bj0, bj1, bl);
          gx0 = __builtin_fmaf(lw.cwx[r], bv, gx0);
          gx1 = __builtin_fmaf(lw.cwy[r], bv, gx1);
          tx[4 * ib + r] = __builtin_fmaf(bv, cx0, bj0);  // dW0[o][0] / 2
          ty[4 * ib + r] = __builtin_fmaf(bv, cx1, bj1);  // dW0[o][1] / 2
          tb[4 * ib + r] = bv;                            // db0[o] / c
          if (r == 3 && ib < 3) lw = layer0_weights(s_small, ib + 1, g);
        });
        add_sums(dw[0], sign, sums);
        sum[0] += sign * row_reduce_scatter16(tx, m_pick);
        sum[1] += sign * row_reduce_scatter16(ty, m_pick);
        sum[2] += sign * row_reduce_scatter16(tb, m_pick);
        gx0 = sum_lane_groups(gx0);
        gx1 = sum_lane_groups(gx1);
        if (g == 0 && active && grad_coordinates != nullptr) {
          grad_coordinates[2 * point] = sign * gx0;
          grad_coordinates[2 * point + 1] = sign * gx1;
        }
      }
      clock.mark(kClockLayer1);
      clock.count(kClockTiles);
    }
    load_dw(dw_lane, dw[1]);
    load_dw(dw_lane + 4 * kBwdWaves * kWave, dw[2]);
    // A split tile's point sums into this wave's owned-neuron lanes (owned_neuron): the wave's rows
    // only; the point sums shared by the 4 waves from wave 0 alone.
    auto add_split = [&](const SplitSums& s, int m_pick) {
      const bool own = (m_pick >> 2) == w;
      sum[0] += own ? s.w0x : 0.f;
      sum[1] += own ? s.w0y : 0.f;
      sum[2] += own ? s.b0 : 0.f;
      sum[3] += own ? s.wout : 0.f;
#pragma unroll
      for (int l = 0; l < 3; ++l) sum[4 + l] += own ? s.bh[l] : 0.f;
      if (w == 0) {
        sum_bout += s.bout;
        sum_loss += s.loss;
        sum_bloss += s.bloss;
      }
    };
    // kRest: interior points past the last whole round of 64-point tiles, as 16-point tiles
    // whose rows are split over the 4 waves (split_tile); one takes 9.7 us, a 64-point tile 22 (see
    // interior_tiles_for). The scratch
    // overlays the dW staging buffer: the barrier waits for the last 64-point tile's readers.
    // (A separate instantiation: with this loop in the kernel the compiler schedules the
    // 64-point loop differently, so whole rounds run without it.)
    if (kRest && tile < interior_end) {  // uniform per workgroup
      __syncthreads();
      for (; tile < interior_end; tile += slots, ++round) {
        keep_lds_reads_in_loop();
        const int m_pick = opaque(m);
        const TileInputs in = next;
        if (tile + slots < tiles) {
          next = load_tile_inputs<kLoss, kRest>(coordinates, grad_output, grad_laplacian, batch, whole,
                                         seed, tile + slots, w, m);
        }
        const int64_t point = whole * kBwdTile + (tile - whole) * kTile + m;
        SplitSums s{};
        split_tile<4, kLoss>(w_lane, w_t, s_small, s_x.split, minus_one, w, g, m_pick, in.x0, in.x1,
                             kLoss ? 0.f : in.a, kLoss ? 0.f : in.b, kLoss ? in.a : 0.f,
                             point < batch, walk_sign(slot, round), point, grad_coordinates, seed, dw, s);
        add_split(s, m_pick);
        deliver(next);
      }
      clock.mark(kClockRest);
    }
    if (kBoundary && tile < tiles) {  // boundary tiles (uniform per workgroup)
      __syncthreads();
      for (; tile < tiles; tile += slots, ++round) {
        keep_lds_reads_in_loop();
        const int m_pick = opaque(m);
        const TileInputs in = next;
        if (tile + slots < tiles) {
          next = load_tile_inputs<kLoss, kRest>(coordinates, grad_output, grad_laplacian, batch, whole, seed,
                                         tile + slots, w, m);
        }
        const int64_t point = (tile - seed.interior_tiles) * kTile + m;
        SplitSums s{};
        split_tile<1, kLoss>(w_lane, w_t, s_small, s_x.split, minus_one, w, g, m_pick, in.x0, in.x1, 0.f,
                             0.f, 0.f, point < seed.boundary_count, walk_sign(slot, round), point, nullptr, seed, dw, s);
        add_split(s, m_pick);
        deliver(next);
        clock.mark(kClockBoundary);
        clock.count(kClockBoundaryTiles);
      }
    }

    // ---- this slot's partial row: every entry written by exactly one lane ----
    float* row = partials + static_cast<int64_t>(slot) * kRowStride;
    store_dw(row, w, lane, dw);
    // Per-wave sums (lane = owned neuron) combined over the 4 waves in a fixed order.
    __syncthreads();  // every wave is done with the staging buffer
    {
      const int o = owned_neuron(m, g);
#pragma unroll
      for (int q = 0; q < kCombined; ++q) s_x.comb[q][w][o] = sum[q];
      if (lane == 0) {
        s_red[0][w] = sum_bout;
        s_red[1][w] = sum_loss;
        s_red[2][w] = sum_bloss;
      }
      __syncthreads();
      const int n = lane;  // neuron; this wave stores quantities w and w + 4
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int q = w + 4 * i;
        if (q < kCombined) {
          const float total = ((s_x.comb[q][0][n] + s_x.comb[q][1][n]) + s_x.comb[q][2][n]) + s_x.comb[q][3][n];
          // dW0 / 2, db0 / c, dw_out, hidden db / c
          const int dst = q < 2 ? kInputs * n + q
                          : q == 2 ? kLayer0Bias + n
                          : q == 3 ? kOutputBase + n
                                   : kHiddenBase + (q - 4) * kHiddenStride + kHidden * kHidden + n;
          __builtin_nontemporal_store((q < 2 ? 2.0f : q == 3 ? 1.0f : kC) * total, &row[dst]);
        }
      }
      if (threadIdx.x < (kLoss ? 3 : 1)) {
        const float* red = s_red[threadIdx.x];
        const int col = threadIdx.x == 0 ? kOutputBase + kHidden : kLossColumn + threadIdx.x - 1;
        __builtin_nontemporal_store(((red[0] + red[1]) + red[2]) + red[3], &row[col]);
      }
    }
    __syncthreads();  // s_red and the staging buffer are reused by the next slot
    clock.mark(kClockPartials);
  }
  clock.store(w);
}

// ---------------------------------------------------------------------------------------------
// Small-batch backward. backward_kernel carries 16 points per wave through the whole walk, so a
// batch with at most one workgroup tile per CU costs that latency whatever its size. Here a
// workgroup of 4 waves runs one 16-point tile at a time with rows split over the waves
// (split_tile; boundary tiles with the value channel alone).
//   * Each wave owns distinct entries of the slot's partial row (its rows of the vectors, its
//     block of every dW), so the partial row needs no combine across waves.
// Slots and the fixed-order reduction are those of backward_kernel with 16-point tiles. The
// choice between the two kernels depends only on the batch, so results do not depend on the
// device. The tanh-jet, adjoint and loss arithmetic is backward_kernel's; the sums over points
// are grouped differently, so the two kernels agree to rounding, not bitwise.
template <bool kLoss>
__global__ void __launch_bounds__(kSplitWaves * kWave, 1)
backward_split_kernel(const float* __restrict__ coordinates, const float* __restrict__ params,
                      const float* __restrict__ grad_output,
                      const float* __restrict__ grad_laplacian,
                      float* __restrict__ grad_coordinates, float* __restrict__ partials,
                      int64_t batch, int64_t tiles, int slots, LossSeed seed) {
  __shared__ u4 s_w[3 * kLayerU4];
  __shared__ __attribute__((aligned(16))) float s_small[kSmallFloats];
  __shared__ SplitScratch s_x;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x / kWave;
  const int m = lane & 15;
  const int g = lane >> 4;
  // Per-point inputs of 16-point tiles (load_tile_inputs with no 64-point tiles): the first
  // slot's first tile's are read before the staging and each next tile's during the current
  // one, so no tile starts with a wait on global memory (a call here is a few tiles long).
  TileInputs next{0.f, 0.f, 0.f, 0.f};
  if (static_cast<int>(blockIdx.x) < slots) {
    next = load_tile_inputs<kLoss, true>(coordinates, grad_output, grad_laplacian, batch, 0, seed,
                                         blockIdx.x, w, m);
  }
  const float step_count = kLoss ? seed.step[0] : 0.0f;  // advanced below, as in backward_kernel
  const SmallLoads small = load_small<kSplitWaves * kWave>(params, threadIdx.x);
  stage_operand_weights<kSplitWaves * kWave>(params, s_w, threadIdx.x);
  store_small(s_small, threadIdx.x, small);
  __syncthreads();
  if (kLoss && blockIdx.x == 0 && threadIdx.x == 0) seed.step[0] = step_count + 1.0f;

  const u2 minus_one = minus_identity(m, g);
  const int entry = operand_entry(m, g);
  const u4* w_lane = s_w + entry;
  const u4* w_t = s_w + transposed_entry(m, g);
  for (int slot = blockIdx.x; slot < slots; slot += gridDim.x) {
    f16 dw[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
#pragma unroll
      for (int r = 0; r < 16; ++r) dw[l][r] = 0.0f;
    }
    SplitSums sums{};
    if (slot != static_cast<int>(blockIdx.x)) {
      next = load_tile_inputs<kLoss, true>(coordinates, grad_output, grad_laplacian, batch, 0,
                                           seed, slot, w, m);
    }
    // Interior tiles, then (kLoss) boundary tiles.
    const int64_t interior_end = kLoss ? std::min<int64_t>(tiles, seed.interior_tiles) : tiles;
    int64_t tile = slot;
    int round = 0;  // tiles of this slot so far (walk_sign)
    for (; tile < interior_end; tile += slots, ++round) {
      keep_lds_reads_in_loop();
      const TileInputs in = next;
      if (tile + slots < tiles) {
        next = load_tile_inputs<kLoss, true>(coordinates, grad_output, grad_laplacian, batch, 0,
                                             seed, tile + slots, w, m);
      }
      const int64_t point = tile * kTile + m;
      split_tile<4, kLoss>(w_lane, w_t, s_small, s_x, minus_one, w, g, m, in.x0, in.x1,
                           kLoss ? 0.f : in.a, kLoss ? 0.f : in.b, kLoss ? in.a : 0.f, point < batch,
                           walk_sign(slot, round), point, grad_coordinates, seed, dw, sums);
      deliver(next);
    }
    if (kLoss) {
      for (; tile < tiles; tile += slots, ++round) {
        keep_lds_reads_in_loop();
        const TileInputs in = next;
        if (tile + slots < tiles) {
          next = load_tile_inputs<kLoss, true>(coordinates, grad_output, grad_laplacian, batch, 0,
                                               seed, tile + slots, w, m);
        }
        const int64_t point = (tile - seed.interior_tiles) * kTile + m;
        split_tile<1, kLoss>(w_lane, w_t, s_small, s_x, minus_one, w, g, m, in.x0, in.x1, 0.f, 0.f, 0.f,
                             point < seed.boundary_count, walk_sign(slot, round), point, nullptr, seed, dw,
                             sums);
        deliver(next);
      }
    }

    // ---- this slot's partial row: each wave writes its own rows and blocks ----
    float* row = partials + static_cast<int64_t>(slot) * kRowStride;
    store_dw(row, w, lane, dw);
    if (m < 4) {
      const int n = 16 * w + 4 * g + m;
      row[kInputs * n] = 2.0f * sums.w0x;
      row[kInputs * n + 1] = 2.0f * sums.w0y;
      row[kLayer0Bias + n] = kC * sums.b0;
      row[kOutputBase + n] = sums.wout;
#pragma unroll
      for (int l = 0; l < 3; ++l) {
        row[kHiddenBase + l * kHiddenStride + kHidden * kHidden + n] = kC * sums.bh[l];
      }
    }
    if (w == 0 && lane == 0) {
      row[kOutputBase + kHidden] = sums.bout;
      if (kLoss) {
        row[kLossColumn] = sums.loss;
        row[kLossColumn + 1] = sums.bloss;
      }
    }
  }
}

constexpr int kPerGroup = kMaxSlots / kReduceGroups;  // slots per group of the fixed tree

// Column k's entries of group `group`'s slots, in slot order, as loaded: slot and column are
// clamped to a written row, and fixed_tree_total drops what lies beyond them. The 16 loads are
// issued unconditionally, where this is called, and waited for once, in fixed_tree_total:
// behind per-slot branches the compiler had waited for the first load, and for everything
// issued before it, before it issued the other 15.
__device__ __forceinline__ void load_group_column(const float* __restrict__ partials, int slots,
                                                  int k, int columns, int group,
                                                  float (&v)[kPerGroup]) {
  const int column = k < columns ? k : 0;
#pragma unroll
  for (int i = 0; i < kPerGroup; ++i) {
    const int slot = group * kPerGroup + i;
    v[i] = partials[static_cast<int64_t>(slot < slots ? slot : slots - 1) * kRowStride + column];
  }
}

// The fixed-tree total of column k from load_group_column's entries: each group's entries in
// slot order, then the 16 group sums in group order; complete in the threads of group 0. Slots
// at or beyond `slots` add +0.0f, and a column >= `columns` sums to +0.0f.
__device__ __forceinline__ float fixed_tree_total(float (&v)[kPerGroup], int slots, int k,
                                                  int columns, float (*s_part)[64], int group,
                                                  int col) {
  // An empty asm that reads and writes the 16 values: the loads cannot sink past it (into
  // per-slot branches around the selects below), so they stay where they were issued.
  __asm__ volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]),
                   "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]), "+v"(v[10]), "+v"(v[11]),
                   "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
  static_assert(kPerGroup == 16, "the asm above names 16 values");
  float acc = 0.0f;
#pragma unroll
  for (int i = 0; i < kPerGroup; ++i) {
    const int slot = group * kPerGroup + i;
    acc += k < columns && slot < slots ? v[i] : 0.0f;
  }
  s_part[group][col] = acc;
  __syncthreads();
  float total = 0.0f;
  if (group == 0) {
#pragma unroll
    for (int i = 0; i < kReduceGroups; ++i) total += s_part[i][col];
  }
  return total;
}

// grad[k] = sum over slots of partials[slot][k], in a fixed tree: 16 groups of 16 consecutive
// slots are summed in slot order, then the 16 group sums in group order. Slots at or beyond
// `slots` are skipped (they would add +0.0f).
__global__ void __launch_bounds__(kReduceGroups * 64)
reduce_partials_kernel(const float* __restrict__ partials, int slots, float* __restrict__ grad) {
  __shared__ float s_part[kReduceGroups][64];
  const int col = threadIdx.x & 63;
  const int group = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + col;
  float v[kPerGroup];
  load_group_column(partials, slots, k, kParameterCount, group, v);
  const float total = fixed_tree_total(v, slots, k, kParameterCount, s_part, group, col);
  if (group == 0 && k < kParameterCount) grad[k] = total;
}

// Adam (torch.optim.Adam, amsgrad = False, maximize = False) on the flat parameter buffer.
struct AdamArgs {
  float* params;
  float* exp_avg;
  float* exp_avg_sq;
  const float* step;  // already advanced for this step by the gradient kernel
  float* loss;        // mean r^2 + w mean u_b^2
  float* grad;        // optional copy of the summed gradient (nullptr: none)
  double lr, beta1, beta2, eps, weight_decay;
  float inv_batch;       // fl(1 / B)
  float inv_boundary;    // fl(1 / B_b), 0 without boundary points
  float boundary_weight; // fl(w)
};

// The fixed-tree gradient sum of reduce_partials_kernel, then the Adam update of each
// parameter in the same thread, so the summed gradient never goes through memory. Element
// arithmetic follows torch's multi-tensor Adam (torch/optim/adam.py, _multi_tensor_adam):
//   g += wd p;  m = lerp(m, g, 1 - b1);  v = v b2 + (1 - b2) g g;
//   p += -(lr / bc1) m / (sqrt(v) / sqrt(bc2) + eps),  bc_i = 1 - b_i^t,
// with the bias corrections in double and every tensor operation rounded to float. Columns
// kLossColumn and kLossColumn + 1 give loss = fl(sum r^2 / B) + fl(w fl(sum u_b^2 / B_b)).
__global__ void __launch_bounds__(kReduceGroups * 64)
reduce_adam_kernel(const float* __restrict__ partials, int slots, AdamArgs a) {
  __shared__ float s_part[kReduceGroups][64];
  __shared__ float s_loss[2];
  const int col = threadIdx.x & 63;
  const int group = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + col;
  // The Adam state is read before the partial rows, so the two memory round trips overlap.
  const bool updates = group == 0 && k < kParameterCount;
  float p = 0.0f, m = 0.0f, v = 0.0f;
  if (updates) {
    p = a.params[k];
    m = a.exp_avg[k];
    v = a.exp_avg_sq[k];
  }
  const float step_count = a.step[0];
  float parts[kPerGroup];
  load_group_column(partials, slots, k, kLossColumn + 2, group, parts);
  // The bias corrections (two double-precision powers, a long dependent chain) are formed in
  // the updating wave while the partial rows are in flight, not after their sum.
  float step_size = 0.0f, bc2_sqrt = 1.0f;
  if (updates) {
    const double t = static_cast<double>(step_count);
    const double bc1 = 1.0 - pow(a.beta1, t);
    const double bc2 = 1.0 - pow(a.beta2, t);
    step_size = static_cast<float>(-(a.lr / bc1));
    bc2_sqrt = static_cast<float>(sqrt(bc2));
  }
  const float total = fixed_tree_total(parts, slots, k, kLossColumn + 2, s_part, group, col);
  if (group == 0 && (k == kLossColumn || k == kLossColumn + 1)) s_loss[k - kLossColumn] = total;
  __syncthreads();
  if (group != 0) return;
  if (k == kLossColumn) {
    const float interior = s_loss[0] * a.inv_batch;
    a.loss[0] = a.inv_boundary != 0.0f ? interior + a.boundary_weight * (s_loss[1] * a.inv_boundary)
                                       : interior;
    return;
  }
  if (!updates) return;
  if (a.grad) a.grad[k] = total;
  const float w1 = static_cast<float>(1.0 - a.beta1);
  const float b2 = static_cast<float>(a.beta2);
  const float w2 = static_cast<float>(1.0 - a.beta2);
  const float eps = static_cast<float>(a.eps);
  const float wd = static_cast<float>(a.weight_decay);

  float g = total;
  if (wd != 0.0f) g = g + wd * p;
  m = m + w1 * (g - m);  // lerp with weight < 0.5
  v = v * b2;
  v = v + w2 * g * g;
  const float denom = sqrtf(v) / bc2_sqrt + eps;
  p = p + step_size * m / denom;
  a.exp_avg[k] = m;
  a.exp_avg_sq[k] = v;
  a.params[k] = p;
}

__global__ void fill_zero_kernel(float* __restrict__ out, int64_t n) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (k < n) out[k] = 0.0f;
}

// ---------------------------------------------------------------------------------------------
// Host side.

constexpr int kFwdWaves = 8;  // forward workgroup: 2 waves per SIMD
constexpr int kSplitTilesPerCu = 2;  // forward_split_kernel up to this many tiles per CU

thread_local char g_last_error[512] = "";

int fail(int status, const char* fmt, ...) {
  va_list args;
  va_start(args, fmt);
  std::vsnprintf(g_last_error, sizeof(g_last_error), fmt, args);
  va_end(args);
  return status;
}

int check_launch(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) {
    return fail(FHOAD_ERROR_DEVICE, "%s launch failed: %s", what, hipGetErrorString(err));
  }
  return FHOAD_SUCCESS;
}

// Tiles of forward_kernel that run whole: all of them below one round of one tile per SIMD
// (4 per workgroup) or when the rounds are whole, otherwise the whole rounds; the rest run as
// split tiles. FUSED_HOAD_FWD_SPLIT_REST=0 (experiment knob, read per call) runs every tile
// whole.
int64_t forward_whole_tiles(int64_t tiles, int grid) {
  const int64_t round = 4 * static_cast<int64_t>(grid);
  if (const char* env = std::getenv("FUSED_HOAD_FWD_SPLIT_REST")) {
    if (std::atoi(env) == 0) return tiles;
  }
  if (tiles < round || tiles % round == 0) return tiles;
  return tiles - tiles % round;
}

// Compute units of the current device, queried once per device. The cache entries are atomic:
// calls from several host threads may fill the same entry (with the same value).
int current_device_cus(int* cus) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices] = {};
  int device = 0;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "hipGetDevice: %s", hipGetErrorString(err));
  if (device >= 0 && device < kMaxDevices) {
    const int known = cached[device].load(std::memory_order_relaxed);
    if (known > 0) {
      *cus = known;
      return FHOAD_SUCCESS;
    }
  }
  int count = 0;
  err = hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device);
  if (err != hipSuccess) {
    return fail(FHOAD_ERROR_DEVICE, "hipDeviceGetAttribute: %s", hipGetErrorString(err));
  }
  if (count < 1) count = 1;
  if (device >= 0 && device < kMaxDevices) cached[device].store(count, std::memory_order_relaxed);
  *cus = count;
  return FHOAD_SUCCESS;
}

// Workspaces and saved-layer buffers must be 16-byte aligned (part of the ABI: hipMalloc and
// torch allocations are).
int check_workspace_alignment(const void* workspace, const char* what = "workspace") {
  if (reinterpret_cast<uintptr_t>(workspace) % alignof(f4) != 0) {
    return fail(FHOAD_ERROR_MISALIGNED, "%s must be 16-byte aligned", what);
  }
  return FHOAD_SUCCESS;
}

int64_t backward_tiles(int64_t batch) { return (batch + kBwdTile - 1) / kBwdTile; }

int slots_for_tiles(int64_t tiles) { return static_cast<int>(std::min<int64_t>(tiles, kMaxSlots)); }

int backward_slots(int64_t batch) { return slots_for_tiles(backward_tiles(batch)); }

// Workspace of the gradient kernels for `slots` slots: one partial row per slot.
constexpr size_t workspace_bytes_for(int slots) {
  return static_cast<size_t>(slots) * kRowStride * sizeof(float);
}

// Scratch of fhoad_forward_laplacian_backward_noalloc: a file-scope device array, one per GPU
// (each device that loads this code object holds its own copy until the process ends). It is
// sized for kMaxSlots slots, the most any batch uses (both gradient kernels cap their slots
// at kMaxSlots), so every batch fits. Host code never passes `scratch` itself to a kernel:
// the name is a host-side stand-in, and the device address comes from hipGetSymbolAddress
// (noalloc_scratch below).
constexpr size_t kNoAllocScratchBytes = workspace_bytes_for(kMaxSlots);
static_assert(kNoAllocScratchBytes % sizeof(float) == 0, "the scratch holds whole partial rows");
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

int64_t split_tiles(int64_t points) { return (points + kTile - 1) / kTile; }

// Interior tiles of backward_kernel for `batch` points over `slots` slots: 64-point tiles in
// whole rounds of `slots` (`whole` of them), then the remaining points as 16-point tiles whose
// rows are split over the waves (`total` counts both). Below one whole round, or when the
// rounds are whole, every tile is a 64-point one. A split tile takes 0.43 of a 64-point tile's time, so
// a rest of one or two a slot costs less than a round of 64-point tiles would, one of three or four
// more (backward call of 16,384 points 36.4 us, 16,400 44.2, 24,000 57.5, 28,000 67, 32,000 77, and
// 32,768, two whole rounds, 58.6).
struct InteriorTiles {
  int64_t whole, total;
};

InteriorTiles interior_tiles_for(int64_t batch, int slots) {
  const int64_t t64 = backward_tiles(batch);
  const int64_t rounds = t64 / slots;
  if (rounds == 0 || t64 % slots == 0) return {t64, t64};
  const int64_t whole = rounds * slots;
  return {whole, whole + split_tiles(batch - whole * kBwdTile)};
}

// Gradient kernel for `batch` interior and `boundary_count` boundary points:
// backward_split_kernel up to kSplitBwdMaxTiles 16-point tiles, chosen from the batch alone
// so that results do not depend on the device. FUSED_HOAD_BWD_SPLIT=0 / 1 (experiment knob,
// read per call) forces either kernel.
bool use_split_backward(int64_t batch, int64_t boundary_count) {
  if (const char* env = std::getenv("FUSED_HOAD_BWD_SPLIT")) return std::atoi(env) != 0;
  return split_tiles(batch) + split_tiles(boundary_count) <= kSplitBwdMaxTiles;
}

// Workspace for either gradient kernel: one partial row per slot, for the larger slot count of
// the two (a knob can force either kernel).
size_t gradient_workspace_bytes(int64_t batch, int64_t boundary_count) {
  const int64_t boundary_tiles = split_tiles(boundary_count);
  return workspace_bytes_for(slots_for_tiles(
      std::max(backward_tiles(batch), split_tiles(batch)) + boundary_tiles));
}

// Persistent grid of the gradient kernel: one workgroup per CU, at most one per slot.
// FUSED_HOAD_BWD_BLOCKS caps it, as in the reference (fused_backward.cu:873-880). Here it
// changes only which workgroup computes a slot, never the arithmetic, so gradients stay
// bitwise identical.
int backward_grid(int slots, int* grid) {
  int cus = 0;
  if (int st = current_device_cus(&cus)) return st;
  *grid = std::min(slots, cus);
  if (const char* env = std::getenv("FUSED_HOAD_BWD_BLOCKS")) {
    const long cap = std::atol(env);
    if (cap > 0) *grid = static_cast<int>(std::min<long>(*grid, cap));
  }
  return FHOAD_SUCCESS;
}

// Device address of this device's `scratch`, looked up once per device (with that device
// current, on the first no-allocation call there) and kept per device: each GPU holds its own
// copy of the array at its own address. The cache entries are atomic, so calls from several
// host threads may fill one (with the same address).
int noalloc_scratch(void** out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<void*> addresses[kMaxDevices] = {};
  int device = 0;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "hipGetDevice: %s", hipGetErrorString(err));
  if (device < 0 || device >= kMaxDevices) {
    return fail(FHOAD_ERROR_DEVICE, "device %d is beyond the %d devices the scratch table covers",
                device, kMaxDevices);
  }
  void* address = addresses[device].load(std::memory_order_acquire);
  if (address == nullptr) {
    // The first call on a device may come while the caller captures a HIP graph (the callers
    // this entry point is for): the lookup, which may load the code object on this device, runs
    // in the relaxed capture mode, so a global-mode capture in progress neither rejects it nor
    // is invalidated by it. The thread's mode is restored afterwards.
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    err = hipThreadExchangeStreamCaptureMode(&mode);
    if (err != hipSuccess) {
      return fail(FHOAD_ERROR_DEVICE, "hipThreadExchangeStreamCaptureMode: %s", hipGetErrorString(err));
    }
    const hipError_t lookup = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    err = hipThreadExchangeStreamCaptureMode(&mode);
    if (lookup != hipSuccess || address == nullptr) {
      return fail(FHOAD_ERROR_DEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(lookup));
    }
    if (err != hipSuccess) {
      return fail(FHOAD_ERROR_DEVICE, "hipThreadExchangeStreamCaptureMode: %s", hipGetErrorString(err));
    }
    addresses[device].store(address, std::memory_order_release);
  }
  *out = address;
  return FHOAD_SUCCESS;
}

// Backward call on a workspace of `workspace_bytes` bytes (checked by the caller).
int launch_backward(const float* coordinates, const float* parameters, const float* grad_output,
                    const float* grad_laplacian, float* grad_parameters, float* grad_coordinates,
                    void* workspace, int64_t batch, hipStream_t hs);

}  // namespace
}  // namespace fhoad

using namespace fhoad;

extern "C" int fhoad_abi_version(void) { return FHOAD_ABI_VERSION; }

extern "C" int64_t fhoad_parameter_count(void) { return kParameterCount; }

extern "C" const char* fhoad_status_string(int status) {
  switch (status) {
    case FHOAD_SUCCESS: return "success";
    case FHOAD_ERROR_INVALID_VERSION: return "invalid version";
    case FHOAD_ERROR_INVALID_VALUE: return "invalid value";
    case FHOAD_ERROR_MISALIGNED: return "misaligned pointer";
    case FHOAD_ERROR_WORKSPACE: return "workspace too small";
    case FHOAD_ERROR_DEVICE: return "device error";
    default: return "unknown status";
  }
}

extern "C" const char* fhoad_last_error(void) { return g_last_error; }

extern "C" int fhoad_check_device(void* stream) {
  hipError_t err = hipStreamSynchronize(static_cast<hipStream_t>(stream));
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "hipStreamSynchronize: %s", hipGetErrorString(err));
  unsigned status = 0;
  err = hipMemcpyFromSymbol(&status, HIP_SYMBOL(g_device_status), sizeof(status), 0, hipMemcpyDeviceToHost);
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "reading the device status: %s", hipGetErrorString(err));
  if (status == 0) return FHOAD_SUCCESS;
  const unsigned zero = 0;
  err = hipMemcpyToSymbol(HIP_SYMBOL(g_device_status), &zero, sizeof(zero), 0, hipMemcpyHostToDevice);
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "clearing the device status: %s", hipGetErrorString(err));
  return fail(FHOAD_ERROR_DEVICE,
              "a forward split tile's wave gave up waiting for its quad (status 0x%x): that tile's u "
              "and Laplacian were written as NaN",
              status);
}

#ifdef FHOAD_PHASE_CLOCK
// Measurement build only: the shape of backward_kernel's phase-clock table
// ([workgroups][waves][fields] of uint64), its reset and its copy to the host.
extern "C" void fhoad_phase_clock_shape(int* workgroups, int* waves, int* fields) {
  *workgroups = kClockWorkgroups;
  *waves = kBwdWaves;
  *fields = kClockFields;
}

extern "C" int fhoad_phase_clock_reset(void) {
  static const unsigned long long zeros[kClockWorkgroups * kBwdWaves * kClockFields] = {};
  hipError_t err = hipDeviceSynchronize();
  if (err == hipSuccess) err = hipMemcpyToSymbol(HIP_SYMBOL(g_phase_clock), zeros, sizeof(zeros));
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "resetting the phase clock: %s", hipGetErrorString(err));
  return FHOAD_SUCCESS;
}

extern "C" int fhoad_phase_clock_read(unsigned long long* out) {
  hipError_t err = hipDeviceSynchronize();
  if (err == hipSuccess) {
    err = hipMemcpyFromSymbol(out, HIP_SYMBOL(g_phase_clock), sizeof(g_phase_clock), 0,
                              hipMemcpyDeviceToHost);
  }
  if (err != hipSuccess) return fail(FHOAD_ERROR_DEVICE, "reading the phase clock: %s", hipGetErrorString(err));
  return FHOAD_SUCCESS;
}
#endif

namespace fhoad {
namespace {

// The forward launch shared by fhoad_forward_laplacian and fhoad_forward_laplacian_saving.
// batch > 0.
int launch_forward(const float* coordinates, const float* parameters, float* output,
                   float* laplacian, int64_t batch, hipStream_t hs) {
  int cus = 0;
  if (int st = current_device_cus(&cus)) return st;
  const int64_t tiles = (batch + kTile - 1) / kTile;
  const int grid = static_cast<int>(std::min<int64_t>(tiles, cus));
  // Below kSplitTilesPerCu tiles per CU the split kernel runs each tile on a CU's 4 SIMDs.
  // FUSED_HOAD_FWD_SPLIT=0 / 1 (experiment knob, read per call) forces either kernel.
  const char* split_env = std::getenv("FUSED_HOAD_FWD_SPLIT");
  const bool split = split_env ? std::atoi(split_env) != 0 : tiles <= kSplitTilesPerCu * cus;
  if (split) {
    const int split_grid = static_cast<int>(std::min<int64_t>(tiles, kSplitTilesPerCu * cus));
    hipLaunchKernelGGL(forward_split_kernel, dim3(split_grid), dim3(kSplitWaves * kWave), 0, hs,
                       coordinates, parameters, output, laplacian, batch, tiles);
    return check_launch("forward_split_kernel");
  }
  const int64_t whole = forward_whole_tiles(tiles, grid);
  // Polls per quad meeting before a split tile's wave gives up. FUSED_HOAD_QUAD_SPIN_LIMIT
  // (test knob, read per call) lowers it; 0 makes every meeting give up at once, so the tests can
  // check the timeout path (device status word, NaN outputs) with every kernel exiting normally.
  int spin_limit = kQuadSpinLimit;
  if (const char* env = std::getenv("FUSED_HOAD_QUAD_SPIN_LIMIT")) {
    spin_limit = static_cast<int>(std::min<long>(std::max<long>(std::atol(env), 0), kQuadSpinLimit));
  }
  hipLaunchKernelGGL((forward_kernel<kFwdWaves>), dim3(grid), dim3(kFwdWaves * kWave), 0, hs,
                     coordinates, parameters, output, laplacian, batch, whole, tiles, spin_limit);
  return check_launch("forward_kernel");
}

}  // namespace
}  // namespace fhoad

extern "C" int fhoad_forward_laplacian(const float* coordinates, const float* parameters,
                                       float* output, float* laplacian, int64_t batch,
                                       int version, void* stream) {
  if (version < 0 || version > 5) return fail(FHOAD_ERROR_INVALID_VERSION, "version must be 0 to 5");
  if (batch < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be non-negative");
  if (batch == 0) return FHOAD_SUCCESS;
  if (!coordinates || !parameters || !output || !laplacian) {
    return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  }
  return launch_forward(coordinates, parameters, output, laplacian, batch,
                        static_cast<hipStream_t>(stream));
}

// The saved-layer pair checks its buffer as it always did and runs the forward and the backward
// that re-runs it (see fused_hoad.h).
constexpr int64_t kSavedF4PerTile = 3 * 16 * kWave;  // the buffer: h1..h3 of a 16-point tile

extern "C" size_t fhoad_saved_layers_size(int64_t batch) {
  if (batch <= 0) return 0;
  // Unsigned, and saturated: a batch whose buffer would not fit in size_t gets SIZE_MAX, which
  // no buffer can hold, so the saving forward rejects it.
  constexpr uint64_t kTileBytes = static_cast<uint64_t>(kSavedF4PerTile) * sizeof(f4);
  const uint64_t tiles = (static_cast<uint64_t>(batch) + kTile - 1) / kTile;
  if (tiles > SIZE_MAX / kTileBytes) return SIZE_MAX;
  return static_cast<size_t>(tiles * kTileBytes);
}

extern "C" int fhoad_forward_laplacian_saving(const float* coordinates, const float* parameters,
                                              float* output, float* laplacian, void* saved,
                                              size_t saved_bytes, int64_t batch, int version,
                                              void* stream) {
  if (version < 0 || version > 5) return fail(FHOAD_ERROR_INVALID_VERSION, "version must be 0 to 5");
  if (batch < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be non-negative");
  if (batch == 0) return FHOAD_SUCCESS;
  if (!coordinates || !parameters || !output || !laplacian) {
    return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  }
  const size_t needed = fhoad_saved_layers_size(batch);
  if (!saved || saved_bytes < needed) {
    return fail(FHOAD_ERROR_WORKSPACE, "saved-layer buffer holds %zu bytes, %zu needed", saved_bytes,
                needed);
  }
  if (int st = check_workspace_alignment(saved, "saved-layer buffer")) return st;
  return launch_forward(coordinates, parameters, output, laplacian, batch,
                        static_cast<hipStream_t>(stream));
}

extern "C" size_t fhoad_backward_workspace_size(int64_t batch) {
  if (batch <= 0) return 0;
  return gradient_workspace_bytes(batch, 0);
}

extern "C" size_t fhoad_poisson_adam_step_workspace_size(int64_t batch, int64_t boundary_count) {
  if (batch <= 0 || boundary_count < 0) return 0;
  return gradient_workspace_bytes(batch, boundary_count);
}

extern "C" int fhoad_forward_laplacian_backward(const float* coordinates, const float* parameters,
                                                const float* grad_output,
                                                const float* grad_laplacian,
                                                float* grad_parameters, float* grad_coordinates,
                                                void* workspace, size_t workspace_bytes,
                                                int64_t batch, int version, void* stream) {
  if (version < 1 || version > 6) {
    return fail(FHOAD_ERROR_INVALID_VERSION, "backward version must be 1 to 6");
  }
  if (batch < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be non-negative");
  if (!parameters || !grad_parameters) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const hipStream_t hs = static_cast<hipStream_t>(stream);
  if (batch == 0) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3((kParameterCount + 255) / 256), dim3(256), 0, hs,
                       grad_parameters, static_cast<int64_t>(kParameterCount));
    return check_launch("fill_zero_kernel");
  }
  if (!coordinates) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const size_t needed = fhoad_backward_workspace_size(batch);
  if (!workspace || workspace_bytes < needed) {
    return fail(FHOAD_ERROR_WORKSPACE, "workspace holds %zu bytes, %zu needed", workspace_bytes,
                needed);
  }
  if (int st = check_workspace_alignment(workspace)) return st;
  return launch_backward(coordinates, parameters, grad_output, grad_laplacian, grad_parameters,
                         grad_coordinates, workspace, batch, hs);
}

extern "C" int fhoad_forward_laplacian_backward_noalloc(
    const float* coordinates, const float* parameters, const float* grad_output,
    const float* grad_laplacian, float* grad_parameters, float* grad_coordinates, int64_t batch,
    int version, void* stream) {
  if (version < 1 || version > 6) {
    return fail(FHOAD_ERROR_INVALID_VERSION, "backward version must be 1 to 6");
  }
  if (batch < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be non-negative");
  if (!parameters || !grad_parameters) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const hipStream_t hs = static_cast<hipStream_t>(stream);
  if (batch == 0) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3((kParameterCount + 255) / 256), dim3(256), 0, hs,
                       grad_parameters, static_cast<int64_t>(kParameterCount));
    return check_launch("fill_zero_kernel");
  }
  if (!coordinates) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const size_t needed = fhoad_backward_workspace_size(batch);
  if (needed > kNoAllocScratchBytes) {
    return fail(FHOAD_ERROR_WORKSPACE, "batch %lld needs %zu bytes of scratch, the static scratch holds %zu",
                static_cast<long long>(batch), needed, kNoAllocScratchBytes);
  }
  void* device_scratch = nullptr;
  if (int st = noalloc_scratch(&device_scratch)) return st;
  return launch_backward(coordinates, parameters, grad_output, grad_laplacian, grad_parameters,
                         grad_coordinates, device_scratch, batch, hs);
}

extern "C" int fhoad_forward_laplacian_backward_saved(
    const float* coordinates, const float* parameters, const void* saved, size_t saved_bytes,
    const float* grad_output, const float* grad_laplacian, float* grad_parameters,
    float* grad_coordinates, void* workspace, size_t workspace_bytes, int64_t batch, int version,
    void* stream) {
  if (version < 1 || version > 6) {
    return fail(FHOAD_ERROR_INVALID_VERSION, "backward version must be 1 to 6");
  }
  if (batch < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be non-negative");
  if (!parameters || !grad_parameters) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const hipStream_t hs = static_cast<hipStream_t>(stream);
  if (batch == 0) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3((kParameterCount + 255) / 256), dim3(256), 0, hs,
                       grad_parameters, static_cast<int64_t>(kParameterCount));
    return check_launch("fill_zero_kernel");
  }
  if (!coordinates) return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  const size_t saved_needed = fhoad_saved_layers_size(batch);
  if (!saved || saved_bytes < saved_needed) {
    return fail(FHOAD_ERROR_WORKSPACE, "saved-layer buffer holds %zu bytes, %zu needed",
                saved_bytes, saved_needed);
  }
  if (int st = check_workspace_alignment(saved, "saved-layer buffer")) return st;
  const size_t needed = fhoad_backward_workspace_size(batch);
  if (!workspace || workspace_bytes < needed) {
    return fail(FHOAD_ERROR_WORKSPACE, "workspace holds %zu bytes, %zu needed", workspace_bytes,
                needed);
  }
  if (int st = check_workspace_alignment(workspace)) return st;
  return launch_backward(coordinates, parameters, grad_output, grad_laplacian, grad_parameters,
                         grad_coordinates, workspace, batch, hs);
}

namespace fhoad {
namespace {

int launch_backward(const float* coordinates, const float* parameters, const float* grad_output,
                    const float* grad_laplacian, float* grad_parameters, float* grad_coordinates,
                    void* workspace, int64_t batch, hipStream_t hs) {
  float* partials = static_cast<float*>(workspace);
  int slots = 0, grid = 0;
  if (use_split_backward(batch, 0)) {
    const int64_t tiles = split_tiles(batch);
    slots = slots_for_tiles(tiles);
    if (int st = backward_grid(slots, &grid)) return st;
    hipLaunchKernelGGL(backward_split_kernel<false>, dim3(grid), dim3(kSplitWaves * kWave), 0, hs,
                       coordinates, parameters, grad_output, grad_laplacian, grad_coordinates,
                       partials, batch, tiles, slots, LossSeed{});
    if (int st = check_launch("backward_split_kernel")) return st;
  } else {
    slots = backward_slots(batch);
    if (int st = backward_grid(slots, &grid)) return st;
    const InteriorTiles it = interior_tiles_for(batch, slots);
    const dim3 block(kBwdWaves * kWave);
    if (it.whole != it.total) {
      hipLaunchKernelGGL((backward_kernel<false, true, false>), dim3(grid), block, 0, hs, coordinates,
                         parameters, grad_output, grad_laplacian, grad_coordinates, partials, batch,
                         it.whole, it.total, slots, LossSeed{});
    } else {
      hipLaunchKernelGGL((backward_kernel<false, false, false>), dim3(grid), block, 0, hs, coordinates,
                         parameters, grad_output, grad_laplacian, grad_coordinates, partials, batch,
                         it.whole, it.total, slots, LossSeed{});
    }
    if (int st = check_launch("backward_kernel")) return st;
  }
  hipLaunchKernelGGL(reduce_partials_kernel, dim3((kParameterCount + 63) / 64),
                     dim3(kReduceGroups * 64), 0, hs, partials, slots, grad_parameters);
  return check_launch("reduce_partials_kernel");
}

}  // namespace
}  // namespace fhoad

extern "C" int fhoad_poisson_adam_step(const float* coordinates, const float* source,
                                       int64_t batch, const float* boundary,
                                       int64_t boundary_count, double boundary_weight,
                                       float* parameters, float* exp_avg, float* exp_avg_sq,
                                       float* step, float* loss, float* grad_parameters,
                                       float* grad_coordinates, void* workspace,
                                       size_t workspace_bytes, double lr, double beta1,
                                       double beta2, double eps, double weight_decay,
                                       void* stream) {
  if (batch <= 0) return fail(FHOAD_ERROR_INVALID_VALUE, "batch must be positive");
  if (boundary_count < 0) return fail(FHOAD_ERROR_INVALID_VALUE, "boundary_count must be non-negative");
  if (!coordinates || !source || !parameters || !exp_avg || !exp_avg_sq || !step || !loss ||
      (boundary_count > 0 && !boundary)) {
    return fail(FHOAD_ERROR_INVALID_VALUE, "null device pointer");
  }
  if (!(lr >= 0.0) || !(eps >= 0.0) || !(beta1 >= 0.0 && beta1 < 1.0) ||
      !(beta2 >= 0.0 && beta2 < 1.0) || !(weight_decay >= 0.0) || !(boundary_weight >= 0.0)) {
    return fail(FHOAD_ERROR_INVALID_VALUE,
                "Adam needs lr >= 0, eps >= 0, 0 <= betas < 1, weight_decay >= 0 and "
                "boundary_weight >= 0");
  }
  const size_t needed = fhoad_poisson_adam_step_workspace_size(batch, boundary_count);
  if (!workspace || workspace_bytes < needed) {
    return fail(FHOAD_ERROR_WORKSPACE, "workspace holds %zu bytes, %zu needed", workspace_bytes,
                needed);
  }
  if (int st = check_workspace_alignment(workspace)) return st;
  const bool split = use_split_backward(batch, boundary_count);
  const int slots = slots_for_tiles((split ? split_tiles(batch) : backward_tiles(batch)) +
                                    split_tiles(boundary_count));
  const InteriorTiles it =
      split ? InteriorTiles{0, split_tiles(batch)} : interior_tiles_for(batch, slots);
  const int64_t interior_tiles = it.total;
  const int64_t tiles = interior_tiles + split_tiles(boundary_count);  // 16-point boundary tiles
  int grid = 0;
  if (int st = backward_grid(slots, &grid)) return st;
  const hipStream_t hs = static_cast<hipStream_t>(stream);
  const float inv_batch = 1.0f / static_cast<float>(batch);
  const float weight = static_cast<float>(boundary_weight);
  const float boundary_scale = boundary_count > 0 ? weight / static_cast<float>(boundary_count) : 0.0f;
  const float inv_boundary = boundary_count > 0 ? 1.0f / static_cast<float>(boundary_count) : 0.0f;
  float* partials = static_cast<float*>(workspace);
  const LossSeed seed{source, boundary, interior_tiles, boundary_count, inv_batch, boundary_scale, step};
  if (split) {
    hipLaunchKernelGGL(backward_split_kernel<true>, dim3(grid), dim3(kSplitWaves * kWave), 0, hs,
                       coordinates, parameters, nullptr, nullptr, grad_coordinates, partials,
                       batch, tiles, slots, seed);
    if (int st = check_launch("backward_split_kernel")) return st;
  } else {
    if (it.whole != it.total) {
      hipLaunchKernelGGL((backward_kernel<true, true, true>), dim3(grid), dim3(kBwdWaves * kWave),
                         0, hs, coordinates, parameters, nullptr, nullptr, grad_coordinates,
                         partials, batch, it.whole, tiles, slots, seed);
    } else if (boundary_count > 0) {
      hipLaunchKernelGGL((backward_kernel<true, false, true>), dim3(grid), dim3(kBwdWaves * kWave),
                         0, hs, coordinates, parameters, nullptr, nullptr, grad_coordinates,
                         partials, batch, it.whole, tiles, slots, seed);
    } else {
      hipLaunchKernelGGL((backward_kernel<true, false, false>), dim3(grid), dim3(kBwdWaves * kWave),
                         0, hs, coordinates, parameters, nullptr, nullptr, grad_coordinates,
                         partials, batch, it.whole, tiles, slots, seed);
    }
    if (int st = check_launch("backward_kernel")) return st;
  }
  const AdamArgs args{parameters, exp_avg, exp_avg_sq, step, loss, grad_parameters,
                      lr, beta1, beta2, eps, weight_decay, inv_batch, inv_boundary, weight};
  hipLaunchKernelGGL(reduce_adam_kernel, dim3((kLossColumn + 2 + 63) / 64),
                     dim3(kReduceGroups * 64), 0, hs, partials, slots, args);
  return check_launch("reduce_adam_kernel");
}
