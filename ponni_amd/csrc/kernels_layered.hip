// LAYERED kernel family: one dense block over the whole batch on the matrix
// cores.  out[f, b] = epilogue_f(sum_k W[k][f] in[k, b]) for a dense op of the
// GENERIC op list (a generated Dense's bias seeds the sum), the other ops of
// the list running on generic_forward between such launches
// (plan.cpp layered_forward).
//
// Weights are packed in A-fragment order (plan.cpp visit_param_slots, the
// MFMA / FUSED packing), states are [features, batch] rows.  A 256-lane
// workgroup computes 32 MI output features x 32 NJ columns, each of its four
// waves 16 MI x 16 NJ, in contraction steps of KS features.  A step's
// fragments and rows go from memory straight into LDS
// (global_load_lds_dwordx4: no registers, and none of the VALU work that
// does not run beside fp32 / fp64 MFMAs) two steps ahead, into three slots;
// one barrier a step.  16-bit states are contracted on the 16-bit MFMAs: a
// lane's B operand, 4 consecutive features of one column, is one
// ds_read_b64_tr_b16 of the row-major tile.  The usual epilogue steps
// run on the accumulators, one uniform branch a step; any other step, and
// those after it, in a loop over the finished tile in LDS (the run-time
// switch in that loop cost 30 us a tile; unrolled over the accumulators, the
// whole switch held the kernel at one workgroup per CU).  Rows are stored
// from LDS in pieces of 4 columns.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "plan.h"
#include "pointwise.h"

namespace ponni_hip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 b16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 b16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void;
typedef __attribute__((address_space(3))) i16x4* lds_i16x4;

// Storage type -> compute type, A fragment, features per step (one fragment).
template <class S> struct Traits;
template <> struct Traits<float> {
  using C = float;
  using Acc = f32x4;
  using A = f32x4;
  static constexpr int KS = 16;
};
template <> struct Traits<double> {
  using C = double;
  using Acc = f64x4;
  using A = f64x4;
  static constexpr int KS = 16;
};
template <> struct Traits<_Float16> {
  using C = float;
  using Acc = f32x4;
  using A = h16x8;
  using B4 = h16x4;
  static constexpr int KS = 32;
  __device__ static Acc mfma(A a, A b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct Traits<__bf16> {
  using C = float;
  using Acc = f32x4;
  using A = b16x8;
  using B4 = b16x4;
  static constexpr int KS = 32;
  __device__ static Acc mfma(A a, A b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
__device__ inline f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ inline f64x4 mfma4(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// One 16- or 4-byte request per lane into LDS at lds + size * lane (lds
// uniform), as inline asm so that the compiler's wait insertion does not
// wait for every request before each LDS read; the waits below order them
// (the s_nop is the wait state between the write of M0 and its use).
__device__ inline void dma16(void const* g, unsigned lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}
__device__ inline void dma4(void const* g, unsigned lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}
// At most N requests of this wave outstanding, and its LDS accesses done.
template <int N>
__device__ inline void wait_requests() {
  static_assert(N >= 0 && N < 16, "vmcnt field");
  __builtin_amdgcn_s_waitcnt(0x0070 | N);
}
__device__ inline void workgroup_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// How the input rows reach LDS: 16-byte pieces (aligned rows), 4-byte pieces
// (fp32 / fp64 rows at any alignment), or elements through registers (16-bit
// rows at any alignment).
enum InputMode { IN_VEC = 0, IN_DWORD = 1, IN_ELEMENT = 2 };

// The usual activations of fp32 plans on the accumulators.  The hardware forms
// of the generated kernels (pointwise.h) are off by up to an ulp of one near
// zero (tanh) and by |x| / 2 ulp (sigmoid and SiLU of negative x), which libm's
// (GENERIC's) are not: largest relative errors, libm / hardware forms / these,
// tanh on -2..-0.55 1.5e-7 / 3.5e-7 / 2.0e-7, sigmoid on -40..-12 1.8e-7 /
// 1.9e-6 / 2.0e-7.  64-1024-1024-64 tanh, 65,536 columns: 1302 us with the
// hardware forms, 1307 with these, 1325 with libm's; 40-700-30 sigmoid 129, 132, 170.
// e^v: 2^(v log2 e) with the rounding error of the product carried along.
__device__ inline float exp_f32(float v) {
  constexpr float kLog2eRest = 1.9259630e-8f, kLn2 = 0.69314718f;
  float const t = v * kLog2e;
  float const rest = fmaf(v, kLog2eRest, fmaf(v, kLog2e, -t));
  float const e = __builtin_amdgcn_exp2f(t);
  return __builtin_fabsf(t) < 128.0f ? fmaf(e, rest * kLn2, e) : e;
}
// x / (1 + e): the hardware's reciprocal and one correction of the quotient.
__device__ inline float over_one_plus(float x, float e) {
  float const d = 1.0f + e, r = __builtin_amdgcn_rcpf(d), q = x * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, x), r, q), d, x);
}
__device__ inline float sigmoid_f32(float x) { return over_one_plus(1.0f, exp_f32(-x)); }
__device__ inline float silu_f32(float x) { return over_one_plus(x, exp_f32(-x)); }
// ponni_Gelu.h:48-53: x sigmoid(2u), u = sqrt(2/pi) (x + 0.044715 x^3)
__device__ inline float gelu_tanh_f32(float x) {
  constexpr float c = -2.0f * 0.79788456080286535588f;
  return over_one_plus(x, exp_f32(x * fmaf(0.044715f * c, x * x, c)));
}
// 1 - 2 e / (1 + e) of |x|, e = e^(-2|x|); near zero, where that cancels, x p(x^2)
// with p a Chebyshev fit of tanh(x) / x (4.5e-9 on |x| <= 0.55).
__device__ inline float tanh_f32(float x) {
  float const s = x * x;
  float q = fmaf(s, -0.00623885f, 0.02104217f);
  q = fmaf(s, q, -0.05384337f);
  q = fmaf(s, q, 0.13332468f);
  q = fmaf(s, q, -0.33333311f);
  float const a = __builtin_fabsf(x);
  float const e = __builtin_amdgcn_exp2f(-2.0f * kLog2e * a);
  float const r = a <= 0.55f ? fmaf(a * s, q, a) : 1.0f + over_one_plus(-2.0f * e, e);
  return __builtin_copysignf(r, x);
}
// 16-bit plans: the hardware form, and x itself where that is closer than the
// type resolves (below 2^-7 tanh(x) is x to 2e-5; the form's error there is an
// ulp of fp32's one, more than an ulp of a small fp16 result).  fp16
// 24-1100-200, 40,000 columns: 84 us without, 87 with.
__device__ inline float tanh_half(float x) { return __builtin_fabsf(x) < 0.0078125f ? x : act_tanh_fast(x); }

// The epilogue steps that run on the accumulators: each(f) for one of them,
// false for any other.  fp64 keeps libm's, whose code for every accumulator at
// once is too long.
template <class C, bool Precise, class Each>
__device__ inline bool usual_step(Step const& st, Each&& each) {
  C const a = C(st.a);
  switch (st.act) {
    case ACT_RELU: each([](C v) { return act_relu(v); }); return true;
    case ACT_LEAKY_RELU: each([a](C v) { return act_leaky_relu(v, a); }); return true;
    default: break;
  }
  if constexpr (sizeof(C) == 4) {
    switch (st.act) {
      case ACT_TANH: each([](C v) { return Precise ? tanh_f32(v) : tanh_half(v); }); return true;
      case ACT_SIGMOID: each([](C v) { return Precise ? sigmoid_f32(v) : act_sigmoid_fast(v); }); return true;
      case ACT_SILU: each([](C v) { return Precise ? silu_f32(v) : act_silu_fast(v); }); return true;
      case ACT_GELU_TANH: each([](C v) { return Precise ? gelu_tanh_f32(v) : act_gelu_tanh_fast(v); }); return true;
      default: break;
    }
  }
  return false;
}
constexpr int kSlots = 3;      // steps in LDS: computed, landed, in flight

template <class S, int MI, int NJ, int MODE>
__global__ __launch_bounds__(256, 2) void layered_dense(DenseArgs a) {
  using T = Traits<S>;
  using C = typename T::C;
  using Acc = typename T::Acc;
  constexpr int KS = T::KS, ES = sizeof(S);
  constexpr int BO = 32 * MI, BB = 32 * NJ;
  constexpr int FRAG = 64 * sizeof(typename T::A);          // bytes of one fragment
  constexpr int A_BYTES = BO / 16 * FRAG, B_BYTES = KS * BB * ES, SLOT = A_BYTES + B_BYTES;
  constexpr int A_REQ = A_BYTES / 4096;                     // requests per wave and step
  constexpr int PIECE = MODE == IN_VEC ? 16 : 4;            // bytes a lane requests of a row
  constexpr int B_REQ = MODE == IN_ELEMENT ? 0 : B_BYTES / (256 * PIECE);
  constexpr int REQ = A_REQ + B_REQ;
  static_assert(A_BYTES % 4096 == 0 && (MODE == IN_ELEMENT || B_BYTES % (256 * PIECE) == 0), "whole requests");
  // Finished tiles, CH row tiles of each wave at a time, rows padded by 16
  // bytes or more.  (fp32: two at a time keep the LDS at 48 KB, three workgroups per CU.)
  constexpr int CH = ES == 4 ? 2 : MI < 4 ? MI : 4;
  constexpr int LD = 16 * NJ + 4;
  constexpr int EPI = 4 * 16 * CH * LD * int(sizeof(C));
  constexpr int BYTES = kSlots * SLOT > EPI ? kSlots * SLOT : EPI;
  __shared__ __attribute__((aligned(16))) char lds[BYTES];

  int const tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  int const wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int const wo = wave >> 1, wb = wave & 1;
  // Consecutive workgroups go to the eight XCDs in turn; each XCD takes a
  // contiguous share of the tiles, output blocks of one column block first,
  // so that a column block's rows are read into one L2 only.
  int const out_blocks = (a.n_out + BO - 1) / BO;
  int64_t tile;
  {
    int64_t const n = gridDim.x, q = n / 8, r = n % 8, xcd = blockIdx.x % 8;
    tile = xcd * q + (xcd < r ? xcd : r) + blockIdx.x / 8;
  }
  int64_t const col0 = tile / out_blocks * BB;
  int const out0 = int(tile % out_blocks) * BO;
  C const* __restrict__ P = static_cast<C const*>(a.params);
  S const* __restrict__ X = static_cast<S const*>(a.x);
  Step const* __restrict__ steps_ = a.steps + a.epi_begin;
  unsigned const lds0 = static_cast<unsigned>(reinterpret_cast<uint64_t>((lds_void)lds));

  int const steps = (a.n_in + KS - 1) / KS;
  int const out_tiles = (a.n_out + 15) / 16;
  // This lane's part of each request, advanced a step at a time.
  char const* pa[A_REQ];
#pragma unroll
  for (int r = 0; r < A_REQ; r++) {
    int const piece = wave + 4 * r;  // 1 KB pieces of the fragments
    int mo = out0 / 16 + piece * 1024 / FRAG;
    mo = mo < out_tiles ? mo : out_tiles - 1;  // (a tile past the last one is computed and dropped)
    pa[r] = reinterpret_cast<char const*>(P + a.woff) + int64_t(mo) * steps * FRAG + piece * 1024 % FRAG + 16 * lane;
  }
  constexpr int BR = B_REQ > 0 ? B_REQ : 1;
  char const* pb[BR];
  int rb[BR];
#pragma unroll
  for (int r = 0; r < B_REQ; r++) {
    int const p = (wave + 4 * r) * 64 + lane;  // piece of the step's rows
    rb[r] = p / (BB * ES / PIECE);
    int64_t const at = int64_t(p % (BB * ES / PIECE)) * PIECE;  // byte in the row's tile
    // columns past the batch repeat its last ones (PIECE bytes that hold a
    // column of the batch lie in its row)
    int64_t const last = (a.batch - 1) * ES / PIECE * PIECE + (PIECE < ES ? at % ES : 0);
    int64_t byte = col0 * ES + at;
    byte = byte < last || (PIECE < ES && byte < a.batch * ES) ? byte : last;
    pb[r] = reinterpret_cast<char const*>(X) + int64_t(rb[r]) * a.ldx * ES + byte;
  }
  auto request = [&](int s) {
    unsigned const slot = s % kSlots * SLOT;
#pragma unroll
    for (int r = 0; r < A_REQ; r++) {
      dma16(pa[r], lds0 + slot + (wave + 4 * r) * 1024);
      pa[r] += FRAG;
    }
    if constexpr (MODE == IN_ELEMENT) {
      S v[KS * BB / 256];
#pragma unroll
      for (int i = 0; i < KS * BB / 256; i++) {
        int const idx = 256 * i + tid, k = s * KS + idx / BB;
        int64_t const col = col0 + idx % BB;
        v[i] = k < a.n_in && col < a.batch ? X[int64_t(k) * a.ldx + col] : S(0.0f);
      }
#pragma unroll
      for (int i = 0; i < KS * BB / 256; i++) reinterpret_cast<S*>(lds + slot + A_BYTES)[256 * i + tid] = v[i];
    } else {
#pragma unroll
      for (int r = 0; r < B_REQ; r++) {
        unsigned const at = slot + A_BYTES + (wave + 4 * r) * 64 * PIECE;
        // rows past the input are zero (their weights are, but not their product with an infinity)
        if (s * KS + rb[r] < a.n_in) {
          if (PIECE == 16) dma16(pb[r], lds0 + at);
          else dma4(pb[r], lds0 + at);
        } else if (PIECE == 16) {
          *reinterpret_cast<f32x4*>(lds + at + 16 * lane) = f32x4{0, 0, 0, 0};
        } else {
          *reinterpret_cast<float*>(lds + at + 4 * lane) = 0.0f;
        }
        pb[r] += int64_t(KS) * a.ldx * ES;
      }
    }
  };
  request(0);
  if (steps > 1) request(1);
  // The lane's 4 entries of a per-feature vector (padded to 16) for row tile i.
  auto rows = [&](int off, int i) {
    int mo = out0 / 16 + MI * wo + i;
    mo = mo < out_tiles ? mo : out_tiles - 1;
    return *reinterpret_cast<Acc const*>(P + off + 16 * mo + 4 * g);
  };
  Acc acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; i++) {
    Acc const seed = a.bias_first ? rows(steps_[0].off, i) : Acc{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[i][j] = seed;
  }
  for (int s = 0; s < steps; s++) {
    // This wave's requests for step s have landed once only those for step
    // s + 1 are outstanding; the barrier makes that true of every wave, and
    // ends every wave's reads of the slot that step s + 2 takes.  (A last step
    // with rows past the input may have made fewer requests: waited for whole.)
    if (MODE != IN_ELEMENT && s + 1 < steps && (s + 2 < steps || a.n_in % KS == 0)) wait_requests<REQ>();
    else wait_requests<0>();
    workgroup_barrier();
    if (s + 2 < steps) request(s + 2);
    char const* __restrict__ As = lds + s % kSlots * SLOT + MI * wo * FRAG;
    S const* __restrict__ Bs = reinterpret_cast<S const*>(lds + s % kSlots * SLOT + A_BYTES) + 16 * NJ * wb;
    typename T::A av[MI];
#pragma unroll
    for (int i = 0; i < MI; i++) av[i] = reinterpret_cast<typename T::A const*>(As + i * FRAG)[lane];
    if constexpr (ES == 2) {
      typename T::A bv[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        typename T::B4 h[2];
#pragma unroll
        for (int m = 0; m < 2; m++)
          h[m] = __builtin_bit_cast(typename T::B4,
                                    __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4)(
                                        Bs + (16 * m + 4 * g + (c >> 2)) * BB + 16 * j + 4 * (c & 3))));
        bv[j] = __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < MI; i++) acc[i][j] = T::mfma(av[i], bv[j], acc[i][j]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        C bv[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) bv[j] = Bs[(4 * g + e) * BB + 16 * j + c];
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
          for (int j = 0; j < NJ; j++) acc[i][j] = mfma4(av[i][e], bv[j], acc[i][j]);
      }
    }
  }
  wait_requests<0>();
  workgroup_barrier();
  // Epilogue (ponni_Inference.h:431-444): the steps in order, the usual ones on
  // the accumulators, the rest (from step k on) on 4 columns of one row at a time.
  int k0 = a.bias_first;
  for (; k0 < a.epi_count; k0++) {
    Step const st = steps_[k0];
    if (st.act == ACT_BIAS) {
#pragma unroll
      for (int i = 0; i < MI; i++) {
        Acc const b = rows(st.off, i);
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] += b;
      }
      continue;
    }
    bool const done = usual_step<C, ES == 4>(st, [&](auto f) {
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][j][e] = f(acc[i][j][e]);
    });
    if (!done) break;
  }
  S* __restrict__ Y = static_cast<S*>(a.y);
  typedef S S4 __attribute__((ext_vector_type(4)));
  typedef C C4 __attribute__((ext_vector_type(4)));
  bool const yvec = (reinterpret_cast<uint64_t>(Y) | uint64_t(a.ldy) * ES) % (4 * ES) == 0;
  C* __restrict__ out = reinterpret_cast<C*>(lds) + wave * 16 * CH * LD;
  constexpr int LPR = 4 * NJ;  // lanes per row
#pragma unroll
  for (int i0 = 0; i0 < MI; i0 += CH) {
#pragma unroll
    for (int i = 0; i < CH; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) out[(16 * i + 4 * g + e) * LD + 16 * j + c] = acc[i0 + i][j][e];
    int64_t const col = col0 + 16 * NJ * wb + 4 * (lane % LPR);
    // this lane's 4 columns of its rows, in order
    auto each_row = [&](auto f) {
#pragma unroll 1
      for (int r = lane / LPR; r < 16 * CH; r += 64 / LPR) f(r, *reinterpret_cast<C4*>(out + r * LD + 4 * (lane % LPR)));
    };
#pragma unroll 1
    for (int k = k0; k < a.epi_count; k++) {
      Step const st = steps_[k];
      if (st.act >= ACT_RELU && st.act <= ACT_MISH) {
        map_activation<C>(st.act, C(st.a), C(st.b), [&](auto f) {
          each_row([&](int, C4& v) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
              C t = v[e];
              f(t);
              v[e] = t;
            }
          });
        });
        continue;
      }
      each_row([&](int r, C4& v) {
        int const f = out0 + 16 * (MI * wo + i0) + r;
        C const bias = act_has_param(st.act) && f < a.n_out ? P[st.off + f] : C(0);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = apply_step<C>(st.act, v[e], bias, C(st.a), C(st.b));
      });
    }
    each_row([&](int r, C4& v) {
      int const f = out0 + 16 * (MI * wo + i0) + r;
      if (f >= a.n_out || col >= a.batch) return;
      S* __restrict__ y = Y + int64_t(f) * a.ldy + col;
      S4 const o = __builtin_convertvector(v, S4);
      if (yvec && col + 4 <= a.batch) {
        *reinterpret_cast<S4*>(y) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (col + e < a.batch) y[e] = o[e];
      }
    });
  }
}

template <class S, int MI, int NJ>
hipError_t launch(DenseArgs const& a, hipStream_t stream) {
  constexpr int BO = 32 * MI, BB = 32 * NJ, ES = sizeof(S);
  int64_t const blocks = (a.batch + BB - 1) / BB * ((a.n_out + BO - 1) / BO);
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  dim3 const grid(static_cast<unsigned>(blocks)), block(256);
  bool const vec = (reinterpret_cast<uint64_t>(a.x) | uint64_t(a.ldx) * ES) % 16 == 0;
  constexpr int other = ES == 2 ? IN_ELEMENT : IN_DWORD;
  if (vec) hipLaunchKernelGGL((layered_dense<S, MI, NJ, IN_VEC>), grid, block, 0, stream, a);
  else hipLaunchKernelGGL((layered_dense<S, MI, NJ, other>), grid, block, 0, stream, a);
  return hipGetLastError();
}

// Do the op's input and output rows share memory?
bool overlap(DenseArgs const& a, size_t es) {
  auto const x = reinterpret_cast<uint64_t>(a.x), y = reinterpret_cast<uint64_t>(a.y);
  uint64_t const x_end = x + (uint64_t(a.n_in - 1) * a.ldx + a.batch) * es;
  uint64_t const y_end = y + (uint64_t(a.n_out - 1) * a.ldy + a.batch) * es;
  return x < y_end && y < x_end;
}

// The large tile where it fills the 256 CUs, two workgroups each; otherwise
// the small one, four times as many workgroups.  An op whose output takes its
// input's place (a chain of one, called in place) has all its outputs in one
// workgroup's tile if either tile holds them: it reads its columns before it stores.
template <class S, int MI, int NJ, int MS, int NS>
hipError_t launch_sized(DenseArgs const& a, hipStream_t stream) {
  int64_t const large = (a.batch + 32 * NJ - 1) / (32 * NJ) * ((a.n_out + 32 * MI - 1) / (32 * MI));
  bool const fits = a.n_out <= 32 * MS;  // (the large tile would be half empty)
  bool const whole = !fits && a.n_out <= 32 * MI && overlap(a, sizeof(S));
  return (large >= 512 && !fits) || whole ? launch<S, MI, NJ>(a, stream) : launch<S, MS, NS>(a, stream);
}

}  // namespace

hipError_t launch_layered_dense(int dtype, DenseArgs const& a, hipStream_t stream) {
  if (a.batch <= 0) return hipSuccess;
  switch (dtype) {
    case PONNI_F64: return launch_sized<double, 4, 2, 2, 2>(a, stream);
    case PONNI_F16: return launch_sized<_Float16, 8, 4, 4, 2>(a, stream);
    case PONNI_BF16: return launch_sized<__bf16, 8, 4, 4, 2>(a, stream);
    default: return launch_sized<float, 4, 4, 2, 2>(a, stream);
  }
}

}  // namespace ponni_hip
