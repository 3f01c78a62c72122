// FUSED path, small batches: the columns of one tile shared by a whole
// workgroup.
//
// The throughput kernels (fused_f32.h dense_ep, fused_f16.h dense_hs) give
// every wave its own columns, so a batch that does not fill the chip that
// way still pays one wave's full pass over every layer.  Here all W waves of
// a workgroup own the same 16 NT columns: each wave holds the whole state in
// registers (the same tiles, in the same layout), a dense layer's output
// tiles are dealt to the waves round robin (wave w computes tiles w, w + W,
// ...), and the finished tiles pass through LDS, lane to same lane, so that
// every wave holds the next state.  Operations that are not contractions run
// in every wave alike.  Weights go straight from L2 to the registers of the
// one wave that uses them; the first kRing fragments of the next contraction
// are requested before the exchange that ends the last one.
#pragma once

namespace ponni_hip {
namespace fused {

// A-fragment ring of a wave's contraction: 16 KB in flight per wave.
constexpr int kRing = 16;

// Every wave's LDS writes made, then all waves here: the exchange buffers
// are the only LDS memory written after the prologue.
__device__ inline void exchange_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// How a wave's OWN output tiles of a contraction are computed: GT at a time,
// one accumulation chain each (and per column tile).
constexpr int split_group(int own) { return own <= 4 ? own : own % 4 == 0 ? 4 : own % 3 == 0 ? 3 : own % 2 == 0 ? 2 : 1; }

// The wave's A fragments of a contraction over TI input blocks, in the order
// it consumes them: own tiles in groups of GT, input blocks within a group,
// tiles within a block.  Own tile o is the layer's tile wave + W o (a wave
// without a last tile repeats the layer's last one, unused).
template <class F, int TI, int TO, int W>
struct Frags {
  static constexpr int OWN = (TO + W - 1) / W;
  static constexpr int GT = split_group(OWN);
  static constexpr int NF = OWN * TI;
  static constexpr int R = kRing < NF ? kRing : NF;
  F const* w;  // the layer's fragments, this lane's element of each
  int wave;
  F ring[R];
  __device__ F load(int i) const {
    int const own = i / (GT * TI) * GT + i % GT, m = i / GT % TI;
    int mo = wave + W * own;
    if (TO % W != 0 && own == OWN - 1) mo = mo < TO ? mo : TO - 1;
    return w[(mo * TI + m) * 64];
  }
  __device__ void begin(F const* frags, int wave_, int lane) {
    w = frags + lane;
    wave = wave_;
#pragma unroll
    for (int i = 0; i < R; i++) ring[i] = load(i);
  }
  __device__ F take(int i) {
    F const f = ring[i % R];
    if (i + R < NF) ring[i % R] = load(i + R);
    return f;
  }
  // does the wave hold own tile o
  __device__ bool has(int o) const { return TO % W == 0 || o < OWN - 1 || wave + W * o < TO; }
};

template <int TI, int TO, int W>
using FragsR = Frags<realx4, TI, TO, W>;

// The wave's output tiles of W^T in (fp32 / fp64), each finished by
// epi(mo, tile).  init(mo) is the accumulator's seed; KS as in dense_ep.
template <int TO, int W, int KS, int TI, int NT, class Init, class Epi>
__device__ inline S<(TO + W - 1) / W, NT> split_dense(S<TI, NT> const& in, FragsR<TI, TO, W>& f, Init init, Epi epi) {
  using FR = FragsR<TI, TO, W>;
  constexpr int GT = FR::GT;
  S<FR::OWN, NT> own;
#pragma unroll
  for (int o0 = 0; o0 < FR::OWN; o0 += GT) {
    if (GT == 1 && !f.has(o0)) continue;
#pragma unroll
    for (int q = 0; q < GT; q++) {
      realx4 const seed = init(f.has(o0 + q) ? f.wave + W * (o0 + q) : 0);
#pragma unroll
      for (int n = 0; n < NT; n++) own.v[o0 + q][n] = seed;
    }
#pragma unroll
    for (int m = 0; m < TI; m++) {
      realx4 a[GT];
#pragma unroll
      for (int q = 0; q < GT; q++) a[q] = f.take((o0 / GT * TI + m) * GT + q);
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (4 * m + e < KS)
#pragma unroll
          for (int q = 0; q < GT; q++)
#pragma unroll
            for (int n = 0; n < NT; n++) own.v[o0 + q][n] = mfma4(a[q][e], in.v[m][n][e], own.v[o0 + q][n]);
    }
#pragma unroll
    for (int q = 0; q < GT; q++)
      if (f.has(o0 + q)) epi(f.wave + W * (o0 + q), own.v[o0 + q]);
  }
  return own;
}

// Own tiles into the exchange buffer, and the whole state out of it.
template <int TO, int W, int OWN, int NT>
__device__ inline void split_put(realx4* __restrict__ buf, S<OWN, NT> const& own, int wave, Lane const& L) {
#pragma unroll
  for (int o = 0; o < OWN; o++) {
    int const mo = wave + W * o;
    if (TO % W != 0 && o == OWN - 1 && mo >= TO) continue;
#pragma unroll
    for (int n = 0; n < NT; n++) buf[(mo * NT + n) * 64 + L.lane] = own.v[o][n];
  }
}
template <int TO, int NT = kNT>
__device__ inline S<TO, NT> split_get(realx4 const* __restrict__ buf, Lane const& L) {
  S<TO, NT> s;
#pragma unroll
  for (int m = 0; m < TO; m++)
#pragma unroll
    for (int n = 0; n < NT; n++) s.v[m][n] = buf[(m * NT + n) * 64 + L.lane];
  return s;
}

// Own tiles of the model's output straight to y.
template <int N, int TO, int W, int OWN, int NT>
__device__ inline void split_store(S<OWN, NT> const& own, real* __restrict__ y, int64_t ld, int wave, Lane const& L) {
  real* __restrict__ yl = y + lane_offset(L, ld) + L.col0;
#pragma unroll
  for (int o = 0; o < OWN; o++) {
    int const mo = wave + W * o;
#pragma unroll
    for (int n = 0; n < NT; n++) {
      bool const col_ok = L.col0 + 16 * n + L.c < L.batch;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        int const f = 16 * mo + 4 * L.g + e;
        if (f < N && col_ok) yl[int64_t(16 * mo + e) * ld + 16 * n] = own.v[o][n][e];
      }
    }
  }
}

// t += tile mo of s, mo uniform across the wave but not a constant.
template <int T, int NT>
__device__ inline void tile_add_state_at(realx4 (&t)[NT], S<T, NT> const& s, int mo) {
#pragma unroll
  for (int m = 0; m < T; m++)
    if (m == mo)
#pragma unroll
      for (int n = 0; n < NT; n++) t[n] += s.v[m][n];
}

#ifdef PONNI_SPLIT_HALF
// ---- fp16 / bf16 states ---------------------------------------------------
template <class E, int TI, int TO, int W>
using FragsH = Frags<typename Vec<E>::x8, (TI + 1) / 2, TO, W>;

// As dense_hs: fp32 accumulators seeded by init(mo) and finished by
// epi(mo, t, o), which rounds the tile to the 16-bit state o; TR swaps the
// MFMA operands (a transposed output tile, store_rows_ht).
template <int TO, int W, bool TR, int TI, int NT, class E, class Init, class Epi>
__device__ inline H<(TO + W - 1) / W, NT, E> split_dense_h(H<TI, NT, E> const& in, FragsH<E, TI, TO, W>& f, Init init,
                                                           Epi epi) {
  using FR = FragsH<E, TI, TO, W>;
  using V4 = typename Vec<E>::x4;
  constexpr int TS = (TI + 1) / 2, GT = FR::GT;
  H<FR::OWN, NT, E> own;
#pragma unroll
  for (int o0 = 0; o0 < FR::OWN; o0 += GT) {
    if (GT == 1 && !f.has(o0)) continue;
    floatx4 acc[GT][NT];
#pragma unroll
    for (int q = 0; q < GT; q++) {
      floatx4 const seed = init(f.has(o0 + q) ? f.wave + W * (o0 + q) : 0);
#pragma unroll
      for (int n = 0; n < NT; n++) acc[q][n] = seed;
    }
#pragma unroll
    for (int t = 0; t < TS; t++) {
      typename Vec<E>::x8 a[GT];
#pragma unroll
      for (int q = 0; q < GT; q++) a[q] = f.take((o0 / GT * TS + t) * GT + q);
#pragma unroll
      for (int n = 0; n < NT; n++) {
        V4 const lo = in.v[2 * t][n];
        V4 const hi = (2 * t + 1 < TI) ? in.v[(2 * t + 1 < TI) ? 2 * t + 1 : 2 * t][n]
                                       : V4{E(0.0f), E(0.0f), E(0.0f), E(0.0f)};
        auto const b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int q = 0; q < GT; q++) acc[q][n] = TR ? Vec<E>::mfma(b, a[q], acc[q][n]) : Vec<E>::mfma(a[q], b, acc[q][n]);
      }
    }
#pragma unroll
    for (int q = 0; q < GT; q++)
      if (f.has(o0 + q)) epi(f.wave + W * (o0 + q), acc[q], own.v[o0 + q]);
  }
  return own;
}

// 16-bit tiles 2t and 2t + 1 of a lane sit side by side (16 bytes).
template <int TO, int W, int OWN, int NT, class E>
__device__ inline void split_put(typename Vec<E>::x4* __restrict__ buf, H<OWN, NT, E> const& own, int wave,
                                 Lane const& L) {
#pragma unroll
  for (int o = 0; o < OWN; o++) {
    int const mo = wave + W * o;
    if (TO % W != 0 && o == OWN - 1 && mo >= TO) continue;
#pragma unroll
    for (int n = 0; n < NT; n++) buf[(((mo >> 1) * NT + n) * 64 + L.lane) * 2 + (mo & 1)] = own.v[o][n];
  }
}
template <int TO, class E, int NT = kNT>
__device__ inline H<TO, NT, E> split_get_h(typename Vec<E>::x4 const* __restrict__ buf, Lane const& L) {
  using V8 = typename Vec<E>::x8;
  H<TO, NT, E> s;
#pragma unroll
  for (int t = 0; t < (TO + 1) / 2; t++)
#pragma unroll
    for (int n = 0; n < NT; n++) {
      V8 const v = *reinterpret_cast<V8 const*>(buf + ((t * NT + n) * 64 + L.lane) * 2);
      s.v[2 * t][n] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
      if (2 * t + 1 < TO) s.v[2 * t + 1 < TO ? 2 * t + 1 : 2 * t][n] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
    }
  return s;
}

// Own tiles of the output: row-major tiles, or transposed ones (TR).
template <int N, int TO, int W, bool TR, int OWN, int NT, class E, class Y>
__device__ inline void split_store_h(H<OWN, NT, E> const& own, Y* __restrict__ y, int64_t ld, int wave,
                                     Lane const& L) {
  using Y4 = typename Vec4Of<Y>::type;
#pragma unroll
  for (int o = 0; o < OWN; o++) {
    int const mo = wave + W * o;
    if (mo >= TO) continue;
    if (TR) {
      int const f = 16 * mo + L.c;
      if (N % 16 != 0 && f >= N) continue;
      Y* __restrict__ yr = y + int64_t(f) * ld + L.col0 + 4 * L.g;
      bool const full = L.col0 + 16 * NT <= L.batch;
#pragma unroll
      for (int n = 0; n < NT; n++) {
        Y4 const v = __builtin_convertvector(own.v[o][n], Y4);
        if (full) {
          *reinterpret_cast<Y4*>(yr + 16 * n) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (L.col0 + 16 * n + 4 * L.g + e < L.batch) yr[16 * n + e] = v[e];
        }
      }
    } else {
      Y* __restrict__ yl = y + (int64_t(16 * mo + 4 * L.g) * ld + L.col0 + L.c);
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (16 * mo + 4 * L.g + e < N && L.col0 + 16 * n + L.c < L.batch) yl[int64_t(e) * ld + 16 * n] = static_cast<Y>(own.v[o][n][e]);
    }
  }
}

// Projection add in the own tile: the state's tile (widened) plus the fp32
// projection, rounded once (fused_f16.h proj_add_h).
template <int T, int NT, class E>
__device__ inline void tile_add_state_at_h(floatx4 (&t)[NT], H<T, NT, E> const& s, int mo) {
#pragma unroll
  for (int m = 0; m < T; m++)
    if (m == mo)
#pragma unroll
      for (int n = 0; n < NT; n++) t[n] = widen4<E>(s.v[m][n]) + t[n];
}
#endif

}  // namespace fused
}  // namespace ponni_hip
