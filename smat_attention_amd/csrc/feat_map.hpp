// The feature map of src/smat/attention.py:82-106 as a device-side stage, shared
// by the stand-alone featurise kernel and the consumers that compute their
// features in place (scan, Gram sums, query):
//
//   Phi = map(Q W^T),  Psi = map(K W^T) * h,  Vb = [V, 1]
//   map = elu(.) + 1   (kind 0)   or   relu(.) + 1e-3   (kind 1)
//
// in the input dtype with torch's rounding steps: the product rounded to the
// dtype, elu rounded, + 1 rounded, the gate product rounded (fp32 math in
// between, as torch does for 16-bit tensors).
#pragma once

#include <type_traits>

#include "smat_common.hpp"

namespace smat {

// map() of four values of the product, each step rounded to In.  bf16's elu is
// exp2 minus one: its error (1e-7, absolute) only matters where |expm1| is so
// small that the roundings after it, to steps of 2^-8 of 1 + expm1, discard it,
// and map() equals the one on the correctly rounded expm1 for every
// non-positive bf16 input -- an exhaustive check.  It is formed for every lane
// and selected, so no branch keeps the map from interleaving with the MFMAs
// around it (for v > 0 exp2 may be inf), and the conversions go two values to
// an instruction: half the vector work of a form that holds expm1's relative
// error (a polynomial near zero), and the map's vector work weighs on the kernels
// that form their features (the forward from q, k, v at 8 sequences of 131072
// tokens: 1780 -> 1734 us; the feature map alone at 96 of 4096, widths 64:
// 79 -> 71).  fp16, whose 11-bit significand could round that error differently,
// and fp32, where nothing rounds afterwards, take libm's expm1f.
template <typename In, int KIND>
__device__ __forceinline__ typename Traits<In>::half_frag feature_map4(const f32x4& acc) {
  typedef typename Traits<In>::half_frag Half;
  if constexpr (std::is_same<In, bf16>::value) {
    auto rounded = [](const f32x4& x) {
      return __builtin_convertvector(__builtin_convertvector(x, Half), f32x4);
    };
    const f32x4 v = rounded(acc);                              // torch's matmul output
    f32x4 y;
    if constexpr (KIND == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float m = __builtin_amdgcn_exp2f(v[i] * 1.4426950408889634f) - 1.f;
        y[i] = v[i] > 0.f ? v[i] : m;
      }
      y = rounded(y) + 1.0f;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = fmaxf(v[i], 0.f) + 1e-3f;
    }
    return __builtin_convertvector(y, Half);
  } else {
    Half out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v = to_f32(from_f32<In>(acc[i]));
      float y;
      if constexpr (KIND == 0) y = to_f32(from_f32<In>(v > 0.f ? v : expm1f(v))) + 1.0f;
      else y = fmaxf(v, 0.f) + 1e-3f;
      out[i] = from_f32<In>(y);
    }
    return out;
  }
}

// Four mapped values times their row's gate, rounded.
template <typename In>
__device__ __forceinline__ typename Traits<In>::half_frag feature_gate4(
    const typename Traits<In>::half_frag& y, float gate) {
  typename Traits<In>::half_frag out;
#pragma unroll
  for (int i = 0; i < 4; ++i) out[i] = from_f32<In>(to_f32(y[i]) * gate);
  return out;
}

// The feature map handed to a consumer kernel: W (128 x 128, features x d_qk,
// row-major, 16-byte aligned rows), the optional key gate h (nb, T) and kind.
struct FeatArgs {
  const void* W;
  const void* h;
  int64_t h_sb;
  int kind;
  // Where a Gram prepass that forms Psi also stores it, rows of 128 at row
  // stride 128 and sequence stride psi_sb (none when null).
  void* psi_out = nullptr;
  int64_t psi_sb = 0;
};

// Features [16 wf, 16 wf + 16) of W as MFMA A fragments over d_qk = 128: k-block
// kb holds k-slots 32 kb + 8 (lane / 16) + j, j < 8.  A per-wave constant.
template <typename In>
__device__ __forceinline__ void feat_w_load(typename Traits<In>::frag (&wa)[4], const In* W, int wf,
                                            int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const In* row = W + (int64_t)(16 * wf + r16) * 128;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
    wa[kb] = *reinterpret_cast<const typename Traits<In>::frag*>(row + 32 * kb + 8 * g);
}

// Over NRT 16-row tiles starting at row tile rt0 of LDS tiles of 256-byte
// rows whose 16-byte chunk k of row t sits at slot k ^ swz(t): read the rows'
// 128 input values (X = Q or K) from src, form this wave's features
// C = W[16 wf .. +16] X^T on MFMA (lane (t, g) ends with features 16 wf + 4 g
// .. +3 of row t), then write map(C) (times gate[rt] for the lane's row of tile
// rt0 + rt when use_gate) into the row's feature chunk of dst.  In place
// (dst == src) every wave's reads must precede any write: the call then has a
// barrier between the two, which every wave of the workgroup must meet
// (inactive waves only meet it).  The caller places a barrier before the
// feature rows are read.  The MFMA sequence is the stand-alone kernel's
// (k-blocks 0..3 in order), so the features are bitwise the same.
template <typename In, int NRT, typename Swz>
__device__ __forceinline__ void feat_rows(const uint4* src, uint4* dst, int rt0, bool active,
                                          const typename Traits<In>::frag (&wa)[4], int wf,
                                          int kind, bool use_gate, const float (&gate)[NRT],
                                          int lane, Swz swz) {
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Half;
  const int r16 = lane & 15, g = lane >> 4;
  f32x4 acc[NRT];
  if (active) {
    Frag bx[NRT][4];
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int t = 16 * (rt0 + rt) + r16;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        bx[rt][kb] = *reinterpret_cast<const Frag*>(src + t * 16 + ((4 * kb + g) ^ swz(t)));
    }
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      acc[rt] = zero4();
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc[rt] = mma(acc[rt], wa[kb], bx[rt][kb]);
    }
  }
  if (dst == src) lds_barrier();                     // every wave has read its rows
  // one branch on the (uniform) kind around all of the rows' values
  auto put = [&](auto KC) {
    constexpr int KIND = decltype(KC)::value;
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int t = 16 * (rt0 + rt) + r16;
      Half hv = feature_map4<In, KIND>(acc[rt]);
      if (use_gate) hv = feature_gate4<In>(hv, gate[rt]);
      char* p = reinterpret_cast<char*>(dst + t * 16 + ((2 * wf + (g >> 1)) ^ swz(t)));
      *reinterpret_cast<Half*>(p + 8 * (g & 1)) = hv;
    }
  };
  if (active) {
    if (kind == 0)
      put(std::integral_constant<int, 0>{});
    else
      put(std::integral_constant<int, 1>{});
  }
}

// Columns 128..135 of [V, 1] for 64 rows (one 16-byte chunk a row): the ones
// column, then zeros.
template <typename In>
__device__ __forceinline__ void feat_ones_tile(uint4* chunks, int tid, int nthreads) {
  typedef typename Traits<In>::frag Frag;
  for (int t = tid; t < 64; t += nthreads) {
    Frag f;
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = from_f32<In>(j == 0 ? 1.f : 0.f);
    *reinterpret_cast<Frag*>(chunks + t) = f;
  }
}

}  // namespace smat
