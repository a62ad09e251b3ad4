// Fragment helpers of the backward kernels at r = 64 features and p = 65
// value columns (head_dim 64 plus the ones column) on gfx950 MFMA
// (v_mfma_f32_16x16x32 for 16-bit inputs, 16x16x4 for fp32); value column 64
// is kept out of the matrix products, as rank-1 fp32 terms.
//
// LDS layouts: 16-bit tiles of 64 columns as rows of 128 bytes, 16-byte
// chunk k of row t at k ^ (t & 6) -- conflict-free for row-wise 16-byte reads
// (four phases of 16 lanes) and for the transposing ds_read_b64_tr_b16 (two
// phases of 32 lanes); fp32 tiles as rows of kS = 68 floats.
#pragma once

#include "smat_host.hpp"

namespace smat {

namespace cb {

// The (item, sequence) of this workgroup of a (nitems, nseq) grid, with all the
// items of a sequence on one XCD: workgroups are dispatched to the 8 XCDs
// round-robin by linear id, so XCD x takes sequences x, x + 8, ... in turn
// and the rows its items share (a token in several cells' or points' lists)
// are re-read from that XCD's L2 instead of from HBM.  Sequences past the
// last multiple of 8 keep the plain mapping.
__device__ __forceinline__ void xcd_item_seq(int& item, int64_t& seq) {
  const int64_t nitems = gridDim.x, nseq = gridDim.y;
  const int64_t lin = (int64_t)blockIdx.y * nitems + blockIdx.x;
  const int64_t full = (nseq / 8) * 8 * nitems;
  if (lin < full) {
    const int64_t k = lin >> 3;
    seq = (lin & 7) + 8 * (k / nitems);
    item = (int)(k % nitems);
  } else {
    seq = lin / nitems;
    item = (int)(lin % nitems);
  }
}

constexpr int kC = 128;          // tokens per chunk
constexpr int kR = 64;           // features
constexpr int kP = 65;           // value columns incl. the ones column
constexpr int kThreads = 512;
constexpr int kS = 68;           // fp32 LDS row stride (floats)
constexpr int kRowChunks = 8;    // 16-byte chunks per 16-bit row of 64
}  // namespace cb

// 16-byte chunk slot of (row, chunk) in a 128-row x 128-byte tile.
__device__ __forceinline__ int cb_slot(int row, int k) { return row * cb::kRowChunks + (k ^ (row & 6)); }

template <typename In>
__device__ __forceinline__ typename Traits<In>::half_frag cb_tr(const uint4* tile, int row, int k,
                                                                int half) {
  typedef short short4v __attribute__((ext_vector_type(4)));
  const char* p = reinterpret_cast<const char*>(tile + cb_slot(row, k)) + 8 * half;
  short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4v*)(__attribute__((address_space(3))) char*)(p));
  return __builtin_bit_cast(typename Traits<In>::half_frag, v);
}

// The A operand along tokens of a transposed 16-bit tile (Phi^T or Psi^T):
// lane (m = 16 ct + lane % 16, g) gets, as k-slot 4h + e, column m of token
// row 16 tile[h] + 4g + e.  Lane 4e + q of each sixteen addresses row
// 16 tile[h] + 4g + e, columns 16 ct + 4q .. +3.
template <typename In>
__device__ __forceinline__ typename Traits<In>::frag cb_tr_pair(const uint4* tile, int t0, int t1,
                                                               int ct, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const int k = 2 * ct + ((r16 & 3) >> 1), half = r16 & 1;
  const auto a = cb_tr<In>(tile, 16 * t0 + 4 * g + (r16 >> 2), k, half);
  const auto b = cb_tr<In>(tile, 16 * t1 + 4 * g + (r16 >> 2), k, half);
  typename Traits<In>::frag f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f[e] = a[e];
    f[4 + e] = b[e];
  }
  return f;
}

// Row-wise operand of a 16-bit tile: lane (row 16 tile + lane % 16, g) gets
// columns 32 kc + 8g .. +7.
template <typename In>
__device__ __forceinline__ typename Traits<In>::frag cb_row(const uint4* tile, int tile_row, int kc,
                                                           int lane) {
  return *reinterpret_cast<const typename Traits<In>::frag*>(
      tile + cb_slot(16 * tile_row + (lane & 15), 4 * kc + (lane >> 4)));
}

// Row-wise operand of an fp32 LDS tile (rows of kS floats), split hi/lo:
// lane (row, g) gets columns 32 kc + 8g .. +7.
template <typename In>
__device__ __forceinline__ void cb_row32(const float* t, int row, int kc, int g,
                                         typename Traits<In>::frag& hi,
                                         typename Traits<In>::frag& lo) {
  const float4 a = *reinterpret_cast<const float4*>(t + row * cb::kS + 32 * kc + 8 * g);
  const float4 b = *reinterpret_cast<const float4*>(t + row * cb::kS + 32 * kc + 8 * g + 4);
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    In h, l;
    split2<In>(v[e], h, l);
    hi[e] = h;
    lo[e] = l;
  }
}

// hi/lo 16-bit B operand from two accumulator tiles (k-slot 4h + e <- tile h, entry e).
template <typename In>
__device__ __forceinline__ void cb_split_pair(const f32x4& a, const f32x4& b,
                                              typename Traits<In>::frag& hi,
                                              typename Traits<In>::frag& lo) {
  typename Traits<In>::half_frag h0, l0, h1, l1;
  split4<In>(a, h0, l0);
  split4<In>(b, h1, l1);
  hi = __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7);
  lo = __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Four floats, or eight 16-bit values, at their own alignment: rows of 65
// elements start anywhere, and a wide load or store only needs the element's
// alignment (measured: no slower than the scalar accesses it stands for).
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
template <typename In>
__device__ __forceinline__ typename Traits<In>::frag cb_load8(const In* p) {
  typedef In in8u __attribute__((ext_vector_type(8), aligned(sizeof(In))));
  return __builtin_bit_cast(typename Traits<In>::frag, *reinterpret_cast<const in8u*>(p));
}

// Stage one contiguous r x p fp32 matrix in LDS rows of kS, all threads (256)
// of the workgroup: eight threads a row, eight floats each, and column 64.
__device__ __forceinline__ void cb_stage_rp(float* s, const float* src) {
  using namespace cb;
  const int tid = threadIdx.x, row = tid >> 3, k = tid & 7;
  f32x4 v[4];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      v[2 * u + h] = *reinterpret_cast<const f32x4u*>(src + (row + 32 * u) * kP + 8 * k + 4 * h);
  const float c = src[(tid & (kR - 1)) * kP + 64];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      *reinterpret_cast<f32x4*>(s + (row + 32 * u) * kS + 8 * k + 4 * h) = v[2 * u + h];
  if (tid < kR) s[tid * kS + 64] = c;
}

// Gradient rows leave as fp32 or rounded (to nearest even) to the inputs'
// 16-bit type.  Four consecutive values: one 16-byte store of floats, or one
// 8-byte store of 16-bit values (rows 16-byte aligned, the group at a column
// that is a multiple of 4).
__device__ __forceinline__ void store_grad4(float* p, const f32x4& v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
template <typename Out>
__device__ __forceinline__ void store_grad4(Out* p, const f32x4& v) {
  typename Traits<Out>::half_frag h;
#pragma unroll
  for (int i = 0; i < 4; ++i) h[i] = from_f32<Out>(v[i]);
  *reinterpret_cast<typename Traits<Out>::half_frag*>(p) = h;
}
// The same at the element's alignment: four values of a 65-wide row.
template <typename Out>
__device__ __forceinline__ void cb_store4(Out* p, const f32x4& v) {
  typedef Out out4u __attribute__((ext_vector_type(4), aligned(sizeof(Out))));
  out4u o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = from_f32<Out>(v[i]);
  *reinterpret_cast<out4u*>(p) = o;
}
// The code of a gradient output type, as the host entry points take it.
template <typename Out> constexpr int out_code();
template <> constexpr int out_code<float>() { return SMAT_F32; }
template <> constexpr int out_code<bf16>() { return SMAT_BF16; }
template <> constexpr int out_code<f16>() { return SMAT_F16; }

// Sum over the four 16-lane groups of a wave (lanes r16, r16 + 16, +32, +48).
__device__ __forceinline__ float cb_sum_groups(float v) {
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// One step's gather: 32 entries, eight threads per entry (slot = tid / 8,
// sub = tid % 8).  A thread loads columns 8 sub .. +7 of the 64-wide 16-bit
// row and of the 65-wide row, and the latter's column 64.  Loads land in
// registers and the kernel writes them to LDS at the top of the step.
// Issuing the next step's gather before the current step's products, and
// reading the entry ids one step further ahead, keeps both of its latencies
// (entry id, then rows) off the step.  The per-entry token, pair and dot
// partials are read after the step's last barrier, so they alternate
// between two buffers by step parity while the next step's rows are written.
template <typename In> struct CbRow8 {            // eight values of the 65-wide row
  typedef typename Traits<In>::frag type;
  static __device__ __forceinline__ type load(const In* p) { return cb_load8(p); }
};
template <> struct CbRow8<float> {
  typedef f32x8 type;
  static __device__ __forceinline__ type load(const float* p) {
    const f32x4 a = *reinterpret_cast<const f32x4u*>(p);
    const f32x4 b = *reinterpret_cast<const f32x4u*>(p + 4);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

template <typename In, typename Row65>
struct CbGather {
  typedef typename Traits<In>::frag Frag;
  typedef typename CbRow8<Row65>::type Row8;
  int id;                                      // the entry of the next load()
  int tok, pair;
  bool ok;
  Frag r64;
  Row8 r65;
  Row65 c65;
  // The id of this thread's entry in the step at s0 (any entry past the end).
  __device__ __forceinline__ void peek(const int32_t* ent, int64_t s0, int64_t beg, int64_t end,
                                       int tid) {
    const int64_t i = s0 + (tid >> 3);
    id = ent[i < end ? i : beg];
  }
  // The rows of the peeked step at s0.  Entry ids are pair-major, pair * L +
  // token (L tokens a sequence), so each cell's list holds its pair-0 entries
  // first; L = 0: plain token ids.
  __device__ __forceinline__ void load(int64_t s0, int64_t end, int L, const In* rows64,
                                       int64_t st64, const Row65* rows65, int64_t st65, int tid) {
    const int sub = tid & 7;
    ok = s0 + (tid >> 3) < end;
    pair = L ? (int)((unsigned)id / (unsigned)L) : 0;
    tok = id - pair * L;
    r64 = cb_load8(rows64 + (int64_t)tok * st64 + 8 * sub);
    const Row65* r = rows65 + (int64_t)tok * st65;
    r65 = CbRow8<Row65>::load(r + 8 * sub);
    c65 = r[64];
  }
  // Entries past the end become zero rows.
  __device__ __forceinline__ void mask() {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      r64[e] = ok ? r64[e] : from_f32<In>(0.f);
      r65[e] = ok ? r65[e] : from_f32<Row65>(0.f);
    }
    c65 = ok ? c65 : from_f32<Row65>(0.f);
  }
};

// Eight fp32 values as one 16-byte piece each of hi and lo 16-bit values.
template <typename In>
__device__ __forceinline__ void cb_split8(const f32x4& x, const f32x4& y, uint4& hi, uint4& lo) {
  typename Traits<In>::half_frag h0, l0, h1, l1;
  split4<In>(x, h0, l0);
  split4<In>(y, h1, l1);
  hi = __builtin_bit_cast(uint4, __builtin_shufflevector(h0, h1, 0, 1, 2, 3, 4, 5, 6, 7));
  lo = __builtin_bit_cast(uint4, __builtin_shufflevector(l0, l1, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Operand down the 32 rows of a 16-bit tile: lane (m = 16 ct + lane % 16, g),
// k-slot e <- column m of row 8g + e.
template <typename In>
__device__ __forceinline__ typename Traits<In>::frag cb_col32(const uint4* tile, int ct,
                                                             int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  const int k = 2 * ct + ((r16 & 3) >> 1), half = r16 & 1;
  const auto a = cb_tr<In>(tile, 8 * g + (r16 >> 2), k, half);
  const auto b = cb_tr<In>(tile, 8 * g + 4 + (r16 >> 2), k, half);
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// dF's column 64 from the per-thread sums v[e] (feature 8 sub + e over the
// thread's slots): summed over the 32 slots through buf (4 x 64 floats), one
// store a feature.  All 256 threads.
__device__ __forceinline__ void cb_store_col64(const float (&v)[8], float* buf, float* out) {
  const int tid = threadIdx.x, sub = tid & 7;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float t = v[e];
    t += __shfl_xor(t, 8);
    t += __shfl_xor(t, 16);
    t += __shfl_xor(t, 32);
    if ((tid & 63) < 8) buf[(tid >> 6) * 64 + 8 * sub + e] = t;
  }
  __syncthreads();
  if (tid < 64) out[tid * cb::kP + 64] = (buf[tid] + buf[64 + tid]) + (buf[128 + tid] + buf[192 + tid]);
}

}  // namespace smat
