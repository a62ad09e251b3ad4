// Feature map and value packing, src/smat/attention.py:82-106:
//
//   Phi = map(Q W^T),  Psi = map(K W^T) * h,  Vb = [V, 1]
//   map = elu(.) + 1   ("elu1")   or   relu(.) + 1e-3   ("relu")
//
// in the input dtype with torch's rounding steps: the product rounded to the
// dtype, elu rounded, + 1 rounded, the gate product rounded (fp32 math in
// between, as torch does for 16-bit tensors).
//
// One wave computes two 16-row tiles of X (Q or K; one in a small call) at a time
// against all r features as C = W X^T on MFMA (W is the A operand from LDS, rows padded by 16
// bytes so the sixteen feature rows a fragment reads fall in distinct banks;
// the X rows are the B operand, loaded straight from HBM as 16-byte rows).  A
// lane then holds four consecutive features of a row in each feature tile; W's
// rows are ordered so that two tiles give it eight, one 16-byte store (16-bit
// types, r a multiple of 32).  The [V, 1] rows are copied by the same launch.
//
// HBM-bound: 2 (T d_qk + T r) + T (d_v + p) elements per sequence, so what
// counts is bytes in flight against the number of places written at once: at 96
// sequences of 4096 tokens, all widths 64, 71 us (the bytes at a copy's rate:
// 63).  With the longer elu it then had: 79 with four workgroups a CU resident
// and none waiting, 85 with three of them, 84 with twelve in turn, 93 with six
// resident; 99 with one row tile a wave, 8-byte stores and W's LDS sized for 128
// features.
#include <math.h>

#include "feat_map.hpp"
#include "smat_host.hpp"

namespace smat {

namespace ft {
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxDqk = 128;       // d_qk
constexpr int kMaxRank = 128;      // feature rank
// W rows in LDS: whole 32-wide k-steps and 16 bytes, so the sixteen rows a
// fragment reads start four banks apart
__host__ __device__ constexpr int w_stride(int dqk, int elem_bytes) {
  return (dqk + 31) / 32 * 32 + 16 / elem_bytes;
}
}  // namespace ft

// kTiles: 16-row tiles a wave takes at a time.
template <typename In, int kTiles>
__global__ __launch_bounds__(ft::kThreads, sizeof(In) == 2 ? 4 : 2) void featurise_kernel(
    const In* __restrict__ q, const In* __restrict__ k, const In* __restrict__ v,
    const In* __restrict__ W, const In* __restrict__ h, In* __restrict__ phi,
    In* __restrict__ psi, In* __restrict__ vb, int nb, int T, int dqk, int r, int dv, int kind,
    int64_t q_sb, int64_t q_st, int64_t k_sb, int64_t k_st, int64_t v_sb, int64_t v_st,
    int64_t h_sb, int64_t o_sb, int64_t o_st, int64_t vb_sb, int64_t vb_st, int vec) {
  // vec: bit 0 = Q/K rows and W 16-byte aligned (vector loads), bit 1 = Phi/Psi
  // rows aligned to four elements (one store per lane and tile), bit 2 = V and
  // Vb rows 16-byte aligned, bit 3 = Phi/Psi rows 16-byte aligned and r a
  // multiple of 32 (16-bit types: one 16-byte store per lane and two tiles).
  using namespace ft;
  constexpr int kRows = 16 * kTiles;
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Quad;
  constexpr int kE = 16 / (int)sizeof(In);                   // elements per 16 bytes
  const int nks = (dqk + 31) / 32;
  const int nft = (r + 15) / 16;
  const int wst = w_stride(dqk, (int)sizeof(In));              // padded W row (elements)
  extern __shared__ __attribute__((aligned(16))) char w_raw[];
  In* w_lds = reinterpret_cast<In*>(w_raw);

  // W (r x dqk) -> LDS, zero beyond r and dqk.  With bit 3 of vec, feature tiles
  // 2 j and 2 j + 1 hold the features of [32 j, 32 j + 32) in the order that
  // leaves a lane eight consecutive ones, four in each tile.
  const bool pair = sizeof(In) == 2 && (vec & 8);
  const int wch = 32 * nks / kE;
  for (int i = threadIdx.x; i < 16 * nft * wch; i += kThreads) {
    const int m = i / wch, c = (i - m * wch) * kE;
    const int f = pair ? (m & ~31) + 8 * ((m >> 2) & 3) + 4 * ((m >> 4) & 1) + (m & 3) : m;
    In tmp[kE];
    if ((vec & 1) && f < r && c + kE <= dqk) {
      *reinterpret_cast<uint4*>(tmp) = *reinterpret_cast<const uint4*>(W + (int64_t)f * dqk + c);
    } else {
#pragma unroll
      for (int e = 0; e < kE; ++e)
        tmp[e] = (f < r && c + e < dqk) ? W[(int64_t)f * dqk + c + e] : from_f32<In>(0.f);
    }
    *reinterpret_cast<uint4*>(w_lds + m * wst + c) = *reinterpret_cast<const uint4*>(tmp);
  }
  __syncthreads();

  const int lane = lane_id();
  const int r16 = lane & 15, grp = lane >> 4;
  // tiles gwave, + nwaves, ... of the (Q / K / V, sequence, 32 rows) list, as
  // a pair (which * nb + b, tile of the sequence) that each step advances
  const int per = (T + kRows - 1) / kRows;
  const int gwave = (int)blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(wave_id());
  const int nwaves = (int)gridDim.x * kWaves;
  const int step_s = nwaves / per, step_t = nwaves - step_s * per;
  int seq = gwave / per, tile = gwave - seq * per;
  for (; seq < 3 * nb; seq += step_s, tile += step_t) {
    if (tile >= per) {
      tile -= per;
      if (++seq >= 3 * nb) break;
    }
    const int which = seq >= 2 * nb ? 2 : seq >= nb ? 1 : 0;  // 0: Q, 1: K, 2: V
    const int64_t b = seq - which * nb;
    const int t0 = tile * kRows;
    if ((which == 1 && !k) || (which == 2 && !v)) continue;   // wave-uniform
    if (which == 2) {
      // [V, 1]: four lanes a row, 16-byte pieces; a tile's loads before its stores
      const In* src = v + b * v_sb;
      In* dst = vb + b * vb_sb;
      const int npc = dv / kE;
      for (int c = lane & 3; c * kE < dv + 1; c += 4) {
        if ((vec & 4) && c < npc) {
          typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
          u32x4 y[kTiles];
#pragma unroll
          for (int u = 0; u < kTiles; ++u) {
            const int row = t0 + 16 * u + (lane >> 2);
            y[u] = *reinterpret_cast<const u32x4*>(src + (int64_t)(row < T ? row : t0) * v_st +
                                                   c * kE);
          }
#pragma unroll
          for (int u = 0; u < kTiles; ++u) {
            const int row = t0 + 16 * u + (lane >> 2);
            if (row < T) *reinterpret_cast<u32x4*>(dst + (int64_t)row * vb_st + c * kE) = y[u];
          }
          continue;
        }
#pragma unroll
        for (int u = 0; u < kTiles; ++u) {
          const int row = t0 + 16 * u + (lane >> 2);
          if (row >= T) continue;
#pragma unroll
          for (int e = 0; e < kE; ++e) {
            const int col = c * kE + e;
            if (col < dv) dst[(int64_t)row * vb_st + col] = src[(int64_t)row * v_st + col];
            else if (col == dv) dst[(int64_t)row * vb_st + col] = from_f32<In>(1.f);
          }
        }
      }
      continue;
    }
    const In* X = (which == 0 ? q + b * q_sb : k + b * k_sb);
    const int64_t x_st = which == 0 ? q_st : k_st;
    // B operands: row r16 of each 16-row tile, k-slots 32 ks + 8 grp .. + 8
    Frag xb[kTiles][kMaxDqk / 32];
    float hv[kTiles];
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      const int row = t0 + 16 * u + r16;
      const bool live = row < T;
      const In* xr = X + (int64_t)(live ? row : t0) * x_st;
#pragma unroll
      for (int ks = 0; ks < kMaxDqk / 32; ++ks) {
        if (ks < nks) {
          const int c0 = 32 * ks + 8 * grp;
          if ((vec & 1) && c0 + 8 <= dqk) {
            xb[u][ks] = *reinterpret_cast<const Frag*>(xr + c0);
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) xb[u][ks][e] = c0 + e < dqk ? xr[c0 + e] : from_f32<In>(0.f);
          }
        }
      }
      hv[u] = which == 1 && h ? to_f32(h[b * h_sb + (live ? row : t0)]) : 1.f;
    }
    In* O = (which == 0 ? phi : psi) + b * o_sb;
    // the lane's four features of feature tile f, for each row tile (a row past
    // the end computes the tile's first row and stores nothing)
    auto features = [&](int f, Quad (&out)[kTiles]) {
      f32x4 acc[kTiles];
#pragma unroll
      for (int u = 0; u < kTiles; ++u) acc[u] = zero4();
#pragma unroll
      for (int ks = 0; ks < kMaxDqk / 32; ++ks) {
        if (ks < nks) {
          Frag wa;
          const In* wp = w_lds + (16 * f + r16) * wst + 32 * ks + 8 * grp;
#pragma unroll
          for (int e = 0; e < 8; ++e) wa[e] = wp[e];
#pragma unroll
          for (int u = 0; u < kTiles; ++u) acc[u] = mma(acc[u], wa, xb[u][ks]);
        }
      }
#pragma unroll
      for (int u = 0; u < kTiles; ++u) {
        out[u] = kind == 0 ? feature_map4<In, 0>(acc[u]) : feature_map4<In, 1>(acc[u]);
        if (which == 1 && h) out[u] = feature_gate4<In>(out[u], hv[u]);
      }
    };
    if (pair) {
#pragma unroll 1
      for (int f = 0; f < nft; f += 2) {
        Quad a[kTiles], c[kTiles];
        features(f, a);
        features(f + 1, c);
#pragma unroll
        for (int u = 0; u < kTiles; ++u) {
          const int row = t0 + 16 * u + r16;
          if (row < T)
            *reinterpret_cast<Frag*>(O + (int64_t)row * o_st + 16 * f + 8 * grp) =
                __builtin_shufflevector(a[u], c[u], 0, 1, 2, 3, 4, 5, 6, 7);
        }
      }
      continue;
    }
#pragma unroll 1
    for (int f = 0; f < nft; ++f) {
      Quad out[kTiles];
      features(f, out);
      const int c0 = 16 * f + 4 * grp;
#pragma unroll
      for (int u = 0; u < kTiles; ++u) {
        const int row = t0 + 16 * u + r16;
        if (row >= T) continue;
        In* o = O + (int64_t)row * o_st + c0;
        if ((vec & 2) && c0 + 3 < r) {
          *reinterpret_cast<Quad*>(o) = out[u];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (c0 + i < r) o[i] = out[u][i];
        }
      }
    }
  }
}

}  // namespace smat

extern "C" int smat_featurise(int dtype, const void* q, const void* k, const void* v,
                              const void* W, const void* h, void* phi, void* psi, void* vb,
                              int nb, int T, int d_qk, int r, int d_v, int kind, int64_t q_sb,
                              int64_t q_st, int64_t k_sb, int64_t k_st, int64_t v_sb,
                              int64_t v_st, int64_t h_sb, int64_t o_sb, int64_t o_st,
                              int64_t vb_sb, int64_t vb_st, void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(q && W && phi, SMAT_EINVAL, "smat_featurise: null pointer");
  SMAT_REQUIRE((!k || psi) && (!v || vb), SMAT_EINVAL, "smat_featurise: k given without psi, or v "
               "without vb");
  SMAT_REQUIRE(nb >= 0 && T >= 0 && d_qk >= 1 && r >= 1 && d_v >= 0, SMAT_EINVAL,
               "smat_featurise: bad sizes");
  SMAT_REQUIRE(d_qk <= ft::kMaxDqk && r <= ft::kMaxRank, SMAT_EUNSUPPORTED,
               "smat_featurise: d_qk=%d r=%d beyond d_qk<=%d, r<=%d", d_qk, r, ft::kMaxDqk,
               ft::kMaxRank);
  SMAT_REQUIRE(kind == 0 || kind == 1, SMAT_EINVAL, "smat_featurise: kind must be 0 (elu1) or 1 "
               "(relu)");
  SMAT_REQUIRE(q_st >= d_qk && (!k || k_st >= d_qk) && (!v || (v_st >= d_v && vb_st > d_v)) &&
                   o_st >= r,
               SMAT_EINVAL, "smat_featurise: row stride too short");
  if (nb == 0 || T == 0) return SMAT_OK;
  const int64_t e16 = 16 / elem_bytes(dtype);
  if (!k) { k = q; k_sb = q_sb; k_st = q_st; psi = phi; }      // alignment checks only
  if (!v) { v = q; vb = phi; v_st = d_v; vb_st = d_v + 1; v_sb = vb_sb = 0; }
  const bool have_k = k != q || psi != phi, have_v = vb != phi;
  const int vec = ((aligned16(q) && aligned16(k) && aligned16(W) && q_st % e16 == 0 &&
                    k_st % e16 == 0 && q_sb % e16 == 0 && k_sb % e16 == 0 && d_qk % e16 == 0)
                       ? 1 : 0) |
                  ((((uintptr_t)phi | (uintptr_t)psi) % (4 * elem_bytes(dtype)) == 0 &&
                    o_st % 4 == 0 && o_sb % 4 == 0) ? 2 : 0) |
                  ((aligned16(v) && aligned16(vb) && v_st % e16 == 0 && v_sb % e16 == 0 &&
                    vb_st % e16 == 0 && vb_sb % e16 == 0) ? 4 : 0) |
                  ((aligned16(phi) && aligned16(psi) && o_st % 8 == 0 && o_sb % 8 == 0 &&
                    r % 32 == 0) ? 8 : 0);
  int dev = 0, ncu = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  // Workgroups a CU: four, or as many as W's LDS leaves room for.  Up to a 16-row
  // tile for each of their waves (a third of it where only Q is mapped), two a wave
  // would only be a longer chain: a sequence of 1000, widths 128, fp32 14.5 us
  // against 22.0, fp16 9.2 against 13.1; past it 16 of 2048 in fp32 57 and 48 us.
  const int eb = elem_bytes(dtype);
  const int64_t lds = (int64_t)((r + 15) / 16 * 16) * ft::w_stride(d_qk, eb) * eb;
  const int64_t wgs = ncu * std::min<int64_t>(4, (160 << 10) / lds);
  const int64_t lists = (int64_t)nb * (have_v ? 3 : have_k ? 2 : 1);
  const bool two = lists * ((T + 15) / 16) > wgs * ft::kWaves;
  const int64_t tiles = lists * (two ? (T + 31) / 32 : (T + 15) / 16);
  const int64_t want = (tiles + ft::kWaves - 1) / ft::kWaves;
  const unsigned grid = (unsigned)std::min<int64_t>(want, (int64_t)ncu * 4);
  hipStream_t st = (hipStream_t)stream;
  const void* kk = have_k ? k : nullptr;
  const void* vv = have_v ? v : nullptr;
#define SMAT_FT(T_)                                                                            \
  smat::launch(two ? featurise_kernel<T_, 2> : featurise_kernel<T_, 1>, dim3(grid),            \
                     dim3(ft::kThreads),                                                         \
                     (uint32_t)lds, st, (const T_*)q,                                            \
                     (const T_*)kk, (const T_*)vv, (const T_*)W, (const T_*)h, (T_*)phi, (T_*)psi, \
                     (T_*)vb, nb, T, d_qk, r, d_v, kind, q_sb, q_st, k_sb, k_st, v_sb, v_st,     \
                     h_sb, o_sb, o_st, vb_sb, vb_st, vec)
  switch (dtype) {
    case SMAT_BF16: SMAT_FT(bf16); break;
    case SMAT_F16: SMAT_FT(f16); break;
    case SMAT_F32: SMAT_FT(float); break;
    default:
      set_error("smat_featurise: unknown dtype %d", dtype);
      return SMAT_EINVAL;
  }
#undef SMAT_FT
  return launch_status("smat_featurise");
}
