// Fused backward of the intra-chunk causal scan for 16-bit inputs at
// r = 64 features and p = 65 value columns (head_dim 64 plus the ones column),
// chunks of C = 128 tokens -- the training shape.  Per chunk, with the
// chunk's incoming state Sin (r x p) and the state Q flowing backwards from
// the later chunks of its segment (r x p, the exclusive reverse scan of
// Phi^T dH):
//
//   A  = tril(Phi Psi^T),   dA = tril(dH Vb^T)               (C x C, on chip)
//   dPhi = dA Psi + dH Sin^T
//   dPsi = dA^T Phi + Vb Q^T
//   dVb  = A^T dH + Psi Q
//
// (the gradient of src/smat/attention.py:134-192 inside one chunk; the
// reference fuses the same products in src/smat/kernels/triton_bwd.py:49-147
// as a row-parallel dPhi kernel and a column-parallel dPsi/dVb kernel.)
//
// One persistent workgroup of eight waves per CU walks the (sequence, chunk)
// list.  The chunk's Phi, Psi, Vb, dH, Sin and Q are staged in LDS once, and
// the next chunk's loads are in flight in registers during its products.
// Wave w does two passes:
//
//   * row pass, row tile i = w (tokens 16w .. 16w+15): for every column tile
//     s <= i it forms the 16 x 16 block of dA^T = Vb dH^T in MFMA
//     accumulators and feeds it, split hi/lo, straight back in as the B
//     operand of dPhi^T = Psi^T dA^T (+ Sin dH^T);
//   * column pass, column tile j = w: for every row tile t >= j it forms the
//     blocks of dA = dH Vb^T and A = Phi Psi^T the same way and feeds them to
//     dPsi^T = Phi^T dA (+ Q Vb^T) and dVb^T = dH^T A (+ Q^T Psi^T).
//
// The row pass of wave w visits w + 1 tiles and the column pass 8 - w, so
// every wave does the same work.  The outputs are formed transposed so that
// each lane ends with four consecutive columns of one token row.
//
// k-slot order.  A 16 x 16 accumulator tile gives lane (n, g) rows 4g .. 4g+3;
// two tiles give it {4g + e, 16 + 4g + e}.  The MFMA contracts over any order
// of its 32 k-slots as long as both operands use it, so a pair of
// accumulator tiles is a B operand as it stands, and the matching A operand
// is read from LDS along those tokens: the gfx950 transposing read
// ds_read_b64_tr_b16 returns four consecutive token rows of one column per
// lane.
//
// Precision: Phi, Psi and Vb are exact in the MFMA's 16-bit inputs; every
// fp32 operand (dH, Sin, Q, A, dA) goes in as hi + lo (about 2^-17
// relative), and a product of two fp32 operands takes hi.hi + hi.lo + lo.hi.
// Value column 64 (the ones column) stays fp32: its rank-1 terms start the
// accumulators of the contractions over p, and dVb's column 64 is summed
// lane by lane from the blocks of A.
//
// LDS: columns 0..63 of every operand as 16-bit rows of 128 bytes (dH, Sin
// and Q once as hi and once as lo), 16-byte chunk k of row t at k ^ (t & 6),
// which keeps both the row-wise 16-byte reads and the transposing reads free
// of bank conflicts; the columns 64 as fp32 arrays.
//
// Bound by HBM: 1.7 KB of operands and gradients a token, more with added
// terms.  One workgroup a chunk, all of whose loads ended before its products
// began, each fp32 value placed in LDS by itself, took 254 us with added
// terms and 237 without at 96 sequences of 4096 tokens; the prefetch and the
// row-wise staging 198 and 179; column 64 off the MFMA tails, four values a
// split and one LDS address per operand and pass 185 and 165 (143 with the
// passes over the tiles left out; the bytes at a copy's rate: 136 and 105).
#include "bwd_common.hpp"

namespace smat {

constexpr int kBwdCUs = 256;   // one persistent workgroup per CU

struct ChunkBwdArgs {
  int nb, nc;                   // sequences, chunks per sequence
  int64_t q_sb, q_st, k_sb, k_st, v_sb, v_st;   // Phi, Psi, Vb (elements)
  int64_t h_sb, h_st;           // dH (floats)
  int64_t d_sb, d_st;           // dPhi and dPsi (elements of Out)
  int64_t e_sb, e_st;           // dVb (elements of Out)
  // optional fp32 terms added before the store (NULL: none): add_phi on rows
  // [add_split, add_end) of dPhi, add_psi and add_vb on rows [0, add_split)
  // of dPsi and dVb; rows are addressed by their absolute index
  const float* add_phi;
  const float* add_psi;
  const float* add_vb;
  int64_t ap_sb, ap_st, ak_sb, ak_st, av_sb, av_st;
  int64_t add_split, add_end;
};

// One thread's share of a chunk, in flight between global memory and LDS: the
// 16-byte pieces (row, k) = (u / 8, u % 8), u = tid + 512 i, of Phi, Psi and Vb
// and the eight floats there of dH (i < 2) and of Sin and Q (i < 1); and one
// value each of the columns 64: fp32 of dH (tid < 128), Sin (128 .. 191) or
// Q (192 .. 255), and Vb's.  The fp32 rows lie at any float stride: their
// sixteen-byte loads need only the floats' own alignment.
template <typename In>
struct ChunkBwdStage {
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Half;
  Frag phi[2], psi[2], vb[2];
  f32x4 dh[4], sn[2], qq[2];
  float c64;
  In v64;

  __device__ __forceinline__ void load(const In* phib, const In* psib, const In* vbb,
                                       const float* dHb, const float* Sinb, const float* Qb,
                                       const ChunkBwdArgs& a, int tid) {
    using namespace cb;
    const int k = tid & 7;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = (tid >> 3) + 64 * u;
      phi[u] = *reinterpret_cast<const Frag*>(phib + row * a.q_st + 8 * k);
      psi[u] = *reinterpret_cast<const Frag*>(psib + row * a.k_st + 8 * k);
      vb[u] = cb_load8(vbb + row * a.v_st + 8 * k);
      const float* y = dHb + row * a.h_st + 8 * k;
      dh[2 * u] = *reinterpret_cast<const f32x4u*>(y);
      dh[2 * u + 1] = *reinterpret_cast<const f32x4u*>(y + 4);
    }
    const int o = (tid >> 3) * kP + 8 * k;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      sn[e] = *reinterpret_cast<const f32x4u*>(Sinb + o + 4 * e);
      qq[e] = *reinterpret_cast<const f32x4u*>(Qb + o + 4 * e);
    }
    const int r = tid & (kR - 1);
    const float* c = tid < 128 ? dHb + tid * a.h_st : (tid < 192 ? Sinb : Qb) + r * kP;
    c64 = c[64];
    v64 = vbb[(tid & (kC - 1)) * a.v_st + 64];
  }
};

template <typename In, typename Out>
__global__ __launch_bounds__(cb::kThreads, 1) void chunk_bwd_kernel(
    const In* __restrict__ phi, const In* __restrict__ psi, const In* __restrict__ vb,
    const float* __restrict__ dH, const float* __restrict__ Sin, const float* __restrict__ Qs,
    Out* __restrict__ dPhi, Out* __restrict__ dPsi, Out* __restrict__ dVb, ChunkBwdArgs a) {
  using namespace cb;
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Half;
  // Phi's and dH's tiles end in sixteen rows of zeros: the row tile past the
  // last one, where a pair of row tiles has no second
  __shared__ __attribute__((aligned(16))) uint4 sPhi[(kC + 16) * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sPsi[kC * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sVb[kC * kRowChunks];
  // the fp32 operands split once into 16-bit hi and lo tiles, laid out as the
  // 16-bit ones (columns 0..63 swizzled)
  __shared__ __attribute__((aligned(16))) uint4 sdHh[(kC + 16) * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sdHl[(kC + 16) * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sSinh[kR * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sSinl[kR * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sQh[kR * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sQl[kR * kRowChunks];
  // columns 64, fp32
  __shared__ __attribute__((aligned(16))) float sVb64[kC], sdH64[kC + 16], sSin64[kR], sQ64[kR];

  ChunkBwdStage<In> sg;
  auto load = [&](int64_t b, int c, int tid) {
    const int64_t t0 = (int64_t)c * kC;
    const int64_t so = (b * a.nc + c) * (kR * kP);
    sg.load(phi + b * a.q_sb + t0 * a.q_st, psi + b * a.k_sb + t0 * a.k_st,
            vb + b * a.v_sb + t0 * a.v_st, dH + b * a.h_sb + t0 * a.h_st, Sin + so, Qs + so, a,
            tid);
  };
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  // the chunks blockIdx.x, + gridDim.x, ... of the (sequence, chunk) list
  const int step_b = (int)gridDim.x / a.nc, step_c = (int)gridDim.x - step_b * a.nc;
  int64_t b = (int)blockIdx.x / a.nc;
  int c = (int)blockIdx.x - (int)b * a.nc;
  if (b < a.nb) load(b, c, threadIdx.x);
  if (threadIdx.x < 16 * kRowChunks) {
    const int z = kC * kRowChunks + (int)threadIdx.x;
    sPhi[z] = sdHh[z] = sdHl[z] = make_uint4(0, 0, 0, 0);
    if (threadIdx.x < 16) sdH64[kC + threadIdx.x] = 0.f;
  }
  while (b < a.nb) {
    // opaque to the compiler, so that the LDS addresses of a whole pass are
    // formed in it instead of held in registers across all of them
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int r16 = lane & 15, g = lane >> 4;
    // byte offsets in a 16-bit tile of this lane's row-wise operand (row r16,
    // chunk 4 kc + g; see cb_row) and of its transposing read (cb_tr_pair);
    // row tile t lies 2048 t bytes on
    int off_r[2], off_t[4];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) off_r[kc] = 16 * cb_slot(r16, 4 * kc + g);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
      off_t[ct] = 16 * cb_slot(4 * g + (r16 >> 2), 2 * ct + ((r16 & 3) >> 1)) + 8 * (r16 & 1);
    auto row_op = [&](const uint4* tile, int t, int kc) {
      return *reinterpret_cast<const Frag*>(reinterpret_cast<const char*>(tile) + off_r[kc] +
                                            2048 * t);
    };
    auto tr_op = [&](const uint4* tile, int t0, int t1, int ct) {
      typedef short short4v __attribute__((ext_vector_type(4)));
      typedef __attribute__((address_space(3))) short4v* lds4;
      const char* p = reinterpret_cast<const char*>(tile) + off_t[ct];
      const Half x = __builtin_bit_cast(
          Half, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds4)(__attribute__((address_space(3))) char*)(p + 2048 * t0)));
      const Half y = __builtin_bit_cast(
          Half, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (lds4)(__attribute__((address_space(3))) char*)(p + 2048 * t1)));
      return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto four = [](const float* t, int row) { return *reinterpret_cast<const f32x4*>(t + row); };
    // A operand down 8 consecutive rows row0 + 8g .. +7 of a 16-bit tile: lane
    // (m = 16 ct + lane % 16, g), k-slot e <- column m of row row0 + 8g + e
    auto col8 = [&](const uint4* tile, int row0, int ct) {
      const int k = 2 * ct + ((r16 & 3) >> 1), half = r16 & 1;
      const Half lo4 = cb_tr<In>(tile, row0 + 8 * g + (r16 >> 2), k, half);
      const Half hi4 = cb_tr<In>(tile, row0 + 8 * g + 4 + (r16 >> 2), k, half);
      Frag f;
  #pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = lo4[e];
        f[4 + e] = hi4[e];
      }
      return f;
    };

    const int64_t t0 = (int64_t)c * kC;
    {
      const int k = tid & 7;
  #pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int s = cb_slot((tid >> 3) + 64 * u, k);
        sPhi[s] = __builtin_bit_cast(uint4, sg.phi[u]);
        sPsi[s] = __builtin_bit_cast(uint4, sg.psi[u]);
        sVb[s] = __builtin_bit_cast(uint4, sg.vb[u]);
        cb_split8<In>(sg.dh[2 * u], sg.dh[2 * u + 1], sdHh[s], sdHl[s]);
      }
      const int s = cb_slot(tid >> 3, k);
      cb_split8<In>(sg.sn[0], sg.sn[1], sSinh[s], sSinl[s]);
      cb_split8<In>(sg.qq[0], sg.qq[1], sQh[s], sQl[s]);
      if (tid < 128) {
        sdH64[tid] = sg.c64;
        sVb64[tid] = to_f32(sg.v64);
      } else if (tid < 192) {
        sSin64[tid - 128] = sg.c64;
      } else if (tid < 256) {
        sQ64[tid - 192] = sg.c64;
      }
    }
    __syncthreads();
    // the added terms of this lane's token row (row 16w + r16 of the chunk in
    // both passes): dPhi's from row add_split on, dPsi's and dVb's before it
    const int64_t row = t0 + 16 * w + r16;
    const bool head = row < a.add_split;
    const float* ad1 = nullptr;
    if (head && a.add_psi != nullptr) ad1 = a.add_psi + b * a.ak_sb + row * a.ak_st;
    if (!head && row < a.add_end && a.add_phi != nullptr)
      ad1 = a.add_phi + b * a.ap_sb + row * a.ap_st;
    f32x4 add1[4], add2[4];
    float add64 = 0.f;
#pragma unroll
    for (int at = 0; at < 4; ++at) add1[at] = add2[at] = zero4();
    if (ad1 != nullptr) {
#pragma unroll
      for (int at = 0; at < 4; ++at)
        add1[at] = *reinterpret_cast<const f32x4*>(ad1 + 16 * at + 4 * g);
    }
    if (head && a.add_vb != nullptr) {
      const float* ad2 = a.add_vb + b * a.av_sb + row * a.av_st;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        add2[ct] = *reinterpret_cast<const f32x4u*>(ad2 + 16 * ct + 4 * g);
      add64 = ad2[64];
    }
    // the next chunk's loads, in flight during this one's products
    int64_t nxt_b = b + step_b;
    int nxt_c = c + step_c;
    if (nxt_c >= a.nc) {
      nxt_c -= a.nc;
      ++nxt_b;
    }
    if (nxt_b < a.nb) load(nxt_b, nxt_c, tid);

    // ---- row pass: dPhi rows of tile i = w ----------------------------------
    {
      const int i = w;
      Frag dh_hi[2], dh_lo[2];
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        dh_hi[kc] = row_op(sdHh, i, kc);
        dh_lo[kc] = row_op(sdHl, i, kc);
      }
      const float dh64 = sdH64[16 * i + r16];

      f32x4 acc[4];
      // dPhi^T += Sin dH^T: A = Sin rows a (k = value column), B = dH^T
#pragma unroll
      for (int at = 0; at < 4; ++at) {
        f32x4 s = four(sSin64, 16 * at + 4 * g) * dh64;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
          const Frag hi = row_op(sSinh, at, kc);
          const Frag lo = row_op(sSinl, at, kc);
          s = mma(s, hi, dh_hi[kc]);
          s = mma(s, hi, dh_lo[kc]);
          s = mma(s, lo, dh_hi[kc]);
        }
        acc[at] = s;
      }
      // dPhi^T += Psi^T dA^T over column tiles s <= i, two at a time
      for (int sp = 0; 2 * sp <= i; ++sp) {
        f32x4 dat[2];
        // dA^T[s][t] = sum_c Vb[s][c] dH[t][c]: A = Vb rows s, B = dH^T
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4 d = four(sVb64, 32 * sp + 16 * h + 4 * g) * dh64;
#pragma unroll
          for (int kc = 0; kc < 2; ++kc) {
            const Frag vf = row_op(sVb, 2 * sp + h, kc);
            d = mma(d, vf, dh_hi[kc]);
            d = mma(d, vf, dh_lo[kc]);
          }
          dat[h] = d;
        }
        if (2 * sp + 1 >= i) {
          // lane (t = r16, g) holds s = 16 (2 sp + h) + 4g + e: keep s <= t
          const int t = 16 * (i - 2 * sp) + r16;
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) dat[h][e] = 16 * h + 4 * g + e <= t ? dat[h][e] : 0.f;
        }
        Frag bh, bl;
        cb_split_pair<In>(dat[0], dat[1], bh, bl);
#pragma unroll
        for (int at = 0; at < 4; ++at) {
          const Frag pa = tr_op(sPsi, 2 * sp, 2 * sp + 1, at);
          acc[at] = mma(acc[at], pa, bh);
          acc[at] = mma(acc[at], pa, bl);
        }
      }
      // lane (t, g) holds dPhi[t][16 at + 4g + e]
      if (!head) {
#pragma unroll
        for (int at = 0; at < 4; ++at) acc[at] += add1[at];
      }
      Out* out = dPhi + b * a.d_sb + row * a.d_st;
  #pragma unroll
      for (int at = 0; at < 4; ++at) store_grad4(out + 16 * at + 4 * g, acc[at]);
    }

    // ---- column pass: dPsi and dVb rows of tile j = w -----------------------
    {
      const int j = w;
      Frag vf[2], pf[2];
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        vf[kc] = row_op(sVb, j, kc);
        pf[kc] = row_op(sPsi, j, kc);
      }
      const float vb64 = sVb64[16 * j + r16];

      f32x4 accq[4], accv[4];
      // dPsi^T += Q Vb^T: A = Q rows a, B = Vb^T
#pragma unroll
      for (int at = 0; at < 4; ++at) {
        f32x4 s = four(sQ64, 16 * at + 4 * g) * vb64;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
          s = mma(s, row_op(sQh, at, kc), vf[kc]);
          s = mma(s, row_op(sQl, at, kc), vf[kc]);
        }
        accq[at] = s;
      }
      // dVb^T += Q^T Psi^T: A = Q^T (rows = value column c, k = feature a):
      // lane (c, g), k-slot e <- Q[32 ka + 8g + e][c]
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
        f32x4 s = zero4();
#pragma unroll
        for (int ka = 0; ka < 2; ++ka) {
          s = mma(s, col8(sQh, 32 * ka, ct), pf[ka]);
          s = mma(s, col8(sQl, 32 * ka, ct), pf[ka]);
        }
        accv[ct] = s;
      }
      // dVb's column 64, summed over this lane's features and row-tile entries
      // and at the end over the lane groups
      float v64 = 0.f;
#pragma unroll
      for (int ka = 0; ka < 2; ++ka)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 q = four(sQ64, 32 * ka + 8 * g + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) v64 += to_f32(pf[ka][4 * h + e]) * q[e];
        }
      // over row tiles t >= j, two at a time
      for (int tp = 0; j + 2 * tp < 8; ++tp) {
        const int tt = j + 2 * tp;
        f32x4 da[2], aa[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 y = four(sdH64, 16 * (tt + h) + 4 * g);
          f32x4 d = y * vb64, s = zero4();
          // dA[t][s] = sum_c dH[t][c] Vb[s][c]: A = dH rows t, B = Vb^T
          // A[t][s] = sum_a Phi[t][a] Psi[s][a]
#pragma unroll
          for (int kc = 0; kc < 2; ++kc) {
            d = mma(d, row_op(sdHh, tt + h, kc), vf[kc]);
            s = mma(s, row_op(sPhi, tt + h, kc), pf[kc]);
            d = mma(d, row_op(sdHl, tt + h, kc), vf[kc]);
          }
          if (h == 0 && tp == 0) {
            // lane (s = r16, g) holds t = 16 tt + 4g + e: keep t >= s
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const bool keep = 4 * g + e >= r16;
              d[e] = keep ? d[e] : 0.f;
              s[e] = keep ? s[e] : 0.f;
            }
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) v64 += s[e] * y[e];
          da[h] = d;
          aa[h] = s;
        }
        Frag dah, dal, aah, aal;
        cb_split_pair<In>(da[0], da[1], dah, dal);
        cb_split_pair<In>(aa[0], aa[1], aah, aal);
        // dPsi^T += Phi^T dA
#pragma unroll
        for (int at = 0; at < 4; ++at) {
          const Frag pa = tr_op(sPhi, tt, tt + 1, at);
          accq[at] = mma(accq[at], pa, dah);
          accq[at] = mma(accq[at], pa, dal);
        }
        // dVb^T += dH^T A: A operand = dH^T (rows = value column c, k = token t)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
          const Frag hi = tr_op(sdHh, tt, tt + 1, ct);
          const Frag lo = tr_op(sdHl, tt, tt + 1, ct);
          accv[ct] = mma(accv[ct], hi, aah);
          accv[ct] = mma(accv[ct], hi, aal);
          accv[ct] = mma(accv[ct], lo, aah);
        }
      }
      v64 = cb_sum_groups(v64);
      // lane (s, g) holds dPsi[s][16 at + 4g + e] and dVb[s][16 ct + 4g + e]
      if (head) {
#pragma unroll
        for (int at = 0; at < 4; ++at) {
          accq[at] += add1[at];
          accv[at] += add2[at];
        }
        v64 += add64;
      }
      Out* op = dPsi + b * a.d_sb + row * a.d_st;
  #pragma unroll
      for (int at = 0; at < 4; ++at) store_grad4(op + 16 * at + 4 * g, accq[at]);
      Out* ov = dVb + b * a.e_sb + row * a.e_st;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) cb_store4(ov + 16 * ct + 4 * g, accv[ct]);
      if (g == 0) ov[64] = from_f32<Out>(v64);
    }
    b = nxt_b;
    c = nxt_c;
    __syncthreads();                                   // this chunk's readers are done
  }
}

bool chunk_bwd_ok(int dtype, int out_dtype, const void* phi, const void* psi, int r, int p,
                  int C, int64_t q_sb, int64_t q_st, int64_t k_sb, int64_t k_st, int64_t d_sb,
                  int64_t d_st, const void* dphi, const void* dpsi) {
  if (dtype != SMAT_BF16 && dtype != SMAT_F16) return false;
  if (out_dtype != SMAT_F32 && out_dtype != dtype) return false;
  if (r != cb::kR || p != cb::kP || C != cb::kC) return false;
  const int ob = elem_bytes(out_dtype);
  return rows_vec_ok(phi, q_sb, q_st, 2) && rows_vec_ok(psi, k_sb, k_st, 2) &&
         rows_vec_ok(dphi, d_sb, d_st, ob) && rows_vec_ok(dpsi, d_sb, d_st, ob);
}

template <typename In, typename Out>
static void chunk_bwd_launch(const void* phi, const void* psi, const void* vb, const float* dH,
                             const float* Sin, const float* Q, void* dPhi, void* dPsi, void* dVb,
                             const ChunkBwdArgs& a, hipStream_t st) {
  const int64_t items = (int64_t)a.nb * a.nc;
  const int grid = (int)(items < kBwdCUs ? items : kBwdCUs);
  hipLaunchKernelGGL((chunk_bwd_kernel<In, Out>), dim3(grid), dim3(cb::kThreads), 0, st,
                     (const In*)phi, (const In*)psi, (const In*)vb, dH, Sin, Q, (Out*)dPhi,
                     (Out*)dPsi, (Out*)dVb, a);
}

// ---------------------------------------------------------------------------
// The per-chunk state gradient Dr_c = Phi_c^T dH_c (r x p fp32, one matrix per
// (sequence, chunk); the input of the reverse scan that gives Q), one
// workgroup of four waves per item.  Phi's chunk is staged as 16-bit rows
// (swizzled), dH's split into 16-bit hi/lo tiles as in chunk_bwd_kernel.
// Wave w forms rows 16w .. 16w+15 of Dr (features) across five value-column
// tiles: A = Phi^T and B = dH, both read down the chunk's tokens with the
// transposing reads, 32 tokens a product; lane (c, g) ends with
// Dr[16w + 4g + e][c].
// ---------------------------------------------------------------------------
namespace cds {
constexpr int kThreads = 256;
}  // namespace cds

template <typename In>
__global__ __launch_bounds__(cds::kThreads) void chunk_dstate_kernel(
    const In* __restrict__ phi, const float* __restrict__ dH, float* __restrict__ Dr, int nc,
    int vec_dh, int64_t q_sb, int64_t q_st, int64_t h_sb, int64_t h_st) {
  using namespace cb;
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Half;
  __shared__ __attribute__((aligned(16))) uint4 sPhi[kC * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sdHh[kC * kRowChunks];
  __shared__ __attribute__((aligned(16))) uint4 sdHl[kC * kRowChunks];
  __shared__ In sdH64h[kC], sdH64l[kC];

  const int c = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int tid = threadIdx.x;
  const int64_t t0 = (int64_t)c * kC;
  const In* phib = phi + b * q_sb + t0 * q_st;
  const float* dHb = dH + b * h_sb + t0 * h_st;
  constexpr int kN = kC * kP;                       // 8320 dH values
  constexpr int kPhiIt = kC * kRowChunks / cds::kThreads;   // 4
  constexpr int kH4 = kN / 4;                       // 2080 float4s
  constexpr int kH4It = (kH4 + cds::kThreads - 1) / cds::kThreads;   // 9
  constexpr int kHIt = (kN + cds::kThreads - 1) / cds::kThreads;     // 33

  auto put = [&](int e, In h, In l) {
    const int row = e / kP, col = e - row * kP;
    if (col < 64) {
      reinterpret_cast<In*>(sdHh + cb_slot(row, col >> 3))[col & 7] = h;
      reinterpret_cast<In*>(sdHl + cb_slot(row, col >> 3))[col & 7] = l;
    } else {
      sdH64h[row] = h;
      sdH64l[row] = l;
    }
  };
  // Phi's rows straight to LDS (issued after dH's loads, which stay in flight)
  auto put_phi = [&]() {
#pragma unroll
    for (int u = 0; u < kPhiIt; ++u) {
      const int e = tid + cds::kThreads * u;
      sPhi[cb_slot(e >> 3, e & 7)] =
          *reinterpret_cast<const uint4*>(phib + (e >> 3) * q_st + 8 * (e & 7));
    }
  };
  if (vec_dh) {
    float4 rdh[kH4It];
#pragma unroll
    for (int u = 0; u < kH4It; ++u) {
      const int e4 = tid + cds::kThreads * u;
      rdh[u] = reinterpret_cast<const float4*>(dHb)[e4 < kH4 ? e4 : 0];
    }
    put_phi();
#pragma unroll
    for (int u = 0; u < kH4It; ++u) {
      const int e4 = tid + cds::kThreads * u;
      if (e4 < kH4) {
        Half h, l;
        split4<In>(f32x4{rdh[u].x, rdh[u].y, rdh[u].z, rdh[u].w}, h, l);
#pragma unroll
        for (int q = 0; q < 4; ++q) put(4 * e4 + q, h[q], l[q]);
      }
    }
  } else {
    put_phi();
    for (int u = 0; u < kHIt; ++u) {
      const int e = tid + cds::kThreads * u;
      if (e < kN) {
        const int row = e / kP, col = e - row * kP;
        In h, l;
        split2<In>(dHb[row * h_st + col], h, l);
        put(e, h, l);
      }
    }
  }
  __syncthreads();

  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  // lane (m = 16 ct + lane % 16, g), k-slot e <- column m of row row0 + 8g + e
  auto col8 = [&](const uint4* tile, int row0, int ct) {
    const int k = 2 * ct + ((r16 & 3) >> 1), half = r16 & 1;
    const Half lo4 = cb_tr<In>(tile, row0 + 8 * g + (r16 >> 2), k, half);
    const Half hi4 = cb_tr<In>(tile, row0 + 8 * g + 4 + (r16 >> 2), k, half);
    Frag f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = lo4[e];
      f[4 + e] = hi4[e];
    }
    return f;
  };
  f32x4 acc[5];
#pragma unroll
  for (int ct = 0; ct < 5; ++ct) acc[ct] = zero4();
#pragma unroll
  for (int ks = 0; ks < kC / 32; ++ks) {
    const Frag pa = col8(sPhi, 32 * ks, w);          // Phi^T rows 16w + r16
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      acc[ct] = mma(acc[ct], pa, col8(sdHh, 32 * ks, ct));
      acc[ct] = mma(acc[ct], pa, col8(sdHl, 32 * ks, ct));
    }
    Frag bh, bl;                                     // column 64: lane r16 = 0
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = 32 * ks + 8 * g + e;
      bh[e] = r16 == 0 ? sdH64h[t] : from_f32<In>(0.f);
      bl[e] = r16 == 0 ? sdH64l[t] : from_f32<In>(0.f);
    }
    acc[4] = mma(acc[4], pa, bh);
    acc[4] = mma(acc[4], pa, bl);
  }
  float* out = Dr + ((int64_t)b * nc + c) * (kR * kP);
#pragma unroll
  for (int ct = 0; ct < 5; ++ct) {
    const int col = 16 * ct + r16;
    if (col < kP) {
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(16 * w + 4 * g + e) * kP + col] = acc[ct][e];
    }
  }
}

}  // namespace smat

extern "C" int smat_chunk_backward(int dtype, int out_dtype, const void* phi, const void* psi,
                                   const void* vb, const float* dH, const float* Sin,
                                   const float* Q, void* dPhi, void* dPsi, void* dVb, int nb,
                                   int nc, int r, int p, int C,
                                   int64_t q_sb, int64_t q_st, int64_t k_sb, int64_t k_st,
                                   int64_t v_sb, int64_t v_st, int64_t h_sb, int64_t h_st,
                                   int64_t d_sb, int64_t d_st, int64_t e_sb, int64_t e_st,
                                   const float* add_phi, const float* add_psi,
                                   const float* add_vb, int64_t ap_sb, int64_t ap_st,
                                   int64_t ak_sb, int64_t ak_st, int64_t av_sb, int64_t av_st,
                                   int64_t add_split, int64_t add_end, void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(phi && psi && vb && dH && Sin && Q && dPhi && dPsi && dVb, SMAT_EINVAL,
               "smat_chunk_backward: null pointer");
  SMAT_REQUIRE(nb >= 0 && nc >= 0, SMAT_EINVAL, "smat_chunk_backward: bad sizes");
  SMAT_REQUIRE(nc < 65536 * 32 && nb < 65536, SMAT_EUNSUPPORTED,
               "smat_chunk_backward: grid %d x %d too large", nc, nb);
  SMAT_REQUIRE(chunk_bwd_ok(dtype, out_dtype, phi, psi, r, p, C, q_sb, q_st, k_sb, k_st, d_sb,
                            d_st, dPhi, dPsi),
               SMAT_EUNSUPPORTED,
               "smat_chunk_backward: needs 16-bit inputs, fp32 or input-typed gradients, r=64, "
               "p=65, C=128 and 16-byte aligned rows of Phi, Psi, dPhi and dPsi (got dtype=%d "
               "out_dtype=%d r=%d p=%d C=%d)",
               dtype, out_dtype, r, p, C);
  SMAT_REQUIRE(v_st >= p && h_st >= p && e_st >= p && d_st >= r, SMAT_EINVAL,
               "smat_chunk_backward: row stride too short");
  SMAT_REQUIRE(0 <= add_split && add_split <= add_end && add_end <= (int64_t)nc * C &&
                   (!add_phi || (rows_vec_ok(add_phi, ap_sb, ap_st, 4) && ap_st >= r)) &&
                   (!add_psi || (rows_vec_ok(add_psi, ak_sb, ak_st, 4) && ak_st >= r)) &&
                   (!add_vb || av_st >= p),
               SMAT_EINVAL,
               "smat_chunk_backward: added terms need 0 <= add_split <= add_end <= nc*C, "
               "16-byte aligned rows for Phi and Psi and full rows");
  if (nb == 0 || nc == 0) return SMAT_OK;
  SMAT_REQUIRE(aligned16(Sin) && aligned16(Q), SMAT_EINVAL,
               "smat_chunk_backward: Sin and Q must be 16-byte aligned");
  ChunkBwdArgs a{nb,    nc,     q_sb,  q_st,  k_sb,    k_st,    v_sb,    v_st,
                 h_sb,  h_st,   d_sb,  d_st,  e_sb,    e_st,    add_phi, add_psi, add_vb,
                 ap_sb, ap_st,  ak_sb, ak_st, av_sb,   av_st,   add_split, add_end};
  hipStream_t st = (hipStream_t)stream;
  const bool f32 = out_dtype == SMAT_F32;
  if (dtype == SMAT_BF16)
    (f32 ? chunk_bwd_launch<bf16, float> : chunk_bwd_launch<bf16, bf16>)(
        phi, psi, vb, dH, Sin, Q, dPhi, dPsi, dVb, a, st);
  else
    (f32 ? chunk_bwd_launch<f16, float> : chunk_bwd_launch<f16, f16>)(
        phi, psi, vb, dH, Sin, Q, dPhi, dPsi, dVb, a, st);
  return launch_status("smat_chunk_backward");
}

extern "C" int smat_chunk_dstates(int dtype, const void* phi, const float* dH, float* Dr, int nb,
                                  int nc, int r, int p, int C, int64_t q_sb, int64_t q_st,
                                  int64_t h_sb, int64_t h_st, void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(phi && dH && Dr, SMAT_EINVAL, "smat_chunk_dstates: null pointer");
  SMAT_REQUIRE(nb >= 0 && nc >= 0, SMAT_EINVAL, "smat_chunk_dstates: bad sizes");
  SMAT_REQUIRE(nc < 65536 * 32 && nb < 65536, SMAT_EUNSUPPORTED,
               "smat_chunk_dstates: grid %d x %d too large", nc, nb);
  SMAT_REQUIRE((dtype == SMAT_BF16 || dtype == SMAT_F16) && r == cb::kR && p == cb::kP &&
                   C == cb::kC && rows_vec_ok(phi, q_sb, q_st, 2) && h_st >= p && aligned16(Dr),
               SMAT_EUNSUPPORTED,
               "smat_chunk_dstates: needs 16-bit Phi with 16-byte aligned rows, r=64, p=65, "
               "C=128 (got dtype=%d r=%d p=%d C=%d)",
               dtype, r, p, C);
  if (nb == 0 || nc == 0) return SMAT_OK;
  const int vec_dh = h_st == p && h_sb % 4 == 0 && aligned16(dH);
  const dim3 grid((unsigned)nc, (unsigned)nb);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SMAT_BF16)
    hipLaunchKernelGGL(chunk_dstate_kernel<bf16>, grid, dim3(cds::kThreads), 0, st,
                       (const bf16*)phi, dH, Dr, nc, vec_dh, q_sb, q_st, h_sb, h_st);
  else
    hipLaunchKernelGGL(chunk_dstate_kernel<f16>, grid, dim3(cds::kThreads), 0, st,
                       (const f16*)phi, dH, Dr, nc, vec_dh, q_sb, q_st, h_sb, h_st);
  return launch_status("smat_chunk_dstates");
}
