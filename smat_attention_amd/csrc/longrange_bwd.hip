// Backward of the pooled long-range branch at the training shape (16-bit
// inputs, r = 64 features, p = 65 value columns).  The forward (attention.py:
// 196-330) pools F_x = sum_{j in profile x} Psi_j^T Vb_j, sums U_h =
// sum_{x in H_h} F_x (+ F_glob), and adds Y_i = Phi_i U_{h(i)} to recent row
// i, h(i) = (i - n) mod B.  Given dY = dH on the recent rows:
//
//   smat_lr_dphi        dPhi_i += dY_i U_h^T                     per row type h
//   smat_lr_dfeat       dF_x = sum_{h : x in H_h} sum_{i in R_h} Phi_i^T dY_i
//                       (dU_h = sum_{i in R_h} Phi_i^T dY_i, then C^T dU, in
//                       one pass: dU never reaches HBM); the global channel's
//                       dF_glob = sum over every recent row
//   smat_pool_backward  dPsi_j += Vb_j dF_x^T,  dVb_j += Psi_j dF_x
//                       per profile x, dF_x read once for both
//
// Each launch streams one r x p fp32 matrix per item (U_h, dF_x) against the
// few token rows of that item -- bandwidth kernels whose waves mostly wait
// on their loads, so the list gram and the pool backward cap their registers
// for five workgroups a CU, every launch has its token rows in flight while the
// matrix is staged, and rows are read eight values at a time wherever they
// start.  At 96 sequences of 4096 tokens, d = 3 (T_R = 2048): the query's dPhi
// 107 -> 91 us (its 390 MB at a copy's rate: 80), the list gram 226 -> 140
// (1 GB of rows from L2; the split of dY once per gathered row instead of by
// every wave, and column 64 off one wave, took it from the LDS and the VALU),
// the pool backward 164 -> 97 (420 MB: 86).  The products run on 16-bit
// MFMA with fp32 operands split hi/lo, except the query's dPhi (fp32 MFMA, see
// there) and the terms of value column 64, which are fp32.  The reference differentiates
// the query and incidence with torch and fuses the pool backward in
// src/smat/kernels/triton_bwd.py:203-237 ("dF_x loaded once"); the
// incidence backward there is the forward kernel over C^T (:262-276).
#include "bwd_common.hpp"

namespace smat {

namespace lr {
constexpr int kThreads = 256;       // four waves; wave w owns 16-wide tile w
constexpr int kRP = cb::kR * cb::kP;   // 4160 floats per r x p matrix
constexpr int kStep = 32;           // tokens per K step of the list gram
}  // namespace lr

// ---------------------------------------------------------------------------
// dPhi[n + h + kB] += dY[n + h + kB] U_h^T, one workgroup per (h, sequence).
// Wave w forms feature tile w of the transposed product, dPhi^T = U_h dY^T:
// A = U_h rows (LDS, loaded once), B = dY^T from the token rows, 16 at a time
// (the first sixteen in flight while U_h is staged); lane (row, g) ends with
// dPhi[row][16w + 4g .. +3].
//
// This product runs on fp32 MFMA (v_mfma_f32_16x16x4_f32, column 32 kc + 8g + j
// for frag element j): its sum over value columns cancels the normaliser column
// against the values (the quotient rule of the final division), and U_h holds
// large pooled sums, so hi/lo 16-bit operands (~2^-16) would leave an error
// of order 1e-3 of the result.
// ---------------------------------------------------------------------------
template <typename In>
__global__ __launch_bounds__(lr::kThreads) void lr_dphi_kernel(
    const float* __restrict__ dH, const float* __restrict__ U, float* __restrict__ dPhi,
    int T_R, int B, int n, int64_t h_sb, int64_t h_st, int64_t u_sb, int64_t d_sb,
    int64_t d_st, int accumulate) {
  using namespace cb;
  __shared__ __attribute__((aligned(16))) float sU[kR * kS];
  const int h = blockIdx.x;
  const int64_t b = blockIdx.y;
  const int cnt = h < T_R ? (T_R - h + B - 1) / B : 0;
  if (cnt == 0) return;                              // uniform over the workgroup
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  const float* dHb = dH + b * h_sb;
  float* dPb = dPhi + b * d_sb;
  // this lane's row of row tile rt (a row past the end reads the first one and
  // is not stored): columns 32 kc + 8g .. +7, and 64
  f32x8 yb[2];
  float yt;
  auto load = [&](int rt) {
    const int k = 16 * rt + r16;
    const float* y = dHb + (n + h + (int64_t)(k < cnt ? k : 0) * B) * h_st;
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) yb[kc] = CbRow8<float>::load(y + 32 * kc + 8 * g);
    yt = y[64];
  };
  load(0);
  cb_stage_rp(sU, U + b * u_sb + (int64_t)h * lr::kRP);
  __syncthreads();

  const int arow = 16 * w + r16;
  f32x8 ua[2];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc)
#pragma unroll
    for (int j = 0; j < 8; ++j) ua[kc][j] = sU[arow * kS + 32 * kc + 8 * g + j];
  f32x4 ut;                                          // column 64 of rows 16w + 4g + i
#pragma unroll
  for (int i = 0; i < 4; ++i) ut[i] = sU[(16 * w + 4 * g + i) * kS + 64];

  for (int rt = 0; 16 * rt < cnt; ++rt) {
    const int k = 16 * rt + r16;
    const bool ok = k < cnt;
    const int64_t row = n + h + (int64_t)(ok ? k : 0) * B;
    f32x4 acc = ut * yt;
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) acc = mma(acc, ua[kc], yb[kc]);
    if (16 * (rt + 1) < cnt) load(rt + 1);
    if (ok) {
      float4* o = reinterpret_cast<float4*>(dPb + row * d_st + 16 * w + 4 * g);
      float4 cur = accumulate ? *o : make_float4(0.f, 0.f, 0.f, 0.f);
      cur.x += acc[0];
      cur.y += acc[1];
      cur.z += acc[2];
      cur.w += acc[3];
      *o = cur;
    }
  }
}

// ---------------------------------------------------------------------------
// dF[x] = sum over the token list of item x of Phi_t^T dY_t, one workgroup
// per (item, sequence): 32 tokens a step are gathered into LDS as 16-bit rows
// (Phi, and dY split hi/lo once; eight threads a token, the next step's gather
// in flight during the products, two buffers and one barrier a step), then
// D[a][c] += Phi^T dY with both operands by transposing reads (k-slot 8g + e =
// token slot).  Wave w owns value-column tile w for all four feature tiles;
// column 64 is summed in fp32 by the threads that gather.
// ---------------------------------------------------------------------------
template <typename In>
__global__ __launch_bounds__(lr::kThreads, 5) void lr_dfeat_kernel(
    const In* __restrict__ phi, const float* __restrict__ dH, const int32_t* __restrict__ tptr,
    const int32_t* __restrict__ tok, float* __restrict__ dF, int64_t q_sb, int64_t q_st,
    int64_t h_sb, int64_t h_st, int64_t f_sb) {
  using namespace cb;
  typedef typename Traits<In>::frag Frag;
  __shared__ __attribute__((aligned(16))) uint4 sT[2][3][lr::kStep * kRowChunks];
  int x;
  int64_t b;
  xcd_item_seq(x, b);
  const int tid = threadIdx.x;
  const int64_t beg = tptr[x], end = tptr[x + 1];
  const In* phib = phi + b * q_sb;
  const float* dHb = dH + b * h_sb;
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int lane = lane_id(), r16 = lane & 15, g = lane >> 4;

  f32x4 acc[4];
  float c64[8];
#pragma unroll
  for (int at = 0; at < 4; ++at) acc[at] = zero4();
#pragma unroll
  for (int e = 0; e < 8; ++e) c64[e] = 0.f;
  CbGather<In, float> ga;
  if (beg < end) {
    ga.peek(tok, beg, beg, end, tid);
    ga.load(beg, end, 0, phib, q_st, dHb, h_st, tid);
    ga.peek(tok, beg + lr::kStep, beg, end, tid);
  }
  for (int64_t s0 = beg; s0 < end; s0 += lr::kStep) {
    uint4 (*buf)[lr::kStep * kRowChunks] = sT[((s0 - beg) / lr::kStep) & 1];
    if (s0 + lr::kStep > end) ga.mask();
    {
      const int s = cb_slot(tid >> 3, tid & 7);
      buf[0][s] = __builtin_bit_cast(uint4, ga.r64);
      cb_split8<In>(__builtin_shufflevector(ga.r65, ga.r65, 0, 1, 2, 3),
                    __builtin_shufflevector(ga.r65, ga.r65, 4, 5, 6, 7), buf[1][s], buf[2][s]);
#pragma unroll
      for (int e = 0; e < 8; ++e) c64[e] += to_f32(ga.r64[e]) * ga.c65;
    }
    // a wave writes the other buffer only after this barrier, which every wave
    // reaches after its products of the step before
    __syncthreads();
    if (s0 + lr::kStep < end) {
      ga.load(s0 + lr::kStep, end, 0, phib, q_st, dHb, h_st, tid);
      ga.peek(tok, s0 + 2 * lr::kStep, beg, end, tid);
    }
    const Frag bh = cb_col32<In>(buf[1], w, lane), bl = cb_col32<In>(buf[2], w, lane);
#pragma unroll
    for (int at = 0; at < 4; ++at) {
      const Frag pa = cb_col32<In>(buf[0], at, lane);
      acc[at] = mma(acc[at], pa, bh);
      acc[at] = mma(acc[at], pa, bl);
    }
  }
  // lane (c = 16 w + r16, g) holds dF[16 at + 4g + e][c]
  float* out = dF + b * f_sb + (int64_t)x * lr::kRP;
#pragma unroll
  for (int at = 0; at < 4; ++at)
#pragma unroll
    for (int e = 0; e < 4; ++e) out[(16 * at + 4 * g + e) * kP + 16 * w + r16] = acc[at][e];
  __syncthreads();
  cb_store_col64(c64, reinterpret_cast<float*>(sT), out);
}

// ---------------------------------------------------------------------------
// Pool backward, one workgroup per (profile x, sequence): profile x < N0
// holds tokens n_P + x + s N0 < n; item N0 (the global channel, when n_P > 0)
// holds tokens 0 .. n_P - 1 with dF row N0 = dF_glob.  dF_x is staged once;
// wave w forms
//   dPsi^T tile w = dF_x Vb^T       (A = dF rows, B = Vb rows)
//   dVb^T  tile w = dF_x^T Psi^T    (A = dF columns, B = Psi rows)
// for the tokens, 16 at a time, and stores them or adds them in; dVb's column
// 64 is an fp32 sum by one wave.
// ---------------------------------------------------------------------------
template <typename In>
__global__ __launch_bounds__(lr::kThreads, 5) void lr_pool_bwd_kernel(
    const In* __restrict__ psi, const In* __restrict__ vb, const float* __restrict__ dF,
    float* __restrict__ dPsi, float* __restrict__ dVb, int N0, int n, int n_P, int64_t k_sb,
    int64_t k_st, int64_t v_sb, int64_t v_st, int64_t f_sb, int64_t d_sb, int64_t d_st,
    int64_t e_sb, int64_t e_st, int accumulate) {
  using namespace cb;
  typedef typename Traits<In>::frag Frag;
  __shared__ __attribute__((aligned(16))) float sF[kR * kS];
  int x;
  int64_t b;
  xcd_item_seq(x, b);
  const int64_t start = x < N0 ? (int64_t)n_P + x : 0;
  const int64_t stride = x < N0 ? N0 : 1;
  const int nX = n - n_P;
  const int cnt = x < N0 ? (x < nX ? (nX - x + N0 - 1) / N0 : 0) : n_P;
  if (cnt == 0) return;                              // uniform over the workgroup
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int lane = lane_id(), r16 = lane & 15, g = lane >> 4;
  const In* psib = psi + b * k_sb;
  const In* vbb = vb + b * v_sb;
  // B operands along this lane's token row of row tile rt (a row past the end
  // reads the first one and is not stored)
  Frag vf[2], pf[2];
  In vt;
  auto load = [&](int rt) {
    const int k = 16 * rt + r16;
    const int64_t j = start + (int64_t)(k < cnt ? k : 0) * stride;
    const In* vrow = vbb + j * v_st;
    const In* prow = psib + j * k_st;
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      pf[kc] = *reinterpret_cast<const Frag*>(prow + 32 * kc + 8 * g);
      vf[kc] = cb_load8(vrow + 32 * kc + 8 * g);
    }
    vt = vrow[64];
  };
  load(0);
  cb_stage_rp(sF, dF + b * f_sb + (int64_t)x * lr::kRP);
  __syncthreads();

  // dPsi: A = dF rows a = 16w + r16 (hi/lo), columns 32 kc + 8g + e, and
  // column 64 of rows 16w + 4g + i
  Frag fh[2], fl[2];
#pragma unroll
  for (int kc = 0; kc < 2; ++kc) cb_row32<In>(sF, 16 * w + r16, kc, g, fh[kc], fl[kc]);
  f32x4 ft;
#pragma unroll
  for (int i = 0; i < 4; ++i) ft[i] = sF[(16 * w + 4 * g + i) * kS + 64];
  // dVb: A = dF^T rows c (value column), k = feature 32 ka + 8g + e
  Frag ch[2], cl[2];
#pragma unroll
  for (int ka = 0; ka < 2; ++ka)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = sF[(32 * ka + 8 * g + 4 * h + e) * kS + 16 * w + r16];
      typename Traits<In>::half_frag hh, ll;
      split4<In>(v, hh, ll);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ch[ka][4 * h + e] = hh[e];
        cl[ka][4 * h + e] = ll[e];
      }
    }

  float* dPb = dPsi + b * d_sb;
  float* dVbb = dVb + b * e_sb;
  for (int rt = 0; 16 * rt < cnt; ++rt) {
    const int k = 16 * rt + r16;
    const bool ok = k < cnt;
    const int64_t j = start + (int64_t)(ok ? k : 0) * stride;
    f32x4 ap = ft * to_f32(vt), av = zero4();
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      ap = mma(ap, fh[kc], vf[kc]);
      ap = mma(ap, fl[kc], vf[kc]);
      av = mma(av, ch[kc], pf[kc]);
      av = mma(av, cl[kc], pf[kc]);
    }
    // dVb's column 64, a sum over the features in fp32, by one wave of the four
    const bool mine = (rt & 3) == w;
    float v64 = 0.f;
    if (mine) {
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v64 += sF[(32 * kc + 8 * g + e) * kS + 64] * to_f32(pf[kc][e]);
      v64 = cb_sum_groups(v64);
    }
    if (16 * (rt + 1) < cnt) load(rt + 1);
    if (ok) {
      // lane (j, g): dPsi[j][16w + 4g + e], dVb[j][16w + 4g + e] (and dVb[j][64])
      float4* o = reinterpret_cast<float4*>(dPb + j * d_st + 16 * w + 4 * g);
      float4 cur = accumulate ? *o : make_float4(0.f, 0.f, 0.f, 0.f);
      cur.x += ap[0];
      cur.y += ap[1];
      cur.z += ap[2];
      cur.w += ap[3];
      *o = cur;
      f32x4u* ov = reinterpret_cast<f32x4u*>(dVbb + j * e_st + 16 * w + 4 * g);
      *ov = accumulate ? *ov + av : av;
      if (mine && g == 0) dVbb[j * e_st + 64] = (accumulate ? dVbb[j * e_st + 64] : 0.f) + v64;
    }
  }
}

static bool lr_shape_ok(int dtype, int r, int p) {
  return (dtype == SMAT_BF16 || dtype == SMAT_F16) && r == cb::kR && p == cb::kP;
}

}  // namespace smat

extern "C" int smat_lr_dphi(int dtype, const float* dH, const float* U, float* dPhi, int nb,
                            int T_R, int B, int n, int r, int p, int64_t h_sb, int64_t h_st,
                            int64_t u_sb, int64_t d_sb, int64_t d_st, int accumulate,
                            void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(dH && U && dPhi, SMAT_EINVAL, "smat_lr_dphi: null pointer");
  SMAT_REQUIRE(nb >= 0 && T_R >= 0 && B >= 1 && n >= 0, SMAT_EINVAL, "smat_lr_dphi: bad sizes");
  SMAT_REQUIRE(lr_shape_ok(dtype, r, p), SMAT_EUNSUPPORTED,
               "smat_lr_dphi: needs dtype bf16/f16, r=64, p=65 (got %d, %d, %d)", dtype, r, p);
  SMAT_REQUIRE(aligned16(U) && u_sb % 4 == 0 && rows_vec_ok(dPhi, d_sb, d_st, 4) &&
                   h_st >= p && d_st >= r,
               SMAT_EINVAL, "smat_lr_dphi: U and dPhi rows must be 16-byte aligned");
  SMAT_REQUIRE(B < 65536 * 32 && nb < 65536, SMAT_EUNSUPPORTED, "smat_lr_dphi: grid too large");
  if (nb == 0 || T_R == 0) return SMAT_OK;
  const dim3 grid((unsigned)B, (unsigned)nb);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SMAT_BF16)
    hipLaunchKernelGGL(lr_dphi_kernel<bf16>, grid, dim3(lr::kThreads), 0, st, dH, U, dPhi, T_R, B,
                       n, h_sb, h_st, u_sb, d_sb, d_st, accumulate);
  else
    hipLaunchKernelGGL(lr_dphi_kernel<f16>, grid, dim3(lr::kThreads), 0, st, dH, U, dPhi, T_R, B,
                       n, h_sb, h_st, u_sb, d_sb, d_st, accumulate);
  return launch_status("smat_lr_dphi");
}

extern "C" int smat_lr_dfeat(int dtype, const void* phi, const float* dH, const int32_t* tptr,
                             const int32_t* tok, float* dF, int nb, int nitems, int r, int p,
                             int64_t q_sb, int64_t q_st, int64_t h_sb, int64_t h_st, int64_t f_sb,
                             void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(phi && dH && tptr && tok && dF, SMAT_EINVAL, "smat_lr_dfeat: null pointer");
  SMAT_REQUIRE(nb >= 0 && nitems >= 0, SMAT_EINVAL, "smat_lr_dfeat: bad sizes");
  SMAT_REQUIRE(lr_shape_ok(dtype, r, p), SMAT_EUNSUPPORTED,
               "smat_lr_dfeat: needs dtype bf16/f16, r=64, p=65 (got %d, %d, %d)", dtype, r, p);
  SMAT_REQUIRE(rows_vec_ok(phi, q_sb, q_st, 2) && h_st >= p && f_sb >= (int64_t)nitems * r * p,
               SMAT_EINVAL, "smat_lr_dfeat: Phi rows must be 16-byte aligned");
  SMAT_REQUIRE(nitems < 65536 * 32 && nb < 65536, SMAT_EUNSUPPORTED,
               "smat_lr_dfeat: grid too large");
  if (nb == 0 || nitems == 0) return SMAT_OK;
  const dim3 grid((unsigned)nitems, (unsigned)nb);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SMAT_BF16)
    hipLaunchKernelGGL(lr_dfeat_kernel<bf16>, grid, dim3(lr::kThreads), 0, st, (const bf16*)phi,
                       dH, tptr, tok, dF, q_sb, q_st, h_sb, h_st, f_sb);
  else
    hipLaunchKernelGGL(lr_dfeat_kernel<f16>, grid, dim3(lr::kThreads), 0, st, (const f16*)phi,
                       dH, tptr, tok, dF, q_sb, q_st, h_sb, h_st, f_sb);
  return launch_status("smat_lr_dfeat");
}

extern "C" int smat_pool_backward(int dtype, const void* psi, const void* vb, const float* dF,
                                  float* dPsi, float* dVb, int nb, int N0, int n, int n_P, int r,
                                  int p, int64_t k_sb, int64_t k_st, int64_t v_sb, int64_t v_st,
                                  int64_t f_sb, int64_t d_sb, int64_t d_st, int64_t e_sb,
                                  int64_t e_st, int accumulate, void* stream) {
  using namespace smat;
  clear_error();
  SMAT_REQUIRE(psi && vb && dF && dPsi && dVb, SMAT_EINVAL, "smat_pool_backward: null pointer");
  SMAT_REQUIRE(nb >= 0 && N0 >= 1 && n_P >= 0 && n >= n_P, SMAT_EINVAL,
               "smat_pool_backward: bad sizes");
  SMAT_REQUIRE(lr_shape_ok(dtype, r, p), SMAT_EUNSUPPORTED,
               "smat_pool_backward: needs dtype bf16/f16, r=64, p=65 (got %d, %d, %d)", dtype, r,
               p);
  SMAT_REQUIRE(rows_vec_ok(psi, k_sb, k_st, 2) && rows_vec_ok(dPsi, d_sb, d_st, 4) &&
                   aligned16(dF) && f_sb % 4 == 0 && v_st >= p && e_st >= p && d_st >= r,
               SMAT_EINVAL, "smat_pool_backward: Psi, dPsi and dF must be 16-byte aligned");
  const int nitems = N0 + (n_P > 0 ? 1 : 0);
  SMAT_REQUIRE(nitems < 65536 * 32 && nb < 65536, SMAT_EUNSUPPORTED,
               "smat_pool_backward: grid too large");
  if (nb == 0) return SMAT_OK;
  const dim3 grid((unsigned)nitems, (unsigned)nb);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == SMAT_BF16)
    hipLaunchKernelGGL(lr_pool_bwd_kernel<bf16>, grid, dim3(lr::kThreads), 0, st,
                       (const bf16*)psi, (const bf16*)vb, dF, dPsi, dVb, N0, n, n_P, k_sb, k_st,
                       v_sb, v_st, f_sb, d_sb, d_st, e_sb, e_st, accumulate);
  else
    hipLaunchKernelGGL(lr_pool_bwd_kernel<f16>, grid, dim3(lr::kThreads), 0, st, (const f16*)psi,
                       (const f16*)vb, dF, dPsi, dVb, N0, n, n_P, k_sb, k_st, v_sb, v_st, f_sb,
                       d_sb, d_st, e_sb, e_st, accumulate);
  return launch_status("smat_pool_backward");
}
