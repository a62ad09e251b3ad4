// The causal pass of the schedule for the common head shapes -- 16-bit inputs,
// r = 64, 80, 96, 112 or 128 features, p = r + 1 value columns (the head's plus
// the ones column), n and the chunk multiples of 64 -- streamed through LDS.
// Same contract as scan_fused_kernel (src/smat/attention.py:134-192 and
// :446-453): segmented chunked scan with one reset at n, the long-range term
// Y added to recent rows, division by the normaliser column, optional gate; or
// H itself.  The description below is of r = 128, eight waves; r = 16 NW takes
// NW waves and NW column tiles, rows of eight chunks and two buffers at r = 64.
//
//   * One workgroup of eight waves walks one group of chunks; the group's
//     incoming state comes from the same prepass (Gram sums per group, shifted
//     exclusive scan over groups) as scan_fused_kernel.
//   * Tokens advance 64 per step.  The Phi, Psi and Vb rows of the next step
//     are copied HBM -> LDS by global_load_lds_dwordx4 while the current step
//     computes: double-buffered, no registers and no VALU spent on staging.
//   * Wave w owns value columns 16w .. 16w+15.  It keeps S[:, cols] (128 x 16,
//     fp32) in MFMA accumulators and produces the transposed output
//         O^T[cols][t] = S^T Phi^T + Vb^T A^T ,
//     because (k-slot bijection) the accumulator tiles of S[a][c], split into
//     hi + lo 16-bit parts, are exactly the A operand of S^T Phi^T -- S never
//     goes through LDS -- and the O^T accumulator layout gives each lane four
//     consecutive columns of one row: 16-byte output stores.
//   * Columns 128..143 (the normaliser column and padding) are a ninth
//     column tile whose state every wave keeps; waves 0..3 each produce the
//     normaliser of one 16-row tile and share it through LDS.
//   * The within-step scores A^T = Psi Phi^T (the causal 16 x 16 tiles of the
//     64 x 64 block) are computed once, split over the waves, masked, rounded
//     to the input dtype as the reference does, and shared through LDS.
//   * Psi and Vb feed the MFMAs along the token axis through the gfx950
//     transposing LDS read ds_read_b64_tr_b16: within each 16-lane group,
//     lane i receives element (i & 3) of the 8 bytes addressed by lane
//     4j + (i >> 2) as its element j.
//
// LDS layout.  The LDS has 64 banks of 4 bytes.  A 16-byte read is served
// in four phases of 16 lanes: lanes 32h + 4j .. 32h + 4j + 3 go in phase
// (h, parity of j) for j = 0..7.  An 8-byte read, transposing or not, is
// served in two phases of 32 consecutive lanes.  A phase is conflict-free
// when its lanes' bytes fall in distinct banks (lanes reading the same
// address share the access).  Phi, Psi and Vb columns 0..127 are tiles of
// 64 rows of 256 bytes (sixteen 16-byte chunks); chunk k of row t is stored
// at slot k ^ swz16(t).  That one XOR satisfies all three reads of a tile: a
// row-wise 16-byte fragment read (16 rows, chunk 4 kk + lane/16), a
// row-wise 8-byte read (16 rows x 2 halves), and a transposing read (8 rows
// x 2 chunks x 2 halves).  Vb columns 128..135 (the normaliser column and
// padding) are a separate tile of 64 rows of 16 bytes.  The score share is
// 64 rows of 128 bytes with chunk k of row t at k ^ swz8(t).  The normaliser
// partials are 64 rows of 32 bytes whose two halves swap in rows 8..15 of
// every 16, so a phase's 16 rows cover the 256 bytes of the banks once.
#include <stdlib.h>

#include <type_traits>

#include "feat_map.hpp"
#include "smat_host.hpp"

namespace smat {

namespace ss {
constexpr int kStep = 64;                      // tokens per step
constexpr int kRowChunks = 16;                 // 16-byte chunks per LDS row of the Gram sums
constexpr int kTileChunks = kStep * kRowChunks;    // 1024
constexpr int kVbTileChunks = kTileChunks + kStep; // + the normaliser chunk of each row
constexpr int kPhiLoads = kTileChunks / 64;        // wave-wide DMA loads per tile: 16
constexpr int kVbLoads = kVbTileChunks / 64;       // 17

// The scan at r = 16 NW features: NW waves, one 16-column tile of Vb each.
// LDS rows hold 16 chunks of 16 bytes (r > 64, of which 2 NW are used) or 8.
// kLoads wave-wide copies bring a step's rows (Phi, Psi, Vb and Vb's
// normaliser chunks); copy I goes to wave I % NW, so wave w issues kBase of
// them, one more for w < kExtra.  Three row buffers at r > 64 (a workgroup a
// CU); two at r = 64, whose 59 KB let two workgroups share a CU.
template <int NW, bool FEAT>
struct Scan {
  static constexpr int kThreads = 64 * NW;
  static constexpr int kRC = NW > 4 ? 16 : 8;
  static constexpr int kTile = kStep * kRC;
  static constexpr int kVbTile = kTile + kStep;
  static constexpr int kLoads = 3 * kRC + (FEAT ? 0 : 1);
  static constexpr int kBase = kLoads / NW, kExtra = kLoads % NW;
  static constexpr int kSlots = (kLoads + NW - 1) / NW;
  static constexpr int kBufs = NW > 4 ? 3 : 2;
};
}  // namespace ss

#define SMAT_LDS __attribute__((address_space(3)))
typedef short short4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int swz16(int t) {
  return (((t & 7) << 1) | ((t >> 3) & 1)) ^ (t & 8);
}
__device__ __forceinline__ int swz8(int t) { return (t >> 1) & 7; }
// The same for rows of eight chunks (r = 64): t's bits 2, 1, 3, so that the
// even (and the odd) rows of a phase of any of the three reads take distinct
// slots beside their neighbours' half of the banks.
template <int RC>
__device__ __forceinline__ int swz_row(int t) {
  return RC == 16 ? swz16(t) : ((t >> 2) & 1) | (t & 2) | ((t >> 1) & 4);
}
// Float index of wave w's normaliser partial of row t: 8 floats a row, the two
// 4-float halves swapped in rows 8..15 of every 16.
__device__ __forceinline__ int norm_slot(int t, int w) {
  return t * 8 + 4 * ((w >> 2) ^ ((t >> 3) & 1)) + (w & 3);
}

// Global loads the compiler does not track: their values may be used only
// after a wait_vmcnt that covers them and an opaque redefinition (asm "+v"),
// so no compiler-placed wait -- which would be vmcnt(0) with DMA loads and
// stores pending beside them -- drains the DMA issued after them.  "memory"
// keeps them in program order with the DMA, which the counts rely on.
__device__ __forceinline__ f32x4 load4_untracked(const void* p) {
  f32x4 v;
  asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(v) : "v"(p) : "memory");
  return v;
}
__device__ __forceinline__ float load1_untracked(const void* p) {
  float v;
  asm volatile("global_load_dword %0, %1, off" : "=&v"(v) : "v"(p) : "memory");
  return v;
}
// A 16-bit element, zero-extended into a 32-bit register, untracked likewise.
__device__ __forceinline__ uint32_t load_u16_untracked(const void* p) {
  uint32_t v;
  asm volatile("global_load_ushort %0, %1, off" : "=&v"(v) : "v"(p) : "memory");
  return v;
}

// 8 bytes of a swizzled row of RC chunks (t, chunk k, half h).
template <typename In, int RC>
__device__ __forceinline__ typename Traits<In>::half_frag row_half(const uint4* tile, int t, int k,
                                                                    int h) {
  const char* p = reinterpret_cast<const char*>(tile + t * RC + (k ^ swz_row<RC>(t))) + 8 * h;
  return *reinterpret_cast<const typename Traits<In>::half_frag*>(p);
}
// 16 bytes (one chunk) of a swizzled row.
template <typename In, int RC>
__device__ __forceinline__ typename Traits<In>::frag row_chunk(const uint4* tile, int t, int k) {
  return *reinterpret_cast<const typename Traits<In>::frag*>(tile + t * RC + (k ^ swz_row<RC>(t)));
}

// The state's hi and lo parts.  WIDE, in fp16: hi ends at the largest value and lo
// holds what is left.  The state is read every 64 tokens, so a segment's last state
// sums 64 tokens more than the general kernel's last one does, and a sum that fits
// there up to 65504 may pass that here (rounded then, up to twice it, to 2^-12 of
// it).  One instruction a value, 3 % of a pass over 128 features.
template <typename In, bool WIDE>
__device__ __forceinline__ void split_state(const f32x4& x, typename Traits<In>::half_frag& hi,
                                            typename Traits<In>::half_frag& lo) {
  if constexpr (WIDE && __is_same(In, f16)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      hi[i] = from_f32<f16>(__builtin_amdgcn_fmed3f(x[i], -65504.f, 65504.f));
      lo[i] = from_f32<f16>(x[i] - to_f32(hi[i]));
    }
  } else {
    split4<In>(x, hi, lo);
  }
}

template <typename In>
__device__ __forceinline__ typename Traits<In>::half_frag tr_read(const char* addr) {
  short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (SMAT_LDS short4v*)(SMAT_LDS char*)(addr));
  return __builtin_bit_cast(typename Traits<In>::half_frag, v);
}

template <typename In>
__device__ __forceinline__ typename Traits<In>::frag join(typename Traits<In>::half_frag lo,
                                                          typename Traits<In>::half_frag hi) {
  typename Traits<In>::frag f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[j] = lo[j];
    f[4 + j] = hi[j];
  }
  return f;
}

// A fragment of Psi^T (rows a = 16*at + lane%16, k-slots = tokens
// 32*ks + 8*grp + j) from a swizzled Psi tile, by two transposing reads.
template <typename In, int RC = ss::kRowChunks>
__device__ __forceinline__ typename Traits<In>::frag psi_tr(const uint4* tile, int at, int ks,
                                                            int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  typename Traits<In>::half_frag h2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 32 * ks + 8 * g + 4 * h + (r16 >> 2);
    const int k = 2 * at + ((r16 & 3) >> 1);
    const char* p =
        reinterpret_cast<const char*>(tile + row * RC + (k ^ swz_row<RC>(row))) + 8 * (r16 & 1);
    h2[h] = tr_read<In>(p);
  }
  return join<In>(h2[0], h2[1]);
}

// The normaliser tile of Vb along tokens (column d_v + lane%16, k-slots =
// tokens 32*ks + 8*grp + j) from the 16-byte rows of columns d_v .. d_v + 7 after
// the tile: the ones column and seven columns of padding; lanes 8..15 repeat
// them in place of columns no caller keeps.
template <typename In, int RC = ss::kRowChunks>
__device__ __forceinline__ typename Traits<In>::frag vb_norm_tr(const uint4* tile, int ks,
                                                                int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  typename Traits<In>::half_frag h2[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 32 * ks + 8 * g + 4 * h + (r16 >> 2);
    const char* p = reinterpret_cast<const char*>(tile + ss::kStep * RC + row) + 8 * (r16 & 1);
    h2[h] = tr_read<In>(p);
  }
  return join<In>(h2[0], h2[1]);
}

// The DMA of one step's Phi, Psi and Vb rows [ts, ts + 64) into one buffer.
// Copy I of the kLoads goes to wave I % NW as its slot u = I / NW: kRC copies of
// Phi, of Psi, of Vb's columns below r, then (not FEAT) one of the normaliser
// chunks, lane = row.  Each moves 64 x 16 bytes to 1 KB of consecutive LDS;
// which global chunk a lane fetches implements the swizzle (chunks past the
// row's 2 NW re-read one of its own).  That choice does not depend on the
// step, so a lane's byte offset from the step's first row is computed once per
// slot; a step adds it to the wave-uniform row base of the slot's tensor.
template <int NW, bool FEAT>
struct DmaOffsets {
  uint32_t off[ss::Scan<NW, FEAT>::kSlots];
};

// Which tensor copy NW u + w belongs to (0 Phi, 1 Psi, 2 Vb): known at compile
// time unless the slot's copies straddle two tensors.
template <int NW, int RC>
__device__ __forceinline__ int dma_tensor(int u, int w) {
  const int lo = NW * u, hi = NW * u + NW - 1;
  if (hi < RC) return 0;
  if (lo >= RC && hi < 2 * RC) return 1;
  if (lo >= 2 * RC) return 2;
  const int I = NW * u + w;
  return I < RC ? 0 : I < 2 * RC ? 1 : 2;
}

// last: the last row to fetch (rows past it re-read it).
template <typename In, int NW, bool FEAT>
__device__ __forceinline__ uint32_t dma_offset(const ScanArgs& a, int u, int w, int lane,
                                               int last) {
  typedef ss::Scan<NW, FEAT> Sh;
  constexpr int RC = Sh::kRC;
  const int I = w + NW * u;
  if (I >= 3 * RC)                                   // the normaliser chunk of row = lane
    return (uint32_t)(((int64_t)min(lane, last) * a.v_st + 16 * NW) * (int64_t)sizeof(In));
  const int t = dma_tensor<NW, RC>(u, w);
  const int row = (64 / RC) * (I - t * RC) + lane / RC;
  int k = (lane % RC) ^ swz_row<RC>(row);
  if (2 * NW < RC && k >= 2 * NW) k -= 8;
  const int64_t st = t == 0 ? a.q_st : t == 1 ? a.k_st : a.v_st;
  return (uint32_t)((min(row, last) * st + 8 * k) * (int64_t)sizeof(In));
}

// FEAT: the rows are Q, Psi and V (the feature map runs in LDS afterwards), and
// the normaliser tile is the constant [1, 0, ...] written once.  RAG: T is not a
// multiple of 64, and the step that crosses it fetches row T - 1 in place of
// rows past it.
template <typename In, int NW, bool FEAT, bool RAG>
__device__ __forceinline__ void issue_step(uint4* dphi, uint4* dpsi, uint4* dvb, const In* phib,
                                           const In* psib, const In* vbb, int64_t ts,
                                           const ScanArgs& a, int w, int lane,
                                           const DmaOffsets<NW, FEAT>& d) {
  typedef ss::Scan<NW, FEAT> Sh;
  constexpr int RC = Sh::kRC;
  const char* bphi = reinterpret_cast<const char*>(phib + ts * a.q_st);
  const char* bpsi = reinterpret_cast<const char*>(psib + ts * a.k_st);
  const char* bvb = reinterpret_cast<const char*>(vbb + ts * a.v_st);
  const int last = (int)min<int64_t>(ss::kStep, a.T - ts) - 1;
#pragma unroll
  for (int u = 0; u < Sh::kSlots; ++u) {
    const int I = w + NW * u;
    if (I < Sh::kLoads) {
      const int t = dma_tensor<NW, RC>(u, w);
      const char* base = t == 0 ? bphi : t == 1 ? bpsi : bvb;
      uint4* dst = t == 0 ? dphi : t == 1 ? dpsi : dvb;
      const uint32_t off = RAG && last < ss::kStep - 1
                               ? dma_offset<In, NW, FEAT>(a, u, w, lane, last)
                               : d.off[u];
      lds_dma16<true>(reinterpret_cast<const void*>(base + off), dst + 64 * (I - t * RC));
    }
  }
}

// Per-lane byte offsets of the step's Y and output rows from row ts (the
// lane's rows 16 tt + lane % 16 at columns 16 w + 4 g), computed once; a step
// adds them to wave-uniform row bases.  y8 is the normaliser column's offset
// from the lane's Y chunk.
struct RowOffsets {
  uint32_t y[4], o[4];
  int y8;
};

__device__ __forceinline__ void row_offsets(RowOffsets& R, const ScanArgs& a, int w, int lane) {
  const int r16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    R.y[tt] = (uint32_t)(((int64_t)(16 * tt + r16) * a.y_st + 16 * w + 4 * g) * 4);
    R.o[tt] = (uint32_t)(((int64_t)(16 * tt + r16) * a.o_st + 16 * w + 4 * g) * 4);
  }
  R.y8 = (a.p - 1 - 16 * w - 4 * g) * 4;
}

__device__ __forceinline__ f32x4 mma16(f32x4 c, bf16x4 a, bf16x4 b) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a),
                                                   __builtin_bit_cast(s4, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma16(f32x4 c, f16x4 a, f16x4 b) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

// The step's Y rows, its normaliser column and gates in registers, loaded
// untracked (used after a wait that covers them).
struct YRegs {
  f32x4 y[4];      // Y[t][16w + 4g .. +3] for the step's four row tiles
  float y8[4];     // Y[t][p - 1]
  float gv[4];     // gate
};

// NW: r = 16 NW features, p = 16 NW + 1.  FEAT (NW = 8): phi, psi and vb are Q,
// Psi (formed by the prepass, gate applied) and V rows; Phi is formed in place
// over the copied Q tile.  TERMS = false compiles Y and the gate out (launches
// with neither): their pointers and flags would otherwise spill scalar
// registers every step.  RAG: T is not a multiple of 64.  WH: out is H
// (unnormalised, p columns, rows of any alignment).
//
// What bounds it: HBM at r = 128 (4.6 TB/s).  At r = 64 .. 112 it took the place
// of the general kernel, which stages rows through registers into two LDS
// layouts and stores 4-byte elements: forward of 32 x 8192 tokens at r = 64
// 164 -> 119 us, of 12 x 10007 (ragged) at r = 96 403 -> 317 us, the positional
// training step's (H, r = 64) 1825 -> 1766 us.
template <typename In, int NW, bool FEAT, bool TERMS, bool RAG, bool WH>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void scan_stream_kernel(
    const In* __restrict__ phi, const In* __restrict__ psi, const In* __restrict__ vb,
    const float* __restrict__ Sg, const float* __restrict__ Y, const float* __restrict__ gate,
    float* __restrict__ out, ScanArgs a, FeatArgs fa) {
  using namespace ss;
  typedef Scan<NW, FEAT> Sh;
  typedef typename Traits<In>::frag Frag;
  typedef typename Traits<In>::half_frag Half;
  constexpr int RC = Sh::kRC, NBUF = Sh::kBufs, NKB = NW / 2;
  // An odd NW's last 16 features are a k-block whose other half is zero, on the
  // same MFMA as the others: a chain that went on from the 16 x 16 x 32 form to
  // the 16 x 16 x 16 one lost terms of its accumulator (seen on gfx950).
  constexpr bool kOdd = NW % 2 != 0;
  constexpr int kSteps = NKB + (kOdd ? 1 : 0);
  constexpr int kBase = Sh::kBase, kExtra = Sh::kExtra;
  // The shape that has always streamed.  The others took the general kernel's place
  // and keep its range: the whole division, and in fp16 the states it never forms.
  constexpr bool kFirst = NW == 8 && !RAG;
  static_assert(!FEAT || (NW == 8 && !RAG && !WH), "the feature map is 128 x 128");
  static_assert(!(WH && TERMS), "H carries no Y and no gate");
  __shared__ __attribute__((aligned(16))) uint4 phi0[Sh::kTile];
  __shared__ __attribute__((aligned(16))) uint4 psi0[Sh::kTile];
  __shared__ __attribute__((aligned(16))) uint4 vb0[Sh::kVbTile];
  __shared__ __attribute__((aligned(16))) uint4 phi1[Sh::kTile];
  __shared__ __attribute__((aligned(16))) uint4 psi1[Sh::kTile];
  __shared__ __attribute__((aligned(16))) uint4 vb1[Sh::kVbTile];
  // Three buffers (160 768 bytes of LDS in all) keep the rows of steps s + 1
  // and s + 2 in flight while step s computes; with two, step s + 2's copy is
  // issued once every wave is past step s's rows.  Y and
  // the gate are loaded untracked and waited for by count.
  __shared__ __attribute__((aligned(16))) uint4 phi2[NBUF == 3 ? Sh::kTile : 1];
  __shared__ __attribute__((aligned(16))) uint4 psi2[NBUF == 3 ? Sh::kTile : 1];
  __shared__ __attribute__((aligned(16))) uint4 vb2[NBUF == 3 ? Sh::kVbTile : 1];
  __shared__ __attribute__((aligned(16))) uint4 share[kStep * 8];
  // normaliser partials: wave w's share of H[t][p-1] at normp[norm_slot(t, w)]
  __shared__ __attribute__((aligned(16))) float normp[kStep * 8];

  // Groups run last sequence first, last group first: the prepass just read
  // the same Psi and Vb rows in the opposite order, so the first groups here
  // find theirs in the memory-side cache (556 -> 531 us for the causal pass
  // at 8 x 131072 tokens).
  const int grp = gridDim.x - 1 - blockIdx.x;
  const int64_t b = gridDim.y - 1 - blockIdx.y;
  // The wave index in a scalar register: every condition on it below is a
  // scalar branch.  (Under a vector condition the compiler masks EXEC around
  // an MFMA without branching past it, and MFMAs execute regardless of EXEC.)
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  __builtin_assume(w >= 0 && w < NW);
  const int lane = lane_id();
  const int r16 = lane & 15, g = lane >> 4;

  int c0, c1;
  if (grp < a.ng0) {
    c0 = grp * a.K;
    c1 = min(c0 + a.K, a.nc0);
  } else {
    c0 = a.nc0 + (grp - a.ng0) * a.K;
    c1 = min(c0 + a.K, a.nc);
  }
  const int64_t tk0 = (int64_t)c0 * a.C;
  const int64_t tk1 = min((int64_t)c1 * a.C, (int64_t)a.T);
  const int nsteps = (int)((tk1 - tk0 + (RAG ? kStep - 1 : 0)) / kStep);

  const In* phib = phi + b * a.q_sb;
  const In* psib = psi + b * a.k_sb;
  const In* vbb = vb + b * a.v_sb;
  const float* Yb = (TERMS && Y) ? Y + b * a.y_sb : nullptr;
  const float* gb = (TERMS && gate) ? gate + b * a.g_sb : nullptr;
  float* outb = out + b * a.o_sb;
  const float* Sb = Sg + ((int64_t)b * gridDim.x + grp) * (int64_t)(16 * NW) * a.p;

  DmaOffsets<NW, FEAT> dmo;
#pragma unroll
  for (int u = 0; u < Sh::kSlots; ++u)
    dmo.off[u] = w + NW * u < Sh::kLoads ? dma_offset<In, NW, FEAT>(a, u, w, lane, kStep - 1) : 0;
  RowOffsets rof;
  row_offsets(rof, a, w, lane);
  if (nsteps > 0)
    issue_step<In, NW, FEAT, RAG>(phi0, psi0, vb0, phib, psib, vbb, tk0, a, w, lane, dmo);
  Frag wa[4];
  if constexpr (FEAT) {
    feat_w_load<In>(wa, (const In*)fa.W, w, lane);
    feat_ones_tile<In>(vb0 + Sh::kTile, threadIdx.x, Sh::kThreads);
    feat_ones_tile<In>(vb1 + Sh::kTile, threadIdx.x, Sh::kThreads);
    feat_ones_tile<In>(vb2 + Sh::kTile, threadIdx.x, Sh::kThreads);
  }
  // The score tiles (1, 0) and (3, 2) stay zero, and so do the normaliser
  // partials of waves that do not exist (published by step 0's first barrier).
  for (int e = threadIdx.x; e < kStep * 8; e += Sh::kThreads) {
    share[e] = make_uint4(0, 0, 0, 0);
    normp[e] = 0.f;
  }

  // incoming state: S[a][16w + lane%16] for all a, and the normaliser column
  // S[a][16 NW] (in lanes % 16 = 0) for this wave's rows a in [16w, 16w + 16)
  f32x4 accS[NW], accS8;
#pragma unroll
  for (int at = 0; at < NW; ++at)
#pragma unroll
    for (int i = 0; i < 4; ++i) accS[at][i] = Sb[(int64_t)(16 * at + 4 * g + i) * a.p + 16 * w + r16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float v8 = Sb[(int64_t)(16 * w + 4 * g + i) * a.p + (r16 == 0 ? 16 * NW : 0)];
    accS8[i] = r16 == 0 ? v8 : 0.f;
  }
  // Consume the state (and W) loads here, so that no wait for them is placed
  // inside the loop.  The copies are untracked and the compiler's wait here is
  // vmcnt(0), which lands step 0's rows too; step 1's copy goes out after it.
#pragma unroll
  for (int at = 0; at < NW; ++at) asm volatile("" : "+v"(accS[at]));
  asm volatile("" : "+v"(accS8));
  if constexpr (FEAT) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) asm volatile("" : "+v"(wa[kb]));
  }

  // Rows of the step at ts that exist (all 64 except across a ragged T).
  auto rows_left = [&](int64_t ts) { return RAG ? (int)min<int64_t>(kStep, a.T - ts) : kStep; };
  // The Y rows and gates of the step at ts (rows past a ragged T re-read row
  // T - 1's).
  auto issue_y = [&](YRegs& R, int64_t ts) {
    const bool rec = Yb != nullptr && ts >= a.n;
    const int left = rows_left(ts);
    if (rec) {
      const char* yb = reinterpret_cast<const char*>(Yb + (ts - a.n) * a.y_st);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        uint32_t off = rof.y[tt];
        if (RAG && left < kStep)
          off = (uint32_t)((min(16 * tt + r16, left - 1) * a.y_st + 16 * w + 4 * g) * 4);
        R.y[tt] = load4_untracked(yb + off);
        R.y8[tt] = load1_untracked(yb + off + rof.y8);
      }
    }
    if (gb) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const int t = RAG ? min(16 * tt + r16, left - 1) : 16 * tt + r16;
        R.gv[tt] = load1_untracked(gb + ts + t);
      }
    }
  };
  // Until only the step's copy issued last is outstanding (its count differs by
  // one between the waves), or nothing when none was issued.
  auto wait_dma = [&](bool issued) {
    if (!issued)
      wait_vmcnt<0>();
    else if (w < kExtra)
      wait_vmcnt<kBase + 1>();
    else
      wait_vmcnt<kBase>();
  };
  if constexpr (NBUF == 2) wait_vmcnt<0>();
  if (nsteps > 1)
    issue_step<In, NW, FEAT, RAG>(phi1, psi1, vb1, phib, psib, vbb, tk0 + kStep, a, w, lane, dmo);

  auto step = [&](auto BUFC, int s) {
    constexpr int BUF = decltype(BUFC)::value;
    const uint4* tphi = BUF == 2 ? phi2 : BUF ? phi1 : phi0;
    const uint4* tpsi = BUF == 2 ? psi2 : BUF ? psi1 : psi0;
    const uint4* tvb = BUF == 2 ? vb2 : BUF ? vb1 : vb0;
    const int64_t ts = tk0 + (int64_t)s * kStep;
    // An opaque copy of the lane index per step: the LDS addresses derived
    // from it are recomputed inside the step instead of being hoisted out of
    // the loop, where the ~60 distinct swizzled addresses would pin as many
    // registers for the whole kernel.
    int lane = lane_id();
    asm volatile("" : "+v"(lane));
    const int r16 = lane & 15, g = lane >> 4;
    // Loads complete in order, so waiting until only the next step's copy is
    // outstanding lands this step's.  (Two buffers: the previous step's (e), or
    // the prologue, has waited for it.)
    if constexpr (NBUF == 3) wait_dma(s + 1 < nsteps);
    lds_barrier();      // every wave's DMA of this step has landed
    if constexpr (FEAT) {
      // in place: feat_rows reads every wave's rows, then waits, then writes
      const float none[4] = {1.f, 1.f, 1.f, 1.f};
      const auto sw = [](int t) { return swz16(t); };
      uint4* tq = BUF == 2 ? phi2 : BUF ? phi1 : phi0;
      feat_rows<In, 4>(tq, tq, 0, true, wa, w, fa.kind, false, none, lane, sw);
      lds_barrier();    // the step's Phi tile is complete
    }
    // The step's Y rows and gates; the only vector memory issued after them
    // before (e) is the DMA of step s + 2.
    const bool rec = Yb != nullptr && ts >= a.n;
    YRegs yr;
    if constexpr (TERMS) issue_y(yr, ts);

    // (a) this wave's share of the causal score tiles A^T = Psi Phi^T
    //     entries 0..9: (ut, tt) with ut <= tt.  Wave w takes entries w, w + NW,
    //     ...; the fragments of its (up to three) products are read first and
    //     their MFMA chains interleave.
    {
      auto entry = [](int e, int& ut, int& tt) {
        tt = e < 1 ? 0 : e < 3 ? 1 : e < 6 ? 2 : 3;
        ut = e - (tt * (tt + 1)) / 2;
      };
      // acc[i] = A^T[t' = 16ut + 4g + i][t = 16tt + r16] = A[t][t'], masked,
      // rounded to the input type and stored to the share
      auto put = [&](const f32x4& acc, int ut, int tt) {
        Half hv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool keep = ut < tt || 4 * g + i <= r16;
          hv[i] = from_f32<In>(keep ? acc[i] : 0.f);
        }
        const int t = 16 * tt + r16;
        const int k = 2 * ut + (g >> 1);
        char* p = reinterpret_cast<char*>(share + t * 8 + (k ^ swz8(t))) + 8 * (g & 1);
        *reinterpret_cast<Half*>(p) = hv;
      };
      struct Prod {
        Frag fa[kSteps], fb[kSteps];
        int ut, tt;
      };
      auto read = [&](Prod& q, int e) {
        entry(e, q.ut, q.tt);
#pragma unroll
        for (int kk = 0; kk < NKB; ++kk) {
          q.fa[kk] = row_chunk<In, RC>(tpsi, 16 * q.ut + r16, 4 * kk + g);
          q.fb[kk] = row_chunk<In, RC>(tphi, 16 * q.tt + r16, 4 * kk + g);
        }
        if constexpr (kOdd) {
          const int kl = 2 * (NW - 1) + (g >> 1);
          q.fa[NKB] = join<In>(row_half<In, RC>(tpsi, 16 * q.ut + r16, kl, g & 1), Half{});
          q.fb[NKB] = join<In>(row_half<In, RC>(tphi, 16 * q.tt + r16, kl, g & 1), Half{});
        }
      };
      auto mul = [&](f32x4& acc, const Prod& q, int kk) { acc = mma(acc, q.fa[kk], q.fb[kk]); };
      constexpr int kMax = (10 + NW - 1) / NW;       // products a wave: at most 2 or 3
      // wave w has kMax products if w + NW (kMax - 1) < 10, else one fewer
      Prod q0, q1, q2;
      f32x4 s0 = zero4(), s1 = zero4(), s2 = zero4();
      read(q0, w);
      if constexpr (kMax == 3) read(q1, w + NW);
      if (w + NW * (kMax - 1) < 10) {
        if constexpr (kMax == 3)
          read(q2, w + 2 * NW);
        else
          read(q1, w + NW);
#pragma unroll
        for (int kk = 0; kk < kSteps; ++kk) {
          mul(s0, q0, kk);
          mul(s1, q1, kk);
          if constexpr (kMax == 3) mul(s2, q2, kk);
        }
        put(s1, q1.ut, q1.tt);
        if constexpr (kMax == 3) put(s2, q2.ut, q2.tt);
      } else {
#pragma unroll
        for (int kk = 0; kk < kSteps; ++kk) {
          mul(s0, q0, kk);
          if constexpr (kMax == 3) mul(s1, q1, kk);
        }
        if constexpr (kMax == 3) put(s1, q1.ut, q1.tt);
      }
      put(s0, q0.ut, q0.tt);
    }

    // Three buffers: step s + 2's rows go to the buffer step s - 1 used, free
    // since that step's last barrier.  Issued after the score reads: before
    // them, the compiler waits for the whole DMA in one of the three steps.
    if constexpr (NBUF == 3) {
      constexpr int NB = (BUF + 2) % 3;
      if (s + 2 < nsteps)
        issue_step<In, NW, FEAT, RAG>(NB == 2 ? phi2 : NB ? phi1 : phi0,
                                      NB == 2 ? psi2 : NB ? psi1 : psi0,
                                      NB == 2 ? vb2 : NB ? vb1 : vb0, phib, psib, vbb,
                                      ts + 2 * kStep, a, w, lane, dmo);
    }

    // (b) O^T = S^T Phi^T with the state before this step; the normaliser
    //     column's share of this wave's 16 state rows
    f32x4 accO[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) accO[tt] = zero4();
    // Row t = 16 tt + r16 of the Phi tile, one opaque base per tt.  Rows t and
    // t + 16 sit at the same swizzle a constant apart; seen as such, their two
    // 8-byte reads are fused into one ds_read2st64_b64, which the LDS serves at
    // half the rate of two ds_read_b64 and with this pattern's lanes in
    // conflict.  With opaque bases every read stays a ds_read_b64.
    const char* prow[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      uint32_t off = (uint32_t)(16 * tt + r16) * (RC * 16);
      asm volatile("" : "+v"(off));
      prow[tt] = reinterpret_cast<const char*>(tphi) + off;
    }
    const int sw = swz_row<RC>(r16);
    auto phi_half = [&](int tt, int k) {
      return *reinterpret_cast<const Half*>(prow[tt] + ((k ^ sw) * 16 + 8 * (g & 1)));
    };
    // The Phi fragments of k-block kk + 1 are read while block kk's state is
    // split and multiplied, and the hi parts of the four row tiles go before
    // the lo parts, so no MFMA waits on the one before it.
    Frag bfs[2][4];
    auto read_bf = [&](Frag(&dst)[4], int kk) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        dst[tt] = join<In>(phi_half(tt, 4 * kk + (g >> 1)), phi_half(tt, 4 * kk + 2 + (g >> 1)));
    };
    read_bf(bfs[0], 0);
#pragma unroll
    for (int kk = 0; kk < NKB; ++kk) {
      if (kk + 1 < NKB) read_bf(bfs[(kk + 1) & 1], kk + 1);
      Half h0, l0, h1, l1;
      split_state<In, !kFirst>(accS[2 * kk], h0, l0);
      split_state<In, !kFirst>(accS[2 * kk + 1], h1, l1);
      const Frag shi = join<In>(h0, h1), slo = join<In>(l0, l1);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) accO[tt] = mma(accO[tt], shi, bfs[kk & 1][tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) accO[tt] = mma(accO[tt], slo, bfs[kk & 1][tt]);
    }
    if constexpr (kOdd) {
      Half hi, lo;
      Frag bh[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        bh[tt] = join<In>(phi_half(tt, 2 * (NW - 1) + (g >> 1)), Half{});
      split_state<In, !kFirst>(accS[NW - 1], hi, lo);
      const Frag shi = join<In>(hi, Half{}), slo = join<In>(lo, Half{});
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) accO[tt] = mma(accO[tt], shi, bh[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) accO[tt] = mma(accO[tt], slo, bh[tt]);
    }
    float own = 0.f;                       // wave w < 4: its row tile's value, finished in (d)
    {
      Half s8hi, s8lo, bfn[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) bfn[tt] = phi_half(tt, 2 * w + (g >> 1));
      split_state<In, !kFirst>(accS8, s8hi, s8lo);
      f32x4 pn[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) pn[tt] = mma16(zero4(), s8hi, bfn[tt]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) pn[tt] = mma16(pn[tt], s8lo, bfn[tt]);
      if (g == 0) {                        // the normaliser's row of the tile: 0
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          if (tt == w)
            own = pn[tt][0];
          else
            normp[norm_slot(16 * tt + r16, w)] = pn[tt][0];
        }
      }
    }

    // (c) S += Psi^T Vb over the step's 64 tokens
    // The normaliser tile's rows of this wave take the Psi fragment of row tile
    // w once more, outside the loop: a branch on at == w inside it would split
    // the loop into blocks the compiler cannot move a read across.
    // The (ks, at) products run in order with the Psi fragments of the next two
    // read ahead (sched barriers keep the compiler from sinking the reads to
    // their MFMAs).
    Frag vbw[2], vb8[2], pa[3];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      vbw[ks] = psi_tr<In, RC>(tvb, w, ks, lane);
      vb8[ks] = vb_norm_tr<In, RC>(tvb, ks, lane);
    }
    pa[0] = psi_tr<In, RC>(tpsi, 0, 0, lane);
    pa[1] = psi_tr<In, RC>(tpsi, 1, 0, lane);
#pragma unroll
    for (int i = 0; i < 2 * NW; ++i) {
      if (i + 2 < 2 * NW)
        pa[(i + 2) % 3] = psi_tr<In, RC>(tpsi, (i + 2) % NW, (i + 2) / NW, lane);
      __builtin_amdgcn_sched_barrier(0);
      accS[i % NW] = mma(accS[i % NW], pa[i % 3], vbw[i / NW]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) accS8 = mma(accS8, psi_tr<In, RC>(tpsi, w, ks, lane), vb8[ks]);
    lds_barrier();       // the score share is complete
    // Two buffers: every wave is past its reads of this step's rows, so step
    // s + 2's go there, a whole step before (e) of step s + 1 waits for them.
    if constexpr (NBUF == 2) {
      if (s + 2 < nsteps)
        issue_step<In, NW, FEAT, RAG>(BUF ? phi1 : phi0, BUF ? psi1 : psi0, BUF ? vb1 : vb0, phib,
                                      psib, vbb, ts + 2 * kStep, a, w, lane, dmo);
    }

    // (d) O^T += Vb^T A^T within the step; waves 0..3 add the row sums of A
    //     (the ones column) to their row tile's normaliser
    auto share_bf = [&](int t, int ks) {
      return *reinterpret_cast<const Frag*>(share + t * 8 + ((4 * ks + g) ^ swz8(t)));
    };
    {
      Frag sh[4][2];    // the six causal score fragments, read before their MFMAs
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ks = 0; ks <= (tt >> 1); ++ks) sh[tt][ks] = share_bf(16 * tt + r16, ks);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int tt = 2 * ks; tt < 4; ++tt) accO[tt] = mma(accO[tt], vbw[ks], sh[tt][ks]);
    }
    if (w < 4) {        // row tile w's normaliser: the row sums of its score tiles
      const int t = 16 * w + r16;
      f32x4 p8 = mma(zero4(), vb8[0], share_bf(t, 0));
      if (w >= 2) p8 = mma(p8, vb8[1], share_bf(t, 1));
      if (g == 0) normp[norm_slot(t, w)] = own + p8[0];
    }
    lds_barrier();

    // (e) long-range term, normalise, store four columns per lane per row tile
    // Issued after the Y and gate loads: step s + 2's copy.  With two buffers
    // this wait also lands step s + 1's rows.
    if (NBUF == 2 || (TERMS && (rec || gb))) wait_dma(s + 2 < nsteps);
    if (TERMS && (rec || gb)) {
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
        asm volatile("" : "+v"(yr.y[tt]), "+v"(yr.y8[tt]), "+v"(yr.gv[tt]));
    }
    const int left = rows_left(ts);
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      const int t = 16 * tt + r16;
      const float4 n0 = *reinterpret_cast<const float4*>(normp + norm_slot(t, 0));
      float den = (n0.x + n0.y) + (n0.z + n0.w);
      if constexpr (NW > 4) {
        const float4 n1 = *reinterpret_cast<const float4*>(normp + norm_slot(t, 4));
        den += (n1.x + n1.y) + (n1.z + n1.w);
      }
      float4 o;
      o.x = accO[tt][0];
      o.y = accO[tt][1];
      o.z = accO[tt][2];
      o.w = accO[tt][3];
      if constexpr (WH) {
        if (!RAG || t < left) {
          float* h = reinterpret_cast<float*>(reinterpret_cast<char*>(outb + ts * a.o_st) +
                                              rof.o[tt]);
          h[0] = o.x;
          h[1] = o.y;
          h[2] = o.z;
          h[3] = o.w;
          if (tt % NW == w && g == 0) outb[(ts + t) * a.o_st + 16 * NW] = den;
        }
        continue;
      }
      if (TERMS && rec) {
        den += yr.y8[tt];
        o.x += yr.y[tt][0];
        o.y += yr.y[tt][1];
        o.z += yr.y[tt][2];
        o.w += yr.y[tt][3];
      }
      // The gate (1 without) times the reciprocal (1 ulp, zero past 2^126) in place
      // of the IEEE division's ten instructions, or that division, the gate last.
      const float num = TERMS && gb ? yr.gv[tt] : 1.f;
      const float inv = kFirst ? num * __builtin_amdgcn_rcpf(den) : 1.f / den;
      o.x *= inv;
      o.y *= inv;
      o.z *= inv;
      o.w *= inv;
      if (!kFirst && TERMS && gb) {
        o.x *= num;
        o.y *= num;
        o.z *= num;
        o.w *= num;
      }
      if (!RAG || t < left)
        *reinterpret_cast<float4*>(reinterpret_cast<char*>(outb + ts * a.o_st) + rof.o[tt]) = o;
    }
  };

  if constexpr (NBUF == 3) {
    for (int s = 0; s < nsteps; s += 3) {
      step(std::integral_constant<int, 0>{}, s);
      if (s + 1 < nsteps) step(std::integral_constant<int, 1>{}, s + 1);
      if (s + 2 < nsteps) step(std::integral_constant<int, 2>{}, s + 2);
    }
  } else {
    for (int s = 0; s < nsteps; s += 2) {
      step(std::integral_constant<int, 0>{}, s);
      if (s + 1 < nsteps) step(std::integral_constant<int, 1>{}, s + 1);
    }
  }
}

// ---------------------------------------------------------------------------
// Gram sums G = sum_t Psi_t^T Vb_t over a token progression (the chunk-group
// prepass of the causal pass, and the profile pool), same machinery: rows
// of 64 tokens at a time copied HBM -> LDS by DMA (double-buffered), read
// along tokens by transposing LDS reads, wave w accumulating G[:, 16w ..
// 16w+15] and rows [16w, 16w+16) of the normaliser column's tile.  r = 16 NW
// takes NW waves, as in the scan.  Rows past the end of a progression are
// fetched from its first token (in bounds) and zeroed in the Vb fragment, so
// they add nothing.
// ---------------------------------------------------------------------------

// Issue one step's DMA: Psi (16 loads) and Vb (17) for rows
// tok(row) = start + stride * (base + row), row < 64, load I on wave I % NW
// (chunks past the row's 2 NW re-read one of its own).
// FEAT: K and V rows; the normaliser tile is constant, so 32 loads, four a wave.
// Token of term idx: LIST (mode 2) reads it from the item's column list; the
// other modes compute it, with no index loads whose waits (vmcnt(0), placed by
// the compiler at every join after them) would drain the DMA in flight.
template <bool LIST>
__device__ __forceinline__ int64_t gram_token_of(const GramItems& it, int item, int64_t start,
                                                 int64_t stride, int idx) {
  if constexpr (LIST)
    return gram_token(it, item, start, stride, idx);
  else
    return start + (int64_t)idx * stride;
}

template <typename In, int NW, bool FEAT, bool LIST>
__device__ __forceinline__ void issue_gram(uint4* dpsi, uint4* dvb, const In* psib,
                                           const In* vbb, const GramItems& it, int item,
                                           int64_t start, int64_t stride, int base, int count,
                                           int64_t k_st, int64_t v_st, int w, int lane) {
  constexpr int kL = ss::kPhiLoads + ss::kVbLoads - (FEAT ? 1 : 0);     // 33 or 32
  const auto chunk = [](int k) { return 2 * NW < ss::kRowChunks && k >= 2 * NW ? k - 8 : k; };
#pragma unroll
  for (int u = 0; u < (kL + NW - 1) / NW; ++u) {
    const int I = w + NW * u;
    if (I < kL) {
      const In* src;
      uint4* dst;
      if (I < ss::kPhiLoads) {
        const int row = 4 * I + (lane >> 4);
        const int k = chunk((lane & 15) ^ swz16(row));
        const int64_t tok =
            gram_token_of<LIST>(it, item, start, stride, base + row < count ? base + row : 0);
        src = psib + tok * k_st + 8 * k;
        dst = dpsi + 64 * I;
      } else {
        // Vb's value columns swizzled like Psi, then the normaliser chunks, lane = row
        const int li = I - ss::kPhiLoads;
        const int row = li < ss::kPhiLoads ? 4 * li + (lane >> 4) : lane;
        const int col = li < ss::kPhiLoads ? 8 * chunk((lane & 15) ^ swz16(row)) : 16 * NW;
        const int64_t tok =
            gram_token_of<LIST>(it, item, start, stride, base + row < count ? base + row : 0);
        src = vbb + tok * v_st + col;
        dst = dvb + 64 * li;
      }
      // untracked except with the list's token loads, whose own compiler
      // waits drain the copies anyway
      lds_dma16<!LIST>(reinterpret_cast<const void*>(src), dst);
    }
  }
}

// ONE: the profiles of the launch have at most kStep terms (the profile pool at
// long T: (n - n_P) / N0 tokens a profile), so one buffer suffices -- a global
// channel's few steps wait for their rows one by one.  Its
// 35 KB of LDS let three workgroups share a CU instead of two, which is what
// a launch of one-step items -- a load latency, a few MFMAs and a 66 KB
// store each -- is limited by.
// FEAT: psi and vb are K and V rows; each step's Psi tile is formed in place
// from the DMA'd K tile (feat_rows, W in registers, two halves of 32 rows),
// times the key gate.
template <typename In, int NW, bool ONE, bool FEAT, bool LIST>
__global__ __launch_bounds__(64 * NW, (ONE && !FEAT) ? 3 : 2) void gram_stream_kernel(
    const In* __restrict__ psi, const In* __restrict__ vb, float* __restrict__ G,
    float* __restrict__ G_last, GramItems it, int64_t k_sb, int64_t k_st, int64_t v_sb,
    int64_t v_st, int64_t g_sb, int64_t g_si, int64_t gl_sb, FeatArgs fa) {
  using namespace ss;
  typedef typename Traits<In>::frag Frag;
  constexpr int kThreads = 64 * NW;
  constexpr int kP = 16 * NW + 1;                    // = p
  constexpr int kL = kPhiLoads + kVbLoads - (FEAT ? 1 : 0);
  static_assert(!FEAT || NW == 8, "the feature map is 128 x 128");
  static_assert(!(ONE && LIST), "a list's length is not known to the launch");
  // psi0 and vb0 are one array: after the last step it stages the output
  __shared__ __attribute__((aligned(16))) uint4 stage0[kTileChunks + kVbTileChunks];
  static_assert((kTileChunks + kVbTileChunks) * 16 >= 64 * kP * 4, "stage holds 64 rows of G");
  uint4* psi0 = stage0;
  uint4* vb0 = stage0 + kTileChunks;
  __shared__ __attribute__((aligned(16))) uint4 psi1[ONE ? 1 : kTileChunks];
  __shared__ __attribute__((aligned(16))) uint4 vb1[ONE ? 1 : kVbTileChunks];

  // Profiles (mode 1) run point by point across the sequences, so the last
  // rows of F written -- the ones the memory-side cache still holds when the
  // incidence starts -- are spread over all sequences, whose slices the
  // incidence walks on separate XCDs.
  int item = blockIdx.x;
  int64_t b = blockIdx.y;
  if (it.mode == 1) {
    const int64_t lin = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    b = lin % gridDim.y;
    item = (int)(lin / gridDim.y);
  }
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  __builtin_assume(w >= 0 && w < NW);
  int64_t start, stride;
  int count;
  gram_item(it, item, start, stride, count);
  const In* psib = psi + b * k_sb;
  const In* vbb = vb + b * v_sb;
  float* Gout = (it.mode == 1 && item == it.N0) ? G_last + b * gl_sb : G + b * g_sb + item * g_si;
  const int nsteps = (count + kStep - 1) / kStep;

  f32x4 accS[NW], accS8 = zero4();
#pragma unroll
  for (int at = 0; at < NW; ++at) accS[at] = zero4();
  if (nsteps > 0)
    issue_gram<In, NW, FEAT, LIST>(psi0, vb0, psib, vbb, it, item, start, stride, 0, count, k_st, v_st, w,
                         lane_id());
  Frag wa[4];
  const In* hb = nullptr;
  if constexpr (FEAT) {
    feat_w_load<In>(wa, (const In*)fa.W, w, lane_id());
    feat_ones_tile<In>(vb0 + kTileChunks, threadIdx.x, kThreads);
    if (!ONE) feat_ones_tile<In>(vb1 + kTileChunks, threadIdx.x, kThreads);
    hb = fa.h ? (const In*)fa.h + b * fa.h_sb : nullptr;
    // consumed here (the compiler's wait also lands step 0's rows), so no
    // wait for W sits inside the loop
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) asm volatile("" : "+v"(wa[kb]));
  }

  auto step = [&](auto BUFC, int s) {
    constexpr int BUF = decltype(BUFC)::value;
    const uint4* tpsi = BUF ? psi1 : psi0;
    const uint4* tvb = BUF ? vb1 : vb0;
    int lane = lane_id();
    asm volatile("" : "+v"(lane));
    const int g = lane >> 4;
    // FEAT: the key gate of the lane's four rows, loaded untracked before the
    // next step's copy and consumed after the wait that covers it
    uint32_t hraw[4] = {0, 0, 0, 0};
    if constexpr (FEAT) {
      const int r16 = lane & 15;
      if (hb) {
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const int row = s * kStep + 16 * tt + r16;
          hraw[tt] = load_u16_untracked(
              hb + gram_token_of<LIST>(it, item, start, stride, row < count ? row : 0));
        }
      }
    }
    if (!ONE && s + 1 < nsteps) {
      issue_gram<In, NW, FEAT, LIST>(BUF ? psi0 : psi1, BUF ? vb0 : vb1, psib, vbb, it, item, start, stride,
                           (s + 1) * kStep, count, k_st, v_st, w, lane);
      // the gate loads (issued first) are older than this step's DMA loads
      if (w < kL % NW)
        wait_vmcnt<kL / NW + 1>();
      else
        wait_vmcnt<kL / NW>();
    } else {
      wait_vmcnt<0>();
    }
    lds_barrier();
    if constexpr (FEAT) {
      float hv[4] = {1.f, 1.f, 1.f, 1.f};
      if (hb) {
        asm volatile("" : "+v"(hraw[0]), "+v"(hraw[1]), "+v"(hraw[2]), "+v"(hraw[3]));
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) hv[tt] = to_f32(__builtin_bit_cast(In, (uint16_t)hraw[tt]));
      }
      uint4* fpsi = BUF ? psi1 : psi0;
      const auto sw = [](int t) { return swz16(t); };
      const float h01[2] = {hv[0], hv[1]}, h23[2] = {hv[2], hv[3]};
      feat_rows<In, 2>(fpsi, fpsi, 0, true, wa, w, fa.kind, hb != nullptr, h01, lane, sw);
      feat_rows<In, 2>(fpsi, fpsi, 2, true, wa, w, fa.kind, hb != nullptr, h23, lane, sw);
      lds_barrier();    // the step's Psi tile is complete
      if (fa.psi_out != nullptr) {
        // the tile's rows to psi_out: thread (t, c) of 64 rows x 8 pairs of
        // 16-byte chunks, un-swizzled, for the rows that hold tokens
        const int t = threadIdx.x >> 3, c = 2 * (threadIdx.x & 7);
        const int row = s * kStep + t;
        if (row < count) {
          const int64_t tok = gram_token_of<LIST>(it, item, start, stride, row);
          uint4* dst = reinterpret_cast<uint4*>((In*)fa.psi_out + b * fa.psi_sb + tok * 128);
          dst[c] = fpsi[t * kRowChunks + (c ^ swz16(t))];
          dst[c + 1] = fpsi[t * kRowChunks + ((c + 1) ^ swz16(t))];
        }
      }
    }
    const int nvalid = count - s * kStep;        // rows of this step holding tokens
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (32 * ks >= nvalid) continue;
      Frag vbw = psi_tr<In>(tvb, w, ks, lane);
      Frag vb8 = vb_norm_tr<In>(tvb, ks, lane);
      if (nvalid < kStep) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const bool ok = 32 * ks + 8 * g + e < nvalid;
          vbw[e] = ok ? vbw[e] : from_f32<In>(0.f);
          vb8[e] = ok ? vb8[e] : from_f32<In>(0.f);
        }
      }
#pragma unroll
      for (int at = 0; at < NW; ++at) {
        const Frag pa = psi_tr<In>(tpsi, at, ks, lane);
        accS[at] = mma(accS[at], pa, vbw);
        if (at == w) accS8 = mma(accS8, pa, vb8);
      }
    }
    lds_barrier();     // this buffer is free for the next DMA
    if (ONE && s + 1 < nsteps)
      issue_gram<In, NW, FEAT, LIST>(psi0, vb0, psib, vbb, it, item, start, stride,
                                     (s + 1) * kStep, count, k_st, v_st, w, lane);
  };
  if constexpr (ONE) {
    for (int s = 0; s < nsteps; ++s) step(std::integral_constant<int, 0>{}, s);
  } else {
    for (int s = 0; s < nsteps; s += 2) {
      step(std::integral_constant<int, 0>{}, s);
      if (s + 1 < nsteps) step(std::integral_constant<int, 1>{}, s + 1);
    }
  }

  const int lane = lane_id();
  const int r16 = lane & 15, g = lane >> 4;
  if ((reinterpret_cast<uintptr_t>(Gout) & 15) == 0) {
    // The r x p result is one contiguous block.  Stage it 64 rows (33 KB at
    // r = 128) at a time in the idle tile buffer and store each part as
    // consecutive 16-byte stores: whole cache lines, instead of 64-byte runs of
    // 516-byte rows.  Non-temporal: the table (888 MB for the long-prefill
    // pool) is far larger than the last-level cache and is read back only by
    // the next kernel.
    float* st = reinterpret_cast<float*>(stage0);
#pragma unroll
    for (int h = 0; h < (NW + 3) / 4; ++h) {
      const int tiles = min(4, NW - 4 * h);          // row tiles of this part
      lds_barrier();                                 // the tile buffer is free
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        if (4 * h + q4 >= NW) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st[(16 * q4 + 4 * g + i) * kP + 16 * w + r16] = accS[4 * h + q4][i];
      }
      if ((w >> 2) == h && r16 == 0) {               // the last column: rows 16 w + 4 g + i
#pragma unroll
        for (int i = 0; i < 4; ++i) st[(16 * (w & 3) + 4 * g + i) * kP + kP - 1] = accS8[i];
      }
      lds_barrier();
      const float4* src = reinterpret_cast<const float4*>(st);
      float4* dst = reinterpret_cast<float4*>(Gout + h * 64 * kP);
      for (int e = threadIdx.x; e < tiles * 4 * kP; e += kThreads) {
        const float4 v = src[e];
        __builtin_nontemporal_store(v.x, &dst[e].x);
        __builtin_nontemporal_store(v.y, &dst[e].y);
        __builtin_nontemporal_store(v.z, &dst[e].z);
        __builtin_nontemporal_store(v.w, &dst[e].w);
      }
    }
    return;
  }
#pragma unroll
  for (int at = 0; at < NW; ++at)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      Gout[(int64_t)(16 * at + 4 * g + i) * kP + 16 * w + r16] = accS[at][i];
  if (r16 == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) Gout[(int64_t)(16 * w + 4 * g + i) * kP + kP - 1] = accS8[i];
  }
}

bool gram_stream_ok(int dtype, const void* psi, const void* vb, int r, int p, int64_t k_sb,
                    int64_t k_st, int64_t v_sb, int64_t v_st, const GramItems& it, int nitems,
                    int nb) {
  if (dtype != SMAT_BF16 && dtype != SMAT_F16) return false;
  if (r % 16 || r < 80 || r > 128 || p != r + 1 || it.nsplit > 1) return false;
  if (r < 128 && it.mode == 2) return false;           // lists: compiled for r = 128
  // few, long profiles: the split-K kernel (chunk groups are not split)
  if (it.mode != 0 && (int64_t)nitems * nb < 256) return false;
  if (!rows_vec_ok(psi, k_sb, k_st, 2) || !rows_vec_ok(vb, v_sb, v_st, 2) || v_st < r + 8)
    return false;
  return variant(SMAT_VARIANT_GRAM) == 0;
}

template <typename In, int NW, bool FEAT>
static void gram_stream_kernel_launch(const void* psi, const void* vb, float* G, float* G_last,
                                      const GramItems& it, dim3 grid, bool one, int64_t k_sb,
                                      int64_t k_st, int64_t v_sb, int64_t v_st, int64_t g_sb,
                                      int64_t g_si, int64_t gl_sb, const FeatArgs& fa,
                                      hipStream_t stream) {
  const In* k = (const In*)psi;
  const In* v = (const In*)vb;
  const dim3 blk(64 * NW);
  // lists (r = 128) have no form with the feature map
  if constexpr (!FEAT && NW == 8) {
    if (it.mode == 2) {
      smat::launch((gram_stream_kernel<In, 8, false, false, true>), grid, blk, 0, stream, k, v, G,
                   G_last, it, k_sb, k_st, v_sb, v_st, g_sb, g_si, gl_sb, fa);
      return;
    }
  }
  if (one)
    smat::launch((gram_stream_kernel<In, NW, true, FEAT, false>), grid, blk, 0, stream, k, v, G,
                 G_last, it, k_sb, k_st, v_sb, v_st, g_sb, g_si, gl_sb, fa);
  else
    smat::launch((gram_stream_kernel<In, NW, false, FEAT, false>), grid, blk, 0, stream, k, v, G,
                 G_last, it, k_sb, k_st, v_sb, v_st, g_sb, g_si, gl_sb, fa);
}

// Whether the profiles, of ceil((n - n_P) / N0) terms, fit one step, and the
// global channel (item N0, when launched), of n_P, a few: 128 of them beside
// profiles of 14 tokens in two buffers held the pool of 12 x 10007 tokens of 96
// to 72 us.
static bool gram_one_step(const GramItems& it, int nitems) {
  if (it.mode != 1) return false;
  const int64_t maxc = it.N0 > 0 ? ((int64_t)it.n - it.n_P + it.N0 - 1) / it.N0 : 0;
  return maxc <= ss::kStep && (nitems <= it.N0 || it.n_P <= 8 * ss::kStep);
}

int gram_stream_launch(int dtype, const void* psi, const void* vb, float* G, float* G_last,
                       const GramItems& it, int nitems, int nb, int p, int64_t k_sb,
                       int64_t k_st, int64_t v_sb, int64_t v_st, int64_t g_sb, int64_t g_si,
                       int64_t gl_sb, hipStream_t stream, const char* who) {
  const dim3 grid((unsigned)nitems, (unsigned)nb);
  const bool one = gram_one_step(it, nitems);
  const FeatArgs fa{};
#define SMAT_GRAM_NW(NWV)                                                                      \
  case NWV:                                                                                    \
    if (dtype == SMAT_BF16)                                                                    \
      gram_stream_kernel_launch<bf16, NWV, false>(psi, vb, G, G_last, it, grid, one, k_sb,     \
                                                  k_st, v_sb, v_st, g_sb, g_si, gl_sb, fa,     \
                                                  stream);                                     \
    else                                                                                       \
      gram_stream_kernel_launch<f16, NWV, false>(psi, vb, G, G_last, it, grid, one, k_sb,      \
                                                 k_st, v_sb, v_st, g_sb, g_si, gl_sb, fa,      \
                                                 stream);                                      \
    break;
  switch (p / 16) {
    SMAT_GRAM_NW(5)
    SMAT_GRAM_NW(6)
    SMAT_GRAM_NW(7)
    SMAT_GRAM_NW(8)
    default:
      set_error("%s: no streaming Gram kernel for p=%d", who, p);
      return SMAT_EUNSUPPORTED;
  }
#undef SMAT_GRAM_NW
  return launch_status(who);
}

// The Gram sums with the feature map in place: k, v are K and V rows
// (d_qk = d_v = 128, 16-byte aligned rows); any item count (no split-K).
int gram_stream_launch_feat(int dtype, const void* k, const void* v, float* G, float* G_last,
                            const GramItems& it, int nitems, int nb, int64_t k_sb, int64_t k_st,
                            int64_t v_sb, int64_t v_st, int64_t g_sb, int64_t g_si,
                            int64_t gl_sb, const FeatArgs& fa, hipStream_t stream,
                            const char* who) {
  if (nitems == 0 || nb == 0) return SMAT_OK;
  if (it.mode == 2) {                  // compiled for profiles and chunk groups only
    set_error("%s: the feature map is not fused into list Gram sums", who);
    return SMAT_EUNSUPPORTED;
  }
  const dim3 grid((unsigned)nitems, (unsigned)nb);
  const bool one = gram_one_step(it, nitems);
  if (dtype == SMAT_BF16)
    gram_stream_kernel_launch<bf16, 8, true>(k, v, G, G_last, it, grid, one, k_sb, k_st, v_sb,
                                             v_st, g_sb, g_si, gl_sb, fa, stream);
  else
    gram_stream_kernel_launch<f16, 8, true>(k, v, G, G_last, it, grid, one, k_sb, k_st, v_sb,
                                            v_st, g_sb, g_si, gl_sb, fa, stream);
  return launch_status(who);
}

// The shapes this kernel serves; everything else runs scan_fused_kernel.
bool scan_stream_ok(int dtype, const void* phi, const void* psi, const void* vb, const float* Y,
                    const float* out, const ScanArgs& a) {
  if (dtype != SMAT_BF16 && dtype != SMAT_F16) return false;
  if (a.r % 16 || a.r < 64 || a.r > 128 || a.p != a.r + 1) return false;
  if (a.C % ss::kStep || a.n % ss::kStep) return false;
  if (!rows_vec_ok(phi, a.q_sb, a.q_st, 2) || !rows_vec_ok(psi, a.k_sb, a.k_st, 2) ||
      !rows_vec_ok(vb, a.v_sb, a.v_st, 2) || a.v_st < a.r + 8)
    return false;
  // H only at r = 64, the width of the fused backward.  There a training step's bits
  // depend on Vb's rows, as a forward's do at every width here: those that are not
  // 16-byte aligned take the general kernel, which rounds 16-bit scores inside its
  // chunk of 128 tokens instead of inside steps of 64.  Wider H takes the general
  // kernel for every row stride.
  if (a.write_H ? a.r != 64 : !rows_vec_ok(out, a.o_sb, a.o_st, 4)) return false;
  if (Y && !rows_vec_ok(Y, a.y_sb, a.y_st, 4)) return false;
  // per-lane row offsets are 32-bit bytes over 64 rows
  constexpr int64_t kMaxSt = 1 << 20;
  if (a.q_st >= kMaxSt || a.k_st >= kMaxSt || a.v_st >= kMaxSt || a.o_st >= kMaxSt ||
      a.y_st >= kMaxSt)
    return false;
  return variant(SMAT_VARIANT_SCAN) == 0;
}

template <typename In, int NW>
static void scan_stream_kernel_launch(const void* phi, const void* psi, const void* vb,
                                      const float* Sg, const float* Y, const float* gate,
                                      float* out, dim3 grid, const ScanArgs& a,
                                      hipStream_t stream) {
  const In* q = (const In*)phi;
  const In* k = (const In*)psi;
  const In* v = (const In*)vb;
  const dim3 blk(64 * NW);
  const FeatArgs fa{};
  if constexpr (NW == 4) {
    if (a.write_H) {
      smat::launch((scan_stream_kernel<In, NW, false, false, true, true>), grid, blk, 0, stream,
                   q, k, v, Sg, Y, gate, out, a, fa);
      return;
    }
  }
  if (a.T % ss::kStep)
    smat::launch((scan_stream_kernel<In, NW, false, true, true, false>), grid, blk, 0, stream, q,
                 k, v, Sg, Y, gate, out, a, fa);
  else if (Y || gate)
    smat::launch((scan_stream_kernel<In, NW, false, true, false, false>), grid, blk, 0, stream, q,
                 k, v, Sg, Y, gate, out, a, fa);
  else
    smat::launch((scan_stream_kernel<In, NW, false, false, false, false>), grid, blk, 0, stream,
                 q, k, v, Sg, Y, gate, out, a, fa);
}

template <typename In>
static void scan_stream_shape(const void* phi, const void* psi, const void* vb, const float* Sg,
                              const float* Y, const float* gate, float* out, dim3 grid,
                              const ScanArgs& a, hipStream_t stream) {
  switch (a.r / 16) {
    case 4:
      return scan_stream_kernel_launch<In, 4>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
    case 5:
      return scan_stream_kernel_launch<In, 5>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
    case 6:
      return scan_stream_kernel_launch<In, 6>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
    case 7:
      return scan_stream_kernel_launch<In, 7>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
    default:
      return scan_stream_kernel_launch<In, 8>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
  }
}

int scan_stream_launch(int dtype, const void* phi, const void* psi, const void* vb,
                       const float* Sg, const float* Y, const float* gate, float* out, int nb,
                       int ng, const ScanArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)ng, (unsigned)nb);
  if (dtype == SMAT_BF16)
    scan_stream_shape<bf16>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
  else
    scan_stream_shape<f16>(phi, psi, vb, Sg, Y, gate, out, grid, a, stream);
  return launch_status("smat_causal_scan");
}

// The streaming causal pass with the feature map in place: q and v are Q and V
// rows (r = 128, T a multiple of 64, V rows of 128); psi is the Psi rows (key
// gate applied).
int scan_stream_launch_feat(int dtype, const void* q, const void* psi, const void* v,
                            const float* Sg, const float* Y, const float* gate, float* out,
                            int nb, int ng, const ScanArgs& a, const FeatArgs& fa,
                            hipStream_t stream) {
  const dim3 grid((unsigned)ng, (unsigned)nb), blk(64 * 8);
  if (dtype == SMAT_BF16)
    smat::launch((scan_stream_kernel<bf16, 8, true, true, false, false>), grid, blk, 0, stream,
                 (const bf16*)q, (const bf16*)psi, (const bf16*)v, Sg, Y, gate, out, a, fa);
  else
    smat::launch((scan_stream_kernel<f16, 8, true, true, false, false>), grid, blk, 0, stream,
                 (const f16*)q, (const f16*)psi, (const f16*)v, Sg, Y, gate, out, a, fa);
  return launch_status("smat_causal_scan");
}

}  // namespace smat
