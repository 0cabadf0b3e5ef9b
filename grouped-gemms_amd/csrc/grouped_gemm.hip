// MX-scaled grouped GEMM kernels for gfx950 (CDNA4):
//   * forward / dgrad:  out[s:e] = A[s:e] @ B[g]^T          (kernels/forward.py:81-294)
//   * weight gradient:  out[g]   = GO[:, s:e] @ IA[:, s:e]^T (kernels/backward.py:31-215)
//   * routing table and tile schedule exposed for testing   (kernels/forward.py:31-51, 296-365)
//   * scale re-layout feeding both GEMMs                    (the role of kernels/forward.py:367-397)
//   * split of an under-filled last round along the reduction, with fp32
//     partial tiles and a reduce kernel        (generalises kernels/backward.py:106-215)
//   * a forward last round of few tiles as 128 x 128 quarter tiles where that
//     beats the split (fwd_quad_kernel, fwd_plan)
//   * forward calls of few rows per group as weight-streaming tiles
//     (fwd_stream_kernel)
//
// Both GEMMs are "NT" products whose two operands are contiguous along the
// reduction dimension, so they share one main loop:
//   acc[r][c] = sum_k X[r][k] * W[c][k] * 2**(xs[r][k/32]-127) * 2**(ws[c][k/32]-127)
// with X on the B side and W on the A side of v_mfma_scale_f32_32x32x64_f8f6f4,
// so that every lane of the accumulator holds 4 consecutive output columns.
//
// Main loop (step_mainloop): the reduction runs in 128-element steps, one
// 128-byte line of every e4m3 row, that alternate between two LDS slots.
// While a step's two halves are multiplied out of registers, the next step
// lies in the other slot and the one after it is copied into the slot being
// left.
//   * X and W tiles go global -> LDS directly with 16-byte buffer_load ... lds;
//     chunks outside the reduction range read as zero through the buffer
//     range check.  16-byte chunks are XOR-swizzled by row: conflict-free
//     fragment reads.
//   * e8m0 scales: a re-layout kernel first writes the plain `to_mx` scales
//     step-major, one dword (4 scale bytes = one 128-element step) per row:
//     [step][row].  The scales of a tile for two steps are then a few
//     contiguous 1 KB pieces, copied into a two-slot scale area every two
//     steps (small calls copy the plain scales themselves, 8 steps of a row
//     at a time); each MFMA picks its lane's byte with op_sel.
//   * everything but the MFMAs is kept to about four instructions per MFMA
//     (131 to 136 beside the 32 of a 256 x 256 step): one wave per SIMD issues
//     them all.
#include <mutex>
#include <type_traits>

#include "mxgg_device.h"
#include "mxgg_host.h"

namespace mxgg {

constexpr int STEP = 128;      // reduction elements per step: a scale dword (4 blocks of 32)
constexpr int HALF = 64;       // half a step: reduction elements per MFMA

// Split of the last, partial round.  With T tiles and P workgroups resident
// at once, the rem = T % P tiles of the last round leave most of the chip idle
// for (a fraction of) a tile time.  They can instead be cut into S pieces
// along the reduction (whole 128-element steps, at least kMinSplitSteps per
// piece, at most kMaxSplit pieces per tile, `slots` pieces in all); pieces
// store fp32 partial tiles and a second kernel adds them in piece order and
// rounds once.  Tiles 0 .. dp-1 run whole, tile dp + v as pieces v*S ..
// v*S+S-1.  Up to P / 2 last-round tiles, S <= P / rem keeps the pieces in one
// round.  Past that, S pieces per tile run in ceil(rem * S / P) rounds (160
// tiles on 256 CUs: 3 pieces each, two rounds of a third of the reduction
// instead of one round of all of it).
//
// Only a last round that follows at most kSplitMaxRounds full rounds is
// split (measured: a loss from 5 full rounds on).  Tiles of one launch stay
// in step round after round, so the last round does leave most CUs idle,
// but its few tiles run uncontended at a higher clock, in about 0.6 of a
// full round's tile time, and the pieces, the reduce and two more launches
// cost as much.  S is picked by a cost model
// (nanoseconds, MI355X kernel traces): the last round of n steps costs about
// kTailNsPerStep * n (0.75 of 1.7 us per step; kBusyNsPerStep, 1.7 us, when
// the last round fills more than half the chip); cut into S pieces it costs
// rounds * n / S of that, plus kSplitFixedNs (piece prologue and epilogue, two
// launches) plus the partial traffic, rem * S tiles written and read back
// (kSplitNsPerMiB).  No split unless that saves at least kSplitMinGainNs (the
// model is coarse); reductions shorter than kMinSplitTotal steps are never
// split.  Integer arithmetic: every kernel that recomputes the plan on the
// device gets the same answer, bit for bit.
constexpr int kMinSplitSteps = 4;
constexpr int kMaxSplit = 8;
constexpr int kMinSplitTotal = 32;
constexpr int kSplitMaxRounds = 2;
constexpr int64_t kTailNsPerStep = 1275;
constexpr int64_t kBusyNsPerStep = 1700;
constexpr int64_t kSplitFixedNs = 9000;
constexpr int64_t kSplitNsPerMiB = 400;
constexpr int64_t kSplitMinGainNs = 16000;
constexpr size_t kSplitBytes = (size_t)128 << 20;  // partial-tile area of a full workspace

struct Split {
  int dp;       // tiles computed whole
  int S;        // pieces per split tile (1: no split)
  int units;    // pieces in all (rem * S, or 0)
};

// saved: what the plan saves over whole tiles, by the model (ns; 0: no split).
__host__ __device__ inline Split split_plan(int T, int P, int nsteps, int slots, int tile_kib, int* saved = nullptr) {
  Split sp{T, 1, 0};
  if (saved) *saved = 0;
  if (T <= 0 || P <= 0 || nsteps < kMinSplitTotal || T / P > kSplitMaxRounds) return sp;
  const int rem = T % P;
  if (rem == 0) return sp;
  int smax = 2 * rem > P ? kMaxSplit : P / rem;
  if (smax > kMaxSplit) smax = kMaxSplit;
  if (smax > nsteps / kMinSplitSteps) smax = nsteps / kMinSplitSteps;
  if (smax > slots / rem) smax = slots / rem;
  // int32 throughout: tail <= 1700 * 2^20, rounds * (tail / S) <= tail, and
  // rem * S <= slots <= 4096 with tile_kib <= 256 keeps the staging term
  // below 2^30.  Unrolled, every
  // tail / S has a constant divisor.
  const int per = (int)(2 * rem > P ? kBusyNsPerStep : kTailNsPerStep);
  const int tail = per * (nsteps < (1 << 20) ? nsteps : (1 << 20));
  int best = (int)kSplitMinGainNs;
#pragma unroll
  for (int S = 2; S <= kMaxSplit; ++S) {
    if (S > smax) break;
    const int rounds = (rem * S + P - 1) / P;   // <= S while rem < P
    const int gain =
        tail - rounds * (tail / S) - (int)kSplitFixedNs - rem * S * tile_kib * (int)kSplitNsPerMiB / 1024;
    if (gain > best) {
      best = gain;
      sp.S = S;
    }
  }
  if (sp.S < 2) return sp;
  sp.dp = T - rem;
  sp.units = rem * sp.S;
  if (saved) *saved = best;
  return sp;
}

// Steps [a, b) of piece s out of S over steps [a0, a0 + n).  32-bit
// unsigned arithmetic: n < 2**25 steps and s < S <= kMaxSplit keep n * (s+1)
// below 2**28 (a 64-bit division is a long software sequence on the device).
__host__ __device__ inline void split_range(int a0, int n, int s, int S, int& a, int& b) {
  a = a0 + (int)((uint32_t)n * (uint32_t)s / (uint32_t)S);
  b = a0 + (int)((uint32_t)n * (uint32_t)(s + 1) / (uint32_t)S);
}

template <int BM_, int BN_, int WGM_, int WGN_, int WFMT_, int NH_, bool PS_ = false>
struct Cfg {
  static constexpr int BM = BM_;        // X rows per tile (output rows)
  static constexpr int BN = BN_;        // W rows per tile (output columns)
  static constexpr int WGM = WGM_;      // waves along rows
  static constexpr int WGN = WGN_;      // waves along columns
  static constexpr int WFMT = WFMT_;    // W element format (X is always e4m3)
  static constexpr int NH = NH_;        // 64-element half steps held in LDS
  static constexpr int NS = NH / 2;     // LDS slots (steps)
  // Scale source: false, step-major dwords [step][row] (the re-layout
  // kernel's output or the quantizer's native layout); true, the plain
  // to_mx scales (row r's byte b at r * ld + b, ld a multiple of 16), read
  // directly in 32-byte row pieces of 8 steps.
  static constexpr bool PS = PS_;
  static constexpr bool F4 = WFMT == MXGG_FMT_E2M1;
  static constexpr int NW = WGM * WGN;
  static constexpr int NT = NW * kWave;
  static constexpr int WTM = BM / WGM;
  static constexpr int WTN = BN / WGN;
  static constexpr int FM = WTM / 32;
  static constexpr int FN = WTN / 32;
  static constexpr int NMMA = FM * FN;              // MFMAs per wave and half step
  static constexpr int XROW = STEP;                 // bytes per X row per step
  static constexpr int WROW = F4 ? STEP / 2 : STEP; // bytes per W row per step
  static constexpr int XBYTES = BM * XROW;          // one X slot
  static constexpr int WBYTES = BN * WROW;          // one W slot
  static constexpr int WOFF = NS * XBYTES;          // X slots, then W slots, then scale slots
  static constexpr int SOFF = WOFF + NS * WBYTES;
  // Two scale slots of GSTEPS steps each.  Step-major: GSTEPS x BM X-row
  // dwords ([step][row]) followed by GSTEPS x BN W-row dwords.  Plain: BM X
  // rows then BN W rows of 32 bytes (8 steps of the row from the run's first
  // step on), the two 16-byte halves of rows 8..15 of every 16 swapped
  // (conflict-free reads of one step over 32 rows, two ways apart at most).
  static constexpr int GSTEPS = PS ? 8 : 2;
  static constexpr int SSLOT = GSTEPS * (BM + BN) * 4;
  static constexpr int LDS = SOFF + 2 * SSLOT;
  static constexpr int QX = XBYTES / 1024 / NW;     // 1 KB data copies per wave and step
  static constexpr int QW = WBYTES / 1024 / NW;
  static constexpr int NC = QX + QW;
  static constexpr int XCR = 1024 / XROW;           // rows per copy
  static constexpr int WCR = 1024 / WROW;
  // step-major: 1 KB scale copies of the X part and per group (wave w makes
  // copy w % NSD)
  static constexpr int NSX = PS ? 0 : GSTEPS * BM * 4 / 1024;
  static constexpr int NSD = PS ? 1 : SSLOT / 1024;
  // plain: 1 KB scale copies (32 rows) per wave and group; waves 0 .. NXW-1
  // copy X rows, the others W rows
  static constexpr int SPW = PS ? (BM + BN) / 32 / NW : 0;
  static constexpr int NXW = PS ? BM / 32 / SPW : 0;
  // Schedule of a step's 2 * NMMA MFMAs (see step_pos): reads of the second
  // half step during the first RD, barrier B1 before MFMA PB1, the copies
  // over the NMMA MFMAs from there, barrier B2 before MFMA PB2 and the next
  // step's reads over the RD from there.
  static constexpr int RD = NMMA / 2;
  static constexpr int PB1 = (5 * NMMA + 7) / 8;
  static constexpr int PB2 = 5 * NMMA / 4;
  static_assert(NH == 4, "the main loop alternates between two slots");
  static_assert(XBYTES % (2048 * NW) == 0 && WBYTES % (2048 * NW) == 0, "even numbers of copies per wave");
  static_assert(PS || ((GSTEPS * BM * 4) % 1024 == 0 && (GSTEPS * BN * 4) % 1024 == 0 && NW % NSD == 0),
                "scale copies: one operand each, one per wave");
  static_assert(!PS || ((SPW == 2 || SPW == 4) && (BM + BN) % (32 * NW) == 0 && (BM / 32) % SPW == 0),
                "plain scale copies: whole 32-row pieces, one operand per wave, one per two steps");
  static_assert(SOFF % (2 * SSLOT) == 0, "scale slots are told apart by one address bit");
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile");
  static_assert(LDS <= 160 * 1024, "LDS budget");
  static_assert(XBYTES + 32 * (FM - 1) * XROW < 65536 && WBYTES + 32 * (FN - 1) * WROW < 65536, "ds_read offsets");
  static_assert(PB1 >= RD && PB2 >= NMMA && PB2 + RD <= 2 * NMMA && PB1 + NMMA <= 2 * NMMA && NC + 2 <= 63,
                "step schedule");
};

// 16-byte chunk swizzle of 64-byte rows: bijective on the chunk index for
// every 8-row and every 16-row class; depends on row % 16 only.
__device__ __forceinline__ int swz4(int r) {
  return ((((r >> 2) ^ (r >> 3)) & 1) << 1) | (((r >> 1) ^ (r >> 2)) & 1);
}

// A tile's rows of one operand in global memory, in one of three layouts,
// G = 2**pl rows per group:
//   rows  (pl = 0): byte k of row r at r * ld + k;
//   pairs (pl = 1, e4m3) and quads (pl = 2, packed e2m1): the G rows of a
//         group interleave in P = 128 / G byte pieces -- one 64-element
//         half step of a row -- byte k of row r at (r / G) * G ld +
//         (k / P) * 128 + (r % G) * P + k % P, so the half-step pieces of a group
//         fill one 128-byte line and a copy touches whole lines instead of
//         halves (pairs) or quarters (quads).
// Local row r of the tile is row e = r + shift of the buffer `data`, which
// starts at the group of the tile's first row (shift = row0 % G); the range
// ends after the group of the tile's last row, so reads past the tile's rows
// return 0 except the other rows of that last group.
struct Operand {
  __amdgpu_buffer_rsrc_t data;
  __amdgpu_buffer_rsrc_t dma;    // data, starting kCopyBias bytes earlier (the main loop's copies)
  uint32_t ld;                   // bytes between rows (groups: between groups / G)
  uint32_t pl;                   // log2 G: 0 rows, 1 pairs, 2 quads
  uint32_t shift;                // row0 % G of the tile
};

// Added to the scalar offsets of the copies, and taken off the base, so that
// the offsets stay non-negative less the immediate they are paired with.
constexpr int kCopyBias = 3 * 1024;

// Operand of rows row0 .. row0 + rows - 1 of the matrix at `base`.
__device__ __forceinline__ Operand make_operand(const uint8_t* base, int64_t ld, int pl, int64_t row0, int rows) {
  Operand o;
  o.ld = (uint32_t)ld;
  o.pl = (uint32_t)pl;
  const int64_t mask = ((int64_t)1 << pl) - 1;
  o.shift = (uint32_t)(row0 & mask);
  const int64_t unit = ld << pl;                                  // bytes per group
  const uint32_t units = (uint32_t)(((int64_t)o.shift + rows + mask) >> pl);
  o.data = make_rsrc(base + (row0 >> pl) * unit, units * (uint32_t)unit);
  o.dma = make_rsrc(base + (row0 >> pl) * unit - kCopyBias, units * (uint32_t)unit + kCopyBias);
  return o;
}

// Byte offset in O.data of byte `col` of local row `row` (pieces of
// 2**pb = 128 / G bytes; for rows, pb = 7 leaves col unchanged).
__device__ __forceinline__ uint32_t operand_off(const Operand& O, uint32_t row, uint32_t col) {
  const uint32_t e = row + O.shift;
  const uint32_t pb = 7u - O.pl;
  return (e >> O.pl) * (O.ld << O.pl) + ((col >> pb) << 7) + ((e & ((1u << O.pl) - 1u)) << pb) +
         (col & ((1u << pb) - 1u));
}

// Where a tile's step-major scales live: dword (t, r) of an operand with R
// rows per step is at byte 4 (t R + r) of the buffer `rsrc` (the operand's
// [step][row] array, re-laid into the workspace or written so by the
// quantizer); reads past the buffer return 0.
struct ScaleSrc {
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t rows;    // step-major: R, rows per step of that array; plain: bytes per row
  uint32_t row0;    // first row of the tile
};

#define MXGG_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")
#define MXGG_WAIT_LGKM() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
#define MXGG_BARRIER() asm volatile("s_barrier" ::: "memory")
#define MXGG_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

template <class C>
struct Frags {
  v8i a[C::FN];   // W fragments (MFMA A operand)
  v8i b[C::FM];   // X fragments (MFMA B operand)
};

// Per-wave and per-lane addresses of the main loop.
// Data copy i of a wave fills 1 KB of a slot, rows (wave * Q + i) * R .. of
// R = 1024 / row bytes: 8 rows of 128 bytes, whole cache lines of a row-major
// operand (packed e2m1 W: 16 rows of 64 bytes).  Slot layout, 128-byte rows:
// tile row m at byte 128 m, its 16-byte unit u (elements 16u .. 16u+15 of the
// step) at unit u ^ (m % 8) ^ ((m / 8) % 2), so that one unit over 8
// consecutive rows hits 8 different 16-byte bank groups of 128 bytes, and over
// 16 rows 16 different ones of 256 bytes; the last term alternates from copy
// to copy, hence two lane offsets (even, odd copies).  64-byte rows: unit u
// (32 elements) at u ^ swz4(m).  The K position travels in the lane offsets,
// the rows in scalar offsets that stay constant: copy i also adds 1024 (i % 4)
// to the LDS and (taken off again in the scalar offset) to the global address
// through the instruction's immediate, so M0 changes once in four copies.
template <class C>
struct Plan {
  uint32_t xe, xo, we, wo;           // lane offsets of the X and W copies
  uint32_t xs[C::QX], ws[C::QW];     // scalar offsets
  uint32_t mxe, mxo, mwe, mwo;       // 0, or kOOB where the copy's chunk lies past the end in the last step
  uint32_t xm0, wm0;                 // LDS address of the wave's copies into the slot of the step
  uint32_t xa[4], wa[4];             // LDS addresses of units 2k + lane / 32 of row lane % 32 (F4: k / 2)
                                     // in the slot read next (k / 2: the half step; each read toggles)
  uint32_t sm0;                      // LDS address of the wave's scale copies in slot 0
  uint32_t sx, sw;                   // LDS addresses of the lane's scale dwords in slot 0
  uint32_t sv;                       // lane offset of the scale copies
  uint32_t s_step;                   // step-major: bytes per step; plain: bytes per 32 rows
  int ux, uw;                        // unit of the lane's X (even copies; odd: ux ^ 1) and W chunk
  int sh;                            // 8 * (lane / 32)
};

// Sets M0, the LDS base of the copies that follow (LDS DMA reads M0 one wait
// state after a write at the earliest).  The copies are issued in asm: M0 then
// changes where it must and not per copy, and the compiler, which does not
// see them, adds no waits of its own.  Callers order them with vmcnt waits.
// (M0 is reserved: the compiler keeps no value of its own in it, and warns of a
// declared clobber.)
__device__ __forceinline__ void set_m0(uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" ::"s"(lds));
#endif
}

// 16 bytes per lane global -> LDS at M0 + IMM + 16 lane; global byte voff +
// soff + IMM of rsrc (past its range: zeros).
template <int IMM>
__device__ __forceinline__ void copy16(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen offset:%3 lds" ::"v"(voff), "s"(rsrc), "s"(soff), "n"(IMM)
               : "memory");
#endif
}

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(lds_ptr_t)(const_cast<void*>(p));
}

// Plan of a run that starts at step t0 of the reduction.
template <class C>
__device__ __forceinline__ void make_plan(Plan<C>& P, uint8_t* smem, const Operand& X, const Operand& W,
                                          const ScaleSrc& xss, const ScaleSrc& wss, int t0) {
  const int lane = threadIdx.x % kWave;
  const int wave = wave_id();
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  const uint32_t lds0 = lds_addr(smem);
  {
    const int row = lane / 8;
    P.ux = (lane & 7) ^ row;
    P.xe = operand_off(X, (uint32_t)row, (uint32_t)(t0 * C::XROW + P.ux * 16));
    P.xo = operand_off(X, (uint32_t)row, (uint32_t)(t0 * C::XROW + (P.ux ^ 1) * 16));
  }
  if constexpr (C::F4) {
    const int row = lane / 4;
    P.uw = (lane & 3) ^ swz4(row);
    P.we = P.wo = operand_off(W, (uint32_t)row, (uint32_t)(t0 * C::WROW + P.uw * 16));
  } else {
    const int row = lane / 8;
    P.uw = P.ux;
    P.we = operand_off(W, (uint32_t)row, (uint32_t)(t0 * C::WROW + P.uw * 16));
    P.wo = operand_off(W, (uint32_t)row, (uint32_t)(t0 * C::WROW + (P.uw ^ 1) * 16));
  }
#pragma unroll
  for (int i = 0; i < C::QX; ++i) P.xs[i] = (uint32_t)(C::XCR * (wave * C::QX + i)) * X.ld + (uint32_t)(kCopyBias - 1024 * (i % 4));
#pragma unroll
  for (int i = 0; i < C::QW; ++i) P.ws[i] = (uint32_t)(C::WCR * (wave * C::QW + i)) * W.ld + (uint32_t)(kCopyBias - 1024 * (i % 4));
  P.xm0 = lds0 + (uint32_t)(wave * C::QX * 1024);
  P.wm0 = lds0 + (uint32_t)(C::WOFF + wave * C::QW * 1024);
  const int h = lane >> 5, r32 = lane & 31;
  const int g = (r32 & 7) ^ ((r32 >> 3) & 1);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    P.xa[k] = (uint32_t)((wm * C::WTM + r32) * C::XROW + (((2 * k + h) ^ g) * 16));
    const int uw = C::F4 ? ((2 * (k / 2) + h) ^ swz4(r32)) : ((2 * k + h) ^ g);
    P.wa[k] = (uint32_t)(C::WOFF + (wn * C::WTN + r32) * C::WROW + uw * 16);
  }
  P.sh = 8 * h;
  if constexpr (C::PS) {
    const bool isx = wave < C::NXW;
    const ScaleSrc& S = isx ? xss : wss;
    const int row = (isx ? wave : wave - C::NXW) * C::SPW * 32 + lane / 2;   // operand row of the tile
    const int half = (lane ^ (lane >> 4)) & 1;
    P.sv = (S.row0 + (uint32_t)row) * S.rows + (uint32_t)(4 * t0 + half * 16);
    P.s_step = S.rows * 32u;
    P.sm0 = lds0 + (uint32_t)(C::SOFF + wave * C::SPW * 1024);
    const uint32_t sr = (uint32_t)(C::SOFF + r32 * 32 + ((r32 >> 3) & 1) * 16);
    P.sx = sr + (uint32_t)(wm * C::WTM * 32);
    P.sw = sr + (uint32_t)((C::BM + wn * C::WTN) * 32);
  } else {
    const int wq = wave % C::NSD;
    const bool isx = wq < C::NSX;
    const int R = isx ? C::BM : C::BN;              // tile rows of the lane's operand
    const int q = (isx ? wq : wq - C::NSX) * 256 + 4 * lane;   // first dword of the lane in its part
    const ScaleSrc& S = isx ? xss : wss;
    P.s_step = S.rows * 4u;
    P.sv = (S.row0 + (uint32_t)(q % R)) * 4u + (uint32_t)(t0 + q / R) * P.s_step;
    P.sm0 = lds0 + (uint32_t)(C::SOFF + wq * 1024);
    P.sx = (uint32_t)(C::SOFF + (wm * C::WTM + r32) * 4);
    P.sw = (uint32_t)(C::SOFF + C::GSTEPS * C::BM * 4 + (wn * C::WTN + r32) * 4);
  }
}

// Lane offsets of one step's copies (the plan's, or masked ones).
struct CopyOff {
  uint32_t xe, xo, we, wo;
};

// Offsets of the copies of a step of which only units [xlo, xhi) of X and
// [wlo, whi) of W lie inside the reduction range; the other chunks read as
// zeros without touching memory.
template <class C>
__device__ __forceinline__ CopyOff mask_copies(const Plan<C>& P, int xlo, int xhi, int wlo, int whi) {
  CopyOff o;
  const int xo = P.ux ^ 1, wo = C::F4 ? P.uw : P.uw ^ 1;
  o.xe = (P.ux >= xlo && P.ux < xhi) ? P.xe : kOOB;
  o.xo = (xo >= xlo && xo < xhi) ? P.xo : kOOB;
  o.we = (P.uw >= wlo && P.uw < whi) ? P.we : kOOB;
  o.wo = (wo >= wlo && wo < whi) ? P.wo : kOOB;
  return o;
}

// Copies I .. E-1 of a step (X, then W) into the slot at P.xm0 / P.wm0.
template <class C, int I, int E>
__device__ __forceinline__ void step_copies(const Operand& X, const Operand& W, const Plan<C>& P, const CopyOff& o) {
  if constexpr (I < E) {
    if constexpr (I < C::QX) {
      if constexpr (I % 4 == 0) set_m0(P.xm0 + I * 1024);
      copy16<(I % 4) * 1024>(X.dma, (I & 1) ? o.xo : o.xe, P.xs[I]);
    } else {
      constexpr int J = I - C::QX;
      if constexpr (J % 4 == 0) set_m0(P.wm0 + J * 1024);
      copy16<(J % 4) * 1024>(W.dma, (J & 1) ? o.wo : o.we, P.ws[J]);
    }
    step_copies<C, I + 1, E>(X, W, P, o);
  }
}

// Scale copy issued at step t (relative to the run's first step) when t is
// even, of the group after t's.  Step-major: the wave's 1 KB.  Plain: one
// 32-row piece of the wave (pieces 0 .. SPW-1 over the group's even steps).
// The branch lives inside the asm, so the step stays one basic block for the
// compiler (a branch there costs the register allocator dearly).
template <class C>
__device__ __forceinline__ void issue_scales(__amdgpu_buffer_rsrc_t ssr, const Plan<C>& P, int t) {
  const int g = t / C::GSTEPS + 1;
  const uint32_t i = C::PS ? (uint32_t)((t / 2) % (C::PS ? C::SPW : 1)) : 0u;
  [[maybe_unused]] const uint32_t m0 = P.sm0 + (uint32_t)((g & 1) * C::SSLOT) + i * 1024u;
  [[maybe_unused]] const uint32_t so = C::PS ? P.s_step * i + (uint32_t)(g * 32) : P.s_step * (uint32_t)(g * C::GSTEPS);
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_bitcmp1_b32 %0, 0\n\t"
      "s_cbranch_scc1 1f\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %2, %3, %4 offen lds\n"
      "1:"
      :
      : "s"(t), "s"(m0), "v"(P.sv), "s"(ssr), "s"(so)
      : "memory", "scc");
#endif
}

// Takes the chunks past the end out of the lane offsets when step t is the
// last of the run's n, all of them when it lies past it (branches inside the
// asm, as above).
template <class C>
__device__ __forceinline__ void mask_end(Plan<C>& P, int t, int n) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile(
      "s_cmp_lt_i32 %4, %9\n\t"
      "s_cbranch_scc1 2f\n\t"
      "s_cmp_lg_u32 %4, %9\n\t"
      "s_cbranch_scc1 1f\n\t"
      "v_or_b32 %0, %0, %5\n\t"
      "v_or_b32 %1, %1, %6\n\t"
      "v_or_b32 %2, %2, %7\n\t"
      "v_or_b32 %3, %3, %8\n\t"
      "s_branch 2f\n"
      "1:\n\t"
      "v_mov_b32 %0, %10\n\t"
      "v_mov_b32 %1, %10\n\t"
      "v_mov_b32 %2, %10\n\t"
      "v_mov_b32 %3, %10\n"
      "2:"
      : "+v"(P.xe), "+v"(P.xo), "+v"(P.we), "+v"(P.wo)
      : "s"(t), "v"(P.mxe), "v"(P.mxo), "v"(P.mwe), "v"(P.mwo), "s"(n - 1), "s"(kOOB)
      : "scc");
#endif
}

// Fragments A .. B-1 (W's, then X's) of half step J of the step in the slot
// P.wa / P.xa point to.
// MFMA operand layout: lane half h holds elements 16h .. 16h+15 of the half
// step in dwords 0-3 and 32+16h .. 32+16h+15 in dwords 4-7 (packed e2m1: 32h
// .. 32h+31 in dwords 0-3).
template <class C, int J, int A, int B>
__device__ __forceinline__ void read_frags(const uint8_t* smem, const Plan<C>& P, Frags<C>& F) {
  if constexpr (A < B) {
    if constexpr (A < C::FN) {
      constexpr int off = A * 32 * C::WROW;
      if constexpr (C::F4) {
        const v4i l = *reinterpret_cast<const v4i*>(smem + P.wa[2 * J] + off);
        F.a[A] = (v8i){l[0], l[1], l[2], l[3], 0, 0, 0, 0};
      } else {
        const v4i l = *reinterpret_cast<const v4i*>(smem + P.wa[2 * J] + off);
        const v4i h = *reinterpret_cast<const v4i*>(smem + P.wa[2 * J + 1] + off);
        F.a[A] = (v8i){l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
      }
    } else {
      constexpr int i = A - C::FN;
      constexpr int off = i * 32 * C::XROW;
      const v4i l = *reinterpret_cast<const v4i*>(smem + P.xa[2 * J] + off);
      const v4i h = *reinterpret_cast<const v4i*>(smem + P.xa[2 * J + 1] + off);
      F.b[i] = (v8i){l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
    }
    read_frags<C, J, A + 1, B>(smem, P, F);
  }
}

// Point half step J's read addresses at the other slot.
template <class C, int J>
__device__ __forceinline__ void toggle_reads(Plan<C>& P) {
#pragma unroll
  for (int k = 2 * J; k < 2 * J + 2; ++k) {
    P.xa[k] ^= (uint32_t)C::XBYTES;
    P.wa[k] ^= (uint32_t)C::WBYTES;
  }
}

// The lane's raw scale dwords of step t (relative to the run's first step).
template <class C>
__device__ __forceinline__ void read_scales(const uint8_t* smem, const Plan<C>& P, int t, uint32_t (&xs)[C::FM],
                                            uint32_t (&ws)[C::FN]) {
  const uint32_t slot = (uint32_t)(((t / C::GSTEPS) & 1) * C::SSLOT);
  uint32_t ax, aw;
  constexpr int row = C::PS ? 32 : 4;    // bytes between rows
  if constexpr (C::PS) {
    const uint32_t s = slot | (uint32_t)((t & 7) * 4);
    ax = P.sx ^ s;
    aw = P.sw ^ s;
  } else {
    ax = P.sx + (slot + (uint32_t)((t & 1) * C::BM * 4));
    aw = P.sw + (slot + (uint32_t)((t & 1) * C::BN * 4));
  }
#pragma unroll
  for (int i = 0; i < C::FM; ++i) xs[i] = *reinterpret_cast<const uint32_t*>(smem + ax + i * 32 * row);
#pragma unroll
  for (int j = 0; j < C::FN; ++j) ws[j] = *reinterpret_cast<const uint32_t*>(smem + aw + j * 32 * row);
}

// A step's dword holds the scales of its blocks 0 .. 3; lane half h supplies
// block h of the first and 2 + h of the second half step.  Shifted down by 8h
// they are bytes 0 and 2 on every lane, which op_sel picks per MFMA.  The
// registers the previous MFMA reads its scales from, the last of each array,
// are written last.
template <class C>
__device__ __forceinline__ void shift_scales(const Plan<C>& P, const uint32_t (&xn)[C::FM], const uint32_t (&wn)[C::FN],
                                             uint32_t (&xs)[C::FM], uint32_t (&ws)[C::FN]) {
#pragma unroll
  for (int i = 0; i < C::FM - 1; ++i) xs[i] = xn[i] >> P.sh;
#pragma unroll
  for (int j = 0; j < C::FN - 1; ++j) ws[j] = wn[j] >> P.sh;
  MXGG_SCHED_FENCE();
  xs[C::FM - 1] = xn[C::FM - 1] >> P.sh;
  ws[C::FN - 1] = wn[C::FN - 1] >> P.sh;
}

// Shifted scales of step `ta` (of the whole reduction), the run's first or
// last: blocks wholly outside [lo, hi) get the neutral scale 127, so
// zero-filled data never meets a NaN scale byte.  A block that only partly
// overlaps [lo, hi) (a bound that is not a multiple of 32) keeps its scale:
// its in-range elements are real data.
template <class C>
__device__ __forceinline__ void mask_scales(const Plan<C>& P, int ta, int lo, int hi, uint32_t (&xs)[C::FM],
                                            uint32_t (&ws)[C::FN]) {
  const int k0 = ta * STEP + 4 * P.sh, k1 = k0 + 64;   // block of the lane in each half step
  uint32_t am = 0xffffffffu;
  if (k0 + 32 <= lo || k0 >= hi) am &= 0xffffff00u;
  if (k1 + 32 <= lo || k1 >= hi) am &= 0xff00ffffu;
  const uint32_t om = 0x7f7f7f7fu & ~am;
#pragma unroll
  for (int i = 0; i < C::FM; ++i) xs[i] = (xs[i] & am) | om;
#pragma unroll
  for (int j = 0; j < C::FN; ++j) ws[j] = (ws[j] & am) | om;
}

// MFMA T of a half step (row block T / FN, column block T % FN), scale byte
// OPS of the shifted dwords.
template <class C, int T, int OPS>
__device__ __forceinline__ void mfma1(const Frags<C>& F, const uint32_t (&xs)[C::FM], const uint32_t (&ws)[C::FN],
                                      v16f (&acc)[C::FM][C::FN]) {
  constexpr int i = T / C::FN, j = T % C::FN;
  acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(F.a[j], F.b[i], acc[i][j], C::WFMT, MXGG_FMT_E4M3, OPS,
                                                               (int)ws[j], OPS, (int)xs[i]);
}

// Keep the MFMA operand registers of a region allocated until the region's
// end.  The compiler does not guard the scale operands of v_mfma_scale_* as
// in-flight reads, so a register freed by an MFMA's last use could otherwise be
// rewritten by the very next VALU instruction while the MFMA still reads it.
template <class FR, int NM, int NN>
__device__ __forceinline__ void hold(const FR& F, const uint32_t (&xs)[NM], const uint32_t (&ws)[NN]) {
#if defined(__HIP_DEVICE_COMPILE__)   // VGPR constraints exist only in the device pass
#pragma unroll
  for (int i = 0; i < NM; ++i) asm volatile("" ::"v"(xs[i]), "v"(F.b[i]));
#pragma unroll
  for (int j = 0; j < NN; ++j) asm volatile("" ::"v"(ws[j]), "v"(F.a[j]));
#endif
}

// Keep the accumulators in AGPRs here, as values the compiler knows nothing
// of.  Left alone, the allocator shuffles all 256 of them, and spills
// fragments, on the way into the steps after the loop and into the epilogue;
// and zeros that it knows of it writes once more on the path that skips the
// loop, with 384 moves to bring both paths together (256 x 256 tiles of 512
// elements, one per CU: 16.9 us, pinned after the clearing too 15.9).
template <class C>
__device__ __forceinline__ void pin_acc(v16f (&acc)[C::FM][C::FN]) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) asm volatile("" : "+a"(acc[i][j]));
#endif
}

template <class C>
__device__ __forceinline__ void zero_acc(v16f (&acc)[C::FM][C::FN]) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) acc[i][j] = (v16f){};
}

// MFMAs P0 .. of step t (relative to the run's first), with what is issued
// beside each.  KIND: kStepFull also copies step t + 2 into this step's slot;
// kStepNoCopy, the last but one, does not; kStepLast only multiplies.
//   MFMA 0 .. RD-1:     read the second half step's fragments (F1)
//   before MFMA PB1:    barrier: every wave has read this slot, so
//   MFMA PB1 ..:        the copies of step t + 2 go into it, one per MFMA
//   before MFMA PB2:    the copies of step t + 1 (older than the `issued`
//                       ones of step t + 2) have landed; barrier
//   MFMA PB2 ..:        read the first half step of step t + 1 (F0, free
//                       since MFMA NMMA - 1) and its scales
// A scheduling fence after every MFMA keeps the order.  With a wave alone on
// its SIMD every other instruction between two MFMAs is issue time the matrix
// core waits for: 256 x 256 tiles issue 131 to 136 per step of 32 MFMAs.
constexpr int kStepFull = 0, kStepNoCopy = 1, kStepLast = 2;
template <class C, int KIND, int P0>
__device__ __forceinline__ void step_pos(uint8_t* smem, const Operand& X, const Operand& W, __amdgpu_buffer_rsrc_t ssr,
                                         Plan<C>& P, int t, Frags<C>& F0, Frags<C>& F1, uint32_t (&xc)[C::FM],
                                         uint32_t (&wc)[C::FN], uint32_t (&xn)[C::FM], uint32_t (&wn)[C::FN],
                                         v16f (&acc)[C::FM][C::FN]) {
  if constexpr (P0 < 2 * C::NMMA) {
    constexpr int NF = C::FM + C::FN;
    if constexpr (KIND == kStepFull && P0 == C::PB1) {
      MXGG_WAIT_LGKM();
      MXGG_BARRIER();
      MXGG_SCHED_FENCE();
    }
    if constexpr (KIND != kStepLast && P0 == C::PB2) {
      constexpr int issued = KIND == kStepFull ? C::NC * (C::PB2 - C::PB1) / C::NMMA : 0;
      MXGG_WAIT_VM(issued);
      MXGG_BARRIER();
      MXGG_SCHED_FENCE();
    }
    if constexpr (P0 < C::NMMA)
      mfma1<C, P0, 0>(F0, xc, wc, acc);
    else
      mfma1<C, P0 - C::NMMA, 2>(F1, xc, wc, acc);
    if constexpr (P0 < C::RD) read_frags<C, 1, P0 * NF / C::RD, (P0 + 1) * NF / C::RD>(smem, P, F1);
    if constexpr (P0 == C::RD) toggle_reads<C, 1>(P);
    if constexpr (KIND == kStepFull && P0 >= C::PB1 && P0 < C::PB1 + C::NMMA) {
      constexpr int q = P0 - C::PB1;
      if constexpr (q == 0) issue_scales<C>(ssr, P, t);
      step_copies<C, q * C::NC / C::NMMA, (q + 1) * C::NC / C::NMMA>(X, W, P, CopyOff{P.xe, P.xo, P.we, P.wo});
    }
    if constexpr (KIND != kStepLast && P0 >= C::PB2 && P0 < C::PB2 + C::RD) {
      constexpr int q = P0 - C::PB2;
      read_frags<C, 0, q * NF / C::RD, (q + 1) * NF / C::RD>(smem, P, F0);
      if constexpr (q == C::RD - 1) read_scales<C>(smem, P, t + 1, xn, wn);
    }
    MXGG_SCHED_FENCE();
    step_pos<C, KIND, P0 + 1>(smem, X, W, ssr, P, t, F0, F1, xc, wc, xn, wn, acc);
  }
}

template <class C, int KIND>
__device__ __forceinline__ void run_step(uint8_t* smem, const Operand& X, const Operand& W, __amdgpu_buffer_rsrc_t ssr,
                                         Plan<C>& P, int t, Frags<C>& F0, Frags<C>& F1, uint32_t (&xc)[C::FM],
                                         uint32_t (&wc)[C::FN], v16f (&acc)[C::FM][C::FN]) {
  uint32_t xn[C::FM], wn[C::FN];
  step_pos<C, KIND, 0>(smem, X, W, ssr, P, t, F0, F1, xc, wc, xn, wn, acc);
  hold(F1, xc, wc);
  if constexpr (KIND == kStepFull) {
    toggle_reads<C, 0>(P);
    shift_scales<C>(P, xn, wn, xc, wc);
  } else if constexpr (KIND == kStepNoCopy) {
    // (outside the loop nothing ties the new scales to the old ones' registers:
    // hold those until the new ones are written)
    toggle_reads<C, 0>(P);
    uint32_t xs[C::FM], ws[C::FN];
    shift_scales<C>(P, xn, wn, xs, ws);
    hold(F1, xc, wc);
#pragma unroll
    for (int i = 0; i < C::FM; ++i) xc[i] = xs[i];
#pragma unroll
    for (int j = 0; j < C::FN; ++j) wc[j] = ws[j];
  } else {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");   // the last MFMA reads its scales before they are reused
#endif
  }
  MXGG_SCHED_FENCE();
}

// The plan's lane offsets moved on to the next step.
template <class C>
__device__ __forceinline__ void advance(Plan<C>& P, const Operand& X, const Operand& W) {
  const uint32_t dx = (uint32_t)C::XROW << X.pl, dw = (uint32_t)C::WROW << W.pl;
  P.xe += dx;
  P.xo += dx;
  P.we += dw;
  P.wo += dw;
}

// acc = the reduction over the elements [lo, hi) (chunks and scale blocks
// outside are zero / neutral), run as the whole 128-element steps it touches,
// one at least.  Steps alternate between
// two LDS slots; while step t is multiplied, step t + 1 lies in the other slot
// and the copies of step t + 2 go into t's own as soon as every wave has read
// it, so they have about a step and a half to land.
// Bound by power and MFMA issue: 256 x 256 e4m3 tiles, M = N = K = 8192, 2.9
// PFLOP/s; 64-element stages in a 3- to 4-deep ring, whose 10 to 13
// instructions per MFMA kept the matrix cores waiting, reached 2.45.
template <class C>
__device__ __forceinline__ void step_mainloop(uint8_t* smem, const Operand& X, const Operand& W, const ScaleSrc& xss,
                                              const ScaleSrc& wss, int lo, int hi, v16f (&acc)[C::FM][C::FN]) {
  lo = uniform(lo);
  hi = uniform(hi);
  const int t0 = lo / STEP;
  int n = (hi + STEP - 1) / STEP - t0;   // steps of the run
  if (n < 1) n = 1;
  Plan<C> P;
  make_plan<C>(P, smem, X, W, xss, wss, t0);
  // the scale buffer this wave copies from (wave-uniform)
  const __amdgpu_buffer_rsrc_t ssr =
      (C::PS ? wave_id() < C::NXW : wave_id() % C::NSD < C::NSX) ? xss.rsrc : wss.rsrc;
  // units of X (16 elements) and W (e2m1: 32) of a step inside [lo, hi): of
  // the first step those from xlo / wlo on (and below its own end), of the
  // last those below xhi / whi
  constexpr int WE = C::F4 ? 32 : 16;
  const int r0 = lo - t0 * STEP, h0 = hi - t0 * STEP, h1 = hi - (t0 + n - 1) * STEP;
  const int xhi = h1 > 0 ? h1 / 16 : 0, whi = h1 > 0 ? h1 / WE : 0;
  P.mxe = P.ux < xhi ? 0 : kOOB;
  P.mxo = (P.ux ^ 1) < xhi ? 0 : kOOB;
  P.mwe = P.uw < whi ? 0 : kOOB;
  P.mwo = (C::F4 ? P.uw : P.uw ^ 1) < whi ? 0 : kOOB;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 4" ::: "memory");   // scalar operands of the asm copies written by vector instructions
#endif
#pragma unroll
  for (int i = 0; i < (C::PS ? C::SPW : 1); ++i) {   // scale group 0
    set_m0(P.sm0 + (uint32_t)(i * 1024));
    copy16<0>(ssr, P.sv, P.s_step * (uint32_t)i);
  }
  step_copies<C, 0, C::NC>(X, W, P, mask_copies<C>(P, (r0 + 15) / 16, h0 / 16, (r0 + WE - 1) / WE, h0 / WE));
  P.xm0 ^= (uint32_t)C::XBYTES;
  P.wm0 ^= (uint32_t)C::WBYTES;
  advance<C>(P, X, W);
  mask_end<C>(P, 1, n);
  step_copies<C, 0, C::NC>(X, W, P, CopyOff{P.xe, P.xo, P.we, P.wo});
  MXGG_SCHED_FENCE();
  zero_acc<C>(acc);      // while the copies fly
  pin_acc<C>(acc);
  MXGG_SCHED_FENCE();
  MXGG_WAIT_VM(C::NC);
  MXGG_BARRIER();
  Frags<C> F0, F1;
  uint32_t xc[C::FM], wc[C::FN];
  read_frags<C, 0, 0, C::FM + C::FN>(smem, P, F0);
  toggle_reads<C, 0>(P);
  {
    uint32_t xn[C::FM], wn[C::FN];
    read_scales<C>(smem, P, 0, xn, wn);
    shift_scales<C>(P, xn, wn, xc, wc);
  }
  mask_scales<C>(P, t0, lo, hi, xc, wc);
  MXGG_SCHED_FENCE();
  // A run of one step (a wgrad group inside it, K <= 128) goes straight to the
  // last one: as two steps, the second adding zeros, wgrad (8, 1024, 2048,
  // 2048) of 128 tokens a group took 20.1 us, now 19.4.
  if (n > 1) {
    int t = 0;
#pragma nounroll
    for (; t < n - 2; ++t) {
      advance<C>(P, X, W);
      mask_end<C>(P, t + 2, n);
      P.xm0 ^= (uint32_t)C::XBYTES;
      P.wm0 ^= (uint32_t)C::WBYTES;
      run_step<C, kStepFull>(smem, X, W, ssr, P, t, F0, F1, xc, wc, acc);
    }
    pin_acc<C>(acc);
    run_step<C, kStepNoCopy>(smem, X, W, ssr, P, t, F0, F1, xc, wc, acc);
    mask_scales<C>(P, t0 + n - 1, lo, hi, xc, wc);
    pin_acc<C>(acc);
  }
  run_step<C, kStepLast>(smem, X, W, ssr, P, n - 1, F0, F1, xc, wc, acc);
  pin_acc<C>(acc);
  MXGG_WAIT_VM(0);       // (one step: the second one's zero fills)
}

// The in-range elements of the 16-element chunk at cs (a multiple of 16)
// that straddles a bound of the reduction range [lo, hi).  The main loop copies
// whole chunks only, so a bound that is not a multiple of 16 leaves these
// out; they are added here as one more 64-element MFMA step whose fragments
// are loaded into registers, every element outside [lo, hi) and every other
// chunk of the step zero.  MFMA operand layout (the one read_frags builds):
// lane half h holds elements 16h .. 16h+15 of the step in dwords 0-3 and
// 32+16h .. 32+16h+15 in dwords 4-7, and supplies the scale of the step's
// block h (elements 32h .. 32h+31).  e4m3 on both sides (the weight
// gradient's operands).
template <class C>
__device__ __forceinline__ void edge_chunk(const Operand& X, const Operand& W, const ScaleSrc& xss,
                                           const ScaleSrc& wss, int cs, int lo, int hi,
                                           v16f (&acc)[C::FM][C::FN]) {
  static_assert(!C::F4 && !C::PS, "edge chunks: e4m3 operands, step-major scales only");
  const int wave = wave_id();
  const int lane = threadIdx.x % kWave;
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  const int h = lane >> 5, r32 = lane & 31;
  const int kb = cs & ~(HALF - 1);                 // the half step holding the chunk
  const int ci = (cs - kb) >> 4;                   // chunk of the step: half (ci & 1), dwords 4 (ci >> 1) ..
  const bool mine = h == (ci & 1);
  // bytes b of the chunk with lo <= cs + b < hi
  uint32_t mk[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    uint32_t m = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int k = cs + 4 * d + b;
      m |= (k >= lo && k < hi) ? (0xffu << (8 * b)) : 0u;
    }
    mk[d] = mine ? m : 0u;
  }
  Frags<C> F;
  uint32_t xs[C::FM], ws[C::FN];
  const int t = kb / STEP;
  const int blk = (kb / 32 + h) & 3;               // byte of the lane's block in the step's dword
  const bool live = kb + 32 * h < hi && kb + 32 * h + 32 > lo;
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
    const uint32_t row = (uint32_t)(wm * C::WTM + i * 32 + r32);
    const v4i v =
        __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(X.data, operand_off(X, row, (uint32_t)cs), 0, 0));
    v8i f = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int w = v[d] & (int)mk[d];
      if (ci >> 1) f[4 + d] = w; else f[d] = w;
    }
    F.b[i] = f;
    const uint32_t s = __builtin_amdgcn_raw_buffer_load_b32(xss.rsrc, ((uint32_t)t * xss.rows + xss.row0 + row) * 4u, 0, 0);
    xs[i] = live ? (s >> (8 * blk)) & 0xffu : 127u;
  }
#pragma unroll
  for (int j = 0; j < C::FN; ++j) {
    const uint32_t row = (uint32_t)(wn * C::WTN + j * 32 + r32);
    const v4i v =
        __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(W.data, operand_off(W, row, (uint32_t)cs), 0, 0));
    v8i f = (v8i){0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int w = v[d] & (int)mk[d];
      if (ci >> 1) f[4 + d] = w; else f[d] = w;
    }
    F.a[j] = f;
    const uint32_t s = __builtin_amdgcn_raw_buffer_load_b32(wss.rsrc, ((uint32_t)t * wss.rows + wss.row0 + row) * 4u, 0, 0);
    ws[j] = live ? (s >> (8 * blk)) & 0xffu : 127u;
  }
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(F.a[j], F.b[i], acc[i][j], C::WFMT, MXGG_FMT_E4M3, 0,
                                                                   (int)ws[j], 0, (int)xs[i]);
  hold(F, xs, ws);
  // What follows (a second edge step, the epilogue) may reuse these operand
  // registers at once; the compiler does not count the scale operands as
  // in-flight MFMA reads, so give the last MFMA time to read them.
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#endif
}

// Edge chunks of [lo, hi) (see edge_chunk): the chunk holding lo when lo is
// not a multiple of 16, and the one holding hi when hi is not (once when
// they are the same chunk).
template <class C>
__device__ __forceinline__ void edge_chunks(const Operand& X, const Operand& W, const ScaleSrc& xss,
                                            const ScaleSrc& wss, int lo, int hi, v16f (&acc)[C::FM][C::FN]) {
  if (hi <= lo) return;
  const int clo = lo & ~15, chi = hi & ~15;
  if (lo & 15) edge_chunk<C>(X, W, xss, wss, clo, lo, hi, acc);
  if ((hi & 15) && !((lo & 15) && chi == clo)) edge_chunk<C>(X, W, xss, wss, chi, lo, hi, acc);
}

// Store 4 consecutive output columns c .. c+3 of row r (those below `cols`)
// of a row-major output of element type out_dtype.  vec: rows and `out`
// aligned for one 16-byte (f32) or 8-byte (16-bit) store of the four.
// BF16_ONLY: round to bf16 first whatever the output type (wgrad semantics).
template <bool BF16_ONLY>
__device__ __forceinline__ void store4(uint8_t* out, int64_t ldo, int out_dtype, bool vec, int r, int c,
                                       int cols, float v0, float v1, float v2, float v3) {
  // f32 and f16 outputs of BF16_ONLY hold the bf16-rounded value (f16:
  // converted from it)
  if (out_dtype == MXGG_DTYPE_F32) {
    if (BF16_ONLY) {
      v0 = round_bf16(v0); v1 = round_bf16(v1); v2 = round_bf16(v2); v3 = round_bf16(v3);
    }
    float* p = reinterpret_cast<float*>(out) + (int64_t)r * ldo + c;
    if (vec && c + 3 < cols) {
      *reinterpret_cast<float4*>(p) = make_float4(v0, v1, v2, v3);
    } else {
      if (c + 0 < cols) p[0] = v0;
      if (c + 1 < cols) p[1] = v1;
      if (c + 2 < cols) p[2] = v2;
      if (c + 3 < cols) p[3] = v3;
    }
  } else {
    uint32_t w0, w1;
    if (out_dtype == MXGG_DTYPE_BF16) {
      w0 = pack_bf16x2(v0, v1);
      w1 = pack_bf16x2(v2, v3);
    } else {
      if (BF16_ONLY) {
        v0 = round_bf16(v0); v1 = round_bf16(v1); v2 = round_bf16(v2); v3 = round_bf16(v3);
      }
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      h2 a = {(_Float16)v0, (_Float16)v1}, b = {(_Float16)v2, (_Float16)v3};
      w0 = __builtin_bit_cast(uint32_t, a);
      w1 = __builtin_bit_cast(uint32_t, b);
    }
    uint16_t* p = reinterpret_cast<uint16_t*>(out) + (int64_t)r * ldo + c;
    if (vec && c + 3 < cols) {
      *reinterpret_cast<uint2*>(p) = make_uint2(w0, w1);
    } else {
      if (c + 0 < cols) p[0] = (uint16_t)(w0 & 0xffff);
      if (c + 1 < cols) p[1] = (uint16_t)(w0 >> 16);
      if (c + 2 < cols) p[2] = (uint16_t)(w1 & 0xffff);
      if (c + 3 < cols) p[3] = (uint16_t)(w1 >> 16);
    }
  }
}

__device__ __forceinline__ bool store4_vec(const uint8_t* out, int64_t ldo, int out_dtype) {
  return out_dtype == MXGG_DTYPE_F32 ? ((ldo % 4) == 0 && ((uintptr_t)out % 16) == 0)
                                     : ((ldo % 4) == 0 && ((uintptr_t)out % 8) == 0);
}

// The lane, as an epilogue starts from it.  256 x 256 tiles: a value of its
// own, so that none of the epilogue's addresses is computed, and kept or
// spilled, before the main loop.  Smaller tiles have the registers, and the
// time: their addresses are computed while the first copies fly (wgrad (8,
// 1280, 2048, 2048), 128 x 128 tiles: 20.5 us, 21.1 computed after the loop).
template <class C>
__device__ __forceinline__ int store_lane() {
  int lane = threadIdx.x % kWave;
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (C::FM * C::FN >= 16) asm volatile("" : "+v"(lane));
#endif
  return lane;
}

// Store an accumulator tile.  Lane l of fragment (i, j) holds output row
// wm*WTM + 32i + l%32 and columns wn*WTN + 32j + 8(q/4) + 4(l/32) + q%4.
template <class C, bool BF16_ONLY>
__device__ __forceinline__ void store_tile(const v16f (&acc)[C::FM][C::FN], uint8_t* out,
                                           int64_t ldo, int rows, int cols, int out_dtype) {
  const int wave = wave_id();
  const int lane = store_lane<C>();
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  const bool vec = store4_vec(out, ldo, out_dtype);
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
    const int r = wm * C::WTM + i * 32 + (lane & 31);
    if (r >= rows) continue;
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int c = wn * C::WTN + j * 32 + 8 * q4 + 4 * (lane >> 5);
        store4<BF16_ONLY>(out, ldo, out_dtype, vec, r, c, cols, acc[i][j][4 * q4 + 0], acc[i][j][4 * q4 + 1],
                          acc[i][j][4 * q4 + 2], acc[i][j][4 * q4 + 3]);
      }
    }
  }
}

// fp32 partial tile of a split unit, in accumulator-register order: values
// 4q .. 4q+3 of lane l of fragment f = (wave * FM + i) * FN + j are the float4
// at index (f * 4 + q) * 64 + l of the unit's BM x BN slot, so every store
// instruction writes one contiguous 1 KB run.  (With a lane's 16 values
// contiguous instead, each instruction scatters 64 16-byte pieces over 4 KB
// and the partial store takes about four times as long.)
template <class C>
__device__ __forceinline__ void store_partial(const v16f (&acc)[C::FM][C::FN], float* slot) {
  const int wave = wave_id();
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      float4* d = reinterpret_cast<float4*>(slot) + (int64_t)((wave * C::FM + i) * C::FN + j) * 4 * kWave + lane;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        d[q * kWave] =
            make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
    }
}

// Store an accumulator tile through LDS so that every global store
// instruction writes whole row segments (1 KB of 2 rows of f32, 4 of 16 bits;
// straight from the registers it would be 32 bytes of each of 32 rows: f32
// wgrad (8, 2080, 2048, 2048) 51 us that way and 43 staged): each
// wave transposes its WTM x WTN tile into its own LDS area (rows of WTN output
// elements, 16-byte chunks XOR-swizzled by row), then 64 lanes store 64
// consecutive 16-byte chunks.  Tiles larger than the free LDS go in passes of
// whole 32-row fragment rows.  Requires rows that are multiples of 16 bytes
// and a 16-byte aligned `out`; the caller must have drained every LDS-DMA load
// and the workgroup must be past its last main-loop LDS read (this function
// begins with a workgroup barrier).
// Largest divisor of fm not above lim (fragment rows per staging pass).
constexpr int store_pass_rows(int fm, int lim) {
  int best = 1;
  for (int d = 1; d <= fm; ++d)
    if (fm % d == 0 && d <= lim) best = d;
  return best;
}

// DT: the output type, fixed at compile time so the staging loop carries no
// per-write type test.  RB16 (f16, f32): store the bf16-rounded value (the
// weight gradient's semantics).
template <class C, int DT, bool RB16 = false>
__device__ __forceinline__ void store_tile_lds(const v16f (&acc)[C::FM][C::FN], uint8_t* smem,
                                               uint8_t* out, int64_t ldo, int rows, int cols) {
  constexpr int ES = DT == MXGG_DTYPE_F32 ? 4 : 2;
  constexpr int EPC = 16 / ES;                   // elements per 16-byte chunk
  constexpr int RB = C::WTN * ES;                // staged row bytes
  constexpr int NCH = RB / 16;                   // 16-byte chunks per row
  constexpr int AVAIL = C::LDS / C::NW;           // LDS bytes per wave
  constexpr int FPP = store_pass_rows(C::FM, AVAIL / (32 * RB));   // fragment rows per pass
  static_assert(FPP >= 1 && C::FM % FPP == 0, "store staging");
  static_assert(64 % NCH == 0, "store row width");
  const int wave = wave_id();
  const int lane = store_lane<C>();
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  uint8_t* area = smem + wave * (FPP * 32 * RB);
  // a wave's rows and columns all inside the output: no per-store checks
  const bool whole = (wm + 1) * C::WTM <= rows && (wn + 1) * C::WTN <= cols;
#pragma unroll
  for (int i0 = 0; i0 < C::FM; i0 += FPP) {
    __syncthreads();
#pragma unroll
    for (int ii = 0; ii < FPP; ++ii) {
      const int m = ii * 32 + (lane & 31);
#pragma unroll
      for (int j = 0; j < C::FN; ++j) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const v16f& a = acc[i0 + ii][j];
          float f0 = a[4 * q4 + 0], f1 = a[4 * q4 + 1], f2 = a[4 * q4 + 2], f3 = a[4 * q4 + 3];
          if constexpr (DT == MXGG_DTYPE_F32) {
            const int c = 8 * j + 2 * q4 + (lane >> 5);    // 16-byte chunk (4 columns)
            if constexpr (RB16) {
              const uint32_t w0 = pack_bf16x2(f0, f1), w1 = pack_bf16x2(f2, f3);
              f0 = bf16_to_f32(w0 & 0xffffu);
              f1 = __uint_as_float(w0 & 0xffff0000u);
              f2 = bf16_to_f32(w1 & 0xffffu);
              f3 = __uint_as_float(w1 & 0xffff0000u);
            }
            *reinterpret_cast<float4*>(area + m * RB + ((c ^ (m % NCH)) * 16)) = make_float4(f0, f1, f2, f3);
          } else {
            uint32_t w0, w1;
            if constexpr (DT == MXGG_DTYPE_BF16) {
              w0 = pack_bf16x2(f0, f1);
              w1 = pack_bf16x2(f2, f3);
            } else {
              typedef _Float16 h2 __attribute__((ext_vector_type(2)));
              if constexpr (RB16) {
                f0 = round_bf16(f0); f1 = round_bf16(f1); f2 = round_bf16(f2); f3 = round_bf16(f3);
              }
              h2 x = {(_Float16)f0, (_Float16)f1};
              h2 y = {(_Float16)f2, (_Float16)f3};
              w0 = __builtin_bit_cast(uint32_t, x);
              w1 = __builtin_bit_cast(uint32_t, y);
            }
            const int c = 4 * j + q4;                      // 16-byte chunk (8 columns)
            *reinterpret_cast<uint2*>(area + m * RB + ((c ^ (m % NCH)) * 16) + 8 * (lane >> 5)) =
                make_uint2(w0, w1);
          }
        }
      }
    }
    __syncthreads();
    constexpr int RPI = 64 / NCH;                        // rows per read instruction
    if (whole) {
      // Non-temporal stores: the kernel never reads its output back, while
      // its operand copies depend on L2 hits (same-box A/B over the 36-shape
      // sweep: forward +0.6%, wgrad +1.3% geomean, up to +4% on E=8 wgrad).
#pragma unroll
      for (int it = 0; it < FPP * 32 / RPI; ++it) {
        const int r = it * RPI + lane / NCH;
        const int c = lane % NCH;
        const v4i v = *reinterpret_cast<const v4i*>(area + r * RB + ((c ^ (r % NCH)) * 16));
        const int row = wm * C::WTM + i0 * 32 + r;
        const int col = wn * C::WTN + c * EPC;
        __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(out + ((int64_t)row * ldo + col) * ES));
      }
    } else {
      // Chunks that only partly lie in the output (a column count off the
      // 16-byte grid) are the exception: their per-element branches, skipped
      // one by one, 64 times a wave in f32, cost more than the stores (wgrad
      // (4, 5280, 2880, 736): f32 50.2 us with them, 45.1 behind one test, bf16
      // 45.0 and 38.6).  16-bit rows are read from LDS eight chunks at a time
      // before their stores (forward (16, 11360, 640, 512) 12.8 us one by one,
      // 12.6); f32 gains nothing by that.
      const bool parts = cols % EPC != 0;
      const int col = wn * C::WTN + (lane % NCH) * EPC;
      const bool inside = col + EPC <= cols;             // the lane's chunk of every row
      constexpr int IT = FPP * 32 / RPI, NB = ES == 4 ? 1 : (IT < 8 ? IT : 8);
      static_assert(IT % NB == 0, "store batches");
#pragma unroll
      for (int it0 = 0; it0 < IT; it0 += NB) {
        uint4 v[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int r = (it0 + b) * RPI + lane / NCH;
          v[b] = *reinterpret_cast<const uint4*>(area + r * RB + (((lane % NCH) ^ (r % NCH)) * 16));
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int row = wm * C::WTM + i0 * 32 + (it0 + b) * RPI + lane / NCH;
          uint8_t* p = out + ((int64_t)row * ldo + col) * ES;
          if (row >= rows) continue;
          if (inside) {
            *reinterpret_cast<uint4*>(p) = v[b];
          } else if (parts) {
            const uint32_t w[4] = {v[b].x, v[b].y, v[b].z, v[b].w};
#pragma unroll
            for (int e = 0; e < EPC; ++e)
              if (col + e < cols) {
                if constexpr (ES == 4)
                  reinterpret_cast<uint32_t*>(p)[e] = w[e];
                else
                  reinterpret_cast<uint16_t*>(p)[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
              }
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// scale re-layout: plain (rows, nblk) e8m0 scales -> [batch][step][row] dwords
// ---------------------------------------------------------------------------

// One operand's scales: `batches` blocks of `rows` rows (row r of batch b at
// src + b * ld_b + r * ld_r), nblk = K/32 bytes per row.  Output dword
// (b, t, r) at dst[(b * steps + t) * rows + r] holds bytes 4t .. 4t+3 of the
// row; bytes past nblk are 127 (2**0), so a partial last step needs no
// masking in the GEMM.
struct ScaleJob {
  const uint8_t* src; int64_t ld_r; int64_t ld_b;
  uint32_t* dst; int rows; int batches; int nblk; int steps;
  int tiles_r; int tiles_t;      // 64-row x 16-step tiles per batch
};

// An e4m3 operand copied from rows into row pairs (the layout the GEMM
// copies in whole 128-byte lines): `batches` blocks of `rows` rows (even) of
// `len` bytes, row r of batch b at src + b * ld_b + r * ld_r (16-byte
// aligned); byte k of row r of batch b goes to dst + b * rows * ld_dst +
// (r / 2) * 2 * ld_dst + (k / 64) * 128 + (r % 2) * 64 + k % 64, ld_dst =
// len rounded up to 64, bytes past len zero.
struct PairJob {
  const uint8_t* src; int64_t ld_r; int64_t ld_b;
  uint8_t* dst; int ld_dst; int pairs; int batches; int len;   // pairs = rows / 2
};

struct ScaleJobs {
  ScaleJob j[2];
  int tiles0;                    // workgroups of job 0 (job 1 follows)
  int tiles01;                   // workgroups of jobs 0 and 1 (pair job d follows)
  PairJob d;
  int tiles_d;                   // workgroups of pair job d (pair job d2 follows)
  PairJob d2;
};

// Pair job, workgroup w: row pair q of batch b (w = b * pairs + q), its
// 2 * ld_dst output bytes in 16-byte chunks, consecutive threads on
// consecutive chunks (coalesced stores; four threads read one 64-byte row
// piece).  The source is read once: non-temporal loads.
__device__ __forceinline__ void pair_chunks(const PairJob& J, int w) {
  const int b = w / J.pairs, q = w - b * J.pairs;
  const uint8_t* src = J.src + b * J.ld_b + (int64_t)(2 * q) * J.ld_r;
  uint8_t* dst = J.dst + ((int64_t)b * J.pairs + q) * 2 * J.ld_dst;
  for (int o = 16 * (int)threadIdx.x; o < 2 * J.ld_dst; o += 16 * 256) {
    const int h = (o >> 6) & 1, k = (o >> 7) * 64 + (o & 63);
    v4i v = {0, 0, 0, 0};
    if (k < J.len) v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(src + h * J.ld_r + k));
    *reinterpret_cast<v4i*>(dst + o) = v;
  }
}

// 64 rows x 16 steps per workgroup (256 threads): each thread reads 16
// source bytes of one row (4 steps; one 16-byte load, aligned or not, where
// the chunk lies inside the row -- rows of K/32 = 90 or M/32 = 65, 520 bytes
// are common, and byte loads took 14.9 us for E = 32, M = 16640, N = K = 2880
// where this takes 9.3), the tile is transposed through LDS, and each thread
// writes the dwords of 4 consecutive rows for one step (one 16-byte store
// when aligned and inside the operand).
__global__ __launch_bounds__(256) void scale_relayout_kernel(ScaleJobs js) {
  __shared__ uint32_t tile[16][65];
  int bid = blockIdx.x;
  if (bid >= js.tiles01) {
    bid -= js.tiles01;
    if (bid < js.tiles_d)
      pair_chunks(js.d, bid);
    else
      pair_chunks(js.d2, bid - js.tiles_d);
    return;
  }
  const int which = bid < js.tiles0 ? 0 : 1;
  const ScaleJob& J = js.j[which];
  if (which) bid -= js.tiles0;
  const int per_batch = J.tiles_r * J.tiles_t;
  const int b = bid / per_batch;
  const int rt = (bid % per_batch) % J.tiles_r;
  const int tt = (bid % per_batch) / J.tiles_r;
  const int r0 = rt * 64, t0 = tt * 16;
  {
    const int r = r0 + threadIdx.x / 4;
    const int tq = threadIdx.x % 4;                // steps t0 + 4 tq .. + 3
    const int blk0 = 4 * t0 + 16 * tq;             // first scale byte of the chunk
    uint32_t v[4] = {0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu};
    if (r < J.rows && blk0 < J.nblk) {
      const uint8_t* src = J.src + (int64_t)b * J.ld_b + (int64_t)r * J.ld_r + blk0;
      if (blk0 + 16 <= J.nblk) {
        __builtin_memcpy(v, src, 16);   // one 16-byte load at any alignment
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          uint32_t w = 0;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int i = 4 * s + q;
            const uint32_t byte = blk0 + i < J.nblk ? (uint32_t)src[i] : 127u;
            w |= byte << (8 * q);
          }
          v[s] = w;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) tile[4 * tq + s][threadIdx.x / 4] = v[s];
  }
  __syncthreads();
  {
    const int ts = threadIdx.x / 16;               // step of the tile
    const int rq = threadIdx.x % 16;               // rows 4 rq .. 4 rq + 3
    const int t = t0 + ts;
    const int r = r0 + 4 * rq;
    if (t < J.steps && r < J.rows) {
      uint32_t* out = J.dst + ((int64_t)b * J.steps + t) * J.rows + r;
      if (r + 4 <= J.rows && ((uintptr_t)out & 15) == 0) {
        *(uint4*)out = make_uint4(tile[ts][4 * rq], tile[ts][4 * rq + 1], tile[ts][4 * rq + 2],
                                  tile[ts][4 * rq + 3]);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (r + q < J.rows) out[q] = tile[ts][4 * rq + q];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// forward / dgrad
// ---------------------------------------------------------------------------

struct FwdParams {
  const uint8_t* a; int64_t lda;
  const uint8_t* b; int64_t ldb_n; int64_t ldb_e;
  // A scales: step-major [T][M] dwords (T = cdiv(K, 128)), or (plain-scale
  // kernels, Cfg::PS) to_mx's (M, K/32) bytes with row stride as_ld; B
  // scales: step-major [E][T][N] dwords, or plain (E, N, K/32) with row
  // stride bs_ld.  as_bytes / bs_bytes: bytes of A's / of one expert's scales
  // that may be read; bs_expert: bytes from one expert's scales to the next.
  const uint8_t* as; uint32_t as_bytes;
  const uint8_t* bs; uint32_t bs_bytes; uint32_t bs_expert;
  const int32_t* offs; int E; int64_t M; int64_t N; int64_t K;
  uint8_t* out; int out_dtype; int64_t ldo;
  int grid_n; int group_m; int xcd;
  float* part; int par; int slots;          // split: partial slots, resident workgroups, slot count
  int quads;                                // the last round may run as 128 x 128 quarter tiles (fwd_plan)
  int a_pl; int b_pl;                       // operand layouts: 0 rows, 1 row pairs, 2 row quads (Operand)
  uint32_t as_ld; uint32_t bs_ld;           // plain scales: bytes per row (multiples of 16)
};

// Epilogue of the whole-tile kernels, fixed at compile time so that the
// common case carries none of the others' register pressure (with every
// variant in one kernel the allocator spilled accumulators to scratch and
// reloaded them serially in the epilogue): kEpiBf16 / kEpiF16 / kEpiF32 are
// outputs whose rows are 16-byte aligned (row stride a multiple of 16 bytes,
// 16-byte aligned base), staged through LDS; kEpiBf16Any / kEpiF16Any /
// kEpiF32Any rows off the 16-byte grid, stored from the registers.
constexpr int kEpiBf16 = 1, kEpiF16 = 2, kEpiF32 = 3, kEpiBf16Any = 4, kEpiF16Any = 5, kEpiF32Any = 6;

// Epilogue of a whole-tile launch for this output (host side).
inline int pick_epi(int out_dtype, int64_t ldo, const void* out) {
  const bool f32 = out_dtype == MXGG_DTYPE_F32;
  const bool al16 = ldo % (f32 ? 4 : 8) == 0 && (uintptr_t)out % 16 == 0;
  if (f32) return al16 ? kEpiF32 : kEpiF32Any;
  if (out_dtype == MXGG_DTYPE_BF16) return al16 ? kEpiBf16 : kEpiBf16Any;
  return al16 ? kEpiF16 : kEpiF16Any;
}

// Store tile acc at `out` (the tile's first element) by epilogue EPI.
// BF16_ONLY: the bf16-rounded value whatever the output type (wgrad).
template <class C, int EPI, bool BF16_ONLY>
__device__ __forceinline__ void store_epi(const v16f (&acc)[C::FM][C::FN], uint8_t* smem, uint8_t* out, int64_t ldo,
                                          int rows, int cols) {
  constexpr int dt = EPI == kEpiF32 || EPI == kEpiF32Any ? MXGG_DTYPE_F32
                     : EPI == kEpiF16 || EPI == kEpiF16Any ? MXGG_DTYPE_F16
                                                           : MXGG_DTYPE_BF16;
  if constexpr (EPI == kEpiBf16 || EPI == kEpiF16 || EPI == kEpiF32)
    store_tile_lds<C, dt, BF16_ONLY>(acc, smem, out, ldo, rows, cols);
  else
    store_tile<C, BF16_ONLY>(acc, out, ldo, rows, cols, dt);
}

// Launches `call` (a macro of one epilogue) for every epilogue.
#define MXGG_EPI_SWITCH(epi, call) \
  switch (epi) {                   \
    call(kEpiBf16);                \
    call(kEpiF16);                 \
    call(kEpiF32);                 \
    call(kEpiBf16Any);             \
    call(kEpiF16Any);              \
    call(kEpiF32Any);              \
  }

struct FwdTile {
  int expert;
  int64_t row0; int rows;     // output rows row0 .. row0 + rows - 1 (one group)
  int64_t n0; int cols;       // output columns n0 .. n0 + cols - 1
};

// Tile of logical index lt (0 <= lt < tiles) after the XCD swizzle and the
// expert-aligned band order (route_tile: bands of at most GROUP_M m-blocks
// inside one group); false when it holds no output rows.  Wave-uniform.
// wg: the groups as load_groups read them when E <= 64 (else offs is read).
template <class C>
__device__ __forceinline__ bool fwd_tile(const FwdParams& p, int lt, int tiles, const WaveGroups& wg,
                                         FwdTile& tl) {
  const int t = p.xcd > 1 ? xcd_swizzle(lt, tiles, p.xcd) : lt;
  int pn;
  const TileRoute r = p.E <= kWave ? route_tile(wg, p.E, C::BM, p.grid_n, p.group_m, t, pn)
                                   : route_tile(p.offs, p.E, C::BM, p.grid_n, p.group_m, t, pn);
  if (r.expert < 0) return false;
  tl.expert = r.expert;
  tl.row0 = (int64_t)r.start + (int64_t)r.block * C::BM;
  int64_t rows64 = p.M - tl.row0;
  if (rows64 > r.rows) rows64 = r.rows;
  if (rows64 <= 0) return false;
  tl.rows = (int)rows64;
  tl.n0 = (int64_t)pn * C::BN;
  tl.cols = (int)(p.N - tl.n0 < C::BN ? p.N - tl.n0 : C::BN);
  return true;
}

// The last round of a launch of T tiles of 256 x 256 on P resident workgroups:
// whole, cut along the reduction (split_plan), or, with `quads`, as 128 x 128
// quarter tiles (fwd_quad_kernel: dp < T and no units).  Quarters need no
// partial tiles and no reduce and give a whole tile's bits; up to P / 4 tiles
// they get a CU each, up to 2 P / 5 half a CU.  Priced per step from kernel
// times (MI355X; a 128 x 128 step waits on its copies, 0.6 to 0.85 us: 25 to
// 35 us at K = 5120, 54 at K = 8192 with 8 experts): they must beat the split
// by kQuadMarginNs.  (1, 2080, 8192, 5120): 96.6 us split, 89.9 quartered; (8,
// 16640, 2048, 8192): 253 split, 262 quartered.  A reduction too short to
// split (fewer than kMinSplitTotal steps) takes the quarters whenever they get
// a CU each: a lone round of 256 x 256 tiles at K = 2048 takes about as long
// as a full round.
constexpr int kQuadNsPerStep = 650, kQuad2NsPerStep = 1000, kQuadMarginNs = 8000, kQuadMinGainNs = 3000;

__host__ __device__ inline Split fwd_plan(int T, int P, int nsteps, int slots, int tile_kib, bool quads) {
  int saved;
  const Split sp = split_plan(T, P, nsteps, slots, tile_kib, &saved);
  if (!quads || T <= 0 || P <= 0 || T / P > kSplitMaxRounds) return sp;
  const int rem = T % P;
  if (rem == 0 || 5 * rem > 2 * P) return sp;
  const bool one = 4 * rem <= P;
  const int n = nsteps < (1 << 20) ? nsteps : (1 << 20);
  const int gain = ((int)kTailNsPerStep - (one ? kQuadNsPerStep : kQuad2NsPerStep)) * n;
  if ((one && nsteps < kMinSplitTotal) || gain >= (saved ? saved + kQuadMarginNs : kQuadMinGainNs))
    return Split{T - rem, 1, 0};
  return sp;
}

template <class C>
__device__ __forceinline__ Split fwd_split(const FwdParams& p, int tiles) {
  return fwd_plan(tiles, p.par, (int)((p.K + STEP - 1) / STEP), p.slots, C::BM * C::BN * 4 / 1024, p.quads != 0);
}

// Tile tl whole (PIECES = false; epilogue EPI), or piece `piece` of S of it
// into partial slot `slot` (PIECES = true).
template <class C, bool PIECES, int EPI>
__device__ __forceinline__ void fwd_tile_run(const FwdParams& p, uint8_t* smem, const FwdTile& tl, int piece, int S,
                                             int slot) {
  const int64_t row0 = tl.row0, n0 = tl.n0;
  const int rows = tl.rows, cols = tl.cols;

  const Operand X = make_operand(p.a, p.lda, p.a_pl, row0, rows);
  const Operand W = make_operand(p.b + (int64_t)tl.expert * p.ldb_e, p.ldb_n, p.b_pl, n0, cols);
  const ScaleSrc xs{make_rsrc(p.as, p.as_bytes), C::PS ? p.as_ld : (uint32_t)p.M, (uint32_t)row0};
  const ScaleSrc ws{make_rsrc(p.bs + (int64_t)tl.expert * p.bs_expert, p.bs_bytes), C::PS ? p.bs_ld : (uint32_t)p.N,
                    (uint32_t)n0};

  v16f acc[C::FM][C::FN];   // set by step_mainloop
  const int K = (int)p.K;
  if constexpr (PIECES) {
    int a, b;
    split_range(0, (int)((p.K + STEP - 1) / STEP), piece, S, a, b);
    const int lo = STEP * a;
    const int hi = STEP * b < K ? STEP * b : K;
    step_mainloop<C>(smem, X, W, xs, ws, lo, hi, acc);
    store_partial<C>(acc, p.part + (int64_t)slot * (C::BM * C::BN));
  } else {
    step_mainloop<C>(smem, X, W, xs, ws, 0, K, acc);
    constexpr int es = EPI == kEpiF32 || EPI == kEpiF32Any ? 4 : 2;
    store_epi<C, EPI, false>(acc, smem, p.out + (row0 * p.ldo + n0) * es, p.ldo, rows, cols);
  }
}

// Tile of logical index lt, run as fwd_tile_run describes.
template <class C, bool PIECES, int EPI>
__device__ __forceinline__ void fwd_run(const FwdParams& p, uint8_t* smem, int lt, int piece, int S, int slot,
                                        int tiles, const WaveGroups& wg) {
  FwdTile tl;
  if (fwd_tile<C>(p, lt, tiles, wg, tl)) fwd_tile_run<C, PIECES, EPI>(p, smem, tl, piece, S, slot);
}

// Groups of a forward launch and its m-block count: one read of offs when
// E <= 64 (kept for the tile lookup), else a scan of offs in 64-group chunks.
template <class C>
__device__ __forceinline__ int fwd_groups(const FwdParams& p, WaveGroups& wg) {
  if (p.E <= kWave) {
    wg = load_groups(p.offs, p.E, C::BM);
    return wg.total;
  }
  wg = WaveGroups{0, 0, 0, 0, 0};
  return route_total(p.offs, p.E, C::BM);
}

// PIECES = false: workgroup i < dp computes tile i whole (epilogue EPI).
// PIECES = true: workgroup u < units computes piece u % S of tile dp + u / S
// into partial slot u.  Other workgroups exit.  (Two kernels rather than one
// with both paths: sharing a register allocation slows the whole-tile loop by
// ~2%.)
template <class C, bool PIECES, int EPI = kEpiBf16>
__global__ __launch_bounds__(C::NT) void fwd_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
  WaveGroups wg;
  const int tiles = fwd_groups<C>(p, wg) * p.grid_n;
  const Split sp = fwd_split<C>(p, tiles);
  const int pid = blockIdx.x;
  if constexpr (PIECES) {
    if (pid < sp.units) fwd_run<C, true, kEpiBf16>(p, smem, sp.dp + pid / sp.S, pid % sp.S, sp.S, pid, tiles, wg);
  } else {
    if (pid < sp.dp) fwd_run<C, false, EPI>(p, smem, pid, 0, 1, 0, tiles, wg);
  }
}

// The last round of a launch of C tiles (256 x 256) as Q tiles (128 x 128):
// workgroup u < 4 * (tiles - dp) computes quarter u % 4 (row half u / 2 % 2,
// column half u % 2) of tile dp + u / 4, clipped to the tile; the routing and
// the plan are C's, so the whole-tile kernel and this one agree on dp.
template <class C, class Q, int EPI>
__global__ __launch_bounds__(Q::NT) void fwd_quad_kernel(FwdParams p) {
  static_assert(C::BM == 2 * Q::BM && C::BN == 2 * Q::BN && C::WFMT == Q::WFMT, "quarter tiles");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[Q::LDS];
  WaveGroups wg;
  const int tiles = fwd_groups<C>(p, wg) * p.grid_n;
  const Split sp = fwd_split<C>(p, tiles);
  if (sp.units) return;   // a last round split into pieces is not quartered
  const int dp = sp.dp;
  const int u = blockIdx.x;
  if (u >= 4 * (tiles - dp)) return;
  FwdTile tl;
  if (!fwd_tile<C>(p, dp + u / 4, tiles, wg, tl)) return;
  const int dr = (u & 2) ? Q::BM : 0, dc = (u & 1) ? Q::BN : 0;
  if (tl.rows <= dr || tl.cols <= dc) return;
  tl.row0 += dr;
  tl.rows = tl.rows - dr < Q::BM ? tl.rows - dr : Q::BM;
  tl.n0 += dc;
  tl.cols = tl.cols - dc < Q::BN ? tl.cols - dc : Q::BN;
  fwd_tile_run<Q, false, EPI>(p, smem, tl, 0, 1, 0);
}

// ---------------------------------------------------------------------------
// Few rows per group: weight streaming
// ---------------------------------------------------------------------------

// Tiles of BM_ (32 or 64) rows x 128 columns for groups of few rows, whose
// time is the read of the weight: one wave per 32 columns, NS_ LDS slots of one
// 128-element step with NS_ - 1 steps in flight, scales in two slots of 8
// steps (step-major or plain, as Cfg).  Slot layouts as Cfg's.
template <int BM_, int WFMT_, int NS_, bool PS_>
struct StreamCfg {
  static constexpr int BM = BM_, BN = 128, WGM = 1, WGN = 4, WFMT = WFMT_, NS = NS_;
  static constexpr bool PS = PS_;
  static constexpr bool F4 = WFMT == MXGG_FMT_E2M1;
  static constexpr int NW = 4, NT = NW * kWave;
  static constexpr int WTM = BM, WTN = 32, FM = BM / 32, FN = 1;
  static constexpr int XROW = STEP, WROW = F4 ? STEP / 2 : STEP;
  static constexpr int XBYTES = BM * XROW, WBYTES = BN * WROW, SLOT = XBYTES + WBYTES;
  static constexpr int GSTEPS = 8;
  static constexpr int SXB = GSTEPS * BM * 4, SSLOT = GSTEPS * (BM + BN) * 4;   // X part, slot
  static constexpr int SOFF = NS * SLOT;
  static constexpr int LDS = SOFF + 2 * SSLOT;
  static constexpr int QX = XBYTES / 1024 / NW, QW = WBYTES / 1024 / NW, NC = QX + QW;   // 1 KB copies per wave
  static constexpr int XCR = 1024 / XROW, WCR = 1024 / WROW;                            // rows per copy
  static_assert((QX == 1 || QX == 2) && (QW == 2 || QW == 4), "one M0 per operand and step");
  static_assert(NS >= 3 && NS <= GSTEPS + 1 && (NS - 2) * NC + 2 <= 63 && LDS <= 160 * 1024, "ring");
};

// acc = the whole reduction over K elements, in steps: wait for step t, start
// the copies of step t + NS - 1 into the slot of step t - 1, multiply step t.
// The same MFMAs on the same accumulators in the same order as step_mainloop:
// the same bits.
template <class C>
__device__ __forceinline__ void stream_mainloop(uint8_t* smem, const Operand& X, const Operand& W, const ScaleSrc& xss,
                                                const ScaleSrc& wss, int K, v16f (&acc)[C::FM][C::FN]) {
  const int lane = threadIdx.x % kWave;
  const int wave = wave_id();
  const int h = lane >> 5, r32 = lane & 31;
  const int n = uniform(K > STEP ? (K + STEP - 1) / STEP : 1);
  const int hl = K - (n - 1) * STEP;            // elements of the last step
  const uint32_t lds0 = lds_addr(smem);
  // lane offsets of the even and odd copies (packed e2m1 W: one)
  const int ue = (lane & 7) ^ (lane / 8);
  const int uw = C::F4 ? (lane & 3) ^ swz4(lane / 4) : ue;
  const int wrow = C::F4 ? lane / 4 : lane / 8;
  constexpr int WE = C::F4 ? 32 : 16;
  const int x1 = C::QX == 1 ? (wave & 1) : 0;   // a wave's only X copy is odd on odd waves
  uint32_t xo[2], wo[2], xm[2], wm[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int u = ue ^ (k ^ x1), w = C::F4 ? uw : uw ^ k;
    xo[k] = operand_off(X, (uint32_t)(lane / 8), (uint32_t)(u * 16));
    wo[k] = operand_off(W, (uint32_t)wrow, (uint32_t)(w * 16));
    xm[k] = u < hl / 16 ? 0u : kOOB;
    wm[k] = w < hl / WE ? 0u : kOOB;
  }
  uint32_t xs[C::QX], ws[C::QW];
#pragma unroll
  for (int i = 0; i < C::QX; ++i)
    xs[i] = (uint32_t)(C::XCR * (wave * C::QX + i)) * X.ld + (uint32_t)(kCopyBias - 1024 * i);
#pragma unroll
  for (int i = 0; i < C::QW; ++i)
    ws[i] = (uint32_t)(C::WCR * (wave * C::QW + i)) * W.ld + (uint32_t)(kCopyBias - 1024 * i);
  // scale copies: every wave 1 KB of the W part, waves below BM / 32 also 1 KB of the X part
  const bool sx = wave < C::BM / 32;
  uint32_t svx, svw, sstep_x, sstep_w;          // lane offsets; bytes per group
  if constexpr (C::PS) {
    const uint32_t half = (uint32_t)((lane ^ (lane >> 4)) & 1) * 16u;
    svx = (xss.row0 + (uint32_t)(wave * 32 + lane / 2)) * xss.rows + half;
    svw = (wss.row0 + (uint32_t)(wave * 32 + lane / 2)) * wss.rows + half;
    sstep_x = sstep_w = 32u;
  } else {
    const int qx = 256 * wave + 4 * lane;
    svx = ((uint32_t)(qx / C::BM) * xss.rows + xss.row0 + (uint32_t)(qx % C::BM)) * 4u;
    svw = ((uint32_t)(qx / C::BN) * wss.rows + wss.row0 + (uint32_t)(qx % C::BN)) * 4u;
    sstep_x = xss.rows * 4u * C::GSTEPS;
    sstep_w = wss.rows * 4u * C::GSTEPS;
  }
  const uint32_t dx = (uint32_t)C::XROW << X.pl, dw = (uint32_t)C::WROW << W.pl;
  // copies of step s (s counts up by one per call) into slot s % NS
  auto issue = [&](int s, int slot) {
    if (s >= n - 1) {                           // the last step's end, then nothing at all
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        xo[k] |= s == n - 1 ? xm[k] : kOOB;
        wo[k] |= s == n - 1 ? wm[k] : kOOB;
      }
    }
    const uint32_t sb = lds0 + (uint32_t)(slot * C::SLOT);
    set_m0(sb + (uint32_t)(wave * C::QX * 1024));
    copy16<0>(X.dma, xo[0], xs[0]);
    if constexpr (C::QX > 1) copy16<1024>(X.dma, xo[1], xs[1]);
    set_m0(sb + (uint32_t)(C::XBYTES + wave * C::QW * 1024));
    copy16<0>(W.dma, wo[0], ws[0]);
    copy16<1024>(W.dma, wo[1], ws[1]);
    if constexpr (C::QW > 2) {
      copy16<2048>(W.dma, wo[0], ws[2]);
      copy16<3072>(W.dma, wo[1], ws[3]);
    }
  };
  auto issue_scale_group = [&](int g) {
    const uint32_t sb = lds0 + (uint32_t)(C::SOFF + (g & 1) * C::SSLOT);
    if (sx) {
      set_m0(sb + (uint32_t)(wave * 1024));
      copy16<0>(xss.rsrc, svx, (uint32_t)g * sstep_x);
    }
    set_m0(sb + (uint32_t)(C::SXB + wave * 1024));
    copy16<0>(wss.rsrc, svw, (uint32_t)g * sstep_w);
  };
  auto advance = [&] {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      xo[k] += dx;
      wo[k] += dw;
    }
  };
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_nop 4" ::: "memory");   // scalar operands of the asm copies written by vector instructions
#endif
  issue_scale_group(0);
#pragma unroll
  for (int s = 0; s < C::NS - 1; ++s) {
    if (s) advance();
    issue(s, s);
  }
  zero_acc<C>(acc);
  // LDS read addresses inside a slot
  const int g = (r32 & 7) ^ ((r32 >> 3) & 1);
  uint32_t xa[4], wa[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    xa[k] = (uint32_t)(r32 * C::XROW + (((2 * k + h) ^ g) * 16));
    const int u = C::F4 ? ((2 * (k & 1) + h) ^ swz4(r32)) : ((2 * k + h) ^ g);
    wa[k] = (uint32_t)(C::XBYTES + (wave * 32 + r32) * C::WROW + u * 16);
  }
  const uint32_t sra = C::PS ? (uint32_t)(r32 * 32 + ((r32 >> 3) & 1) * 16) : (uint32_t)(r32 * 4);
  const int sh = 8 * h;
  int slot = 0, next = C::NS - 1;
#pragma nounroll
  for (int t = 0; t < n; ++t) {
    MXGG_WAIT_LGKM();                      // (this wave's reads of step t - 1)
    MXGG_WAIT_VM((C::NS - 2) * C::NC);     // this wave's copies of step t
    MXGG_BARRIER();                        // every wave's; the slot of step t - 1 is free
    MXGG_SCHED_FENCE();
    const uint8_t* sp = smem + slot * C::SLOT;
    const uint8_t* ss = smem + C::SOFF + ((t / C::GSTEPS) & 1) * C::SSLOT;
    const int u = t % C::GSTEPS;
    v8i a[2], b[2][C::FM];
    uint32_t wsc, xsc[C::FM];
    if constexpr (C::PS) {
      wsc = *reinterpret_cast<const uint32_t*>(ss + C::SXB + wave * 1024 + (sra ^ (uint32_t)(4 * u)));
#pragma unroll
      for (int i = 0; i < C::FM; ++i) xsc[i] = *reinterpret_cast<const uint32_t*>(ss + i * 1024 + (sra ^ (uint32_t)(4 * u)));
    } else {
      wsc = *reinterpret_cast<const uint32_t*>(ss + C::SXB + u * C::BN * 4 + wave * 128 + sra);
#pragma unroll
      for (int i = 0; i < C::FM; ++i) xsc[i] = *reinterpret_cast<const uint32_t*>(ss + u * C::BM * 4 + i * 128 + sra);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (C::F4) {
        const v4i l = *reinterpret_cast<const v4i*>(sp + wa[j]);
        a[j] = (v8i){l[0], l[1], l[2], l[3], 0, 0, 0, 0};
      } else {
        const v4i l = *reinterpret_cast<const v4i*>(sp + wa[2 * j]), m = *reinterpret_cast<const v4i*>(sp + wa[2 * j + 1]);
        a[j] = (v8i){l[0], l[1], l[2], l[3], m[0], m[1], m[2], m[3]};
      }
#pragma unroll
      for (int i = 0; i < C::FM; ++i) {
        const v4i l = *reinterpret_cast<const v4i*>(sp + xa[2 * j] + i * 32 * C::XROW);
        const v4i m = *reinterpret_cast<const v4i*>(sp + xa[2 * j + 1] + i * 32 * C::XROW);
        b[j][i] = (v8i){l[0], l[1], l[2], l[3], m[0], m[1], m[2], m[3]};
      }
    }
    MXGG_SCHED_FENCE();
    if (t % C::GSTEPS == 0) issue_scale_group(t / C::GSTEPS + 1);
    advance();
    issue(t + C::NS - 1, next);
    MXGG_SCHED_FENCE();
    wsc >>= sh;
#pragma unroll
    for (int i = 0; i < C::FM; ++i) xsc[i] >>= sh;
    if (t == n - 1) {                      // blocks past K: zero data, neutral scale
      uint32_t am = 0xffffffffu;
      if (32 * h >= hl) am &= 0xffffff00u;
      if (64 + 32 * h >= hl) am &= 0xff00ffffu;
      wsc = (wsc & am) | (0x7f7f7f7fu & ~am);
#pragma unroll
      for (int i = 0; i < C::FM; ++i) xsc[i] = (xsc[i] & am) | (0x7f7f7f7fu & ~am);
    }
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
      acc[i][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[0], b[0][i], acc[i][0], C::WFMT, MXGG_FMT_E4M3, 0,
                                                                   (int)wsc, 0, (int)xsc[i]);
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
      acc[i][0] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[1], b[1][i], acc[i][0], C::WFMT, MXGG_FMT_E4M3, 2,
                                                                   (int)wsc, 2, (int)xsc[i]);
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" ::"v"(wsc), "v"(a[1]));
#pragma unroll
    for (int i = 0; i < C::FM; ++i) asm volatile("" ::"v"(xsc[i]), "v"(b[1][i]));
    asm volatile("" ::"v"(xo[0]), "v"(xo[1]), "v"(wo[0]), "v"(wo[1]));
#endif
    MXGG_SCHED_FENCE();
    slot = slot + 1 == C::NS ? 0 : slot + 1;
    next = next + 1 == C::NS ? 0 : next + 1;
  }
  MXGG_WAIT_LGKM();
  MXGG_WAIT_VM(0);                         // zero fills and scale copies past the end
}

// Workgroup i computes tile i (no tile is split).
template <class C, int EPI>
__global__ __launch_bounds__(C::NT) void fwd_stream_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
  WaveGroups wg;
  const int tiles = fwd_groups<C>(p, wg) * p.grid_n;
  const int pid = blockIdx.x;
  FwdTile tl;
  if (pid >= tiles || !fwd_tile<C>(p, pid, tiles, wg, tl)) return;
  const Operand X = make_operand(p.a, p.lda, p.a_pl, tl.row0, tl.rows);
  const Operand W = make_operand(p.b + (int64_t)tl.expert * p.ldb_e, p.ldb_n, p.b_pl, tl.n0, tl.cols);
  const ScaleSrc xs{make_rsrc(p.as, p.as_bytes), C::PS ? p.as_ld : (uint32_t)p.M, (uint32_t)tl.row0};
  const ScaleSrc ws{make_rsrc(p.bs + (int64_t)tl.expert * p.bs_expert, p.bs_bytes), C::PS ? p.bs_ld : (uint32_t)p.N,
                    (uint32_t)tl.n0};
  v16f acc[C::FM][C::FN];
  stream_mainloop<C>(smem, X, W, xs, ws, (int)p.K, acc);
  constexpr int es = EPI == kEpiF32 || EPI == kEpiF32Any ? 4 : 2;
  store_epi<C, EPI, false>(acc, smem, p.out + (tl.row0 * p.ldo + tl.n0) * es, p.ldo, tl.rows, tl.cols);
}

// Sum over the S pieces (slots base + s * BM * BN, s = 0 .. S-1, in that
// order) of the 16 partial values of lane `lane` of fragment f.
template <class C>
__device__ __forceinline__ void sum_pieces(const float* base, int S, int f, int lane, float (&v)[16]) {
#pragma unroll
  for (int q = 0; q < 16; ++q) v[q] = 0.f;
  const float4* src = reinterpret_cast<const float4*>(base) + (int64_t)f * 4 * kWave + lane;
  for (int s = 0; s < S; ++s) {
    const float4* x = src + (int64_t)s * (C::BM * C::BN / 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 t = x[q * kWave];
      v[4 * q] += t.x; v[4 * q + 1] += t.y; v[4 * q + 2] += t.z; v[4 * q + 3] += t.w;
    }
  }
}

// Store the 16 values of lane `lane` of fragment f of a tile (rows x cols at
// `out`, row stride ldo).
template <class C, bool BF16_ONLY>
__device__ __forceinline__ void store_fragment_lane(const float (&v)[16], int f, int lane, uint8_t* out,
                                                    int64_t ldo, int rows, int cols, int out_dtype) {
  const int wave = f / (C::FM * C::FN), i = (f / C::FN) % C::FM, j = f % C::FN;
  const int wm = wave / C::WGN, wn = wave % C::WGN;
  const int r = wm * C::WTM + i * 32 + (lane & 31);
  if (r >= rows) return;
  const bool vec = store4_vec(out, ldo, out_dtype);
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    const int c = wn * C::WTN + j * 32 + 8 * q4 + 4 * (lane >> 5);
    store4<BF16_ONLY>(out, ldo, out_dtype, vec, r, c, cols, v[4 * q4], v[4 * q4 + 1], v[4 * q4 + 2], v[4 * q4 + 3]);
  }
}

// Fragments per tile and reduce items per tile (4 fragments, one per wave of
// a 256-thread workgroup).
template <class C>
struct ReduceShape {
  static constexpr int NF = C::NW * C::FM * C::FN;
  static constexpr int CH = NF / 4;
  static_assert(NF % 4 == 0, "reduce items");
};

// Store one reduce item: fragments 4c .. 4c+3 of a tile, fragment f = 4c +
// wave of the workgroup, with FN = 4 the column blocks j = 0 .. 3 of row
// block i of wave tile wt, i.e. 32 rows x WTN columns.  16-bit outputs with
// 16-byte aligned rows whose block lies wholly inside the tile go through LDS
// (store_item_lds), so that each global store writes 4 whole row segments of
// WTN * 2 bytes; the per-lane stores (store_fragment_lane) write 16 bytes of
// each of 32 rows instead, and serve every other output and tiles of other
// wave shapes (FN != 4).  Every wave of the workgroup calls it for the same
// item: the LDS path holds workgroup barriers, and its condition is the same
// for the four fragments.
template <class C, bool BF16_ONLY>
__device__ __forceinline__ void store_item_lds(const float (&v)[16], int f, int lane, uint8_t* out, int64_t ldo,
                                               int rows, int cols, int out_dtype, uint8_t* blk) {
  constexpr int RB = C::WTN * 2;                 // staged row bytes
  constexpr int NCH = RB / 16;                   // 16-byte chunks per row (XOR-swizzled by row in blk)
  constexpr int RPI = 64 / NCH;                  // rows per store instruction
  constexpr int RPW = 32 / C::NW;                // rows each wave stores
  static_assert(NCH <= 64 && 64 % NCH == 0 && RPW % RPI == 0, "reduce block shape");
  const int wt = f / (C::FM * C::FN), i = (f / C::FN) % C::FM, j = f % C::FN;
  const int r0 = (wt / C::WGN) * C::WTM + i * 32, c0 = (wt % C::WGN) * C::WTN;
  const bool staged = out_dtype != MXGG_DTYPE_F32 && ldo % 8 == 0 && (uintptr_t)out % 16 == 0 &&
                      r0 + 32 <= rows && c0 + C::WTN <= cols;
  if (!staged) {
    store_fragment_lane<C, BF16_ONLY>(v, f, lane, out, ldo, rows, cols, out_dtype);
    return;
  }
  const int m = lane & 31, h = lane >> 5;
  __syncthreads();                               // the previous item's reads of blk are done
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4) {
    uint32_t w0, w1;
    if (out_dtype == MXGG_DTYPE_BF16) {
      w0 = pack_bf16x2(v[4 * q4], v[4 * q4 + 1]);
      w1 = pack_bf16x2(v[4 * q4 + 2], v[4 * q4 + 3]);
    } else {
      float f0 = v[4 * q4], f1 = v[4 * q4 + 1], f2 = v[4 * q4 + 2], f3 = v[4 * q4 + 3];
      if (BF16_ONLY) {
        f0 = round_bf16(f0); f1 = round_bf16(f1); f2 = round_bf16(f2); f3 = round_bf16(f3);
      }
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      h2 x = {(_Float16)f0, (_Float16)f1}, y = {(_Float16)f2, (_Float16)f3};
      w0 = __builtin_bit_cast(uint32_t, x);
      w1 = __builtin_bit_cast(uint32_t, y);
    }
    const int c = 4 * j + q4;                    // 16-byte chunk (8 columns) of the block row
    *reinterpret_cast<uint2*>(blk + m * RB + ((c ^ (m % NCH)) * 16) + 8 * h) = make_uint2(w0, w1);
  }
  __syncthreads();
  const int wid = wave_id();
#pragma unroll
  for (int it = 0; it < RPW / RPI; ++it) {       // wave wid: rows RPW wid .. RPW wid + RPW - 1
    const int r = wid * RPW + it * RPI + lane / NCH;
    const int c = lane % NCH;
    const v4i val = *reinterpret_cast<const v4i*>(blk + r * RB + ((c ^ (r % NCH)) * 16));
    __builtin_nontemporal_store(
        val, reinterpret_cast<v4i*>(reinterpret_cast<uint16_t*>(out) + (int64_t)(r0 + r) * ldo + c0 + c * 8));
  }
}

template <class C, bool BF16_ONLY>
__device__ __forceinline__ void store_item(const float (&v)[16], int f, int lane, uint8_t* out, int64_t ldo,
                                           int rows, int cols, int out_dtype, uint8_t* blk) {
  if constexpr (C::FN == 4 && C::NW == 4)
    store_item_lds<C, BF16_ONLY>(v, f, lane, out, ldo, rows, cols, out_dtype, blk);
  else
    store_fragment_lane<C, BF16_ONLY>(v, f, lane, out, ldo, rows, cols, out_dtype);
}

// Split tiles of a forward launch: item (v, c) = fragments 4c .. 4c+3 of split
// tile v, summed over its pieces and stored.  The plan is recomputed from
// offs exactly as fwd_kernel computed it.
template <class C>
__global__ __launch_bounds__(256) void fwd_reduce_kernel(FwdParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t blk[32 * C::WTN * 2];
  WaveGroups wg;
  const int tiles = fwd_groups<C>(p, wg) * p.grid_n;
  const Split sp = fwd_split<C>(p, tiles);
  if (sp.units == 0) return;
  constexpr int CH = ReduceShape<C>::CH;
  const int rem = sp.units / sp.S;
  const int lane = threadIdx.x % kWave;
  const int esz = p.out_dtype == MXGG_DTYPE_F32 ? 4 : 2;
  for (int item = blockIdx.x; item < rem * CH; item += gridDim.x) {
    const int v = item / CH, f = (item % CH) * 4 + wave_id();
    FwdTile tl;
    if (!fwd_tile<C>(p, sp.dp + v, tiles, wg, tl)) continue;
    float acc[16];
    sum_pieces<C>(p.part + (int64_t)v * sp.S * (C::BM * C::BN), sp.S, f, lane, acc);
    store_item<C, false>(acc, f, lane, p.out + (tl.row0 * p.ldo + tl.n0) * esz, p.ldo, tl.rows, tl.cols,
                         p.out_dtype, blk);
  }
}

// ---------------------------------------------------------------------------
// weight gradient: one workgroup per (group, N tile, K tile); the group's
// token range is the reduction range (masked at unaligned ends).
// ---------------------------------------------------------------------------

struct WgradParams {
  const uint8_t* go; int64_t ld_go;
  const uint8_t* ia; int64_t ld_ia;
  const uint8_t* gs; uint32_t gs_bytes;     // GO scales, step-major [T][N] dwords (T = cdiv(M, 128))
  const uint8_t* is; uint32_t is_bytes;     // IA scales, step-major [T][K] dwords
  const int32_t* offs; int E; int64_t M; int64_t N; int64_t K;
  uint8_t* out; int out_dtype;
  int tiles_n; int tiles_k;
  float* part; int dp; int S; int units;    // split plan (host): see split_plan
  int dev; int par; int slots;              // dev: plan on the device (wgrad_groups / wgrad_plan) from par, slots
  int go_pl; int ia_pl;                     // operand layouts: 0 rows, 1 row pairs (Operand)
};

struct WgradTile {
  int g;                      // group
  int64_t n0; int rows;       // output rows (n) n0 .. n0 + rows - 1
  int64_t k0; int cols;       // output columns (k) k0 .. k0 + cols - 1
};

template <class C>
__device__ __forceinline__ WgradTile wgrad_tile(const WgradParams& p, int lt) {
  WgradTile t;
  const int per = p.tiles_n * p.tiles_k;
  t.g = lt / per;
  const int x = lt % per;
  t.n0 = (int64_t)(x / p.tiles_k) * C::BM;   // X side: rows of go_t
  t.k0 = (int64_t)(x % p.tiles_k) * C::BN;   // W side: rows of ia_t
  t.rows = (int)(p.N - t.n0 < C::BM ? p.N - t.n0 : C::BM);
  t.cols = (int)(p.K - t.k0 < C::BN ? p.K - t.k0 : C::BN);
  return t;
}

// Reduction steps (of STEP elements) the longest group touches.  Wave-uniform.
__device__ __forceinline__ int wgrad_max_steps(const int32_t* __restrict__ offs, int E, int64_t M) {
  const int lane = threadIdx.x & (kWave - 1);
  int m = 0;
  for (int base = 0; base < E; base += kWave) {
    const int e = base + lane;
    int n = 0;
    if (e < E) {
      int lo = e > 0 ? offs[e - 1] : 0;
      int hi = offs[e];
      if (lo < 0) lo = 0;
      if (hi > M) hi = (int)M;
      n = hi > lo ? (hi + STEP - 1) / STEP - lo / STEP : 0;
    }
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int o = __shfl_xor(n, d, kWave);
      n = o > n ? o : n;
    }
    m = uniform(n) > m ? uniform(n) : m;
  }
  return m;
}

// Split plan of a wgrad launch: the host's (dev = 0), or, for a lone
// under-filled round of several groups (dev = 1), one made here from the
// longest group, which sets the round's length (the host sees only the
// average).  Every kernel of the launch computes the same plan.
template <class C>
__device__ __forceinline__ Split wgrad_plan(const WgradParams& p) {
  if (!p.dev) return Split{p.dp, p.S, p.units};
  const int tiles = p.E * p.tiles_n * p.tiles_k;
  return split_plan(tiles, p.par, wgrad_max_steps(p.offs, p.E, p.M), p.slots, C::BM * C::BN * 4 / 1024);
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int o = __shfl_xor(v, d, kWave);
    v = o > v ? o : v;
  }
  return v;
}

// Per-group split of a lone wgrad round (dev = 1, E <= 64).  Groups differ in
// length, and one piece count for every tile leaves the round as long as the
// longest group's pieces while short groups' tiles idle.  Greedy
// apportionment instead: from one piece per tile, the first group with the
// longest pieces gets one more piece per tile, again and again, while the
// units (E * TNK tiles' pieces, TNK = tiles_n * tiles_k) fit the budget
// min(par, slots), every piece keeps kMinSplitSteps steps and no tile exceeds
// kMaxSplit pieces.  Each candidate is priced with split_plan's cost model,
// the round lasting as long as its longest piece; the best one is kept if it
// saves kSplitMinGainNs, else no tile is split.  Integer, lane-parallel and
// deterministic: every workgroup of every kernel of the launch gets the same
// plan.  Lane g < E holds group g's entries.
struct WgradGroups {
  int s;       // pieces per tile of group `lane` (1: whole, as one piece); 0 past E
  int c0;      // first unit of group `lane`'s tiles (exclusive prefix of TNK * s)
  int units;   // units in all; 0: no tile is split
};

template <class C>
__device__ __forceinline__ WgradGroups wgrad_groups(const WgradParams& p) {
  const int lane = threadIdx.x & (kWave - 1);
  const int tnk = p.tiles_n * p.tiles_k;
  int n = 0;
  if (lane < p.E) {
    int lo = lane > 0 ? p.offs[lane - 1] : 0;
    int hi = p.offs[lane];
    if (lo < 0) lo = 0;
    if (hi > p.M) hi = (int)p.M;
    n = hi > lo ? (hi + STEP - 1) / STEP - lo / STEP : 0;
    if (n > (1 << 20)) n = 1 << 20;   // keeps the cost model's products in int32
  }
  int s = lane < p.E ? 1 : 0, len = n, units = p.E * tnk, best_s = s, best_units = 0;
  const int budget = p.par < p.slots ? p.par : p.slots;
  const int len0 = wave_max(len);
  const int tail = (int)kTailNsPerStep * len0;
  int best = (int)kSplitMinGainNs;
  constexpr int kib = C::BM * C::BN * 4 / 1024;
  if (len0 >= kMinSplitTotal) {
    for (int it = 0; it < kWave && units + tnk <= budget; ++it) {
      const int m = wave_max(len);
      const int g = __builtin_ctzll(__ballot(lane < p.E && len == m));
      const int gn = lane_value(n, g), gs = lane_value(s, g);
      if (gs >= kMaxSplit || gn / (gs + 1) < kMinSplitSteps) break;
      if (lane == g) {
        s = gs + 1;
        len = (n + s - 1) / s;
      }
      units += tnk;
      const int gain = tail - (int)kTailNsPerStep * wave_max(len) - (int)kSplitFixedNs -
                       units * kib * (int)kSplitNsPerMiB / 1024;
      if (gain > best) {
        best = gain;
        best_s = s;
        best_units = units;
      }
    }
  }
  WgradGroups w;
  w.units = best_units;
  w.s = lane < p.E ? (best_units ? best_s : 1) : 0;
  w.c0 = wave_incl_scan(tnk * w.s) - tnk * w.s;
  return w;
}

// Tiles below the returned index run whole (PIECES = false).
template <class C>
__device__ __forceinline__ int wgrad_whole(const WgradParams& p) {
  if (p.dev && p.E <= kWave) return wgrad_groups<C>(p).units ? 0 : p.E * p.tiles_n * p.tiles_k;
  return wgrad_plan<C>(p).dp;
}

// Tile, piece and piece count of unit u of the piece kernel; false past the
// plan's units.  Unit u writes partial slot u; a tile's pieces are
// consecutive units.
template <class C>
__device__ __forceinline__ bool wgrad_unit(const WgradParams& p, int u, int& lt, int& piece, int& S) {
  if (p.dev && p.E <= kWave) {
    const WgradGroups w = wgrad_groups<C>(p);
    if (u >= w.units) return false;
    const int tnk = p.tiles_n * p.tiles_k;
    const int g = __builtin_ctzll(__ballot(w.s > 0 && w.c0 + tnk * w.s > u));
    S = lane_value(w.s, g);
    const int r = u - lane_value(w.c0, g);
    lt = g * tnk + r / S;
    piece = r % S;
    return true;
  }
  const Split sp = wgrad_plan<C>(p);
  if (u >= sp.units) return false;
  lt = sp.dp + u / sp.S;
  piece = u % sp.S;
  S = sp.S;
  return true;
}

// Split tile v of the reduce kernel: its tile, first partial slot and piece
// count; false past the split tiles.
template <class C>
__device__ __forceinline__ bool wgrad_split_tile(const WgradParams& p, int v, int& lt, int& base, int& S) {
  if (p.dev && p.E <= kWave) {
    const WgradGroups w = wgrad_groups<C>(p);
    const int tnk = p.tiles_n * p.tiles_k;
    if (!w.units || v >= p.E * tnk) return false;
    const int g = v / tnk;
    S = lane_value(w.s, g);
    base = lane_value(w.c0, g) + (v - g * tnk) * S;
    lt = v;
    return true;
  }
  const Split sp = wgrad_plan<C>(p);
  if (sp.S < 2 || v >= sp.units / sp.S) return false;
  lt = sp.dp + v;
  base = v * sp.S;
  S = sp.S;
  return true;
}

// Group of dispatch slot y of the whole-tile grid: the groups longest first
// (most reduction steps; ties by index).  The hardware starts workgroups in
// blockIdx order as CUs free up, so with more tiles than CUs this is the
// longest-processing-time-first schedule: a long group's tiles start in the
// first round instead of behind short groups (E=8, N=K=2048 with groups of 3
// to 44 steps: a 44-step tile then bounds the launch, not a short round plus
// a 36-step one).  Which workgroup computes a tile never changes its result.
// E <= 64 (one lane per group); past that, index order.
__device__ __forceinline__ int wgrad_slot_group(const WgradParams& p, int y) {
  if (p.E > kWave || p.E == 1) return y;
  const int lane = threadIdx.x & (kWave - 1);
  int n = -1;
  if (lane < p.E) {
    int lo = lane > 0 ? p.offs[lane - 1] : 0;
    int hi = p.offs[lane];
    if (lo < 0) lo = 0;
    if (hi > p.M) hi = (int)p.M;
    n = hi > lo ? (hi + STEP - 1) / STEP - lo / STEP : 0;
  }
  int rank = 0;
  for (int g = 0; g < p.E; ++g) {
    const int v = lane_value(n, g);
    rank += (v > n || (v == n && g < lane)) ? 1 : 0;
  }
  return __ffsll((long long)__ballot(lane < p.E && rank == y)) - 1;
}

// PIECES = false: grid (tiles_n * tiles_k, E), workgroup (x, y) computes tile
// g * tiles_n * tiles_k + x of group g = wgrad_slot_group(y) whole when below
// wgrad_whole (epilogue EPI); true: workgroup u computes the piece
// wgrad_unit assigns it.
template <class C, bool PIECES, int EPI = kEpiBf16>
__global__ __launch_bounds__(C::NT) void wgrad_kernel(WgradParams p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
  int lt, piece = 0, S = 1;
  if constexpr (PIECES) {
    if (!wgrad_unit<C>(p, (int)blockIdx.x, lt, piece, S)) return;
  } else {
    // (wgrad_whole is every tile or none except for E = 1 or E > 64, where
    // slots map to groups in index order)
    lt = wgrad_slot_group(p, (int)blockIdx.y) * p.tiles_n * p.tiles_k + (int)blockIdx.x;
    if (lt >= wgrad_whole<C>(p)) return;
  }
  const WgradTile tl = wgrad_tile<C>(p, lt);
  const int g = tl.g;
  const int64_t n0 = tl.n0, k0 = tl.k0;
  const int rows = tl.rows, cols = tl.cols;
  int lo = g > 0 ? p.offs[g - 1] : 0;
  int hi = p.offs[g];
  if (lo < 0) lo = 0;
  if (hi > p.M) hi = (int)p.M;
  if (PIECES && hi > lo) {
    // piece of the group's steps lo/STEP .. cdiv(hi, STEP)-1, clipped to [lo, hi)
    const int a0 = lo / STEP;
    int a, b;
    split_range(a0, (hi + STEP - 1) / STEP - a0, piece, S, a, b);
    if (STEP * a > lo) lo = STEP * a;
    if (STEP * b < hi) hi = STEP * b;
  }

  const Operand X = make_operand(p.go, p.ld_go, p.go_pl, n0, rows);
  const Operand W = make_operand(p.ia, p.ld_ia, p.ia_pl, k0, cols);
  const ScaleSrc xs{make_rsrc(p.gs, p.gs_bytes), (uint32_t)p.N, (uint32_t)n0};
  const ScaleSrc ws{make_rsrc(p.is, p.is_bytes), (uint32_t)p.K, (uint32_t)k0};

  v16f acc[C::FM][C::FN];
  if (hi > lo)
    step_mainloop<C>(smem, X, W, xs, ws, lo, hi, acc);
  else
    zero_acc<C>(acc);
  // group bounds that are not multiples of 16 (any offsets are accepted, as
  // in the reference): the straddling chunks' in-group tokens
  if ((lo | hi) & 15) edge_chunks<C>(X, W, xs, ws, lo, hi, acc);

  if constexpr (PIECES) {
    store_partial<C>(acc, p.part + (int64_t)blockIdx.x * (C::BM * C::BN));
    return;
  }
  constexpr int es = EPI == kEpiF32 || EPI == kEpiF32Any ? 4 : 2;
  store_epi<C, EPI, true>(acc, smem, p.out + ((int64_t)g * p.N * p.K + n0 * p.K + k0) * es, p.K, rows, cols);
}

// Split tiles of a wgrad launch: one workgroup per item (v, c), as in
// fwd_reduce_kernel; items past the plan's split tiles exit.
template <class C>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(WgradParams p) {
  __shared__ __attribute__((aligned(16))) uint8_t blk[32 * C::WTN * 2];
  constexpr int CH = ReduceShape<C>::CH;
  const int v = blockIdx.x / CH, f = (blockIdx.x % CH) * 4 + wave_id();
  int lt, base, S;
  if (!wgrad_split_tile<C>(p, v, lt, base, S)) return;
  const int lane = threadIdx.x % kWave;
  const WgradTile tl = wgrad_tile<C>(p, lt);
  float acc[16];
  sum_pieces<C>(p.part + (int64_t)base * (C::BM * C::BN), S, f, lane, acc);
  const int esz = p.out_dtype == MXGG_DTYPE_F32 ? 4 : 2;
  store_item<C, true>(acc, f, lane, p.out + ((int64_t)tl.g * p.N * p.K + tl.n0 * p.K + tl.k0) * esz, p.K, tl.rows,
                      tl.cols, p.out_dtype, blk);
}

// ---------------------------------------------------------------------------
// routing table / tile order: test hooks that run the GEMMs' own device code
// ---------------------------------------------------------------------------

// The reference's routing buffer [hist E | start E | total | map grid_m_ub]
// (kernels/forward.py:320-354), built with the lookup the GEMMs run: with
// one column tile and bands of one m-block, route_tile's order is the
// reference's m-block order, so tile t is m-block t of the map.  One wave.
__global__ __launch_bounds__(64) void routing_kernel(const int32_t* offs, int E, int BM, int grid_m_ub,
                                                     int32_t* out) {
  for (int e = threadIdx.x; e < E; e += kWave) {
    int prev = e > 0 ? offs[e - 1] : 0;
    out[e] = offs[e] - prev;
    out[E + e] = prev;
  }
  WaveGroups wg{0, 0, 0, 0, 0};
  int total;
  if (E <= kWave) {
    wg = load_groups(offs, E, BM);
    total = wg.total;
  } else {
    total = route_total(offs, E, BM);
  }
  if (threadIdx.x == 0) out[2 * E] = total;
  for (int pid = 0; pid < grid_m_ub; ++pid) {
    int pn;
    const TileRoute r = E <= kWave ? route_tile(wg, E, BM, 1, 1, pid, pn) : route_tile(offs, E, BM, 1, 1, pid, pn);
    if (threadIdx.x == 0) out[2 * E + 1 + pid] = r.expert >= 0 ? (r.block << 16) | r.expert : -1;
  }
}

// The forward kernels' tile order: for every program id of the whole-tile
// grid, the tile fwd_tile gives it (the XCD swizzle, then the expert-aligned
// bands of route_tile), as 5 int32s (expert, row0, rows, n0, cols), or -1s
// past the tiles.  One wave per workgroup, programs strided over the grid.
template <class C>
__global__ __launch_bounds__(64) void schedule_kernel(FwdParams p, int programs, int32_t* out) {
  WaveGroups wg;
  const int tiles = fwd_groups<C>(p, wg) * p.grid_n;
  for (int pid = blockIdx.x; pid < programs; pid += gridDim.x) {
    FwdTile tl;
    const bool ok = pid < tiles && fwd_tile<C>(p, pid, tiles, wg, tl);
    if (threadIdx.x < 5) {
      int v = -1;
      if (ok) {
        const int64_t f[5] = {tl.expert, tl.row0, tl.rows, tl.n0, tl.cols};
        v = (int)f[threadIdx.x];
      }
      out[5 * (int64_t)pid + threadIdx.x] = v;
    }
  }
}

}  // namespace mxgg

// ===========================================================================
// C ABI
// ===========================================================================

using namespace mxgg;

// Row stride of a weight staged in row pairs (K bytes rounded up to 64).
static int64_t staged_ld(int64_t K) { return (K + 63) / 64 * 64; }

// Extra workspace for staging an e4m3 weight in row pairs, or 0 where the
// call would not gain from it.  Staging copies the weight once (2 E N K
// bytes of HBM traffic in the re-layout launch the call makes anyway), about
// 400 E / M of the GEMM's time (5 TB/s against 2 PFLOP/s), so E <= M / 8192 at
// least.  The main loop copies whole lines of row-major data too, so a call
// gains less than that now (dgrad (4, 16640, 8192, 8192) 931 us staged, 885
// not): only callers that ask for the room stage.  256 bytes of slack keep the
// staged lines 256-byte aligned.
static size_t fwd_staging_bytes(int E, int64_t M, int64_t N, int64_t K, int b_fmt) {
  if (b_fmt != MXGG_FMT_E4M3 || E <= 0 || N <= 0 || N % 2 || (int64_t)E * 8192 > M) return 0;
  if (K < 2048 || (K < 4096 && N < 4096)) return 0;
  if ((int64_t)E * (N / 2) > (1 << 22) || K >= (1 << 22)) return 0;   // launch grid, int offsets
  return (size_t)E * (size_t)N * (size_t)staged_ld(K) + 256;
}

// Forward calls above this many multiply-adds (1.2e11 flop) may have A staged.
constexpr int64_t kPlainMaxMacs = (int64_t)60000000000;

// Whether a forward call that stages nothing runs on plain scales (where
// plain_scales_ok) instead of after a scale re-layout launch.  The plain-scale
// kernels copy their scales in 32-byte row pieces, four times the requests of
// the step-major dwords: about 5% of the GEMM's time.  The launch takes about
// 4.5 us and 2 (M + E N) K / 32 bytes at 4 TB/s.  The GEMM is priced at 2.3
// PFLOP/s or, with few rows per expert, at one read of the weight at 5 TB/s.
// Measured (MI355X, whole calls, re-laid / plain scales): (32, 2048, 8192,
// 8192) 449 / 434 us, (1, 16640, 2048, 2048) 79.0 / 77.3, (8, 4096, 4096,
// 4096) 99.0 / 98.3; past the line (8, 16640, 2048, 5120) 187 / 189, (8,
// 16640, 8192, 5120) e2m1 552 / 564, (4, 16640, 8192, 8192) 885 / 900.
static bool plain_pays(int E, int64_t M, int64_t N, int64_t K, int b_fmt) {
  const double macs = (double)M * (double)N * (double)K;
  const double weight = (double)E * (double)N * (double)K * (b_fmt == MXGG_FMT_E2M1 ? 0.5 : 1.0);
  const double gemm = macs / 1.15e6 > weight / 5e3 ? macs / 1.15e6 : weight / 5e3;   // ns
  const double relayout = 4500.0 + ((double)M + (double)E * (double)N) * (double)K / 16.0 / 4e3;
  return 0.05 * gemm <= relayout;
}

// The same for A (M, K), or 0: its copy's time over the GEMM's is about
// 400 / N, so N >= 8192.  A is e4m3 whatever the weight's format.  Not on calls
// of at most kPlainMaxMacs, whose re-layout launch alone costs more than row
// pairs could save.
static size_t fwd_staging_bytes_a(int64_t M, int64_t N, int64_t K, int b_fmt) {
  if ((b_fmt != MXGG_FMT_E4M3 && b_fmt != MXGG_FMT_E2M1) || M <= 0 || M % 2 || N < 8192 || K < 2048) return 0;
  if (M / 2 > (1 << 22) || K >= (1 << 22)) return 0;   // launch grid, int offsets
  if (M * N <= kPlainMaxMacs / K) return 0;
  return (size_t)M * (size_t)staged_ld(K) + 256;
}

namespace {

typedef Cfg<256, 256, 2, 2, MXGG_FMT_E4M3, 4> CfgF8_256;
typedef Cfg<128, 128, 2, 2, MXGG_FMT_E4M3, 4> CfgF8_128;
typedef Cfg<256, 256, 2, 2, MXGG_FMT_E2M1, 4> CfgF4_256;
typedef Cfg<128, 128, 2, 2, MXGG_FMT_E2M1, 4> CfgF4_128;
// The same tiles on plain to_mx scales (drop-in calls whose scale rows are
// 16-byte multiples): no scale re-layout launch; 16 KB scale slots of 8 steps
// (8 KB for 128 x 128 tiles).
typedef Cfg<256, 256, 2, 2, MXGG_FMT_E4M3, 4, true> CfgF8_256P;
typedef Cfg<128, 128, 2, 2, MXGG_FMT_E4M3, 4, true> CfgF8_128P;
typedef Cfg<256, 256, 2, 2, MXGG_FMT_E2M1, 4, true> CfgF4_256P;
typedef Cfg<128, 128, 2, 2, MXGG_FMT_E2M1, 4, true> CfgF4_128P;

// The quarter tiles of a 256 x 256 configuration (void: none).
template <class C>
struct QuadCfg {
  typedef typename std::conditional<C::BM == 256, Cfg<128, 128, 2, 2, C::WFMT, C::NH, C::PS>, void>::type type;
};

// The scale-independent kernels of a configuration (the reduce): its
// step-major twin.
template <class C>
using StepCfg = Cfg<C::BM, C::BN, C::WGM, C::WGN, C::WFMT, C::NH>;

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct FwdChoice {
  int bm, bn, group_m, xcd;
  bool split;   // the last round may be split along K (workspace permitting)
};

struct TunedFwd {
  int E, M, N, K, b_fmt, bm, bn, group_m, xcd, split;
};

#include "tuned_fwd.h"

// Tuned entry for (E, M, N, K, b_fmt): same E, N, K and format, M within a
// factor of two of the swept M; null when the sweep did not cover the shape.
const TunedFwd* find_tuned(int E, int64_t M, int64_t N, int64_t K, int b_fmt) {
  for (const TunedFwd* t = kTunedFwd; t->E; ++t)
    if (t->E == E && t->N == N && t->K == K && t->b_fmt == b_fmt && 2 * M >= t->M && M <= 2 * (int64_t)t->M)
      return t;
  return nullptr;
}

// A tuned entry when the sweep covered the shape.  Otherwise 256 x 256
// tiles, the 8-XCD swizzle and expert-aligned bands of at most 12 m-blocks
// (route_tile; 12 beat 8 and 16 on the sweep's jagged groups, and the
// 256 x 256 tile beats 128 x 128 even at N = K = 2048); 128 x 128 tiles for
// problems too small to fill half the chip with 256 x 256 tiles, unless
// the 256 x 256 plan splits that lone round along K.
// Requests (nonzero bm, bn, gm, xcd) override field by field, and any request
// leaves the split to the workspace (a tuned "whole tiles only" applies to
// calls that request nothing).
template <class C>
int fwd_resident();

// A tuned entry applies whole on every operand layout: calls on different
// layouts give the same bits, and the tile order can change them -- the tiles of a split last round are the last ones in that order.
FwdChoice pick_fwd(int E, int64_t M, int64_t N, int64_t K, int b_fmt, int bm, int bn, int gm, int xcd) {
  FwdChoice c{256, 256, 12, 8, true};
  const int64_t tiles256 = (cdiv(M, 256) + E - 1) * cdiv(N, 256);
  const TunedFwd* t = find_tuned(E, M, N, K, b_fmt);
  if (t) {
    c = FwdChoice{t->bm, t->bn, t->group_m, t->xcd, t->split != 0};
  } else if (M <= 100 * (int64_t)E && E > 1) {
    // Groups that mostly fit 128 rows: (8, 512, 8192, 5120) 80.7 us as 256 x
    // 256 tiles and 72.9 as 128 x 128, (8, 768) 83.9 and 80.6, (32, 2048, 2880,
    // 2880) 95 and 86; 128 rows on average (8, 1024) 85.7 and 109.
    c.bm = 128;
    c.bn = 128;
  } else if (tiles256 < 128) {
    // Under half a chip of 256 x 256 tiles: 128 x 128 tiles (two per CU)
    // spread the work over 4x the workgroups, unless the 256 x 256 launch
    // splits its lone round along K (a long reduction; judged for the full
    // workspace that mxgg_grouped_mm_workspace_size recommends; the launch may
    // then still prefer quarter tiles, see fwd_plan).  E=1, M=2080 (one GPU's
    // share of E=8 under 8-way expert parallelism), N=2048: K=5120 77 -> 54 us;
    // K=8192 splits (70 us, against 76 us as 128 x 128).
    const int par = fwd_resident<CfgF8_256>();
    const int slots = (int)(kSplitBytes / ((size_t)256 * 256 * 4));
    if (split_plan((int)tiles256, par > 0 ? par : 256, (int)cdiv(K, STEP), slots, 256).units == 0) {
      c.bm = 128;
      c.bn = 128;
    }
  }
  if (bm || bn || gm || xcd) c.split = true;
  if (bm) c.bm = bm;
  if (bn) c.bn = bn;
  if (gm) c.group_m = gm;
  if (xcd) c.xcd = xcd;
  return c;
}

// Whether the choice's tile may run: 256 x 256, or 128 x 128 -- beside an e2m1
// weight only in calls for which the library picks it by itself (so that its
// answer, mxgg_grouped_mm_config's, may be passed back as a request).
bool tile_built(const FwdChoice& c, int E, int64_t M, int64_t N, int64_t K, int b_fmt) {
  if (c.bm == 256 && c.bn == 256) return true;
  if (c.bm != 128 || c.bn != 128) return false;
  return b_fmt == MXGG_FMT_E4M3 || pick_fwd(E, M, N, K, b_fmt, 0, 0, 0, 0).bm == 128;
}

// Workgroups of `kernel` (nt threads) resident on the current device at
// once: CUs x per-CU occupancy (LDS, registers).  Cached per device.
template <class KF>
int resident_workgroups(KF kernel, int nt, int (&cache)[64]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (dev >= 0 && dev < 64 && cache[dev]) return cache[dev];
  int cus = 0, per = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, nt, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  const int r = cus * (per > 0 ? per : 1);
  if (dev >= 0 && dev < 64) cache[dev] = r;
  return r;
}

template <class C>
int fwd_resident() {
  static int cache[64];
  return resident_workgroups(fwd_kernel<C, false>, C::NT, cache);
}

// Partial slots of BM x BN fp32 available in `bytes` (capped).
template <class C>
int split_slots(size_t bytes) {
  const size_t n = bytes / ((size_t)C::BM * C::BN * 4);
  return n > 4096 ? 4096 : (int)n;
}

// Rows of the streaming tiles (StreamCfg) of a forward call that requests no
// tile, or 0: the general tiles.  By the average rows per group, which is
// what the host knows; a group of more rows takes several tiles.  Measured
// (MI355X, whole calls, general tiles / 32 / 64 rows): (8, 64, 8192, 5120)
// 73.4 / 64.3 / 63.9 us, its bytes at 5.5 TB/s 63; with e2m1 weights 57.9 /
// 37.7 / 39.9; (16, 50, 544, 5216) e2m1 56 / 20 / 23; (1, 16, 2048, 8192) 28.6
// / 23.3 / 28.3; (8, 256, 8192, 5120) 76.5 / 80 / 66.6, (8, 384) 78.7 / 86 /
// 68.9, (32, 1024, 2880, 2880) 90 / 79 / 70.5; 64 rows per group (8, 512) 80.7
// / 102 / 86: not past 48.  The average is of balanced routing: with half the
// rows in one group 64-row and 128 x 128 tiles are level ((8, 384, 8192, 5120)
// 80 / 95, (32, 1024, 2880, 2880) 69 / 67, (32, 1536, 8192, 5120) 304 / 297, even
// groups 252 / 264), with all of them in one, where they re-read its weight once
// per 64 rows, 64-row tiles lose ((8, 384) 38 / 25 us, (32, 1536) 116 / 68).
static int stream_rows(int E, int64_t M) {
  if (M <= 32 || M <= 8 * (int64_t)E) return 32;
  return M <= 48 * (int64_t)E ? 64 : 0;
}

template <class C>
static int launch_stream(const FwdParams& p0, int gm, int xcd, hipStream_t st) {
  FwdParams p = p0;
  p.grid_n = (int)cdiv(p.N, C::BN);
  p.group_m = gm;
  p.xcd = xcd;
  const int64_t tiles_ub = (cdiv(p.M, C::BM) + p.E - 1) * p.grid_n;
  if (tiles_ub > INT32_MAX) return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: grid too large");
#define MXGG_STREAM(E) \
  case E: hipLaunchKernelGGL((fwd_stream_kernel<C, E>), dim3((unsigned)tiles_ub), dim3(C::NT), 0, st, p); break
  MXGG_EPI_SWITCH(pick_epi(p.out_dtype, p.ldo, p.out), MXGG_STREAM)
#undef MXGG_STREAM
  return launch_status("grouped_mm");
}

// 32-row tiles: two workgroups per CU, 4 (e4m3) or 8 (e2m1) steps in flight
// on it; 64-row tiles: one, with 3.  (A 7-slot ring, one workgroup per CU: 2-4%
// slower at 8 experts, 5-10% faster only where a call has 64 tiles.)
template <int WFMT, bool PS>
static int launch_stream_rows(const FwdParams& p, int bm, int gm, int xcd, hipStream_t st) {
  if (bm == 32) return launch_stream<StreamCfg<32, WFMT, WFMT == MXGG_FMT_E2M1 ? 5 : 3, PS>>(p, gm, xcd, st);
  return launch_stream<StreamCfg<64, WFMT, 4, PS>>(p, gm, xcd, st);
}

// Forward launch: the whole tiles (grid: every possible tile; those at or
// past dp exit), then, when the workspace allows a split at all, the pieces
// (grid: the most pieces a plan can have) and the reduce of the split tiles.
// The plan itself depends on offs and is made on the device.
template <class C>
int launch_fwd(const FwdParams& p0, int grid_m_ub, int gm, int xcd, size_t part_bytes, hipStream_t st) {
  FwdParams p = p0;
  p.grid_n = (int)cdiv(p.N, C::BN);
  p.group_m = gm;
  p.xcd = xcd;
  p.par = fwd_resident<C>();
  p.slots = p.part ? split_slots<C>(part_bytes) : 0;
  const int nsteps = (int)cdiv(p.K, STEP);
  if (p.par <= 0 || p.slots < 2 || nsteps < kMinSplitTotal) p.slots = 0;
  // Rows of every group add up to M in the usual MoE call, with half a tile
  // of padding per group on average: what the plan does with that many tiles
  // decides which launches are made (p.slots = 0 / p.quads = 0 make the device
  // plan, from the real count, agree).  A wrong guess costs time, never
  // correctness.
  typedef typename QuadCfg<C>::type Q;
  constexpr bool kQuads = !std::is_void<Q>::value;
  const int64_t est = (cdiv(p.M, C::BM) + (p.E - 1) / 2) * p.grid_n;
  p.quads = 0;
  if (est > INT32_MAX || p.par <= 0) {
    p.slots = 0;
  } else {
    const Split e = fwd_plan((int)est, p.par, nsteps, p.slots, C::BM * C::BN * 4 / 1024, kQuads);
    p.quads = kQuads && e.units == 0 && e.dp < est;
    if (e.units == 0) p.slots = 0;
  }
  const int64_t tiles_ub = (int64_t)grid_m_ub * p.grid_n;
  if (tiles_ub <= 0) return MXGG_OK;
  if (tiles_ub > INT32_MAX) return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: grid too large");
  // The device's tile count is m * grid_n for some m <= grid_m_ub (each
  // group adds whole m-blocks of grid_n tiles).  When every such count is
  // below one round and its plan splits or quarters it, no tile runs whole: the
  // whole-tile launch would only route and exit (4.5 us on the expert-parallel
  // shard's N = 2048, K = 8192 call), so it is left out.  (E = 1, M = N = 2048,
  // K = 8192, quarter tiles: 41.0 us with that launch, 39.7 without, 51.0 split.)
  bool whole = true;
  if ((p.slots || p.quads) && tiles_ub < p.par) {
    whole = false;
    for (int m = 1; m <= grid_m_ub && !whole; ++m)
      if (fwd_plan(m * p.grid_n, p.par, nsteps, p.slots, C::BM * C::BN * 4 / 1024, p.quads != 0).dp != 0) whole = true;
  }
  const int epi = pick_epi(p.out_dtype, p.ldo, p.out);
#define MXGG_WHOLE(E) \
  case E: hipLaunchKernelGGL((fwd_kernel<C, false, E>), dim3((unsigned)tiles_ub), dim3(C::NT), 0, st, p); break
  if (whole) MXGG_EPI_SWITCH(epi, MXGG_WHOLE)
#undef MXGG_WHOLE
  if (int rc = launch_status("grouped_mm")) return rc;
  if constexpr (kQuads) {
    if (p.quads) {   // 4 * (T % P) < 2 P quarters
#define MXGG_QUAD(E)                                                                                        \
  case E:                                                                                                   \
    hipLaunchKernelGGL((fwd_quad_kernel<C, Q, E>), dim3((unsigned)(2 * p.par)), dim3(Q::NT), 0, st, p);     \
    break
      MXGG_EPI_SWITCH(epi, MXGG_QUAD)
#undef MXGG_QUAD
      if (int rc = launch_status("grouped_mm")) return rc;
    }
  }
  if (!p.slots) return MXGG_OK;
  const int pieces = p.slots;   // units = rem * S <= slots
  hipLaunchKernelGGL((fwd_kernel<C, true>), dim3((unsigned)pieces), dim3(C::NT), 0, st, p);
  if (int rc = launch_status("grouped_mm")) return rc;
  // a split needs rem <= par / 2 tiles of ReduceShape::CH items each; the
  // grid strides over them.  One workgroup per item of the split the host
  // expects (at least 128, which costs little when the device plan differs):
  // a 72-tile split (1152 items) took 21 us on 128 workgroups.
  const int64_t items = (int64_t)(p.par / 2) * ReduceShape<C>::CH;
  const Split esp = split_plan((int)(est < INT32_MAX ? est : INT32_MAX), p.par, nsteps, p.slots,
                               C::BM * C::BN * 4 / 1024);
  int64_t rgrid = esp.S > 0 ? (int64_t)(esp.units / esp.S) * ReduceShape<C>::CH : 0;
  if (rgrid < 128) rgrid = 128;
  if (rgrid > items) rgrid = items;
  if (rgrid <= 0) return MXGG_OK;
  hipLaunchKernelGGL((fwd_reduce_kernel<StepCfg<C>>), dim3((unsigned)rgrid), dim3(256), 0, st, p);
  return launch_status("grouped_mm");
}

ScaleJob scale_job(const uint8_t* src, int64_t ld_r, int64_t ld_b, uint32_t* dst, int64_t rows,
                   int batches, int64_t nblk, int64_t steps) {
  ScaleJob j{src, ld_r, ld_b, dst, (int)rows, batches, (int)nblk, (int)steps,
             (int)cdiv(rows, 64), (int)cdiv(steps, 16)};
  return j;
}

// Re-lay two operands' scales into the workspace, and, given pair jobs,
// one or two operands' data into row pairs (one launch).
int launch_relayout(const ScaleJob& a, const ScaleJob& b, hipStream_t st, const char* what,
                    const PairJob* d = nullptr, const PairJob* d2 = nullptr) {
  ScaleJobs js;
  js.j[0] = a;
  js.j[1] = b;
  js.tiles0 = a.batches * a.tiles_r * a.tiles_t;
  const int64_t t01 = (int64_t)js.tiles0 + (int64_t)b.batches * b.tiles_r * b.tiles_t;
  if (t01 > INT32_MAX) return fail(MXGG_ERR_UNSUPPORTED, "%s: scale re-layout grid too large", what);
  js.tiles01 = (int)t01;
  js.d = d ? *d : PairJob{};
  js.tiles_d = d ? d->batches * d->pairs : 0;
  js.d2 = d2 ? *d2 : PairJob{};
  const int64_t grid = t01 + js.tiles_d + (d2 ? (int64_t)d2->batches * d2->pairs : 0);
  if (grid <= 0) return MXGG_OK;
  if (grid > (int64_t)(UINT32_MAX / 256)) return fail(MXGG_ERR_UNSUPPORTED, "%s: re-layout grid too large", what);
  if (grid > INT32_MAX) return fail(MXGG_ERR_UNSUPPORTED, "%s: scale re-layout grid too large", what);
  hipLaunchKernelGGL(scale_relayout_kernel, dim3((unsigned)grid), dim3(256), 0, st, js);
  return launch_status(what);
}

}  // namespace

extern "C" int64_t mxgg_routing_words(int E, int64_t M, int block_m) {
  if (E <= 0 || M < 0 || block_m <= 0) return 0;
  return 2 * (int64_t)E + 1 + cdiv(M, block_m) + (E > 1 ? E - 1 : 0);
}

extern "C" int mxgg_build_routing(const int32_t* offs, int E, int64_t M, int block_m, int32_t* out,
                                  void* stream) {
  clear_error();
  if (E <= 0 || E > 65535) return fail(MXGG_ERR_INVALID_ARG, "build_routing: E=%d out of range", E);
  if (M < 0 || M > INT32_MAX) return fail(MXGG_ERR_INVALID_ARG, "build_routing: M out of range");
  if (block_m <= 0) return fail(MXGG_ERR_INVALID_ARG, "build_routing: block_m must be positive");
  if (!offs || !out) return fail(MXGG_ERR_INVALID_ARG, "build_routing: null pointer");
  if (int rc = require_device()) return rc;
  const int64_t ub = cdiv(M, block_m) + (E > 1 ? E - 1 : 0);
  hipLaunchKernelGGL(routing_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, offs, E, block_m,
                     (int)ub, out);
  return launch_status("build_routing");
}

extern "C" int64_t mxgg_schedule_programs(int E, int64_t M, int64_t N, int block_m, int block_n) {
  if (E <= 0 || M < 0 || N < 0 || block_m <= 0 || block_n <= 0) return 0;
  return (cdiv(M, block_m) + (E > 1 ? E - 1 : 0)) * cdiv(N, block_n);
}

extern "C" int mxgg_tile_schedule(const int32_t* offs, int E, int64_t M, int64_t N, int block_m,
                                  int block_n, int group_m, int xcd_swizzle, int32_t* out,
                                  void* stream) {
  clear_error();
  if (E <= 0 || E > 65535) return fail(MXGG_ERR_INVALID_ARG, "tile_schedule: E=%d out of range", E);
  if (M < 0 || N < 0 || M > INT32_MAX || N > INT32_MAX)
    return fail(MXGG_ERR_INVALID_ARG, "tile_schedule: M, N out of range");
  if (group_m <= 0 || xcd_swizzle <= 0)
    return fail(MXGG_ERR_INVALID_ARG, "tile_schedule: group_m and xcd_swizzle must be positive");
  if (!((block_m == 256 && block_n == 256) || (block_m == 128 && block_n == 128)))
    return fail(MXGG_ERR_UNSUPPORTED, "tile_schedule: tile %dx%d not built", block_m, block_n);
  const int64_t programs = mxgg_schedule_programs(E, M, N, block_m, block_n);
  if (programs > INT32_MAX / 5) return fail(MXGG_ERR_INVALID_ARG, "tile_schedule: too many programs");
  if (!offs || !out) return fail(MXGG_ERR_INVALID_ARG, "tile_schedule: null pointer");
  if (int rc = require_device()) return rc;
  if (programs == 0) return MXGG_OK;
  FwdParams p{};
  p.offs = offs;
  p.E = E;
  p.M = M;
  p.N = N;
  p.grid_n = (int)cdiv(N, block_n);
  p.group_m = group_m;
  p.xcd = xcd_swizzle;
  const unsigned grid = (unsigned)(programs < 1024 ? programs : 1024);
  if (block_m == 256)
    hipLaunchKernelGGL(schedule_kernel<CfgF8_256>, dim3(grid), dim3(64), 0, (hipStream_t)stream, p, (int)programs,
                       out);
  else
    hipLaunchKernelGGL(schedule_kernel<CfgF8_128>, dim3(grid), dim3(64), 0, (hipStream_t)stream, p, (int)programs,
                       out);
  return launch_status("tile_schedule");
}

static bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Re-laid scales of a forward call: A [T][M], then B [E][T][N] dwords.
static size_t fwd_scale_bytes(int E, int64_t M, int64_t N, int64_t K) {
  return (size_t)4 * (size_t)cdiv(K, STEP) * ((size_t)M + (size_t)E * (size_t)N);
}

// Partial-tile area worth reserving: up to kSplitBytes, no more than `tiles`
// tiles of `tile_bytes` cut into the most pieces a reduction of `nsteps`
// steps allows.
static size_t split_area(int64_t tiles, size_t tile_bytes, int64_t nsteps) {
  if (nsteps < kMinSplitTotal || tiles <= 0) return 0;
  int64_t smax = nsteps / kMinSplitSteps;
  if (smax > kMaxSplit) smax = kMaxSplit;
  const double want = (double)tiles * (double)smax * (double)tile_bytes;
  return want < (double)kSplitBytes ? (size_t)want : kSplitBytes;
}

// Extra workspace for staging both wgrad operands (go_t (N, M), ia_t (K, M))
// in row pairs, or 0 where that would not pay.  The copy moves 2 (N + K) M
// bytes in the scale re-layout launch, about 2000 (N + K) / (N K) of the
// GEMM's time, so it is offered at N = K = 8192 and, with 8 or more groups, at
// N + K >= 10240.  Row-major operands are copied in whole lines too: staging
// costs 7-9% of a call more than it saves, so only callers that ask for the
// room stage.
static size_t wgrad_staging_bytes(int E, int64_t M, int64_t N, int64_t K) {
  if (E <= 0 || M <= 0 || M % 32 || N <= 0 || K <= 0 || N % 2 || K % 2) return 0;
  if (!((N >= 8192 && K >= 8192) || (E >= 8 && N + K >= 10240))) return 0;
  if (M >= (1 << 22) || N / 2 + K / 2 > (1 << 22)) return 0;   // int offsets, launch grid
  return (size_t)(N + K) * (size_t)staged_ld(M) + 512;
}

extern "C" size_t mxgg_wgrad_staging_size(int E, int64_t M, int64_t N, int64_t K) {
  return wgrad_staging_bytes(E, M, N, K);
}

extern "C" size_t mxgg_grouped_mm_staging_size(int E, int64_t M, int64_t N, int64_t K, int b_fmt) {
  if (M < 0 || K < 0 || K % 32 || E <= 0) return 0;
  return fwd_staging_bytes(E, M, N, K, b_fmt) + fwd_staging_bytes_a(M, N, K, b_fmt);
}

// Partial-tile room of a forward call: the most a split plan of the call can
// use (256 x 256 or 128 x 128 tiles, whichever needs more).  Calls given more
// use no more, so every call with at least this room makes the same plan.
static size_t fwd_part_cap(int E, int64_t M, int64_t N, int64_t K) {
  if (E <= 0 || M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t nsteps = cdiv(K, STEP);
  const size_t a = split_area((cdiv(M, 256) + E - 1) * cdiv(N, 256), (size_t)256 * 256 * 4, nsteps);
  const size_t b = split_area((cdiv(M, 128) + E - 1) * cdiv(N, 128), (size_t)128 * 128 * 4, nsteps);
  return a > b ? a : b;
}

extern "C" size_t mxgg_grouped_mm_workspace_size(int E, int64_t M, int64_t N, int64_t K) {
  if (E <= 0 || M < 0 || N < 0 || K < 0) return 0;
  const size_t sc = fwd_scale_bytes(E, M, N, K);
  if (sc == 0 || M == 0 || N == 0) return sc;
  const size_t part = fwd_part_cap(E, M, N, K);
  return part ? align256(sc) + part : sc;
}

extern "C" size_t mxgg_grouped_mm_tile_workspace_size(int E, int64_t M, int64_t N, int64_t K, int block_m,
                                                      int block_n) {
  if (E <= 0 || M < 0 || N < 0 || K < 0) return 0;
  if (!block_m && !block_n && stream_rows(E, M)) return fwd_scale_bytes(E, M, N, K);   // never split
  return mxgg_grouped_mm_workspace_size(E, M, N, K);
}

// Where the parts of a caller's workspace go (plain-scale entry points): the
// re-laid scales (`need` bytes) first; then, 256-byte aligned, the partial
// tiles, given at most `cap` bytes; then, from the bytes past those, the
// staged operands (`stage` bytes, carved from the end).  A workspace of the
// recommended size therefore stages nothing, and a larger one stages without
// taking room from the partial tiles: the split plan, and the bits, are those
// of the unstaged call.
struct WsLayout {
  size_t part_off;    // first byte of the partial area
  size_t part;        // its bytes (0: no tile is split)
  size_t extra;       // bytes past the scales and the partial area
};

static WsLayout ws_layout(size_t ws_bytes, size_t need, size_t cap) {
  WsLayout w{align256(need), 0, 0};
  const size_t avail = ws_bytes > w.part_off ? ws_bytes - w.part_off : 0;
  w.part = avail < cap ? avail : cap;
  const size_t used = w.part ? w.part_off + w.part : need;
  w.extra = ws_bytes > used ? ws_bytes - used : 0;
  return w;
}

// Bytes a row of `len` bytes takes in an operand stored in pieces of `piece`
// bytes (64 for row pairs, 32 for row quads, 1 for rows).
static int64_t operand_row_bytes(int64_t len, int64_t piece) { return (len + piece - 1) / piece * piece; }

// Argument checks of a forward call shared by the entry points; MXGG_OK
// when the call may go ahead (check *empty: nothing to compute).
// plain: A_s / B_s are plain scales with these strides (else step-major,
// strides unused).  layout: MXGG_A_PAIRS / MXGG_B_PAIRS flags.
static int check_grouped_mm(const uint8_t* A, int64_t lda, const uint8_t* A_s, int64_t ldas, const uint8_t* B,
                            int b_fmt, int64_t ldb_n, int64_t ldb_e, const uint8_t* B_s, int64_t ldbs_n,
                            int64_t ldbs_e, const int32_t* offs, int E, int64_t M, int64_t N, int64_t K,
                            const void* out, int out_dtype, int64_t ldo, bool plain, int layout, bool* empty) {
  *empty = false;
  if (b_fmt != MXGG_FMT_E4M3 && b_fmt != MXGG_FMT_E2M1)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: weight format %d not E4M3/E2M1", b_fmt);
  if (layout & ~(MXGG_A_PAIRS | MXGG_B_PAIRS | MXGG_B_QUADS) || (layout & MXGG_B_PAIRS && layout & MXGG_B_QUADS))
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: unknown operand layout flags %d", layout);
  const bool ap = layout & MXGG_A_PAIRS, bp = layout & MXGG_B_PAIRS, bq = layout & MXGG_B_QUADS;
  if (bp && b_fmt != MXGG_FMT_E4M3)
    return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: row pairs are built for e4m3 weights only (e2m1: row quads)");
  if (bq && b_fmt != MXGG_FMT_E2M1)
    return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: row quads are built for packed e2m1 weights only (e4m3: row pairs)");
  if ((ap && M % 2) || (bp && N % 2) || (bq && N % 4))
    return fail(MXGG_ERR_INVALID_ARG,
                "grouped_mm: an operand in row pairs / quads needs a row count divisible by 2 / 4 (M=%lld, N=%lld)",
                (long long)M, (long long)N);
  if (out_dtype != MXGG_DTYPE_BF16 && out_dtype != MXGG_DTYPE_F16 && out_dtype != MXGG_DTYPE_F32)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: out_dtype %d not BF16/F16/F32", out_dtype);
  if (E <= 0 || E > 65535) return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: E=%d out of range", E);
  if (M < 0 || N < 0 || K < 0) return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: negative shape");
  if (K % 32) return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: K=%lld must be a multiple of 32", (long long)K);
  const int64_t kb = b_fmt == MXGG_FMT_E2M1 ? K / 2 : K;
  if (lda < operand_row_bytes(K, ap ? 64 : 1) || ldb_n < operand_row_bytes(kb, bp ? 64 : (bq ? 32 : 1)) || ldo < N ||
      (plain && (ldas < K / 32 || ldbs_n < K / 32)))
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: a row stride is smaller than its row");
  if (E > 1 && (ldb_e < N * ldb_n || (plain && ldbs_e < N * ldbs_n)))
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: expert stride smaller than one expert");
  if (lda % 16 || ldb_n % 16 || !aligned16(A) || !aligned16(B))
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: A/B rows must be 16-byte aligned");
  if (lda >= (1 << 23) || ldb_n >= (1 << 23))
    return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: row strides must be below 2**23 bytes");
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
    return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: dimension above 2**31");
  if (M == 0 || N == 0) {
    *empty = true;
    return MXGG_OK;
  }
  if (!A || !A_s || !B || !B_s || !offs || !out)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm: null pointer");
  if (fwd_scale_bytes(E, M, N, K) >= ((size_t)1 << 31))
    return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: problem too large");
  return MXGG_OK;
}

// Plain to_mx scales the GEMMs can read directly (plain-scale kernels): rows
// of 16-byte multiples, 16-byte aligned buffers, byte ranges below 2**31.
static bool plain_scales_ok(const uint8_t* A_s, int64_t ldas, const uint8_t* B_s, int64_t ldbs_n, int64_t ldbs_e,
                            int E, int64_t M, int64_t N) {
  if (ldas % 16 || ldbs_n % 16 || (E > 1 && ldbs_e % 16) || !aligned16(A_s) || !aligned16(B_s)) return false;
  const int64_t bexp = E > 1 ? ldbs_e : N * ldbs_n;
  return M * ldas < ((int64_t)1 << 31) && bexp < ((int64_t)1 << 31) && (int64_t)(E - 1) * bexp < ((int64_t)1 << 40);
}

// The GEMM launches of a checked forward call on step-major scales (as: A
// [T][M], bs: B [E][T][N] dwords), or, with `plain`, on plain to_mx scales
// (as: A (M, K/32) with row stride ldas, bs: B (E, N, K/32) with strides
// ldbs_n, ldbs_e; plain_scales_ok holds); part / part_bytes: room for the fp32
// partial tiles of a split last round (none: no tile is split).
static int launch_grouped_mm(const uint8_t* A, int64_t lda, const uint8_t* as, const uint8_t* B, int b_fmt,
                             int64_t ldb_n, int64_t ldb_e, const uint8_t* bs, const int32_t* offs, int E, int64_t M,
                             int64_t N, int64_t K, void* out, int out_dtype, int64_t ldo, int block_m, int block_n,
                             int group_m, int xcd, int layout, void* part_area, size_t part_bytes, hipStream_t st,
                             bool plain = false, int64_t ldas = 0, int64_t ldbs_n = 0, int64_t ldbs_e = 0) {
  FwdChoice c = pick_fwd(E, M, N, K, b_fmt, block_m, block_n, group_m, xcd);
  if (!tile_built(c, E, M, N, K, b_fmt)) return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm: tile %dx%d not built", c.bm, c.bn);
  const int64_t T = cdiv(K, STEP);
  float* part = c.split && part_area && part_bytes ? (float*)part_area : nullptr;
  FwdParams p{A, lda, B, ldb_n, ldb_e, as, (uint32_t)(4 * T * M), bs, (uint32_t)(4 * T * N), (uint32_t)(4 * T * N),
              offs, E, M, N, K, (uint8_t*)out, out_dtype, ldo, 0, 0, 0, part, 0, 0, 0,
              (layout & MXGG_A_PAIRS) ? 1 : 0, (layout & MXGG_B_PAIRS) ? 1 : ((layout & MXGG_B_QUADS) ? 2 : 0)};
  // no more room than the split plans of this shape can use (ws_layout)
  const size_t cap = fwd_part_cap(E, M, N, K);
  const size_t pb = part ? (part_bytes < cap ? part_bytes : cap) : 0;
  if (!pb) part = nullptr;
  p.part = part;
  const int bm_stream = block_m || block_n ? 0 : stream_rows(E, M);   // not a tile of pick_fwd's
  const int gm256 = (int)(cdiv(M, 256) + E - 1), gm128 = (int)(cdiv(M, 128) + E - 1);
  if (plain) {
    // Up to the end of the last row's last 16-byte chunk: copies run past the
    // rows, K and N of a tile, and what lies behind the last row of a view (its
    // row stride's rest, the gap to a next expert) need not be the caller's.
    const int64_t row = (K / 32 + 15) / 16 * 16;
    p.as_bytes = (uint32_t)((M - 1) * ldas + row);
    p.bs_bytes = (uint32_t)((N - 1) * ldbs_n + row);
    p.bs_expert = (uint32_t)(E > 1 ? ldbs_e : 0);
    p.as_ld = (uint32_t)ldas;
    p.bs_ld = (uint32_t)ldbs_n;
    if (bm_stream)
      return b_fmt == MXGG_FMT_E2M1 ? launch_stream_rows<MXGG_FMT_E2M1, true>(p, bm_stream, c.group_m, c.xcd, st)
                                    : launch_stream_rows<MXGG_FMT_E4M3, true>(p, bm_stream, c.group_m, c.xcd, st);
    if (b_fmt == MXGG_FMT_E2M1 && c.bm == 128) return launch_fwd<CfgF4_128P>(p, gm128, c.group_m, c.xcd, pb, st);
    if (b_fmt == MXGG_FMT_E2M1) return launch_fwd<CfgF4_256P>(p, gm256, c.group_m, c.xcd, pb, st);
    if (c.bm == 256) return launch_fwd<CfgF8_256P>(p, gm256, c.group_m, c.xcd, pb, st);
    return launch_fwd<CfgF8_128P>(p, gm128, c.group_m, c.xcd, pb, st);
  }
  if (bm_stream)
    return b_fmt == MXGG_FMT_E2M1 ? launch_stream_rows<MXGG_FMT_E2M1, false>(p, bm_stream, c.group_m, c.xcd, st)
                                  : launch_stream_rows<MXGG_FMT_E4M3, false>(p, bm_stream, c.group_m, c.xcd, st);
  if (b_fmt == MXGG_FMT_E2M1 && c.bm == 128) return launch_fwd<CfgF4_128>(p, gm128, c.group_m, c.xcd, pb, st);
  if (b_fmt == MXGG_FMT_E2M1) return launch_fwd<CfgF4_256>(p, gm256, c.group_m, c.xcd, pb, st);
  if (c.bm == 256) return launch_fwd<CfgF8_256>(p, gm256, c.group_m, c.xcd, pb, st);
  return launch_fwd<CfgF8_128>(p, gm128, c.group_m, c.xcd, pb, st);
}

// A checked forward call on plain scales: the GEMM launches, on the plain
// scales where plain_scales_ok holds, else after re-laying them step-major
// into the workspace (the partial tiles follow the room of those scales in
// either case, so both ways make the same split plan and the same bits).
static int run_grouped_mm(const uint8_t* A, int64_t lda, const uint8_t* A_s, int64_t ldas, const uint8_t* B,
                          int b_fmt, int64_t ldb_n, int64_t ldb_e, const uint8_t* B_s, int64_t ldbs_n,
                          int64_t ldbs_e, const int32_t* offs, int E, int64_t M, int64_t N, int64_t K, void* out,
                          int out_dtype, int64_t ldo, int block_m, int block_n, int group_m, int xcd,
                          void* workspace, size_t ws_bytes, void* stream) {
  const size_t need = fwd_scale_bytes(E, M, N, K);
  hipStream_t st = (hipStream_t)stream;
  const int64_t T = cdiv(K, STEP);
  uint32_t* wsd = (uint32_t*)workspace;
  const WsLayout wl = ws_layout(ws_bytes, need, fwd_part_cap(E, M, N, K));
  // The weight, then A, in row pairs, staged at the end of the workspace
  // (the weight last) from the bytes past the partial area (ws_layout).
  const size_t stage_b = fwd_staging_bytes(E, M, N, K, b_fmt), stage_a = fwd_staging_bytes_a(M, N, K, b_fmt);
  const int ldp = (int)staged_ld(K);
  // (each staging size holds 256 bytes of slack for aligning its start)
  uint8_t* const end = (uint8_t*)workspace + ws_bytes;
  PairJob pb{}, pa{};
  const bool staged_b = T > 0 && stage_b && wl.extra >= stage_b;
  if (staged_b) pb = PairJob{B, ldb_n, ldb_e, (uint8_t*)align256((size_t)(end - stage_b)), ldp, (int)(N / 2), E, (int)K};
  const size_t used_b = staged_b ? stage_b : 0;
  const bool staged_a = T > 0 && stage_a && wl.extra >= used_b + stage_a;
  if (staged_a)
    pa = PairJob{A, lda, 0, (uint8_t*)align256((size_t)(end - used_b - stage_a)), ldp, (int)(M / 2), 1, (int)K};
  const bool plain = !staged_a && !staged_b && plain_pays(E, M, N, K, b_fmt) &&
                     plain_scales_ok(A_s, ldas, B_s, ldbs_n, ldbs_e, E, M, N);
  if (T > 0 && !plain) {
    if (int rc = launch_relayout(scale_job(A_s, ldas, 0, wsd, M, 1, K / 32, T),
                                 scale_job(B_s, ldbs_n, ldbs_e, wsd + T * M, N, E, K / 32, T), st, "grouped_mm",
                                 staged_b ? &pb : nullptr, staged_a ? &pa : nullptr))
      return rc;
  }
  void* part = wl.part ? (void*)((uint8_t*)workspace + wl.part_off) : nullptr;
  return launch_grouped_mm(staged_a ? pa.dst : A, staged_a ? (int64_t)ldp : lda,
                           plain ? A_s : (const uint8_t*)wsd, staged_b ? pb.dst : B, b_fmt,
                           staged_b ? (int64_t)ldp : ldb_n, staged_b ? N * ldp : ldb_e,
                           plain ? B_s : (const uint8_t*)(wsd + T * M), offs, E, M, N, K, out, out_dtype, ldo,
                           block_m, block_n, group_m, xcd, (staged_b ? MXGG_B_PAIRS : 0) | (staged_a ? MXGG_A_PAIRS : 0),
                           part, wl.part, st, plain, ldas, ldbs_n, ldbs_e);
}

extern "C" int mxgg_grouped_mm(const uint8_t* A, int64_t lda, const uint8_t* A_s, int64_t ldas,
                               const uint8_t* B, int b_fmt, int64_t ldb_n, int64_t ldb_e,
                               const uint8_t* B_s, int64_t ldbs_n, int64_t ldbs_e,
                               const int32_t* offs, int E, int64_t M, int64_t N, int64_t K,
                               void* out, int out_dtype, int64_t ldo, int block_m, int block_n,
                               int group_m, int xcd, void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  bool empty;
  if (int rc = check_grouped_mm(A, lda, A_s, ldas, B, b_fmt, ldb_n, ldb_e, B_s, ldbs_n, ldbs_e, offs, E, M, N, K,
                                out, out_dtype, ldo, true, 0, &empty))
    return rc;
  if (empty) return MXGG_OK;
  const size_t need = fwd_scale_bytes(E, M, N, K);
  if (need && (!workspace || ws_bytes < need))
    return fail(MXGG_ERR_WORKSPACE, "grouped_mm: workspace of at least %zu bytes needed, %zu given", need,
                workspace ? ws_bytes : (size_t)0);
  if (int rc = require_device()) return rc;
  return run_grouped_mm(A, lda, A_s, ldas, B, b_fmt, ldb_n, ldb_e, B_s, ldbs_n, ldbs_e, offs, E, M, N, K, out,
                        out_dtype, ldo, block_m, block_n, group_m, xcd, workspace, ws_bytes, stream);
}

extern "C" int mxgg_grouped_mm_steps(const uint8_t* A, int64_t lda, const uint32_t* A_ss, const uint8_t* B,
                                     int b_fmt, int64_t ldb_n, int64_t ldb_e, const uint32_t* B_ss,
                                     const int32_t* offs, int E, int64_t M, int64_t N, int64_t K, void* out,
                                     int out_dtype, int64_t ldo, int block_m, int block_n, int group_m, int xcd,
                                     int layout, void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  bool empty;
  if (int rc = check_grouped_mm(A, lda, (const uint8_t*)A_ss, 0, B, b_fmt, ldb_n, ldb_e, (const uint8_t*)B_ss, 0, 0,
                                offs, E, M, N, K, out, out_dtype, ldo, false, layout, &empty))
    return rc;
  if (empty) return MXGG_OK;
  if (((uintptr_t)A_ss | (uintptr_t)B_ss) & 3)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm_steps: step-major scales must be 4-byte aligned");
  if (int rc = require_device()) return rc;
  return launch_grouped_mm(A, lda, (const uint8_t*)A_ss, B, b_fmt, ldb_n, ldb_e, (const uint8_t*)B_ss, offs, E, M,
                           N, K, out, out_dtype, ldo, block_m, block_n, group_m, xcd, layout, workspace,
                           workspace ? ws_bytes : 0, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// allocation-free forward entry point: the workspace is a device array of
// this library (one per GPU) instead of caller memory
// ---------------------------------------------------------------------------

// MXGG_NOALLOC_SCRATCH_BYTES per device, held from the library's load to the
// end of the process: the re-laid scales of a call (4 * cdiv(K, 128) *
// (M + E*N) bytes; 21 MB for the largest sweep shape) and after them the fp32
// partial tiles of a split last round.  Nothing in it needs clearing: every
// call writes the scales before reading them, and a split call writes every
// partial tile before the reduce reads it.
static __device__ __align__(256) uint8_t scratch[MXGG_NOALLOC_SCRATCH_BYTES];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[64];   // device address of `scratch` per device; null until looked up
}  // namespace

// This device's copy of `scratch` (the host-side name is not a device
// address): looked up once per device, with that device current.
static int scratch_for_device(void** ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MXGG_ERR_NO_DEVICE, "grouped_mm_noalloc: no HIP device: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= 64) return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm_noalloc: device %d above 63", dev);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(e != hipSuccess ? (int)e : MXGG_ERR_UNSUPPORTED, "grouped_mm_noalloc: hipGetSymbolAddress: %s",
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return MXGG_OK;
}

extern "C" int mxgg_grouped_mm_noalloc(const uint8_t* A, int64_t lda, const uint8_t* A_s, int64_t ldas,
                                       const uint8_t* B, int b_fmt, int64_t ldb_n, int64_t ldb_e,
                                       const uint8_t* B_s, int64_t ldbs_n, int64_t ldbs_e,
                                       const int32_t* offs, int E, int64_t M, int64_t N, int64_t K,
                                       void* out, int out_dtype, int64_t ldo, int block_m, int block_n,
                                       int group_m, int xcd, void* stream) {
  clear_error();
  bool empty;
  if (int rc = check_grouped_mm(A, lda, A_s, ldas, B, b_fmt, ldb_n, ldb_e, B_s, ldbs_n, ldbs_e, offs, E, M, N, K,
                                out, out_dtype, ldo, true, 0, &empty))
    return rc;
  if (empty) return MXGG_OK;
  const size_t need = fwd_scale_bytes(E, M, N, K);
  if (need > (size_t)MXGG_NOALLOC_SCRATCH_BYTES)
    return fail(MXGG_ERR_WORKSPACE,
                "grouped_mm_noalloc: the re-laid scales need %zu bytes, more than the %zu-byte scratch "
                "(4 * cdiv(K, 128) * (M + E*N) must stay within it)",
                need, (size_t)MXGG_NOALLOC_SCRATCH_BYTES);
  if (int rc = require_device()) return rc;
  void* ws = nullptr;
  if (int rc = scratch_for_device(&ws)) return rc;
  // the recommended size where it fits: no operand is staged (the copy costs
  // more than it saves)
  size_t bytes = mxgg_grouped_mm_workspace_size(E, M, N, K);
  if (bytes > (size_t)MXGG_NOALLOC_SCRATCH_BYTES) bytes = (size_t)MXGG_NOALLOC_SCRATCH_BYTES;
  return run_grouped_mm(A, lda, A_s, ldas, B, b_fmt, ldb_n, ldb_e, B_s, ldbs_n, ldbs_e, offs, E, M, N, K, out,
                        out_dtype, ldo, block_m, block_n, group_m, xcd, ws, bytes, stream);
}

extern "C" int mxgg_grouped_mm_config(int E, int64_t M, int64_t N, int64_t K, int b_fmt, int* block_m,
                                      int* block_n, int* group_m, int* xcd_swizzle) {
  clear_error();
  if (!block_m || !block_n || !group_m || !xcd_swizzle)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm_config: null output pointer");
  if (b_fmt != MXGG_FMT_E4M3 && b_fmt != MXGG_FMT_E2M1)
    return fail(MXGG_ERR_INVALID_ARG, "grouped_mm_config: weight format %d not E4M3/E2M1", b_fmt);
  FwdChoice c = pick_fwd(E, M, N, K, b_fmt, *block_m, *block_n, *group_m,
                         *xcd_swizzle);
  *block_m = c.bm;
  *block_n = c.bn;
  *group_m = c.group_m;
  *xcd_swizzle = c.xcd;
  if (!tile_built(c, E, M, N, K, b_fmt)) return fail(MXGG_ERR_UNSUPPORTED, "grouped_mm_config: tile %dx%d not built", c.bm, c.bn);
  return MXGG_OK;
}

// Re-laid scales of a wgrad call: GO [T][N], then IA [T][K] dwords.
static size_t wgrad_scale_bytes(int64_t M, int64_t N, int64_t K) {
  return (size_t)4 * (size_t)cdiv(M, STEP) * ((size_t)N + (size_t)K);
}

// Reduction steps of an average group (what the split plan is sized for).
static int64_t wgrad_group_steps(int E, int64_t M) {
  const int64_t n = cdiv(M, (int64_t)E * STEP);
  return n > 0 ? n : 1;
}

// Partial-tile room of a wgrad call: the most its split plan can use.  With
// several groups the kernels plan a lone under-filled round from the longest
// group, which may hold all M tokens: room for that plan.
static size_t wgrad_part_cap(int E, int64_t M, int64_t N, int64_t K) {
  if (E <= 0 || M <= 0 || N <= 0 || K <= 0) return 0;
  return split_area((int64_t)E * cdiv(N, 256) * cdiv(K, 256), (size_t)256 * 256 * 4,
                    E > 1 ? cdiv(M, STEP) : wgrad_group_steps(E, M));
}

extern "C" size_t mxgg_wgrad_workspace_size(int E, int64_t M, int64_t N, int64_t K) {
  if (E <= 0 || M < 0 || N < 0 || K < 0) return 0;
  const size_t sc = wgrad_scale_bytes(M, N, K);
  if (sc == 0 || N == 0 || K == 0) return sc;
  const size_t part = wgrad_part_cap(E, M, N, K);
  return part ? align256(sc) + part : sc;
}

// Argument checks of a wgrad call (plain: go_s / ia_s are plain scales with
// these strides); *empty: nothing to compute.
static int check_wgrad(const uint8_t* go_t, int64_t ld_go, const uint8_t* go_s, int64_t ld_gos, const uint8_t* ia_t,
                       int64_t ld_ia, const uint8_t* ia_s, int64_t ld_ias, const int32_t* offs, int E, int64_t M,
                       int64_t N, int64_t K, const void* out, int out_dtype, bool plain, int layout, bool* empty) {
  *empty = false;
  if (out_dtype != MXGG_DTYPE_BF16 && out_dtype != MXGG_DTYPE_F16 && out_dtype != MXGG_DTYPE_F32)
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: out_dtype %d not BF16/F16/F32", out_dtype);
  if (E <= 0 || E > 65535) return fail(MXGG_ERR_INVALID_ARG, "wgrad: E=%d out of range", E);
  if (M < 0 || N < 0 || K < 0) return fail(MXGG_ERR_INVALID_ARG, "wgrad: negative shape");
  if (M % 32) return fail(MXGG_ERR_INVALID_ARG, "wgrad: M=%lld must be a multiple of 32", (long long)M);
  if (layout & ~(MXGG_A_PAIRS | MXGG_B_PAIRS))
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: unknown operand layout flags %d", layout);
  const bool gp = layout & MXGG_A_PAIRS, ip = layout & MXGG_B_PAIRS;
  if ((gp && N % 2) || (ip && K % 2))
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: an operand in row pairs needs an even row count (N=%lld, K=%lld)",
                (long long)N, (long long)K);
  if (ld_go < operand_row_bytes(M, gp ? 64 : 1) || ld_ia < operand_row_bytes(M, ip ? 64 : 1) ||
      (plain && (ld_gos < M / 32 || ld_ias < M / 32)))
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: a row stride is smaller than its row");
  if (ld_go % 16 || ld_ia % 16 || !aligned16(go_t) || !aligned16(ia_t))
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: operand rows must be 16-byte aligned");
  if (ld_go >= (1 << 23) || ld_ia >= (1 << 23))
    return fail(MXGG_ERR_UNSUPPORTED, "wgrad: row strides must be below 2**23 bytes");
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
    return fail(MXGG_ERR_UNSUPPORTED, "wgrad: dimension above 2**31");
  if (N == 0 || K == 0) {
    *empty = true;
    return MXGG_OK;
  }
  if (!go_t || !go_s || !ia_t || !ia_s || !offs || !out)
    return fail(MXGG_ERR_INVALID_ARG, "wgrad: null pointer");
  if (wgrad_scale_bytes(M, N, K) >= ((size_t)1 << 31)) return fail(MXGG_ERR_UNSUPPORTED, "wgrad: problem too large");
  return MXGG_OK;
}

// A wgrad launch whose 256 x 256 tiles would fill at most half the chip and
// whose plan cuts none of them (a reduction too short to split, e.g. one GPU's
// expert-parallel share, 2080 tokens, at N = K = 2048: 64 tiles on 256 CUs),
// or whose 128 x 128 tiles fill at least one round even where a split is
// planned (E = 2, N = K = 2048: 512 tiles for 2 x 256 resident workgroups;
// row-major operands 7% faster than the split 256 x 256 launch, row pairs 3%
// slower, taken on both so that the bits do not depend on the layout):
// 128 x 128 tiles instead, four times as many, two workgroups per CU, whole.
// So do calls of at most kSmallTokens tokens per group with few outputs:
// kSmallOutputs, or kSmallOutputs8 with at most 8 groups.  Most of such a
// tile's time is its start and its store, which the second workgroup of a CU
// covers; 256 x 256 tiles read half as much and win in longer launches, the
// sooner the more groups there are.  Time as 256 x 256 over time as 128 x 128
// tiles, groups of 64 to 320 tokens, even and uneven (MI355X):
//   outputs   E = 8          E = 16         E = 32
//   3.4e7     1.01 .. 1.29
//   7e7       1.01 .. 1.17   0.95 .. 1.22
//   1.3e8     0.98 .. 1.10                  0.90 .. 1.00
//   1.5e8                    0.91 .. 1.00
//   2.1e8     1.04
//   2.7e8                    0.94 .. 1.01
//   3.0e8                                   0.90 .. 0.95
//   3.4e8     1.03
// E = 4 to 6.7e7 outputs 0.98 .. 1.32.  Whole training steps agree in sign
// where they differ by more than 1%: (8, 2080, 5120, 5120) 495 / 488 us, (32,
// 2080, 4096, 4096) 1090 / 1110, (32, 5824, 3968, 3104) 943 / 958; (16, 3616,
// 5504, 4480) 903 / 893, its gradient alone 275 / 298.  More tokens: (16, 5120,
// 4096, 4096) 184 / 192, (32, 16640, 2880, 2880) 261 / 293.
// p: the call's parameters with the 256 x 256 tile counts (replaced here).
constexpr int64_t kSmallTokens = 320, kSmallOutputs = (int64_t)100 * 1000 * 1000,
                  kSmallOutputs8 = (int64_t)350 * 1000 * 1000;

static int launch_wgrad_small(WgradParams p, hipStream_t st) {
  typedef CfgF8_128 Q;
  p.tiles_n = (int)cdiv(p.N, Q::BM);
  p.tiles_k = (int)cdiv(p.K, Q::BN);
  p.part = nullptr;
  p.dp = p.E * p.tiles_n * p.tiles_k;
  p.S = 1;
  p.units = 0;
  p.dev = 0;
  const dim3 grid((unsigned)(p.tiles_n * p.tiles_k), (unsigned)p.E);
#define MXGG_WGRAD(E) \
  case E: hipLaunchKernelGGL((wgrad_kernel<Q, false, E>), grid, dim3(Q::NT), 0, st, p); break
  MXGG_EPI_SWITCH(pick_epi(p.out_dtype, p.K, p.out), MXGG_WGRAD)
#undef MXGG_WGRAD
  return launch_status("wgrad");
}

// The plan of a wgrad call of `tiles` 256 x 256 tiles with `par` resident
// workgroups and `slots` partial-tile slots (0: no room): the host plan, and
// whether the kernels plan on the device and whether the call runs as 128 x
// 128 whole tiles instead (launch_wgrad_small).
struct WgradChoice {
  Split sp;
  bool dev;
  bool small;
};

static WgradChoice wgrad_choice(int E, int64_t M, int64_t N, int64_t K, int64_t tiles, int par, int slots) {
  constexpr int kib = CfgF8_256::BM * CfgF8_256::BN * 4 / 1024;
  WgradChoice w{split_plan((int)tiles, par, (int)wgrad_group_steps(E, M), slots, kib), false, false};
  // A lone round of several groups lasts as long as the longest group, which
  // only the device knows: the kernels plan from the groups' lengths
  // (wgrad_groups, or wgrad_plan past 64 groups) whenever a group of all M
  // rows would be split.
  w.dev = E > 1 && slots > 0 && split_plan((int)tiles, par, (int)cdiv(M, STEP) + 1, slots, kib).units > 0;
  const int64_t tiles128 = (int64_t)E * cdiv(N, 128) * cdiv(K, 128);
  w.small = (!w.dev && w.sp.units == 0 && 2 * tiles <= par) || (2 * tiles <= par && tiles128 >= 2 * par) ||
            (!w.dev && w.sp.units == 0 && M <= kSmallTokens * (int64_t)E &&
             (double)E * (double)N * (double)K <= (double)(E <= 8 ? kSmallOutputs8 : kSmallOutputs));
  return w;
}

// The wgrad launches of a checked call on step-major scales (gs: GO [T][N],
// is: IA [T][K] dwords); part / part_bytes: room for the fp32 partial tiles
// of tiles cut along the tokens (none: no tile is cut).
static int launch_wgrad(const uint8_t* go_t, int64_t ld_go, const uint8_t* gs, const uint8_t* ia_t, int64_t ld_ia,
                        const uint8_t* is, const int32_t* offs, int E, int64_t M, int64_t N, int64_t K, void* out,
                        int out_dtype, int layout, void* part_area, size_t part_bytes, hipStream_t st) {
  typedef CfgF8_256 C;
  const int64_t T = cdiv(M, STEP);
  // no more room than the split plans of this shape can use (ws_layout)
  const size_t cap = wgrad_part_cap(E, M, N, K);
  if (part_bytes > cap) part_bytes = cap;
  float* part = part_area && part_bytes ? (float*)part_area : nullptr;
  WgradParams p{go_t, ld_go, ia_t, ld_ia, gs, (uint32_t)(4 * T * N), is, (uint32_t)(4 * T * K), offs, E, M, N, K,
                (uint8_t*)out, out_dtype, (int)cdiv(N, C::BM), (int)cdiv(K, C::BN), part, 0, 1, 0, 0, 0, 0,
                (layout & MXGG_A_PAIRS) ? 1 : 0, (layout & MXGG_B_PAIRS) ? 1 : 0};
  const int64_t tiles = (int64_t)E * p.tiles_n * p.tiles_k;
  if (tiles > INT32_MAX / 2) return fail(MXGG_ERR_UNSUPPORTED, "wgrad: grid too large");
  static int resident_cache[64];
  const int par = resident_workgroups(wgrad_kernel<C, false>, C::NT, resident_cache);
  // groups differ in length, and with them the tiles' run times: with E > 1
  // only a lone under-filled round is split (its tiles all start at once)
  const bool may_split = E == 1 || tiles < par;
  const int slots = part && may_split ? split_slots<C>(part_bytes) : 0;
  const WgradChoice wc = wgrad_choice(E, M, N, K, tiles, par, slots);
  const Split& sp = wc.sp;
  p.dp = sp.dp;
  p.S = sp.S;
  p.units = sp.units;
  // device plan: the grids cover any such plan, every tile whole, or at most
  // min(par, slots) pieces and every tile reduced
  if (wc.dev) {
    p.dev = 1;
    p.par = par;
    p.slots = slots;
  }
  if (wc.small) return launch_wgrad_small(p, st);
  const int64_t whole_ub = p.dev ? tiles : sp.dp;
  const int64_t units_ub = p.dev ? slots : sp.units;
  const int64_t split_tiles_ub = p.dev ? tiles : (sp.units ? sp.units / sp.S : 0);
  if (whole_ub > 0) {
    const dim3 grid((unsigned)(p.tiles_n * p.tiles_k), (unsigned)E);
#define MXGG_WGRAD(E) \
  case E: hipLaunchKernelGGL((wgrad_kernel<C, false, E>), grid, dim3(C::NT), 0, st, p); break
    MXGG_EPI_SWITCH(pick_epi(out_dtype, K, out), MXGG_WGRAD)
#undef MXGG_WGRAD
    if (int rc = launch_status("wgrad")) return rc;
  }
  if (units_ub <= 0) return MXGG_OK;
  hipLaunchKernelGGL((wgrad_kernel<C, true>), dim3((unsigned)units_ub), dim3(C::NT), 0, st, p);
  if (int rc = launch_status("wgrad")) return rc;
  hipLaunchKernelGGL((wgrad_reduce_kernel<StepCfg<C>>), dim3((unsigned)(split_tiles_ub * ReduceShape<C>::CH)),
                     dim3(256), 0, st, p);
  return launch_status("wgrad");
}

extern "C" int mxgg_wgrad_config(int E, int64_t M, int64_t N, int64_t K, int* block) {
  clear_error();
  if (!block) return fail(MXGG_ERR_INVALID_ARG, "wgrad_config: null output pointer");
  if (E <= 0 || E > 65535 || M < 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
    return fail(MXGG_ERR_INVALID_ARG, "wgrad_config: shape out of range");
  typedef CfgF8_256 C;
  const int64_t tiles = (int64_t)E * cdiv(N, C::BM) * cdiv(K, C::BN);
  if (tiles > INT32_MAX / 2) return fail(MXGG_ERR_UNSUPPORTED, "wgrad_config: grid too large");
  if (int rc = require_device()) return rc;
  static int resident_cache[64];
  const int par = resident_workgroups(wgrad_kernel<C, false>, C::NT, resident_cache);
  if (par <= 0) return fail(MXGG_ERR_NO_DEVICE, "wgrad_config: resident workgroups unknown");
  const size_t part = wgrad_part_cap(E, M, N, K);
  const int slots = part && (E == 1 || tiles < par) ? split_slots<C>(part) : 0;
  *block = wgrad_choice(E, M, N, K, tiles, par, slots).small ? 128 : 256;
  return MXGG_OK;
}

extern "C" int mxgg_wgrad(const uint8_t* go_t, int64_t ld_go, const uint8_t* go_s, int64_t ld_gos,
                          const uint8_t* ia_t, int64_t ld_ia, const uint8_t* ia_s, int64_t ld_ias,
                          const int32_t* offs, int E, int64_t M, int64_t N, int64_t K, void* out,
                          int out_dtype, void* workspace, size_t ws_bytes, void* stream) {
  clear_error();
  bool empty;
  if (int rc = check_wgrad(go_t, ld_go, go_s, ld_gos, ia_t, ld_ia, ia_s, ld_ias, offs, E, M, N, K, out, out_dtype,
                           true, 0, &empty))
    return rc;
  if (empty) return MXGG_OK;
  const size_t need = wgrad_scale_bytes(M, N, K);
  if (need && (!workspace || ws_bytes < need))
    return fail(MXGG_ERR_WORKSPACE, "wgrad: workspace of at least %zu bytes needed, %zu given", need,
                workspace ? ws_bytes : (size_t)0);
  if (int rc = require_device()) return rc;
  hipStream_t st = (hipStream_t)stream;
  const int64_t T = cdiv(M, STEP);
  uint32_t* wsd = (uint32_t*)workspace;
  const WsLayout wl = ws_layout(ws_bytes, need, wgrad_part_cap(E, M, N, K));
  // Both operands in row pairs, staged at the end of the workspace from the
  // bytes past the partial area (ws_layout; 512 bytes of slack align both).
  const size_t stage = wgrad_staging_bytes(E, M, N, K);
  const bool staged = T > 0 && stage && wl.extra >= stage;
  PairJob pg{}, pi{};
  if (staged) {
    const int ldp = (int)staged_ld(M);
    uint8_t* dg = (uint8_t*)align256((size_t)((uint8_t*)workspace + ws_bytes - stage));
    uint8_t* di = (uint8_t*)align256((size_t)(dg + (size_t)N * ldp));
    pg = PairJob{go_t, ld_go, 0, dg, ldp, (int)(N / 2), 1, (int)M};
    pi = PairJob{ia_t, ld_ia, 0, di, ldp, (int)(K / 2), 1, (int)M};
  }
  if (T > 0) {
    if (int rc = launch_relayout(scale_job(go_s, ld_gos, 0, wsd, N, 1, M / 32, T),
                                 scale_job(ia_s, ld_ias, 0, wsd + T * N, K, 1, M / 32, T), st, "wgrad",
                                 staged ? &pg : nullptr, staged ? &pi : nullptr))
      return rc;
  }
  void* part = wl.part ? (void*)((uint8_t*)workspace + wl.part_off) : nullptr;
  return launch_wgrad(staged ? pg.dst : go_t, staged ? (int64_t)pg.ld_dst : ld_go, (const uint8_t*)wsd,
                      staged ? pi.dst : ia_t, staged ? (int64_t)pi.ld_dst : ld_ia, (const uint8_t*)(wsd + T * N), offs,
                      E, M, N, K, out, out_dtype, staged ? (MXGG_A_PAIRS | MXGG_B_PAIRS) : 0, part, wl.part, st);
}

extern "C" int mxgg_wgrad_steps(const uint8_t* go_t, int64_t ld_go, const uint32_t* go_ss, const uint8_t* ia_t,
                                int64_t ld_ia, const uint32_t* ia_ss, const int32_t* offs, int E, int64_t M,
                                int64_t N, int64_t K, void* out, int out_dtype, int layout, void* workspace,
                                size_t ws_bytes, void* stream) {
  clear_error();
  bool empty;
  if (int rc = check_wgrad(go_t, ld_go, (const uint8_t*)go_ss, 0, ia_t, ld_ia, (const uint8_t*)ia_ss, 0, offs, E, M,
                           N, K, out, out_dtype, false, layout, &empty))
    return rc;
  if (empty) return MXGG_OK;
  if (((uintptr_t)go_ss | (uintptr_t)ia_ss) & 3)
    return fail(MXGG_ERR_INVALID_ARG, "wgrad_steps: step-major scales must be 4-byte aligned");
  if (int rc = require_device()) return rc;
  return launch_wgrad(go_t, ld_go, (const uint8_t*)go_ss, ia_t, ld_ia, (const uint8_t*)ia_ss, offs, E, M, N, K, out,
                      out_dtype, layout, workspace, workspace ? ws_bytes : 0, (hipStream_t)stream);
}
