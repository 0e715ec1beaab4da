// Main loop and tile family of the GEMMs with few and middling rows (1 to about 1000 tokens, more of narrow products over
// a deep K), shared by ring.hip (FFN products) and ring_qkv.hip (Q/K/V projection).
//
// What bounds them: streaming the weights once.  The LDS is one ring of NST stages, each holding a 64-deep k tile of both
// operands, and a stage is requested again as soon as the barrier has freed it, so that NST - 1 tiles are on their way
// whatever else a CU does.  (The large-tile loop of gemm_core.h keeps its activations in two buffers and loads complete in
// order, so its weights are never more than about one tile ahead: 64 rows x [4096, 28672] 59 us there and in the split-K
// kernel, 44 us here = 5.3 TB/s; 128 rows 64 -> 51 us.)  How many it takes was measured for 32 x 128 tiles with a CU to
// themselves, 16 rows x [4096, 14336 x 2], 224 workgroups: 32 KB of weights on their way per CU (three stages) 43.0 us, 48 KB
// (four) 44.5, 64 KB 44.7, 96 KB 45.2 - but with fewer workgroups, or other distances in memory, 48 KB (ring_fourth_stage).
//
// 64-deep k tiles: an activation row, and a K-contiguous weight column, is then read in whole 128-byte lines.
// Both operands go global -> LDS without passing through registers (1 KB per wave instruction), XOR-swizzled by the
// choice of the chunk each lane fetches:
//   activations [BM][64], K-contiguous weights [BN][64]: chunk c (8 per row) of row r at slot c ^ ((r >> 1) & 7)
//   row-major weights [64][BN]: chunk c of row k at slot c ^ ((k & 3) << 2), or c ^ (((k >> 1) & 1) << 2) where a
//   row is not a multiple of 256 bytes - the four rows of a transpose read then fall on different banks.
// One barrier per k tile, in front of its last k16 step, when the next tile must have landed; the loads of a tile are
// spread one by one between the MFMAs of the four steps after the barrier that freed their stage, or (RingTile::NP) are left
// to waves that do nothing else.
#if (defined(TRI_BF16) && !defined(TRI_RING_H_BF16)) || (!defined(TRI_BF16) && !defined(TRI_RING_H_F16))
#ifdef TRI_BF16
#define TRI_RING_H_BF16
#else
#define TRI_RING_H_F16
#endif
#include "gemm_core.h"
#include "launch.h"

namespace tri {

// NTW: the weights are requested non-temporally (each line is wanted once: a single row block).
// NP: that many further waves do nothing but request tiles; the WM x WN waves then only read fragments and multiply.
template <int BM_, int BN_, int WM_, int WN_, int NST_, bool NTW_ = false, int NP_ = 0>
struct RingTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NST = NST_, BK = 64, NP = NP_;
  static constexpr bool NTW = NTW_;
  static constexpr int NW = WM * WN, NT = (NW + NP) * 64, LW = NP > 0 ? NP : NW;  // LW: waves that request tiles
  static constexpr int TM = BM / WM, TN = BN / WN, MI = TM / 32, NI = TN / 32;
  static constexpr int X_HALFS = BM * BK, STAGE = (BM + BN) * BK;
  static constexpr int LDS_BYTES = NST * STAGE * 2;
  static constexpr int XI = BM / 8 / LW, WI = BN / 8 / LW, L = XI + WI;  // 1 KB load instructions per loading wave and k tile
  static constexpr int CPR = BN / 8;                                     // 16-byte chunks per row-major weight row
  static_assert(BM % (8 * LW) == 0 && BN % (8 * LW) == 0 && TM % 32 == 0 && TN % 32 == 0, "tile split");
  static_assert(NST >= 3 && LDS_BYTES <= 160 * 1024, "LDS budget");
  static_assert(NP > 0 ? (NST - 1) * L < 64 : (NST - 2) * L + L / 4 < 64, "loads in flight fit vmcnt");
};

// The family (planned by ring_plan below).  Waves are arranged so that every tile has at least one wave per SIMD
// and an accumulator of at most 160 registers; eight waves where the tile is large enough to share (they hide each
// other's LDS reads: 128 x 256 at 512 rows 138 -> 136 us, 64 x 128 at 64 rows of [4096, 14336 x 2] 44.7 -> 44.2 us).
// Tiles of 24 K to 36 K outputs but for 128 x 256: four waves multiply and four do nothing but load.  A wave that does both
// stalls with its MFMAs behind a load that the CU has no room for (a CU keeps 32 KB of misses in flight, however deep the
// ring: a kernel that only streams gets 13 bytes a clock and CU from HBM, 31 from the last-level cache, 63 from its L2); a loop
// without MFMAs and fragment reads takes as long as the whole one then.  192 x 128, 192 x 192 and 256 x 128 are in the family
// because of it: 150 rows x [4096, 14336 x 2] 68 -> 62 us, 192 x [14336, 4096] in eight parts 41.6 -> 38.4, 333 x [18176, 4544]
// in parts 74.7 -> 72.9, 1000 x [4544, 4672] 52.4 -> 48.3 (the best of the family without / with them); 128 x 192 in place
// of four waves that do both 48.0 -> 46.5 (800 x [4096, 6144]); 128 x 256 with four loading waves is level with eight waves
// that do both (333 x [4544, 18176] 64.0 and 64.2), 128 x 128 behind it, 96 x 256 behind 192 x 128.  Two loading waves are
// too few (loads alone, all from the L2, 38 against 31 us).
// Non-temporal weights where one block of at most 32 rows sees them: 16 rows x [18176, 4544] in 7 parts 29.6 -> 27.1 us
// (6.1 TB/s), x [14336, 4096] in 8 parts 22.6 -> 21.2 us; at 64 rows the gain is gone (42.7 -> 43.6, 25.1 -> 23.6 us).
// That tile has three stages, or four (ring_fourth_stage).
#define TRI_RING_TILES(X)            \
  X(0, 32, 128, 1, 4, 3, true, 0)    \
  X(1, 64, 64, 2, 2, 5, false, 0)    \
  X(2, 64, 128, 2, 4, 3, false, 0)   \
  X(3, 96, 128, 1, 4, 5, false, 0)   \
  X(4, 128, 128, 2, 4, 5, false, 0)  \
  X(5, 128, 192, 2, 2, 3, false, 4)  \
  X(6, 128, 256, 2, 4, 3, false, 0)  \
  X(7, 160, 256, 1, 4, 3, false, 0)  \
  X(8, 192, 128, 2, 2, 3, false, 4)  \
  X(9, 192, 192, 2, 2, 3, false, 4)  \
  X(10, 256, 128, 2, 2, 3, false, 4)
constexpr int kRingTiles = 11;
constexpr int kRingTileOneBlock = 0;  // the non-temporal tile, for a single row block of up to 32 rows
// That tile with a fourth stage: 48 KB of weights on their way per workgroup in place of 32.  A CU with two workgroups has
// enough with three stages, and more costs time; one with a single workgroup, or none, leaves memory bandwidth unused, the
// more so the faster the memory is at the distance between rows.  What counts is the last round of workgroups (two a CU).
// us with three / four stages, one row unless said otherwise:
//   K-contiguous: [3072, 11008 x 2] in 4 parts, 688 workgroups, 32.1 / 28.9, [2048, 5632 x 2], 176, 14.9 / 14.2, [5120, 13824 x 2],
//     216, 46.4 / 44.4, [14336, 8192 x 2] in 4 parts, 512, 77.2 / 80.7; columns a multiple of 4 KB apart and parts of as many, from 384
//     on: [6144, 9728 x 2] in three, 456, 51.6 / 49.1, [14336, 4544 x 2] in seven, 497, 58.1 / 54.1, [2048, 28672 x 2], 448, 47.4 / 44.1,
//     but [6144, 17408 x 2], 272, 97.8 / 102.3; a power of two of 8 KB and more: 16 rows x [8192, 5120 x 2] in three parts, 240, 36.3 /
//     38.1, [4096, 12288 x 2] in four, 768, 44.6 / 43.0, [8192, 28672 x 2], 448, 156 / 167, [8192, 8192 x 2], 512, 68.1 / 73.0, but parts of
//     4096, 4 rows x [16384, 15904] in four, 500, 109 / 102, [4096, 32400 x 2], 507, 108 / 96.  (22 KB, K = 11008, would have four
//     there too: 4 rows x [11008, 28672 x 2], 448, 223 / 214.)
//   rows no multiple of 256 bytes: 16 rows x [4544, 4544], 216, 13.2 / 12.9, [4096, 13632], 107, 30.6 / 25.2, [4096, 12288] out of
//     18112, 288, 24.4 / 25.4, 16 rows x [18176, 4672], 481, 1.1 % slower; up to eight rows and nearly two on every CU level or better:
//     [18176, 4544], 504, the whole Falcon-7B FFN 63.1 / 62.8; no multiple of 1 KB: [4544, 9088 x 2], 142, 36.1 / 32.0, [4096, 18176],
//     142, 32.2 / 28.4, [4096, 32000], 250, 40.8 / 42.2
//   else: [4096, 8192], 64, 29.1 / 26.3, [4096, 12288], 192, 22.1 / 22.1, 16 rows x [4096, 6144], 240, 14.1 / 14.6, x [4096, 28672],
//     224, 38.4 / 39.6; halves (a tile takes 128 bytes of a row from each of two matrices) [4096, 8192 x 2], 128, 35.6 / 36.2
// Over 960 K-contiguous and 1170 row-major plans (K 1024 to 18176, 1 to 32 rows) the rule's choice is on average 0.3 and 0.1 %
// slower than the better of the two, at worst 10 % (K-contiguous, K = 14336 in 7 parts, 504 workgroups) and 2.5 %; three
// everywhere 2.3 and 0.4 %, four everywhere 0.7 and 1.5 %.  A column view whose first element is 128 bytes into a line of 256
// changes nothing ([4096, 4096] three / four 11.6 / 11.9 with it, 11.8 / 12.0 without).
using RingTileFour = RingTile<32, 128, 1, 4, 4, true>;
// Q/K/V projections of more than 32 rows in one part and one round (ring_fine_plan): the only tile that takes whole 128-wide heads,
// or 130 to 160 rows of 6144 columns, without parts, whose merge norms and scatters.
using RingTileFine = RingTile<32, 128, 1, 4, 4>;
constexpr int kRingTileFine = kRingTiles;
// K-contiguous columns a power of two of 8 KB and more apart: the memory is slow there.
inline bool ring_slow_columns(int64_t ld) { return ld >= 4096 && (ld & (ld - 1)) == 0; }
// (ld: distances between rows or columns, several or-ed together; k_part: K of a workgroup)
inline bool ring_fourth_stage(int rows, int workgroups, int64_t ld, int k_part, bool kcontig, bool halves) {
  const int last = (workgroups - 1) % 512 + 1;
  if (kcontig) {
    if (ring_slow_columns(ld)) return last < (workgroups <= 256 ? 224 : 257) || (last >= 384 && k_part == 4096);
    return last <= 256 || (last >= 384 && ld % 2048 == 0 && k_part % 2048 == 0);
  }
  if ((ld & 127) != 0) return last < 256 || (rows <= 8 && last > 480);
  if ((ld & 511) != 0) return last < 224;
  return !halves && workgroups < 176;
}
// K-contiguous weights whose columns lie a multiple of 8 KB apart, up to 32 rows (ring_takes_narrow): two waves, 64 columns, and
// an XCD's workgroups on neighbouring columns.  At such distances the memory is slow (a kernel that only reads [4096, 28672]: 45.4 us
// with 224 workgroups of 128 columns, 39.9 with 448 of 64, 37.9 with neighbours on one XCD).
using RingTileKContig = RingTile<32, 64, 1, 2, 5, true>;

// Workgroup id -> (row block, column tile, split): row blocks fastest, so that the workgroups that stream the same
// weights for different rows run together, then columns.  With several row blocks, or tiles of 96 rows and more, the
// round robin of workgroups over the XCDs is undone first: an XCD's L2 then sees the weights once for all its row
// blocks and one run of the activations (100 rows, K = 18176: 42.5 -> 37.7 us).  A single block of few rows has
// nothing to share, and neighbouring columns on different XCDs consume whole DRAM pages together (16 rows,
// K = 4096, 28672 columns: 42.0 -> 40.3 us).
__device__ __forceinline__ void ring_coords(int pid, int nrb, int ntn, int ksplit, bool chunked, int& rb, int& tn, int& split) {
  if (chunked) {
    const int total = nrb * ntn * ksplit, per = total >> 3, rem = total & 7, xcd = pid & 7;
    pid = xcd * per + (xcd < rem ? xcd : rem) + (pid >> 3);
  }
  rb = pid % nrb;
  pid /= nrb;
  tn = pid % ntn;
  split = pid / ntn;
}

// acc[ni][mi] = W-tile^T x X-tile over k in [0, K) of the given pointers (K % 32 == 0, K >= 64).
//   wmap(c, ldw): NTL (K-contiguous weights): c = LDS row of the weight tile -> start of that column's k run;
//   otherwise c = column chunk of the tile -> its first element at k = 0, ldw = distance between k rows.
// SWAP exchanges the MFMA operands (rows = tokens in the registers, columns across the lanes).
// K % 64 == 32: the last k tile starts at K - 64 and its first two k16 steps, already done, are left out.
template <class T, bool NTL, bool SWAP, class WMap>
__device__ __forceinline__ void gemm_mainloop_ring(const half_t* __restrict__ x, int64_t ldx, int m0, int M, int K,
                                                   WMap wmap, half_t* lds, float16v (&acc)[T::NI][T::MI]) {
  constexpr int NW = T::NW, LW = T::LW, BK = T::BK, BN = T::BN, NST = T::NST, XI = T::XI, WI = T::WI, L = T::L, CPR = T::CPR;
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave % T::WM, wn = wave / T::WM;
  const int l32 = lane & 31, g = lane >> 5;
  const int KT = (K + BK - 1) / BK;
  const int lw = T::NP > 0 ? max(wave - NW, 0) : wave;  // which of the loading waves

  const half_t* xsrc[XI];
  const half_t* wsrc[WI];
  // a lane keeps its column chunk, and with it the distance between k rows, over all instructions - unless a row is not
  // a divisor of 64 chunks (BN = 192), where a tile across two weight matrices needs the distance per instruction
  constexpr int NLD = (!NTL && 64 % CPR != 0) ? WI : 1;
  int64_t ldw[NLD];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int rloc = (i * LW + lw) * 8 + (lane >> 3);
    int row = m0 + rloc;
    row = row < M ? row : M - 1;
    xsrc[i] = x + (int64_t)row * ldx + ((lane & 7) ^ ((rloc >> 1) & 7)) * 8;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    if constexpr (NTL) {
      const int nloc = (i * LW + lw) * 8 + (lane >> 3);
      wsrc[i] = wmap(nloc, ldw[0]) + ((lane & 7) ^ ((nloc >> 1) & 7)) * 8;
    } else {
      const int p = (i * LW + lw) * 64 + lane;
      const int krow = p / CPR, slot = p % CPR;
      const int chunk = CPR % 16 == 0 ? slot ^ ((krow & 3) << 2) : slot ^ (((krow >> 1) & 1) << 2);
      wsrc[i] = wmap(chunk, ldw[i % NLD]) + (int64_t)krow * ldw[i % NLD];
    }
  }
  // first k of tile kt; past the end the loop keeps its load count (the waits assume it): the last tile again
  auto koff = [&](int kt) { return min(kt * BK, K - BK); };
  // position of a k tile in both operands, carried from tile to tile (a product per lane and tile would cost as many
  // instructions as the loads themselves where a tile crosses two weight matrices)
  struct KPos {
    int k;
    int64_t w[NLD];
  };
  int64_t wstep[NLD];  // 64 rows on
#pragma unroll
  for (int j = 0; j < NLD; ++j) wstep[j] = NTL ? BK : BK * ldw[j];
  auto advance = [&](KPos& o, int kt) {  // to tile kt, from the tile before
    const int k = koff(kt), d = k - o.k;  // uniform: 64, then 32 at an odd end, then 0
    o.k = k;
    if (d == BK) {
#pragma unroll
      for (int j = 0; j < NLD; ++j) o.w[j] += wstep[j];
    } else if (d != 0) {
#pragma unroll
      for (int j = 0; j < NLD; ++j) o.w[j] += wstep[j] / 2;
    }
  };
  auto load_one = [&](const KPos& o, int st, int i) {
    half_t* b = lds + st * T::STAGE;
    if (i < XI) load_to_lds16(xsrc[i] + o.k, b + (i * LW + lw) * 512);
    else load_to_lds16<T::NTW>(wsrc[i - XI] + o.w[(i - XI) % NLD], b + T::X_HALFS + ((i - XI) * LW + lw) * 512);
  };
  KPos pos;
  pos.k = 0;
#pragma unroll
  for (int j = 0; j < NLD; ++j) pos.w[j] = 0;

  // ---- waves that only load: a tile goes out as soon as the barrier has freed its stage, and the barrier of tile kt waits for
  // their loads of tile kt + 1.  (Barriers: one before tile 0, then one per tile but the last - the others' below.)
  if (T::NP > 0 && wave >= NW) {
    auto load_tile = [&](int st) {
#pragma unroll
      for (int i = 0; i < L; ++i) load_one(pos, st, i);
    };
#pragma unroll
    for (int s = 0; s < NST; ++s) {
      load_tile(s);
      advance(pos, s + 1);
    }
    TRI_WAIT_VMCNT((NST - 1) * L);
    __builtin_amdgcn_s_barrier();
    int st = 0;
    for (int kt = 0; kt < KT - 1; ++kt) {
      TRI_WAIT_VMCNT((NST - 2) * L);
      __builtin_amdgcn_s_barrier();
      load_tile(st);  // tile kt + NST
      advance(pos, kt + NST + 1);
      st = st == NST - 1 ? 0 : st + 1;
    }
    TRI_WAIT_VMCNT(0);
    return;
  }

  // ---- fragment read offsets (halfs)
  const int sx = (l32 >> 1) & 7;
  int xoff[4], woff_t[4], woff_n[T::NI];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    xoff[kk] = (wm * T::TM + l32) * BK + (((kk * 2 + g) ^ sx) << 3);
    woff_t[kk] = T::X_HALFS + (wn * T::TN + l32) * BK + (((kk * 2 + g) ^ sx) << 3);
  }
  const int j4 = (lane & 15) >> 2;
#pragma unroll
  for (int ni = 0; ni < T::NI; ++ni) {
    const int chunk = (wn * T::TN + ni * 32) / 8 + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    const int slot = CPR % 16 == 0 ? chunk ^ (j4 << 2) : chunk ^ (((j4 >> 1) & 1) << 2);
    woff_n[ni] = T::X_HALFS + (g * 8 + j4) * BN + (slot << 3) + (lane & 1) * 4;
  }
  half8v wf[2][T::NI], xf[2][T::MI];
  auto read_one = [&](int st, int kk, int buf, int i) {
    const half_t* b = lds + st * T::STAGE;
    if (i < T::NI) {
      if constexpr (NTL) {
        wf[buf][i] = lds_read8(b + woff_t[kk] + i * 32 * BK);
      } else {
        const half_t* p = b + woff_n[i] + kk * 16 * BN;
        wf[buf][i] = cat8(lds_read_tr16(p), lds_read_tr16(p + 4 * BN));
      }
    } else {
      xf[buf][i - T::NI] = lds_read8(b + xoff[kk] + (i - T::NI) * 32 * BK);
    }
  };
  constexpr int NM = T::NI * T::MI, NF = T::NI + T::MI;
  auto mfma_one = [&](int buf, int i) {
    const int ni = i / T::MI, mq = i % T::MI;
    const int mi = (ni & 1) ? T::MI - 1 - mq : mq;  // serpentine: consecutive MFMAs share a source operand
    acc[ni][mi] = SWAP ? mfma32(xf[buf][mi], wf[buf][ni], acc[ni][mi]) : mfma32(wf[buf][ni], xf[buf][mi], acc[ni][mi]);
  };
  // one k16 step, slot by slot (a schedule fence after each): MFMA i on set `buf`, its share of the loads [lo, hi) of
  // the tile at `o` into stage st and of the fragment reads of step rkk of stage rst into the other set (rkk < 0: none)
  auto step = [&](int buf, const KPos& o, int st, int lo, int hi, int rst, int rkk) {
    const int n = hi - lo;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      mfma_one(buf, i);
#pragma unroll
      for (int j = lo + i * n / NM; j < lo + (i + 1) * n / NM; ++j) load_one(o, st, j);
      if (rkk >= 0) {
#pragma unroll
        for (int j = i * NF / NM; j < (i + 1) * NF / NM; ++j) read_one(rst, rkk, buf ^ 1, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int ni = 0; ni < T::NI; ++ni)
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[ni][mi][r] = 0.f;

  // a quarter of tile kt + NST's loads is issued in the last step of tile kt, the rest in the first three of kt + 1
  constexpr int LE = T::NP > 0 ? 0 : L, L0 = LE / 4, L1 = LE / 2, L2 = 3 * LE / 4;
  if constexpr (T::NP == 0) {
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) {
#pragma unroll
      for (int i = 0; i < L; ++i) load_one(pos, s, i);
      advance(pos, s + 1);
    }
#pragma unroll
    for (int i = 0; i < L0; ++i) load_one(pos, NST - 1, i);
    TRI_WAIT_VMCNT((NST - 2) * L + L0);
  }
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < NF; ++i) read_one(0, 0, 0, i);
  int st = 0;
  for (int kt = 0; kt < KT - 1; ++kt) {
    const int sn = st == NST - 1 ? 0 : st + 1;
    const int sp = st == 0 ? NST - 1 : st - 1;  // the stage of tile kt - 1, taken by tile kt + NST - 1
    __builtin_amdgcn_sched_barrier(0);
    step(0, pos, sp, L0, L1, st, 1);
    step(1, pos, sp, L1, L2, st, 2);
    step(0, pos, sp, L2, LE, st, 3);
    if constexpr (T::NP > 0) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's reads of tile kt are over
      __builtin_amdgcn_s_barrier();
    } else {
      // this wave's reads of tile kt are over and its share of tile kt + 1 has landed; kt + 2 .. kt + NST - 1 in flight
      constexpr int V = (NST - 2) * L;
      __builtin_amdgcn_s_waitcnt((V & 15) | ((V >> 4) << 14) | 0x0070);  // vmcnt(V) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      advance(pos, kt + NST);
    }
    __builtin_amdgcn_sched_barrier(0);
    step(1, pos, st, 0, L0, sn, 0);
    st = sn;
  }
  if (K % BK == 0) {
    step(0, pos, 0, 0, 0, st, 1);
    step(1, pos, 0, 0, 0, st, 2);
  } else {
#pragma unroll
    for (int i = 0; i < NF; ++i) read_one(st, 2, 0, i);
  }
  step(0, pos, 0, 0, 0, st, 3);
  step(1, pos, 0, 0, 0, st, -1);
  if constexpr (T::NP == 0) TRI_WAIT_VMCNT(0);
}

// k tiles per part of a plan (the last part takes what is left, and the odd 32 of a K that is not a multiple of 64)
inline int ring_kt_per_part(int K, int ksplit) { return (K / 64 + ksplit - 1) / ksplit; }

struct RingArgs {
  const half_t* x;
  int64_t ldx;
  const half_t* w[3];  // column segments, concatenated logically
  int64_t ldw[3];      // distance between k rows (row-major) or between columns (K-contiguous)
  int seg_begin[3];    // first logical column of each segment (unused segments start at ncols)
  int M, K, ncols, ksplit;
  float* partial;      // [ksplit][M][ncols]
};
// fp32 partial results of the plan's parts
int launch_ring_partial(const RingArgs& a, int tile, bool kcontig, hipStream_t stream);

}  // namespace tri

#endif  // once per element type
