// Per-key accumulators over queries for RoCo (sum p, sum p^2) and KeyFormer
// (sum of the noise-perturbed probabilities).
//
// Key-major column reduction: a workgroup owns 128 keys of one query head
// (4 waves x 32 keys, K fragments held in registers) and walks the query axis
// in tiles of 64 that go global -> LDS directly.  The score tile is recomputed
// with MFMA in the transposed orientation S^T[key, query], the row normaliser
// comes from the log-sum-exp written by the attention kernel, and each lane
// accumulates its sixteen keys over all queries it meets; one cross-lane
// reduction at the very end.  Nothing of size [heads, S, S] ever reaches HBM.
//
// Under the causal mask key block b only meets queries >= its first key, so
// the work per block falls linearly with b: the longest blocks are dispatched
// first.  (Pairs of blocks b and n - 1 - b, all equally long, remain where a
// workgroup would have too little to do, see score_form.)
//
// Where such workgroups leave CUs empty (up to 1024 keys x 32 heads) the kernel's time is one workgroup's chain of
// tiles: there a workgroup owns 64 keys, its waves are two groups of keys times two query groups that take the tiles of
// the query axis in turn, a step moves a pair of tiles, and the two groups' sums meet in LDS (QG = 2).
#include "common.h"
#include "launch.h"
#include "philox.h"


namespace tri {

constexpr int kQTile = 64;
constexpr int kKeysPerWg = 128;  // (half of them with two query groups)

constexpr int kScoreStages = 4;         // steps (a Q tile per query group) in LDS
constexpr int kScoreMergeFloats = 64;   // sums a wave of the second query group hands over
constexpr int kScoreRound = 256;        // workgroups that have a CU each
constexpr int kScoreBlockTiles = 4, kScoreHandTiles = 1, kScorePairWorkgroups = 768;  // (score_form; the last per query tile)

// s_waitcnt vmcnt(n) leaving the other counters unconstrained (gfx9 encoding)
#define TRI_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0x0F70)

// x + (x of the lane that the DPP pattern CTRL names); rows outside ROW_MASK keep x
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROW_MASK, 0xF, true));
}

// Sum over the 32 lanes of each half of the wave, in lanes 16..31 of the half (the other lanes hold the sum of
// their own 16).  Five vector instructions with lane patterns; the same through __shfl_xor is five LDS
// permutes, each with a wait for the LDS, and a key block ends with 32 such sums per lane.
__device__ __forceinline__ float half_wave_sum_dpp(float x) {
  x = dpp_add<0xB1, 0xF>(x);   // quad_perm [1,0,3,2]
  x = dpp_add<0x4E, 0xF>(x);   // quad_perm [2,3,0,1]
  x = dpp_add<0x141, 0xF>(x);  // row_half_mirror: the other quad of the eight
  x = dpp_add<0x140, 0xF>(x);  // row_mirror: the other eight of the row of 16
  x = dpp_add<0x142, 0xA>(x);  // row_bcast:15 into rows 1 and 3: the sum of the row before
  return x;
}

// MODE_ 0: RoCo; 1: KeyFormer; 2: KeyFormer with seeded noise at temperature 1 (a compile-time variant: left as
// a run-time flag, the compiler computes both noise transforms for every element and selects)
//
// Schedule.  A wave's unit of work is a half tile: S^T of its 32 keys against 32 queries (a chain of D / 16
// MFMAs into one accumulator) and the exponentials and sums of those 16 scores per lane.  The MFMA chain of half
// tile n + 1 is interleaved, instruction slot by slot, with the vector arithmetic of half tile n: one MFMA, the
// LDS read of a Q fragment three slots ahead, two scores' worth of arithmetic, and a scheduling fence - left to
// itself the compiler puts all MFMAs of a tile first, each waiting for its LDS read, and the arithmetic after.
// The chain of (tile t + 1, first half) runs during step t, so a Q tile must be in LDS one step before its own:
// four LDS stages, tiles loaded three steps ahead (tiles past the last one read as zero and are never used).
//
// LONE: a workgroup takes one key block, not two.  (A template parameter: as a field of the arguments it left the loop's
// instructions as they are and cost RoCo 13 % all the same - 10 heads of 128, 1500 tokens, the kernel alone, pairs 27.5 -> 31.0 us,
// single blocks 21.6 -> 25.0; 71 heads of 64, 300 against 9000 keys, single blocks 71.5 -> 77.8; KeyFormer 31.1 -> 31.6.)
template <int D, int MODE_, int QG, bool LONE>
__device__ __forceinline__ void score_body(const ScoreArgs& a, half_t* lds) {
  constexpr int MODE = MODE_ == 0 ? 0 : 1;
  constexpr bool kf_fast = MODE_ == 2;  // seeded noise at temperature 1: exp(s + g) = exp(s) / (-ln u)
  constexpr int TILE = kQTile * D;   // halfs; unpadded, XOR-swizzled (chunk c of row r at slot c ^ f(r))
  constexpr int STAGE = QG * TILE;   // a step's tiles, one per query group
  constexpr int KEYS = kKeysPerWg / QG, KWAVES = 4 / QG;
  constexpr int KSTEPS = D / 16;
  constexpr int CPR = D / 8, INSTR = QG * kQTile * D * 2 / 1024 / 4;
  constexpr int PD = 3, RING = 4;  // LDS reads run PD slots ahead of their MFMAs
  constexpr int GPS = 8 / KSTEPS;  // groups of two scores per MFMA slot
  static_assert(KSTEPS % RING == 0 && PD < KSTEPS, "the fragment ring keeps its phase from chain to chain");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kgroup = wave % KWAVES, qgroup = wave / KWAVES;
  const int l32 = lane & 31, g = lane >> 5;
  const int Ltot = a.P + a.S;
  const int nkb = (Ltot + KEYS - 1) / KEYS;
  // Linear workgroup id -> (head, key block or pair of them).  Workgroups go to the eight XCDs round-robin by id; with a
  // multiple of eight heads XCD x takes heads [x Hq / 8, (x + 1) Hq / 8), so that its L2 streams the Q rows of
  // those heads only (all workgroups of a head read the same Q).  Other head counts: pairs head by head; single blocks by
  // length, all heads' longest first (head by head the last heads' long blocks start last: whole calls, 71 heads of 64, RoCo 2048
  // tokens 207 -> 188 us, 4096 548 -> 482, KeyFormer 1000 127 -> 111, 4096 904 -> 760; 20 of 128 on 4, KeyFormer 4096 441 -> 365; level
  // behind long prefixes, where all blocks are as long).
  const int nbx = LONE ? nkb : (nkb + 1) / 2;
  int h, bx;
  if (a.Hq % 8 == 0) {
    const int x = (int)blockIdx.x % 8, sidx = (int)blockIdx.x / 8;
    const int hx = a.Hq / 8;
    h = x * hx + (LONE ? sidx % hx : sidx / nbx);
    bx = LONE ? sidx / hx : sidx % nbx;
  } else {
    h = LONE ? (int)blockIdx.x % a.Hq : (int)blockIdx.x / nbx;
    bx = LONE ? (int)blockIdx.x / a.Hq : (int)blockIdx.x % nbx;
  }
  const int hk = h / (a.Hq / a.Hkv);
  // the wave's slot on its SIMD (HW_ID bits 3:0): the waves that share a SIMD differ in it
  const int slot = __builtin_amdgcn_s_getreg(4 | (0 << 6) | (3 << 11));
  const float c2 = a.scale * kLog2e;
  const float cp2 = kLog2e / a.tau;
  const uint32_t seed_lo = (uint32_t)a.seed, seed_hi = (uint32_t)(a.seed >> 32);
  auto swz = [](int row) { return D == 128 ? (row & 15) : ((row >> 1) & 7); };

  // Q tiles: buffer-descriptor loads straight into LDS; rows past S read as zero
  const __amdgpu_buffer_rsrc_t qrsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<half_t*>(a.q + h * D), 0, (int)(((int64_t)(a.S - 1) * a.ldq + D) * 2), 0x00020000);
  int ld_off[INSTR];
#pragma unroll
  for (int i = 0; i < INSTR; ++i) {
    const int p = (i * 4 + wave) * 64 + lane;
    const int row = p / CPR, slot = p % CPR;
    ld_off[i] = (row * (int)a.ldq + (slot ^ swz(row)) * 8) * 2;
  }
  const int qtile_bytes = kQTile * (int)a.ldq * 2;
  // Q fragment of k step ks: chunk (2 ks + g) ^ swz of row l32 - the k step only flips bits of the chunk index.
  // (Byte offsets, one register per k step behind an empty asm statement: the compiler would otherwise keep one
  // per (k step, half, stage).)
  int qb[KSTEPS];
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) {
    qb[ks] = (qgroup * TILE + l32 * D + (((ks * 2 + g) ^ swz(l32)) << 3)) * 2;
    asm volatile("" : "+v"(qb[ks]));
  }
  const char* const ldsb = reinterpret_cast<const char*>(lds);
  // fragment (this wave's tile of step st, query half u, k step ks)
  auto frag = [&](int st, int u, int ks) {
    return *reinterpret_cast<const half8v*>(ldsb + qb[ks] + ((st & (kScoreStages - 1)) * STAGE + u * 32 * D) * 2);
  };

  for (int half = 0; half < 2; ++half) {
    // the two key blocks of this workgroup: b and n-1-b (the middle one only once)
    const int kb = half == 0 ? bx : nkb - 1 - bx;
    if (half == 1 && (LONE || kb <= bx)) break;
    const int kb0 = kb * KEYS;
    const int kw0 = kb0 + kgroup * 32;

    // K fragments: MFMA source 0, rows = this wave's 32 keys
    half8v kf[KSTEPS];
    {
      int key = kw0 + l32;
      key = key < Ltot ? key : Ltot - 1;
      const half_t* kp = a.k + (int64_t)hk * a.k_sh + (int64_t)key * a.k_sr + g * 8;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) kf[ks] = *reinterpret_cast<const half8v*>(kp + ks * 16);
    }
    // queries that can see any key of this block
    int qstart = 0;
    if (a.causal) {
      qstart = kb0 - a.P;
      qstart = qstart > 0 ? (qstart / kQTile) * kQTile : 0;
    }
    const int nqt = qstart < a.S ? (a.S - qstart + kQTile - 1) / kQTile : 0;
    const int nsteps = (nqt + QG - 1) / QG;
    auto issue = [&](int st) {   // (st may lie past the last step: those rows are past S and read as zero)
#pragma unroll
      for (int i = 0; i < INSTR; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            qrsrc, (TRI_LDS void*)(lds + (st & (kScoreStages - 1)) * STAGE + (i * 4 + wave) * 512), 16,
            // (unsigned: steps up to three past the last one are issued, and for a Q buffer close to 2 GiB their
            // offsets pass 2^31; they stay beyond the descriptor's size and read as zero)
            (int)((uint32_t)ld_off[i] + (uint32_t)(qstart / kQTile + st * QG) * (uint32_t)qtile_bytes), 0, 0, 0);
    };
    auto tile_of = [&](int st) { return st * QG + qgroup; };  // the wave's tile of a step
    auto load_lse = [&](int st, float (&v)[2]) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        int q = qstart + tile_of(st) * kQTile + nt * 32 + l32;
        q = q < a.S ? q : a.S - 1;
        v[nt] = a.lse[(int64_t)h * a.S + q];
      }
    };

    float acc1[16], acc2[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) { acc1[r] = 0.f; acc2[r] = 0.f; }

    // vector arithmetic of scores 2 i and 2 i + 1 of a half tile (step n, query half u); st: its S^T block
    uint32_t rnd[4] = {0u, 0u, 0u, 0u};
    auto group = [&](const float16v& st, int n, int u, float lse_q, int i, const bool MASK) {
      const int q = qstart + tile_of(n) * kQTile + u * 32 + l32;
      const int qq = q < a.S ? q : a.S - 1;
      const int qlim = a.causal ? a.P + qq : Ltot;
      const float lse2 = lse_q * kLog2e;
      const int rq = i / 2, rp = i / 4;  // the lane's keys kw0 + 8 rq + 4 g + e; groups rq = 2 rp and 2 rp + 1 are
                                         // the two halves of one generator call
      if (MODE == 1 && (i % 4) == 0 && (kf_fast || a.noise == nullptr))
        philox4x32(noise_counter(kw0 + rp * 16 + g * 4), (uint32_t)qq, (uint32_t)h, 0u, seed_lo, seed_hi, rnd);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int r = 2 * i + x, e = r % 4;
        const int key = kw0 + rq * 8 + g * 4 + e;
        float gn = 0.f;
        if (MODE == 1) {
          if (!kf_fast && a.noise != nullptr) {
            gn = (float)a.noise[((int64_t)h * a.S + qq) * Ltot + min(key, Ltot - 1)];
          } else {
            const uint32_t bits = (rq % 2) ? (rnd[e] >> 16) : (rnd[e] & 0xFFFFu);
            gn = kf_fast ? inv_log2_uniform(bits) : gumbel_from_bits(bits);
          }
        }
        float v;
        if (MODE == 1 && !kf_fast) v = (st[r] * a.scale + gn) * cp2 - lse2;
        else v = fmaf(st[r], c2, -lse2);
        float p = fast_exp2(v);
        if (MODE == 1 && kf_fast) p *= gn;
        if (MASK && (q >= a.S || key > qlim || key >= Ltot)) p = 0.f;
        acc1[r] += p;
        if (MODE == 0) acc2[r] = fmaf(p, p, acc2[r]);
      }
    };

    if (nqt > 0) {
      float lse_cur[2], lse_nxt[2];
      half8v fr[RING];
      float16v sa, sb;
      __builtin_amdgcn_s_barrier();  // the previous key block's tiles are no longer read by anyone
      load_lse(0, lse_cur);
      issue(0);
      issue(1);
      issue(2);
      TRI_WAIT_VMCNT(2 * INSTR);     // lse(0) and this wave's share of step 0
      __builtin_amdgcn_s_barrier();
      // ---- S^T of (step 0, first half) on its own; the first fragments of its second half
#pragma unroll
      for (int r = 0; r < 16; ++r) sa[r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) sa = mfma32(kf[ks], frag(0, 0, ks), sa);
#pragma unroll
      for (int j = 0; j < PD; ++j) fr[j] = frag(0, 1, j);

      // One step: [chain (st, second half) beside the arithmetic of (st, first half)], then
      // [chain (st + 1, first half) beside the arithmetic of (st, second half)].
      auto step = [&](int st, const bool MASK) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sb[r] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KSTEPS; ++i) {
          fr[(i + PD) % RING] = (i + PD < KSTEPS) ? frag(st, 1, i + PD) : frag(st + 1, 0, i + PD - KSTEPS);
          sb = mfma32(kf[i], fr[i % RING], sb);
#pragma unroll
          for (int x = 0; x < GPS; ++x) group(sa, st, 0, lse_cur[0], i * GPS + x, MASK);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) sa[r] = 0.f;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KSTEPS; ++i) {
          fr[(i + PD) % RING] = (i + PD < KSTEPS) ? frag(st + 1, 0, i + PD) : frag(st + 1, 1, i + PD - KSTEPS);
          sa = mfma32(kf[i], fr[i % RING], sa);
#pragma unroll
          for (int x = 0; x < GPS; ++x) group(sb, st, 1, lse_cur[1], i * GPS + x, MASK);
          __builtin_amdgcn_sched_barrier(0);
        }
      };

      // Steps [q0, q1), every one with or every one without masking.  The walk over the steps is cut into such
      // runs - the tiles on the causal diagonal come first, a ragged last tile last, and in between nothing is
      // masked - because one loop that chose between the two copies of the step tile by tile made the compiler keep
      // the sums and the S^T blocks in different registers in the two copies and move them at every turn: 62
      // register moves per tile beside 128 instructions of arithmetic (RoCo, S = 4096: 448 -> 440 us).
      auto run = [&](int q0, int q1, const bool MASK) __attribute__((always_inline)) {
        for (int st = q0; st < q1; ++st) {
          // Two workgroups share a CU, and a SIMD serves the older of its two waves first whenever both are ready:
          // left alone, the older workgroup runs at the pace of a lone one, the younger on what is left, and then
          // finishes on its own, one wave per SIMD (S = 4096: one done after 76 us, the other after 110 us).  So the
          // two waves of a SIMD take turns at the higher priority, tile by tile, and stay side by side.
          if ((st ^ slot) & 1) __builtin_amdgcn_s_setprio(1);
          else __builtin_amdgcn_s_setprio(0);
          // this wave's share of step st + 1 has landed (the loads of a wave complete in order; those of step
          // st + 2 may still be in flight)
          TRI_WAIT_VMCNT(INSTR);
          __builtin_amdgcn_s_barrier();  // ... and everybody's; step st - 1 is retired
          load_lse(st + 1, lse_nxt);
          issue(st + 3);
          step(st, MASK);
          lse_cur[0] = lse_nxt[0];
          lse_cur[1] = lse_nxt[1];
        }
      };
      // masking is needed where the causal diagonal crosses this wave's keys - a tile qt with
      // kw0 + 31 > P + qstart + 64 qt - and at the ragged ends (keys past the last one: every tile; queries past
      // S: the last tile, and one past it).  Every wave walks all steps, one barrier each, whatever its runs are.
      auto steps_before = [&](int qt) { return min(nsteps, max(0, (qt - qgroup + QG - 1) / QG)); };  // the wave's, on tiles before qt
      int n_diag = 0;
      if (kw0 + 32 > Ltot) n_diag = nsteps;
      else if (a.causal) n_diag = steps_before(max(0, (kw0 + 31 - a.P - qstart + kQTile - 1) / kQTile));
      const int n_plain_end = max(n_diag, steps_before((qstart + nqt * kQTile > a.S) ? nqt - 1 : nqt));
      run(0, n_diag, true);
      run(n_diag, n_plain_end, false);
      run(n_plain_end, nsteps, true);
      __builtin_amdgcn_s_setprio(0);
      TRI_WAIT_VMCNT(0);  // (the loads past the last step)
    }

    // ---- reduce over the 32 query lanes; lane (l32 == 16) of each half writes
    const float invS = 1.0f / (float)a.S;
    float* const other = reinterpret_cast<float*>(lds + kScoreStages * STAGE) + kgroup * kScoreMergeFloats;  // sums of query group 1
    if (QG == 2) {
      if (qgroup == 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float s1 = half_wave_sum_dpp(acc1[r]), s2 = MODE == 0 ? half_wave_sum_dpp(acc2[r]) : 0.f;
          if (l32 == 16) {
            other[g * 32 + r] = s1;
            if (MODE == 0) other[g * 32 + 16 + r] = s2;
          }
        }
      }
      __syncthreads();  // (the next block's sums are written behind its barriers)
      if (qgroup == 1) continue;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float s1 = half_wave_sum_dpp(acc1[r]), s2 = MODE == 0 ? half_wave_sum_dpp(acc2[r]) : 0.f;
      if (QG == 2) {
        s1 += other[g * 32 + r];
        if (MODE == 0) s2 += other[g * 32 + 16 + r];
      }
      if (MODE == 1 && kf_fast) s1 *= kInvNegLnScale;
      const int key = kw0 + (r >> 2) * 8 + g * 4 + (r & 3);
      if (l32 == 16 && key < Ltot) {
        if (MODE == 0) {
          if (a.mean_var) {
            const float mean = s1 * invS;
            a.o1[(int64_t)h * a.ldo1 + key] = mean;
            a.o2[(int64_t)h * a.ldo2 + key] = s2 * invS - mean * mean;
          } else {
            a.o1[(int64_t)h * a.ldo1 + key] = s1;
            a.o2[(int64_t)h * a.ldo2 + key] = s2;
          }
        } else {
          a.o1[(int64_t)h * a.ldo1 + key] = s1;
        }
      }
    }
  }
}

// (body in a device function: see the note at attn_fwd_kernel)
template <int D, int MODE, int QG, bool LONE>
__global__ __launch_bounds__(256) void score_kernel(ScoreArgs a) {
  extern __shared__ __attribute__((aligned(16))) half_t lds[];
  score_body<D, MODE, QG, LONE>(a, lds);
}

template <int D, int MODE, int QG, bool LONE>
static int launch_score_t(const ScoreArgs& a, hipStream_t stream) {
  constexpr int LDS = kScoreStages * QG * kQTile * D * 2 + (QG == 2 ? 2 * kScoreMergeFloats * 4 : 0);
  constexpr auto kern = score_kernel<D, MODE, QG, LONE>;
  if (set_max_lds<kern, LDS>() != 0) return -1;
  const int nkb = (a.P + a.S + kKeysPerWg / QG - 1) / (kKeysPerWg / QG);
  hipLaunchKernelGGL(kern, dim3((LONE ? nkb : (nkb + 1) / 2) * a.Hq), dim3(256), LDS, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// One block of 128 keys a workgroup, or, where workgroups have a CU each, one or two blocks of 64 with two query groups if
// that chain is shorter, a block's first loads and last sums taken for kScoreBlockTiles tiles and the hand-over between
// two query groups for kScoreHandTiles.  (It counts: without it calls of 65 to 192 tokens took two groups, whole calls of 32
// heads on 8, RoCo 65 tokens 33.7 -> 34.5 us, 192 45.6 -> 46.7, 8 heads, KeyFormer 192 42.1 -> 42.9.  Over 135 calls of 40 to 4000 tokens the
// form taken is 0.3 % slower than the best on average, 0.8 without.)  Pairs of 128-key blocks as the only form -> this, whole
// calls of 32 heads on 8: RoCo, 512 (one of 64, 256 workgroups) 71.9 -> 66.4, 700 (one of 128, 192) 93.9 -> 77.1, 1000
// (two of 64, 256) 109.0 -> 98.5, 300 against 500 keys (one of 128, 224) 68.9 -> 62.7; KeyFormer 256 58.7 -> 54.5, 1000 121.2 ->
// 106.5, 300 against 500 78.3 -> 70.7; 71 heads of 64, RoCo 100 against 100 keys 39.5 -> 35.5.  Beyond a round, one block of
// 128: RoCo 1200 124.3 -> 117.4, 2048 189.2 -> 186.0, 3000 331.2 -> 321.8, 4096 433.3 -> 435.9, KeyFormer 1200 145.8 -> 136.4, 2048 224.2 ->
// 222.1, 3000 416.8 -> 400.2; but pairs where a block meets few query tiles and there are many (one tile, 33 against 3000 keys,
// 768 blocks, 42.4 -> 41.4, 64 against 4000, 1024, 50.6 -> 51.1, 40 against 16000, 4032, 98.8 -> 102.7; two, 100 against 6000, 1536, 71.3 ->
// 70.5; three, 150 against 15000, 3808, 141.2 -> 142.9; five, 300 against 9000, 2336, 157.8 -> 152.9; seven, 71 heads, 400 against
// 15000, 8520, 361.8 -> 363.5; eight, 512 against 16000, 4224, level).
int score_form(int S, int P, int Hq, bool causal) {
  auto blocks = [&](int g) { const int keys = kKeysPerWg / g; return (P + S + keys - 1) / keys; };
  auto chain = [&](int g, int kb) {  // steps of key block kb
    const int q0 = causal ? kb * (kKeysPerWg / g) - P : 0;
    const int tiles = (S - (q0 > 0 ? q0 / kQTile * kQTile : 0) + kQTile - 1) / kQTile;
    return kScoreBlockTiles + (tiles + g - 1) / g + (g - 1) * kScoreHandTiles;
  };
  const int n1 = blocks(1), n2 = blocks(2);
  const int64_t one = (int64_t)n1 * Hq, half = (int64_t)n2 * Hq;
  const int whole = one <= kScoreRound ? chain(1, 0) : 1 << 30;
  if (half <= kScoreRound && chain(2, 0) < whole) return kScoreHalfBlock;
  if (n2 > 1 && (int64_t)(n2 + 1) / 2 * Hq <= kScoreRound && chain(2, 0) + chain(2, n2 - 1) < whole) return kScoreHalfBlockPair;
  return one <= (int64_t)kScorePairWorkgroups * ((S + kQTile - 1) / kQTile) ? kScoreBlock : kScoreBlockPair;
}

template <int D, int MODE>
static int launch_score_d(const ScoreArgs& a, hipStream_t stream) {
  switch (score_form(a.S, a.P, a.Hq, a.causal != 0)) {
    case kScoreHalfBlock: return launch_score_t<D, MODE, 2, true>(a, stream);
    case kScoreHalfBlockPair: return launch_score_t<D, MODE, 2, false>(a, stream);
    case kScoreBlock: return launch_score_t<D, MODE, 1, true>(a, stream);
    default: return launch_score_t<D, MODE, 1, false>(a, stream);
  }
}

int launch_scores(const ScoreArgs& a, hipStream_t stream) {
  if (a.S <= 0) return 0;
  if (a.S <= kFewMaxQueries) {
    const int r = launch_scores_few(a, stream);
    if (r <= 0) return r;
  }
  if (a.D != 64 && a.D != 128) return -1;
  const int mode = a.mode == 1 && a.noise == nullptr && a.tau == 1.0f ? 2 : a.mode;
  switch (mode) {
    case 0: return a.D == 128 ? launch_score_d<128, 0>(a, stream) : launch_score_d<64, 0>(a, stream);
    case 1: return a.D == 128 ? launch_score_d<128, 1>(a, stream) : launch_score_d<64, 1>(a, stream);
    default: return a.D == 128 ? launch_score_d<128, 2>(a, stream) : launch_score_d<64, 2>(a, stream);
  }
}

}  // namespace tri
