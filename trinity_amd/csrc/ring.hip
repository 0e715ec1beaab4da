// GEMMs with few and middling rows (see ring.h for the main loop and what bounds it): the products of the FFNs and of
// the FFN block from 1 to about 1000 tokens, and fp32 partial products for the Q/K/V projection.
//
//   ring_epi_kernel       one workgroup per tile over the whole of K; row scale, activation, residual, one rounding and
//                         whole-row stores in its epilogue
//   ring_partial_kernel   the same tile over a part of K, fp32 partial products [split][row][column] to the workspace
//   ring_finalize_*       sum over the parts in a fixed order (results do not depend on scheduling) and the epilogue
//
// Parts are taken only where whole tiles leave CUs without work: they cost 8 bytes of traffic per output and part
// and a second launch.  ring_plan chooses tile and parts by cost.
#include "ring.h"

#include <math.h>

#include <type_traits>

namespace tri {

template <class T, bool WT>
__global__ __launch_bounds__(T::NT) void ring_partial_kernel(RingArgs a) {
  extern __shared__ __attribute__((aligned(16))) half_t lds[];
  const int nrb = (a.M + T::BM - 1) / T::BM, ntn = (a.ncols + T::BN - 1) / T::BN;
  int rb, tn, split;
  ring_coords(blockIdx.x, nrb, ntn, a.ksplit, nrb > 1 || T::BM >= 96, rb, tn, split);
  const int m0 = rb * T::BM, n0 = tn * T::BN;
  const int per = (a.K / 64 + a.ksplit - 1) / a.ksplit;  // as ring_kt_per_part
  const int k0 = split * per * 64;
  const int kr = split == a.ksplit - 1 ? a.K - k0 : per * 64;
  auto wmap = [&](int c, int64_t& ldw) -> const half_t* {
    int col = n0 + (WT ? c : c * 8);
    col = col < a.ncols ? col : 0;
    const int seg = col >= a.seg_begin[2] ? 2 : (col >= a.seg_begin[1] ? 1 : 0);
    const int64_t ld = seg == 2 ? a.ldw[2] : (seg == 1 ? a.ldw[1] : a.ldw[0]);
    const half_t* w = seg == 2 ? a.w[2] : (seg == 1 ? a.w[1] : a.w[0]);
    col -= seg == 2 ? a.seg_begin[2] : (seg == 1 ? a.seg_begin[1] : a.seg_begin[0]);
    ldw = ld;
    return WT ? w + (int64_t)col * ld + k0 : w + col + (int64_t)k0 * ld;
  };
  float16v acc[T::NI][T::MI];
  gemm_mainloop_ring<T, WT, true>(a.x + k0, a.ldx, m0, a.M, kr, wmap, lds, acc);

  // lanes run along the columns: 128 bytes of a row per half wave and store
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (T::NP > 0 && wave >= T::NW) return;  // (a wave that only loads)
  const int wm = wave % T::WM, wn = wave / T::WM;
  const int l32 = lane & 31, g = lane >> 5;
  float* base = a.partial + (int64_t)split * a.M * a.ncols;
#pragma unroll
  for (int ni = 0; ni < T::NI; ++ni) {
    const int n = n0 + wn * T::TN + ni * 32 + l32;
    if (n >= a.ncols) continue;
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * T::TM + mi * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        if (m < a.M) base[(int64_t)m * a.ncols + n] = acc[ni][mi][r];
      }
  }
}

// out = act(rowscale * X.W) [+ residual].  EPI_SWIGLU: the left half of a tile's columns are gate columns, the right
// half the matching up columns, so the two halves of an output sit in different waves: the up halves pass through LDS
// as fp32 (interleaving gate and up in steps of 16 columns keeps them in one lane, but row-major weights are then read
// in pieces of 32 bytes: 16 rows x [4096, 14336 x 2] 46.0 -> 47.1 us, 128 rows 56.8 -> 60.7 us).
template <class T, int EPI, bool WT>
__global__ __launch_bounds__(T::NT) void ring_epi_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) half_t lds[];
  constexpr bool GATED = EPI == EPI_SWIGLU;
  constexpr int OUT_BN = GATED ? T::BN / 2 : T::BN;
  const int nrb = (a.M + T::BM - 1) / T::BM, ntn = (a.N + OUT_BN - 1) / OUT_BN;
  int rb, tn, split;
  ring_coords(blockIdx.x, nrb, ntn, 1, nrb > 1 || T::BM >= 96 || std::is_same<T, RingTileKContig>::value, rb, tn, split);
  const int m0 = rb * T::BM, n0 = tn * OUT_BN;
  auto wmap = [&](int c, int64_t& ldw) -> const half_t* {
    const int nloc = WT ? c : c * 8;
    int col;
    const half_t* w = a.w;
    ldw = a.ldw;
    if (GATED) {
      col = n0 + nloc % OUT_BN;
      if (nloc >= OUT_BN) { w = a.w2; ldw = a.ldw2; }
    } else {
      col = n0 + nloc;
    }
    col = col < a.N ? col : n0;
    return WT ? w + (int64_t)col * ldw : w + col;
  };
  float16v acc[T::NI][T::MI];
  gemm_mainloop_ring<T, WT, false>(a.x, a.ldx, m0, a.M, a.K, wmap, lds, acc);

  // A lane owns one token and four consecutive columns per register quad: the tile turns around in LDS (free now) and
  // leaves as rows, 16 bytes per lane.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % T::WM, wn = wave / T::WM;
  const int l32 = lane & 31, g = lane >> 5;
  constexpr int RS = OUT_BN + 8;  // halfs per staged row
  constexpr int US = OUT_BN + 4;  // floats per row of the up half
  static_assert(T::BM * RS * 2 <= T::LDS_BYTES && (!GATED || (T::BM * US * 4 <= T::LDS_BYTES && T::WN % 2 == 0)), "the staged tile fits the ring");
  float* up = reinterpret_cast<float*>(lds);
  const bool loader = T::NP > 0 && wave >= T::NW;  // (holds no part of the tile, but stores rows of it below)
  const bool up_wave = GATED && !loader && wn >= T::WN / 2, out_wave = !up_wave && !loader;
  __syncthreads();  // every wave is done with the ring (and every load into it has landed)
  if (up_wave) {
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < T::NI; ++ni)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const float4v v = {acc[ni][mi][rq * 4], acc[ni][mi][rq * 4 + 1], acc[ni][mi][rq * 4 + 2], acc[ni][mi][rq * 4 + 3]};
          *reinterpret_cast<float4v*>(up + (wm * T::TM + mi * 32 + l32) * US + (wn - T::WN / 2) * T::TN + ni * 32 + rq * 8 + g * 4) = v;
        }
  }
  if (GATED) __syncthreads();
  if (out_wave) {
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi) {
      const int mloc = wm * T::TM + mi * 32 + l32, m = m0 + mloc;
      const bool mok = m < a.M;
      const float rs = (a.rowscale != nullptr && mok) ? a.rowscale[m] : 1.0f;
#pragma unroll
      for (int ni = 0; ni < T::NI; ++ni)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const int nloc = wn * T::TN + ni * 32 + rq * 8 + g * 4, n = n0 + nloc;
          float4v u = {0.f, 0.f, 0.f, 0.f};
          if (GATED) u = *reinterpret_cast<const float4v*>(up + mloc * US + nloc);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float c = acc[ni][mi][rq * 4 + e] * rs;
            if (EPI == EPI_GELU) c = gelu_erf(c);
            if (GATED) c = silu(c) * (u[e] * rs);
            acc[ni][mi][rq * 4 + e] = c;
          }
          if (a.residual != nullptr && mok && n < a.N) {
            const half4v rr = *reinterpret_cast<const half4v*>(a.residual + (int64_t)m * a.ldr + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[ni][mi][rq * 4 + e] += (float)rr[e];
          }
        }
    }
  }
  if (GATED) __syncthreads();  // the up half has been read
  if (out_wave) {
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < T::NI; ++ni)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          const half4v h = {(half_t)acc[ni][mi][rq * 4], (half_t)acc[ni][mi][rq * 4 + 1], (half_t)acc[ni][mi][rq * 4 + 2], (half_t)acc[ni][mi][rq * 4 + 3]};
          *reinterpret_cast<half4v*>(lds + (wm * T::TM + mi * 32 + l32) * RS + wn * T::TN + ni * 32 + rq * 8 + g * 4) = h;
        }
  }
  __syncthreads();
  constexpr int CH = OUT_BN / 8;  // 16-byte chunks per staged row
#pragma unroll 4
  for (int idx = threadIdx.x; idx < T::BM * CH; idx += T::NT) {
    const int row = idx / CH, ch = idx % CH;
    const int m = m0 + row, n = n0 + ch * 8;
    // (column counts are multiples of eight: a chunk lies wholly inside or wholly outside)
    if (m < a.M && n < a.N) *reinterpret_cast<half8v*>(a.out + (int64_t)m * a.ldo + n) = *reinterpret_cast<const half8v*>(lds + row * RS + ch * 8);
  }
}

// ---------------------------------------------------------------------------
// merge of the parts
// ---------------------------------------------------------------------------
// out[m, n..n+3] for one thread; the arithmetic mirrors the epilogues above
template <int EPI>
__device__ __forceinline__ half4v finalize_group(const GemmArgs& a, const float* partial, int ksplit, int m, int n, float rs) {
  const int ntot = EPI == EPI_SWIGLU ? 2 * a.N : a.N;
  const int64_t stride = (int64_t)a.M * ntot, off = (int64_t)m * ntot + n;
  float4v v = sum_splits(partial, ksplit, stride, off);
  float4v u = {0.f, 0.f, 0.f, 0.f};
  if (EPI == EPI_SWIGLU) u = sum_splits(partial, ksplit, stride, off + a.N);
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float c = v[e] * rs;
    if (EPI == EPI_GELU) c = gelu_erf(c);
    if (EPI == EPI_SWIGLU) c = silu(c) * (u[e] * rs);
    o[e] = c;
  }
  if (a.residual != nullptr) {
    const half4v rr = *reinterpret_cast<const half4v*>(a.residual + (int64_t)m * a.ldr + n);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += (float)rr[e];
  }
  const half4v h = {(half_t)o[0], (half_t)o[1], (half_t)o[2], (half_t)o[3]};
  *reinterpret_cast<half4v*>(a.out + (int64_t)m * a.ldo + n) = h;
  return h;
}

template <int EPI>
__global__ __launch_bounds__(256) void ring_finalize_kernel(GemmArgs a, const float* partial, int ksplit) {
  const int groups = a.N / 4;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.M * groups) return;
  const int m = idx / groups, n = (idx % groups) * 4;
  finalize_group<EPI>(a, partial, ksplit, m, n, a.rowscale != nullptr ? a.rowscale[m] : 1.0f);
}

// Plain epilogue, one workgroup per row: also leaves the RMSNorm statistic of the finished row in rowstat_out[m].
__global__ __launch_bounds__(1024) void ring_finalize_rowstat_kernel(GemmArgs a, const float* partial, int ksplit) {
  __shared__ float part[16];
  const int m = blockIdx.x, t = threadIdx.x;
  const float rs = a.rowscale != nullptr ? a.rowscale[m] : 1.0f;
  float ss = 0.f;
  for (int g = t; g < a.N / 4; g += 1024) {
    const half4v h = finalize_group<EPI_NONE>(a, partial, ksplit, m, g * 4, rs);
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf((float)h[e], (float)h[e], ss);
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) part[t >> 6] = ss;
  __syncthreads();
  if (t == 0) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += part[i];
    a.rowstat_out[m] = rsqrtf(s / (float)a.N);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <class T, bool WT>
static int launch_partial_t(const RingArgs& a, hipStream_t stream) {
  constexpr auto kern = ring_partial_kernel<T, WT>;
  if (set_max_lds<kern, T::LDS_BYTES>() != 0) return -1;
  const int nrb = (a.M + T::BM - 1) / T::BM, ntn = (a.ncols + T::BN - 1) / T::BN;
  hipLaunchKernelGGL(kern, dim3(nrb * ntn * a.ksplit), dim3(T::NT), T::LDS_BYTES, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_ring_partial(const RingArgs& a, int tile, bool kcontig, hipStream_t stream) {
  if (tile == kRingTileOneBlock && ring_fourth_stage(a.M, (a.ncols + 127) / 128 * a.ksplit, a.ldw[0] | a.ldw[1] | a.ldw[2], ring_kt_per_part(a.K, a.ksplit) * 64, kcontig, false))
    return kcontig ? launch_partial_t<RingTileFour, true>(a, stream) : launch_partial_t<RingTileFour, false>(a, stream);
  switch (tile) {
#define TRI_RING_CASE(id, bm, bn, wm, wn, nst, nt, np)                                                  \
  case id:                                                                                      \
    return kcontig ? launch_partial_t<RingTile<bm, bn, wm, wn, nst, nt, np>, true>(a, stream) \
                   : launch_partial_t<RingTile<bm, bn, wm, wn, nst, nt, np>, false>(a, stream);
    TRI_RING_TILES(TRI_RING_CASE)
#undef TRI_RING_CASE
  }
  return -1;
}

template <class T, int EPI, bool WT>
static int launch_epi_t(const GemmArgs& a, hipStream_t stream) {
  constexpr auto kern = ring_epi_kernel<T, EPI, WT>;
  if (set_max_lds<kern, T::LDS_BYTES>() != 0) return -1;
  constexpr int OUT_BN = EPI == EPI_SWIGLU ? T::BN / 2 : T::BN;
  const int nrb = (a.M + T::BM - 1) / T::BM, ntn = (a.N + OUT_BN - 1) / OUT_BN;
  hipLaunchKernelGGL(kern, dim3(nrb * ntn), dim3(T::NT), T::LDS_BYTES, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

constexpr int kRingTileNarrow = kRingTileFine + 1;  // (not planned by ring_plan: RingTileKContig)

template <int EPI>
static int launch_epi(const GemmArgs& a, int tile, hipStream_t stream) {
  constexpr bool GATED = EPI == EPI_SWIGLU;
  const int64_t ld = a.ldw | (GATED ? a.ldw2 : 0);
  if (tile == kRingTileNarrow) return launch_epi_t<RingTileKContig, EPI, true>(a, stream);
  if (tile == kRingTileOneBlock && ring_fourth_stage(a.M, ((GATED ? 2 : 1) * a.N + 127) / 128, ld, a.K, a.w_kcontig != 0, GATED))
    return a.w_kcontig ? launch_epi_t<RingTileFour, EPI, true>(a, stream) : launch_epi_t<RingTileFour, EPI, false>(a, stream);
  switch (tile) {
#define TRI_RING_CASE(id, bm, bn, wm, wn, nst, nt, np)                                                       \
  case id:                                                                                           \
    return a.w_kcontig ? launch_epi_t<RingTile<bm, bn, wm, wn, nst, nt, np>, EPI, true>(a, stream) \
                       : launch_epi_t<RingTile<bm, bn, wm, wn, nst, nt, np>, EPI, false>(a, stream);
    TRI_RING_TILES(TRI_RING_CASE)
#undef TRI_RING_CASE
  }
  return -1;
}

// Cost of a plan in us.  Three times add up in part (as a 3/2-norm up to 32 rows, as a 2-norm above):
//   memory    the weights once - less fast when the workgroups do not divide evenly over the CUs and some CUs have
//             one more to stream - and what is written;
//   compute   k tiles in a row on the busiest CU, by tile and by whether workgroups share a CU;
//   loads     every byte that passes from L2 to LDS;
// and per wave of workgroups 2 us of first loads and epilogue.  Parts cost a merge and their bytes, and more (parts) per wave of
// workgroups where the tile is large: its fp32 rows are stored by the waves that hold them alone.
// Up to 32 rows: weights at 8 TB/s, loads at 37, fitted to 4100 timings on the card, 16 to 1024 rows, when the 32 x 128 tile had four
// stages throughout; 4 % rms then, the plan it picks 1.3 % slower on average than the best plan of the family.  As that tile
// runs now, ring_fourth_stage, the costs of plans on it are 7 % high, deviation 7, over 1170 row-major ones, 6 and 7 over
// 980 K-contiguous ones, and 4 % low, deviation 9, over 190 with columns 8 or 16 KB apart.
// Above: the constants are those whose picks take least time, not those nearest to the times, and no rates of the chip - the
// weights' 21 TB/s is what the other two times leave of them to be seen.  Chosen over 37700 timings of 1604 products (33 to 1100
// rows, narrow outputs to 8192; K 1024 to 18176, 128 to 28672 columns, plain and gated, both layouts; among them the Q/K/V
// projections and both FFN products inside whole calls).  The pick is 1.3 % slower on average than the best plan, the large
// tiles' included, one in twenty by 7.5 % or more; constants nearest to the times, without the cost of parts by tile, had come to 2.7 %
// and 14.5; over 220 products kept out of the choice 1.8 % for 2.7.  (us with these / with those: 128 rows x [4544, 4544] 23.4 ->
// 21.2, 96 x [4096, 4096] 18.9 -> 17.5, 192 24.4 -> 21.9, 420 32.1 -> 30.7, 900 x [4096, 14336 x 2] 225 -> 211; the other way 230 x
// [14336, 4096] 46.6 -> 49.0, 45 x [4544, 4544] 15.4 -> 16.2.)  Much of what is left is where the weights lie in memory: it moves
// a product by a few percent from one allocation to the next, some with columns 8 KB apart by a fifth.
struct RingCost {
  int bm, bn, per_cu;   // per_cu: workgroups that fit a CU's LDS
  float alone, shared;  // us per k tile of a workgroup with a CU to itself / of each of several
  float parts;          // us per wave of workgroups with parts
  float few_alone, few_shared;  // alone and shared up to 32 rows (0: not for them)
};
#define TRI_RING_PER_CU(bm, bn, nst) ((160 * 1024) / (((bm) + (bn)) * 128 * (nst)))
static const RingCost kRingCost[kRingTiles] = {
    {32, 128, TRI_RING_PER_CU(32, 128, 3), 0.f, 0.f, 0.f, 0.264f, 0.222f},
    {64, 64, TRI_RING_PER_CU(64, 64, 5), 0.294f, 0.338f, -0.59f, 0.215f, 0.181f},
    {64, 128, TRI_RING_PER_CU(64, 128, 3), 0.473f, 0.530f, -0.41f, 0.354f, 0.272f},
    {96, 128, TRI_RING_PER_CU(96, 128, 5), 0.525f, 0.630f, 0.92f, 0.429f, 0.431f},
    {128, 128, TRI_RING_PER_CU(128, 128, 5), 0.606f, 0.709f, 1.72f, 0.f, 0.f},
    {128, 192, TRI_RING_PER_CU(128, 192, 3), 0.763f, 0.959f, 6.78f, 0.f, 0.f},
    {128, 256, TRI_RING_PER_CU(128, 256, 3), 0.969f, 1.085f, 4.82f, 0.f, 0.f},
    {160, 256, TRI_RING_PER_CU(160, 256, 3), 1.081f, 1.170f, 5.40f, 0.f, 0.f},
    {192, 128, TRI_RING_PER_CU(192, 128, 3), 0.707f, 0.873f, 4.81f, 0.f, 0.f},
    {192, 192, TRI_RING_PER_CU(192, 192, 3), 1.027f, 1.145f, 6.07f, 0.f, 0.f},
    {256, 128, TRI_RING_PER_CU(256, 128, 3), 0.879f, 1.080f, 4.79f, 0.f, 0.f}};
// A plan in one part on few workgroups: one streams no faster than about this many bytes of weights per us (16 rows x
// [2048, 5632 x 2] as gate/up, 88 workgroups: 22.0 us, 16.0 in two parts; x [1024, 4096 x 2], 64: 12.0 and 10.1 in four; the
// costs above, fitted where 200 and more workgroups share the memory's rate, say 14.9 and 7.8).  Up to 64 rows and 192
// workgroups; beyond either the costs hold as they are (one row x K-contiguous [4096, 14336 x 2], 224 workgroups, would be
// cut with the bound: the whole FFN 66.3 -> 72.4 us; 48 rows x [2048, 5632 x 2], 176, have to be cut: 22.2 -> 18.7).  What
// the plan picked is slower than the best of the family on average, with this bound and without: gated products of 16 to
// 100 rows, K of 512 to 8192, 2.1 % and 4.7; Q/K/V projections of 768- to 4544-wide models, up to 32 rows, 0.5 and 1.1;
// plain products of such sizes 0.4 either way.
// (Above 32 rows the bound holds up to 96 rows.)
constexpr float kRingStreamRateFew = 34e3f, kRingStreamRate = 37.4e3f;
constexpr int kRingStreamRows = 96, kRingStreamWorkgroups = 192;

static RingPlan ring_plan_search(int M, int K, int ncols, int unit, int min_bn, int64_t ws_bytes, float merge_us) {
  RingPlan best = {-1, 1, 1e30f};
  const int KT = K / 64;
  const float wbytes = 2.0f * (float)K * (float)ncols, obytes = 4.0f * (float)M * (float)ncols;
  const bool few = M <= kRingCost[kRingTileOneBlock].bm;
  for (int tile = 0; tile < kRingTiles; ++tile) {
    const RingCost& c = kRingCost[tile];
    if (c.bn % unit != 0 || c.bn < min_bn) continue;
    if (few ? c.few_alone == 0.f : tile == kRingTileOneBlock) continue;
    const float alone = few ? c.few_alone : c.alone, shared = few ? c.few_shared : c.shared;
    const int tiles = ((M + c.bm - 1) / c.bm) * ((ncols + c.bn - 1) / c.bn);
    int last_per = 0;
    for (int s = 1; s <= 16; ++s) {
      const int per = ring_kt_per_part(K, s);
      if (s > 1 && (per < 4 || s * tiles > 1024 || s * (int64_t)obytes > ws_bytes)) break;
      const int ks = (KT + per - 1) / per;
      if (per == last_per || ks != s) continue;  // (no more parts than before)
      last_per = per;
      const int wg = tiles * ks, share = (wg + 255) / 256;
      const float even = share == 1 ? 1.0f : sqrtf((float)wg / (256.0f * share));
      const float it = share == 1 ? alone : (alone > shared * share ? alone : shared * share);
      float comp = per * it;
      if (ks == 1 && wg <= kRingStreamWorkgroups && M <= kRingStreamRows) comp = fmaxf(comp, per * c.bn * 128.0f / (few ? kRingStreamRateFew : kRingStreamRate));
      const float waves = (float)((share + c.per_cu - 1) / c.per_cu), loaded = (float)wg * per * (c.bm + c.bn) * 128.0f;
      const float written = ks > 1 ? ks * obytes : 0.5f * obytes;
      float us;
      if (few) {
        const float mem = wbytes / (8e6f * even) + written / 3e6f, loads = loaded / 37e6f;
        const float sum = cbrtf(mem * sqrtf(mem) + comp * sqrtf(comp) + loads * sqrtf(loads));
        us = 1.1f + 1.9f * waves + sum * sum + (ks > 1 ? merge_us + ks * obytes / 6e6f : 0.f);
      } else {
        const float mem = wbytes / (21.3e6f * even) + written / 1.81e6f, loads = loaded / 50.4e6f;
        us = 1.37f * waves + sqrtf(mem * mem + comp * comp + loads * loads) +
             (ks > 1 ? merge_us + 1.79f + c.parts * waves + ks * obytes / 14.2e6f : 0.f);
      }
      if (us < best.us) { best.tile = tile; best.ksplit = ks; best.us = us; }
    }
  }
  return best;
}

// RingTileFine, for projections only (its cost chosen over 140 whole calls, with weights from memory and from the last-level
// cache, 192 to 256 workgroups).  Whole calls, the best of the family without it -> this: 131 to 160 rows x [2560, 6144] 26.2 - 27.7 ->
// 24.9 - 26.5 us, x [4096, 6144] 34.2 - 36.2 -> 35.0 - 36.9, but 29.0 -> 26.5 with the weights from the last-level cache; QKNorm of
// 200 to 320 rows x [2048, 3072] 23.8 - 26.5 -> 20.0 - 23.3, 64 to 320 x [1024, 1536] 15.0 - 18.8 -> 13.2 - 17.6.  Not taken: QKNorm
// of 35 to 64 x [4096, 12288] 34.5 -> 36.6, of 131 to 192 x [3072, 5120] 28.0 -> 30.1, of 99 to 128 x [4096, 6144] 30.6 -> 36.2; the
// plain product of 150 x [4096, 6144], whose merge is cheaper, 26.4 -> 28.7.
constexpr float kRingFineTile = 0.37f;  // us per k tile; the rest as in ring_plan_search
bool ring_fine_plan(int M, int K, int ncols, RingPlan& plan) {
  const int tiles = ((M + RingTileFine::BM - 1) / RingTileFine::BM) * ((ncols + RingTileFine::BN - 1) / RingTileFine::BN);
  if (plan.tile < 0 || M <= kRingCost[kRingTileOneBlock].bm || M > kRingMaxRows || tiles > 256) return false;
  const float mem = 2.0f * (float)K * (float)ncols / 21.3e6f + 2.0f * (float)M * (float)ncols / 1.81e6f;
  const float per = (float)ring_kt_per_part(K, 1), loads = (float)tiles * per * (RingTileFine::BM + RingTileFine::BN) * 128.0f / 50.4e6f;
  float comp = per * kRingFineTile;
  if (tiles <= kRingStreamWorkgroups && M <= kRingStreamRows) comp = fmaxf(comp, per * RingTileFine::BN * 128.0f / kRingStreamRate);
  const float us = 1.37f + sqrtf(mem * mem + comp * comp + loads * loads);
  if (us >= plan.us) return false;
  plan = RingPlan{kRingTileFine, 1, us};
  return true;
}

// The search is a pure function of its arguments and takes 5 to 10 us, longer than a launch; each thread keeps the
// answers it was last given.
RingPlan ring_plan(int M, int K, int ncols, int unit, int min_bn, int64_t ws_bytes, float merge_us) {
  if (M < 1 || K % 32 != 0 || K < 64 || ncols < 8) return RingPlan{-1, 1, 1e30f};
  if (M > kRingMaxRows && (M > kRingMaxRowsNarrow || ncols > kRingMaxColsNarrow || K < kRingMinKNarrow)) return RingPlan{-1, 1, 1e30f};
  struct Entry { int M, K, ncols, unit, min_bn; int64_t ws_bytes; float merge_us; RingPlan plan; };
  static thread_local Entry memo[256] = {};
  uint64_t h = (uint64_t)M;
  for (const uint64_t v : {(uint64_t)K, (uint64_t)ncols, (uint64_t)unit, (uint64_t)min_bn, (uint64_t)ws_bytes, (uint64_t)(merge_us * 64.0f)}) h = (h ^ v) * 0x9E3779B97F4A7C15ull;
  Entry& e = memo[h >> 56];
  if (e.M != M || e.K != K || e.ncols != ncols || e.unit != unit || e.min_bn != min_bn || e.ws_bytes != ws_bytes ||
      e.merge_us != merge_us)
    e = Entry{M, K, ncols, unit, min_bn, ws_bytes, merge_us, ring_plan_search(M, K, ncols, unit, min_bn, ws_bytes, merge_us)};
  return e.plan;
}

// out shares memory with x (views of one buffer whose columns do not meet share none)
static bool shares_memory(const GemmArgs& a) {
  const half_t *xend = a.x + (a.M - 1) * a.ldx + a.K, *oend = a.out + (a.M - 1) * a.ldo + a.N;
  if (oend <= a.x || xend <= a.out) return false;
  if (a.M == 1 || a.ldx != a.ldo) return true;  // (the stride of a single row may be anything, zero too)
  const int64_t d = ((a.out - a.x) % a.ldx + a.ldx) % a.ldx;
  return d < a.K || d + a.N > a.ldx;
}

// (Callers have that room up to 64 rows or more, see gemm_workspace_bytes.)
bool ring_gemm_in_place(const GemmArgs& a) {
  return a.ws != nullptr && a.ws_bytes >= (int64_t)a.M * (a.epi == EPI_SWIGLU ? 2 * a.N : a.N) * 4 && shares_memory(a);
}

// Estimated us of a product in one part on RingTileKContig at columns a power of two apart: the 4-norm of its loads on the
// busiest CU and of the weights at 6.3 TB/s (K = 4096 and 8192, 1 to 32 rows, 2048 to 57344 columns: 4.7 % rms).
static float ring_narrow_us(const GemmArgs& a) {
  const int cols = a.epi == EPI_SWIGLU ? 2 * a.N : a.N, share = ((cols + 63) / 64 + 255) / 256;
  const float mem = 2.0f * (float)a.K * (float)cols / 6.3e6f, cu = (float)a.K / 64.0f * (share == 1 ? 0.249f : 0.231f * share);
  const float m2 = mem * mem, c2 = cu * cu;
  return 3.35f + sqrtf(sqrtf(m2 * m2 + c2 * c2));
}

// Whether a product takes RingTileKContig, in one part, in place of its plan (us of the 128-column plan / of this tile, one row
// unless said otherwise).  Columns a power of two apart (8, 16, 32 KB): in place of a plan in one part on 128 columns
// ([4096, 14336 x 2] 45.7 / 42.1, 32 rows 46.7 / 44.0, [4096, 32768] 59.5 / 48.2, [8192, 28672 x 2] 156 / 148, 4 rows x
// [16384, 14336 x 2] 162 / 146) and of any plan that its estimate beats by 5 %, as the plans' costs know nothing of the slow distances
// (in parts [4096, 6912 x 2] 30.5 / 23.2, 32 rows x [4096, 12288 x 2] 50.1 / 40.6, 24 x [4096, 16384] 38.3 / 27.2; of 185 products 67
// take it, none slower; others would be faster, one row x [4096, 12288 x 2] 43.0 / 36.7, but by a margin of 0 some slower, 32 rows x
// [4096, 9728 x 2] 36.9 / 39.7; with few workgroups beyond two a CU the estimate is too low, [4096, 18176 x 2] 60.6 / 63.0).  But not
// where the workgroups just fill the chip (512, two a CU, or 1024) and gate and up columns 8 KB apart also lie a multiple of 8 KB
// from each other, and so meet on the same memory: [4096, 16384 x 2] 56.1 / 58.9, [4096, 32768 x 2] 99.6 / 113, while with up 68 KB
// behind the end of gate [4096, 16384 x 2] is 55.4 / 48.3, and 16 KB apart [8192, 16384 x 2] 116 / 92.6 all the same.  At other
// multiples of 8 KB in place of a plan in one part, gated ones beyond two workgroups a CU: [12288, 28672] 116 / 111, [12288, 17408 x 2] 174 / 163, but
// [12288, 14336 x 2] 109 / 111, [12288, 16384 x 2] 122 / 137, [20480, 14336 x 2] 167 / 175.  12 KB apart it is ahead too, by 3 to 14 %
// (4 rows x [6144, 14336 x 2] 68.2 / 61.3); 4, 20 and 28 KB are mixed ([2048, 14336 x 2] 28.1 / 26.9, [2048, 16384 x 2] 31.5 / 38.5).
static bool ring_takes_narrow(const GemmArgs& a, const RingPlan& plan) {
  const bool gated = a.epi == EPI_SWIGLU;
  const int64_t ld = a.ldw | (gated ? a.ldw2 : 0);
  if (!a.w_kcontig || a.M > RingTileKContig::BM || (ld & 4095) != 0) return false;
  const bool whole = plan.tile == kRingTileOneBlock && plan.ksplit == 1;
  const int wg = ((gated ? 2 : 1) * a.N + RingTileKContig::BN - 1) / RingTileKContig::BN;
  if (!ring_slow_columns(ld)) return whole && (!gated || wg > 512);
  const bool just_full = (wg - 1) % 512 >= 496 || (wg > 512 && wg <= 528);
  if (gated && ld == 4096 && just_full && ((a.w2 - a.w) & 4095) == 0) return false;
  return whole || ((wg <= 512 || wg > 576) && ring_narrow_us(a) < 0.95f * plan.us);
}

// over the whole of K, by the epilogue kernel
static int launch_whole(const GemmArgs& a, int tile, hipStream_t stream) {
  int rc = -1;
  switch (a.epi) {
    case EPI_NONE: rc = launch_epi<EPI_NONE>(a, tile, stream); break;
    case EPI_GELU: rc = launch_epi<EPI_GELU>(a, tile, stream); break;
    case EPI_SWIGLU: rc = launch_epi<EPI_SWIGLU>(a, tile, stream); break;
  }
  if (rc != 0 || a.rowstat_out == nullptr) return rc;
  return launch_rmsnorm(a.out, a.ldo, nullptr, nullptr, 0, a.rowstat_out, a.M, a.N, 0.f, stream);
}

int launch_ring_gemm(const GemmArgs& a, const RingPlan& plan, hipStream_t stream) {
  // the plans' costs are 8 % high for 64 x 64 tiles in one part, 4 to 6 % for most others, and 2 % low at slow distances (strip.hip)
  const float strip = strip_us(a), margin = plan.tile == 1 && plan.ksplit == 1 ? 0.88f : (ring_slow_columns(a.ldw) ? 1.0f : 0.92f);
  const bool narrow = ring_takes_narrow(a, plan);
  if (strip < margin * plan.us && !(narrow && ring_narrow_us(a) < strip) && !shares_memory(a)) return launch_strip(a, stream);
  if (narrow && !shares_memory(a)) return launch_whole(a, kRingTileNarrow, stream);
  const bool gated = a.epi == EPI_SWIGLU;
  // A product that overwrites its own input goes through the workspace also in one part: the tiles of the epilogue
  // kernel would store while others still read.
  if (plan.ksplit == 1 && !ring_gemm_in_place(a)) return launch_whole(a, plan.tile, stream);
  RingArgs r = {};
  r.x = a.x; r.ldx = a.ldx; r.M = a.M; r.K = a.K; r.ncols = gated ? 2 * a.N : a.N; r.ksplit = plan.ksplit; r.partial = a.ws;
  r.w[0] = a.w; r.ldw[0] = a.ldw; r.seg_begin[0] = 0;
  r.w[1] = r.w[2] = gated ? a.w2 : a.w;
  r.ldw[1] = r.ldw[2] = gated ? a.ldw2 : a.ldw;
  r.seg_begin[1] = gated ? a.N : r.ncols;
  r.seg_begin[2] = r.ncols;
  if (launch_ring_partial(r, plan.tile, a.w_kcontig != 0, stream) != 0) return -1;
  if (a.rowstat_out != nullptr && a.epi == EPI_NONE) {
    hipLaunchKernelGGL(ring_finalize_rowstat_kernel, dim3(a.M), dim3(1024), 0, stream, a, a.ws, plan.ksplit);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  const dim3 grid((a.M * (a.N / 4) + 255) / 256), block(256);
  switch (a.epi) {
    case EPI_NONE: hipLaunchKernelGGL(ring_finalize_kernel<EPI_NONE>, grid, block, 0, stream, a, a.ws, plan.ksplit); break;
    case EPI_GELU: hipLaunchKernelGGL(ring_finalize_kernel<EPI_GELU>, grid, block, 0, stream, a, a.ws, plan.ksplit); break;
    case EPI_SWIGLU: hipLaunchKernelGGL(ring_finalize_kernel<EPI_SWIGLU>, grid, block, 0, stream, a, a.ws, plan.ksplit); break;
    default: return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tri
