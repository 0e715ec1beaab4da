// Fused Q/K/V projection for few and middling rows, on the tiles and main loop of ring.h: logical columns
// [q heads | k heads | v heads], per-head RMSNorm of q and k (QKNorm), scatter to q [S, Hq * D] and the head-major
// K / V rows - in the epilogue of a kernel over the whole of K, or in the merge of fp32 partial products.
#include "ring.h"

namespace tri {

template <class T, int D, bool WT>
__global__ __launch_bounds__(T::NT) void ring_qkv_kernel(QkvProjArgs a) {
  extern __shared__ __attribute__((aligned(16))) half_t lds[];
  const int nq = a.Hq * D, nkv = a.Hkv * D, ntot = nq + 2 * nkv;
  const int nrb = (a.S + T::BM - 1) / T::BM, ntn = (ntot + T::BN - 1) / T::BN;
  int rb, tn, split;
  ring_coords(blockIdx.x, nrb, ntn, 1, nrb > 1 || T::BM >= 96, rb, tn, split);
  const int m0 = rb * T::BM, n0 = tn * T::BN;
  auto wmap = [&](int c, int64_t& ldw) -> const half_t* {
    int col = n0 + (WT ? c : c * 8);
    col = col < ntot ? col : 0;
    const half_t* w = a.wq;
    ldw = a.ldwq;
    if (col >= nq + nkv) { w = a.wv; ldw = a.ldwv; col -= nq + nkv; }
    else if (col >= nq) { w = a.wk; ldw = a.ldwk; col -= nq; }
    return WT ? w + (int64_t)col * ldw : w + col;
  };
  float16v acc[T::NI][T::MI];
  gemm_mainloop_ring<T, WT, false>(a.x, a.ldx, m0, a.S, a.K, wmap, lds, acc);

  // the tile turns around in LDS (rounded to 16 bits there) and leaves as 16-byte pieces of rows of one head
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % T::WM, wn = wave / T::WM;
  const int l32 = lane & 31, g = lane >> 5;
  constexpr int RS = T::BN + 8;  // halfs per staged row
  static_assert(T::BM * RS * 2 <= T::LDS_BYTES, "the staged output tile fits the ring");
  __syncthreads();
  if (T::NP == 0 || wave < T::NW) {  // (a wave that only loads holds no part of the tile)
#pragma unroll
    for (int mi = 0; mi < T::MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < T::NI; ++ni)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
          half4v h;
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[ni][mi][rq * 4 + e];
          *reinterpret_cast<half4v*>(lds + (wm * T::TM + mi * 32 + l32) * RS + wn * T::TN + ni * 32 + rq * 8 + g * 4) = h;
        }
  }
  __syncthreads();
  constexpr int CH = T::BN / 8;  // 16-byte chunks per staged row
  static_assert(T::BM * CH % T::NT == 0, "every thread takes part in every pass (head sums run across lanes)");
  for (int idx = threadIdx.x; idx < T::BM * CH; idx += T::NT) {
    const int row = idx / CH, ch = idx % CH;
    const int m = m0 + row, col = n0 + ch * 8;  // a chunk never straddles a head
    half8v h = *reinterpret_cast<const half8v*>(lds + row * RS + ch * 8);
    if (a.qknorm && T::BN % D == 0) {  // D / 8 neighbouring lanes hold a head (the host pairs QKNorm with whole heads)
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf((float)h[e], (float)h[e], ss);
#pragma unroll
      for (int o = D / 16; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      if (col < nq + nkv) {
        const float nrm = rsqrtf(ss / (float)D + a.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = (half_t)((float)h[e] * nrm);
      }
    }
    if (m >= a.S || col >= ntot) continue;
    half_t* dst;
    if (col < nq) {
      dst = a.q + (int64_t)m * a.ldq + col;
    } else if (col < nq + nkv) {
      const int c = col - nq;
      dst = a.k + (int64_t)(c / D) * a.k_sh + (int64_t)(a.P + m) * a.k_sr + c % D;
    } else {
      const int c = col - nq - nkv;
      dst = a.v + (int64_t)(c / D) * a.v_sh + (int64_t)(a.P + m) * a.v_sr + c % D;
    }
    *reinterpret_cast<half8v*>(dst) = h;
  }
}

// Merge of partial products: one group of D/4 consecutive lanes per (row, head): sum the parts, round, optionally
// RMS-normalise the head (q and k only), scatter to q / the cache rows (rows of an fp8 cache: converted on the way).
template <int D>
__global__ __launch_bounds__(256) void ring_finalize_qkv_kernel(QkvProjArgs a, const float* partial, int ksplit) {
  constexpr int LPH = D / 4;  // lanes per head
  const int nq = a.Hq * D, nkv = a.Hkv * D, ntot = nq + 2 * nkv;
  const int heads = a.Hq + 2 * a.Hkv;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  const int grp = idx / LPH, li = idx % LPH;
  const bool live = grp < a.S * heads;
  const int m = live ? grp / heads : 0, hc = live ? grp % heads : 0;
  const int col0 = hc * D;
  float4v v = sum_splits(partial, live ? ksplit : 0, (int64_t)a.S * ntot, (int64_t)m * ntot + col0 + li * 4);
  half_t* dst;
  int seg;
  if (col0 < nq) { seg = 0; dst = a.q + (int64_t)m * a.ldq + col0; }
  else if (col0 < nq + nkv) { seg = 1; dst = a.k + (int64_t)((col0 - nq) / D) * a.k_sh + (int64_t)(a.P + m) * a.k_sr; }
  else { seg = 2; dst = a.v + (int64_t)((col0 - nq - nkv) / D) * a.v_sh + (int64_t)(a.P + m) * a.v_sr; }
  half4v h = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
  if (a.qknorm) {  // uniform; every lane takes part in the reduction
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf((float)h[e], (float)h[e], ss);
#pragma unroll
    for (int o = LPH / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    if (seg < 2) {
      const float nrm = rsqrtf(ss / (float)D + a.eps);
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = (half_t)((float)h[e] * nrm);
    }
  }
  if (!live) return;
  if (a.k8 != nullptr && seg != 0) {
    uint8_t* d8 = seg == 1 ? a.k8 + (int64_t)((col0 - nq) / D) * a.k8_sh + (int64_t)(a.append_row + m) * a.k8_sr
                           : a.v8 + (int64_t)((col0 - nq - nkv) / D) * a.v8_sh + (int64_t)(a.append_row + m) * a.v8_sr;
    *reinterpret_cast<uint32_t*>(d8 + li * 4) = half4_to_fp8x4(h, seg == 1 ? a.k_scale : a.v_scale);
  } else {
    *reinterpret_cast<half4v*>(dst + li * 4) = h;
  }
}

template <class T, int D, bool WT>
static int launch_qkv_t(const QkvProjArgs& a, hipStream_t stream) {
  constexpr auto kern = ring_qkv_kernel<T, D, WT>;
  if (set_max_lds<kern, T::LDS_BYTES>() != 0) return -1;
  const int nrb = (a.S + T::BM - 1) / T::BM, ntn = ((a.Hq + 2 * a.Hkv) * D + T::BN - 1) / T::BN;
  hipLaunchKernelGGL(kern, dim3(nrb * ntn), dim3(T::NT), T::LDS_BYTES, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int D>
static int launch_qkv_tile(const QkvProjArgs& a, int tile, hipStream_t stream) {
  if (tile == kRingTileOneBlock && ring_fourth_stage(a.S, ((a.Hq + 2 * a.Hkv) * D + 127) / 128, a.ldwq | a.ldwk | a.ldwv, a.K, a.w_kcontig != 0, false))
    return a.w_kcontig ? launch_qkv_t<RingTileFour, D, true>(a, stream) : launch_qkv_t<RingTileFour, D, false>(a, stream);
  if (tile == kRingTileFine) return a.w_kcontig ? launch_qkv_t<RingTileFine, D, true>(a, stream) : launch_qkv_t<RingTileFine, D, false>(a, stream);
  switch (tile) {
#define TRI_RING_CASE(id, bm, bn, wm, wn, nst, nt, np)                                                    \
  case id:                                                                                        \
    return a.w_kcontig ? launch_qkv_t<RingTile<bm, bn, wm, wn, nst, nt, np>, D, true>(a, stream) \
                       : launch_qkv_t<RingTile<bm, bn, wm, wn, nst, nt, np>, D, false>(a, stream);
    TRI_RING_TILES(TRI_RING_CASE)
#undef TRI_RING_CASE
  }
  return -1;
}

int launch_ring_qkv(const QkvProjArgs& a, const RingPlan& plan, hipStream_t stream, int* deferred_ksplit, bool* appended) {
  if (plan.ksplit == 1)
    return a.D == 128 ? launch_qkv_tile<128>(a, plan.tile, stream) : launch_qkv_tile<64>(a, plan.tile, stream);
  const int nq = a.Hq * a.D, nkv = a.Hkv * a.D;
  RingArgs r = {};
  r.x = a.x; r.ldx = a.ldx; r.M = a.S; r.K = a.K; r.ncols = nq + 2 * nkv; r.ksplit = plan.ksplit; r.partial = a.ws;
  r.w[0] = a.wq; r.ldw[0] = a.ldwq; r.seg_begin[0] = 0;
  r.w[1] = a.wk; r.ldw[1] = a.ldwk; r.seg_begin[1] = nq;
  r.w[2] = a.wv; r.ldw[2] = a.ldwv; r.seg_begin[2] = nq + nkv;
  if (launch_ring_partial(r, plan.tile, a.w_kcontig != 0, stream) != 0) return -1;
  if (deferred_ksplit != nullptr) {
    *deferred_ksplit = plan.ksplit;
    return 0;
  }
  if (appended != nullptr) *appended = a.k8 != nullptr;
  const int threads = a.S * (a.Hq + 2 * a.Hkv) * (a.D / 4);
  const dim3 grid((threads + 255) / 256), block(256);
  if (a.D == 128) hipLaunchKernelGGL(ring_finalize_qkv_kernel<128>, grid, block, 0, stream, a, a.ws, plan.ksplit);
  else hipLaunchKernelGGL(ring_finalize_qkv_kernel<64>, grid, block, 0, stream, a, a.ws, plan.ksplit);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace tri
