// Products of 1 to 16 rows over K-contiguous weights in one part: a workgroup owns 16 columns over the whole of K, its four
// waves take the 128-deep pieces of K in turn, each through an LDS ring of its own, and add up through LDS at the end.
//
// What bounds it: streaming the weights once.  Columns of 16 leave no CU idle without cutting K into parts, so that the
// merge kernel (4.5 us in a chain of launches) and the partial sums' traffic are gone; a wave that keeps to its own piece
// needs no barrier.  K-contiguous columns make that possible: a piece is 256 bytes of a column however few columns there
// are, where row-major weights would be read 32 bytes of a row at a time (a reader of [14336, 4096]: 5.7 TB/s against 2.7).
#include "gemm_core.h"
#include "launch.h"

#include <math.h>

namespace tri {

// D[16 x 16] += A[16 x 32] * B[32 x 16].  Lane l supplies row (l % 16) of A and column (l % 16) of B, eight consecutive k
// each, k-group (l / 16), and receives column (l % 16), rows 4 * (l / 16) + r of D.
__device__ __forceinline__ float4v mfma16(half8v a, half8v b, float4v c) {
#ifdef TRI_BF16
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#else
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
#endif
}

constexpr int kStripCols = 16, kStripPiece = 128, kStripWaves = 4;
// Three stages: 48 KB, so that three workgroups fit a CU (4 rows x [4544, 18176], 1136 workgroups, 27.3 us, with four 31.9;
// with one workgroup a CU level: one row x [14336, 4096] within 0.3).
constexpr int kStripStages = 3;

// LDS piece [16 columns][128]: 16-byte chunk j (of 16) of column c at slot j ^ c - the lanes of a fragment read (16 columns,
// one chunk) then fall on different banks.  A load instruction fetches 256 bytes of four columns.
template <int EPI, int NST>
__global__ __launch_bounds__(kStripWaves * 64) void strip_kernel(GemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) half_t lds[];
  constexpr int PIECE = kStripCols * kStripPiece;  // halfs
  constexpr int L = 8;                             // load instructions of a piece: four of weights, four of activations
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  // neighbouring columns on one XCD
  const int total = gridDim.x, per = total >> 3, rem = total & 7, xcd = (int)blockIdx.x & 7;
  const int n0 = (xcd * per + (xcd < rem ? xcd : rem) + ((int)blockIdx.x >> 3)) * kStripCols;

  const int np = (a.K + kStripPiece - 1) / kStripPiece;
  const int mine = (np - wave + kStripWaves - 1) / kStripWaves;  // pieces wave, wave + 4, ...
  // first k of a piece; the last one is moved back where K ends within it, past the end it is repeated (the waits count
  // on every load)
  auto kof = [&](int i) { return min((wave + min(i, mine - 1) * kStripWaves) * kStripPiece, a.K - kStripPiece); };
  half_t* ring = lds + wave * NST * PIECE;
  const half_t* wsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = i * 4 + g;
    wsrc[i] = a.w + (int64_t)min(n0 + col, a.N - 1) * a.ldw + (c ^ col) * 8;
  }
  const half_t* xsrc = a.x + (int64_t)min(c, a.M - 1) * a.ldx + g * 8;
  half8v xf[NST][4];
  auto load = [&](int i, int st) __attribute__((always_inline)) {
    const int k = kof(i);
#pragma unroll
    for (int j = 0; j < 4; ++j) load_to_lds16<true>(wsrc[j] + k, ring + st * PIECE + j * 512);
#pragma unroll
    for (int j = 0; j < 4; ++j) xf[st][j] = *reinterpret_cast<const half8v*>(xsrc + k + j * 32);
  };
  auto frag = [&](int st, int j) __attribute__((always_inline)) { return lds_read8(ring + st * PIECE + c * kStripPiece + (((j * 4 + g) ^ c) << 3)); };
  float4v acc = {0.f, 0.f, 0.f, 0.f};
  if (mine > 0) {
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) load(s, s);
    int i0 = 0;
    // (no branches inside: the compiler's own waits for xf then count the loads in flight)
    for (; i0 + NST < mine; i0 += NST) {
#pragma unroll
      for (int st = 0; st < NST; ++st) {
        load(i0 + st + NST - 1, (st + NST - 1) % NST);
        TRI_WAIT_VMCNT((NST - 1) * L);
        __builtin_amdgcn_sched_barrier(0);
        half8v wf[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) wf[j] = frag(st, j);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = mfma16(wf[j], xf[st][j], acc);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage is loaded again next
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // the last one to NST pieces; the very last may begin with steps that the piece before it has done already
    load(i0 + NST - 1, NST - 1);
    TRI_WAIT_VMCNT(0);
#pragma unroll
    for (int st = 0; st < NST; ++st) {
      const int end = (wave + (i0 + st) * kStripWaves + 1) * kStripPiece;
      const int skip = i0 + st >= mine ? 4 : (end > a.K ? (end - a.K) / 32 : 0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j >= skip) acc = mfma16(frag(st, j), xf[st][j], acc);
    }
  }
  TRI_WAIT_VMCNT(0);
  __syncthreads();
  float4v* part = reinterpret_cast<float4v*>(lds);
  if (wave > 0) part[(wave - 1) * 64 + lane] = acc;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < kStripWaves - 1; ++w) acc += part[w * 64 + lane];
  // lane: token c, columns n0 + 4 g .. + 3
  const int n = n0 + g * 4;
  if (c >= a.M || n >= a.N) return;
  const float rs = a.rowscale != nullptr ? a.rowscale[c] : 1.0f;
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[e] = acc[e] * rs;
    if (EPI == EPI_GELU) o[e] = gelu_erf(o[e]);
  }
  if (a.residual != nullptr) {
    const half4v rr = *reinterpret_cast<const half4v*>(a.residual + (int64_t)c * a.ldr + n);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += (float)rr[e];
  }
  const half4v h = {(half_t)o[0], (half_t)o[1], (half_t)o[2], (half_t)o[3]};
  *reinterpret_cast<half4v*>(a.out + (int64_t)c * a.ldo + n) = h;
}

// Estimated us of a product (1e30: not for this kernel), to compare with a ring plan's: of the weights at 12 TB/s and of what the
// busiest CU has to load, activations included, at 58 GB/s the 3/2-norm (up to three workgroups a CU everything is placed at once,
// more even out), and 0.6 us to start each workgroup of a CU.  Over 1690 products (1 to 16 rows, K 512 to 18176, 512 to 32768
// columns) 1 % low on average with a deviation of 7 %; the ring plans' costs are 8 % high there for 64 x 64 tiles in one part, 4 to 6 %
// for most others, and 2 % low, with a deviation of 10, at columns a power of two of 8 KB apart.  Taken below 0.88, 0.92 and 1.0 of
// those (launch_ring_gemm): 940 of the 1690, 56 of them slower than the plan by more than 2 %, at worst 13.  us, and those of the ring
// kernels with their merge: one row x [4096, 4096] 7.6, 13.7, [4096, 14336] 21.0, 29.6, [14336, 4096] 21.9, 24.0, 12 rows 24.7, 23.9, 4 x
// [4544, 18176] 27.6, 32.5, 9 x [16384, 8192] 46.7, 78.8; not taken: 14 x [14336, 4096] 25.6, 23.9, 12 x [2048, 9728] 13.4, 11.8, 10 x
// [512, 4672] 5.5, 4.8, 6 x [14336, 9728] 53.6, 46.3.
float strip_us(const GemmArgs& a) {
  if (!a.w_kcontig || a.epi == EPI_SWIGLU || a.rowstat_out != nullptr || a.M > 16 || a.K < 512 || a.K % 32 != 0 || a.N % 8 != 0) return 1e30f;
  const int wg = (a.N + kStripCols - 1) / kStripCols;
  const float per = (float)wg / 256.0f, share = wg <= 768 ? (float)((wg + 255) / 256) : per + 0.5f;
  const float hbm = 2.0f * (float)a.K * (float)a.N / 12e6f, cu = share * ((float)kStripCols + 1.25f * (float)a.M) * 2.0f * (float)a.K / 58e3f;
  const float sum = cbrtf(hbm * sqrtf(hbm) + cu * sqrtf(cu));
  return 2.8f + 0.6f * per + sum * sum;
}

template <int EPI>
static int launch_strip_t(const GemmArgs& a, hipStream_t stream) {
  constexpr int LDS = kStripWaves * kStripStages * kStripCols * kStripPiece * 2;
  constexpr auto kern = strip_kernel<EPI, kStripStages>;
  if (set_max_lds<kern, LDS>() != 0) return -1;
  hipLaunchKernelGGL(kern, dim3((a.N + kStripCols - 1) / kStripCols), dim3(kStripWaves * 64), LDS, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_strip(const GemmArgs& a, hipStream_t stream) {
  return a.epi == EPI_GELU ? launch_strip_t<EPI_GELU>(a, stream) : launch_strip_t<EPI_NONE>(a, stream);
}

}  // namespace tri
