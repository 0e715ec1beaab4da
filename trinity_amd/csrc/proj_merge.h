// Merge of a split-K Q/K/V projection inside the attention kernels (AttnArgs::pj): the arithmetic and rounding points of
// the projection's own merge kernel (ring_qkv.hip), the results going to LDS and, where asked for, to global memory.
#if (defined(TRI_BF16) && !defined(TRI_PROJ_MERGE_H_BF16)) || (!defined(TRI_BF16) && !defined(TRI_PROJ_MERGE_H_F16))
#ifdef TRI_BF16
#define TRI_PROJ_MERGE_H_BF16
#else
#define TRI_PROJ_MERGE_H_F16
#endif
#include "common.h"
#include "launch.h"

namespace tri {

// One row of D columns to merge: token m, columns [col, col + D) of the partial results.
struct MergeRow {
  int m, col;
  bool normed;       // q or k: RMS-normalised when the call asks for QKNorm
  half_t *lds, *glb; // destinations (glb nullable)
};

// Rows [0, nrows), row i as map(i) says, each the sum of the parts in a fixed order, rounded to the element type.
// Called by all NT threads of the workgroup.  Every thread takes up to R groups of four columns and has the loads of all
// of them in flight together: the partial sums sit in other XCDs' caches, one round trip instead of one per group.
template <int D, int R, int NT, class Map>
__device__ __forceinline__ void merge_projection(const AttnArgs& a, int nrows, Map map) {
  constexpr int LPH = D / 4;  // lanes per row
  const int total = nrows * LPH;
  const int64_t split_stride = (int64_t)a.S * a.pj_ntot;
  for (int base = 0; base < total; base += NT * R) {
    bool live[R];
    int li[R];
    MergeRow row[R];
    const float* src[R];
    float4v acc[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
      const int idx = base + u * NT + (int)threadIdx.x;
      live[u] = idx < total;
      row[u] = map(live[u] ? idx / LPH : 0);
      li[u] = idx % LPH;
      src[u] = a.pj + (int64_t)row[u].m * a.pj_ntot + row[u].col + li[u] * 4;
      acc[u] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    // eight splits at a time (past the last split the last one is re-read and ignored)
    for (int i0 = 0; i0 < a.pj_ksplit; i0 += 8) {
      float4v p[R][8];
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (live[u]) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int i = i0 + j < a.pj_ksplit ? i0 + j : a.pj_ksplit - 1;
            p[u][j] = *reinterpret_cast<const float4v*>(src[u] + i * split_stride);
          }
        }
#pragma unroll
      for (int u = 0; u < R; ++u)
        if (live[u]) {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (i0 + j < a.pj_ksplit) {
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[u][e] += p[u][j][e];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
      half4v h = {(half_t)acc[u][0], (half_t)acc[u][1], (half_t)acc[u][2], (half_t)acc[u][3]};
      if (a.qknorm) {  // uniform; every lane takes part in the reduction
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf((float)h[e], (float)h[e], ss);
#pragma unroll
        for (int o = LPH / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        if (row[u].normed) {
          const float nrm = rsqrtf(ss / (float)D + a.eps);
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half_t)((float)h[e] * nrm);
        }
      }
      if (live[u]) {
        *reinterpret_cast<half4v*>(row[u].lds + li[u] * 4) = h;
        if (row[u].glb != nullptr) *reinterpret_cast<half4v*>(row[u].glb + li[u] * 4) = h;
      }
    }
  }
}

}  // namespace tri

#endif  // once per element type
