// Internal launcher prototypes (host side).  Every launcher enqueues on
// `stream`, allocates nothing, and returns 0 or -1 (the runtime refused).
#if (defined(TRI_BF16) && !defined(TRI_LAUNCH_H_BF16)) || (!defined(TRI_BF16) && !defined(TRI_LAUNCH_H_F16))
#ifdef TRI_BF16
#define TRI_LAUNCH_H_BF16
#else
#define TRI_LAUNCH_H_F16
#endif
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "common.h"

#ifndef TRI_LDS_ATTR_REGISTRY
#define TRI_LDS_ATTR_REGISTRY
// One node per kernel that needs the large-LDS attribute (see LdsAttr below); shared by the fp16 and bf16 copies of
// the kernels, defined in abi.hip.
struct TriLdsAttr;
__attribute__((visibility("hidden"))) void tri_lds_attr_register(TriLdsAttr* node);
__attribute__((visibility("hidden"))) int tri_lds_attr_apply(TriLdsAttr* node);  // current device; 0 or -1
struct TriLdsAttr {
  const void* kern;
  int bytes;
  std::atomic<uint64_t> done{0};
  TriLdsAttr* next = nullptr;
  TriLdsAttr(const void* k, int b) : kern(k), bytes(b) { tri_lds_attr_register(this); }
};
#endif

namespace tri {

// A kernel that wants more than 64 KB of dynamic LDS has to be told so once per device before its first launch.
// Every such kernel owns one TriLdsAttr (a static member of LdsAttr<kernel, bytes>, constructed when the library
// is loaded), which links itself into a list: tri_prepare() walks the list and sets the attribute of every kernel
// for the current device, and a launcher whose kernel has not been prepared on its device does so itself on the
// first call.  Bit d of `done` is set once device d has the attribute; threads racing on the first call repeat
// the same idempotent runtime call.
template <auto Kern, int Bytes>
struct LdsAttr {
  static TriLdsAttr once;
};
template <auto Kern, int Bytes>
TriLdsAttr LdsAttr<Kern, Bytes>::once(reinterpret_cast<const void*>(Kern), Bytes);

template <auto Kern, int Bytes>
inline int set_max_lds() {
  return tri_lds_attr_apply(&LdsAttr<Kern, Bytes>::once);
}

int launch_rmsnorm(const half_t* x, int64_t ldx, const half_t* w, half_t* y, int64_t ldy, float* rstd_out, int rows,
                   int n, float eps, hipStream_t stream);

int launch_add_scaled_rmsnorm(const half_t* a, int64_t lda, const half_t* b, int64_t ldb, const float* bscale,
                              half_t* y, int64_t ldy, int rows, int n, hipStream_t stream);

enum GemmEpi { EPI_NONE = 0, EPI_GELU = 1, EPI_SWIGLU = 2 };

// out[M, N] = act(rowscale[m] * (X[M,K] . W[K,N])) + residual[M,N]
// EPI_SWIGLU: out[M, N] = silu(X.W) * (X.W2), W and W2 both [K, N].
struct GemmArgs {
  const half_t* x;
  int64_t ldx;
  const half_t* w;
  int64_t ldw;
  const half_t* w2;
  int64_t ldw2;
  // weights stored K-contiguous (W^T [N][K]): ldw / ldw2 are then the strides between weight columns.  Needs
  // K % 32 == 0.
  int w_kcontig;
  const float* rowscale;   // nullable, [M]
  const half_t* residual;  // nullable
  int64_t ldr;
  half_t* out;
  int64_t ldo;
  int M, N, K;
  int epi;
  int n_big, big_cols;  // tile plan (filled in by launch_gemm): workgroups and columns covered by big tiles
  float* ws;            // nullable: fp32 workspace for plans that cut K into parts (gemm_workspace_bytes)
  int64_t ws_bytes;
  // nullable: also leave rsqrt(mean(out[m, :]^2)) - the RMSNorm statistic of the finished rows - in rowstat_out[m]
  // (plain epilogue only)
  float* rowstat_out;
};
int launch_gemm(const GemmArgs& a, hipStream_t stream);

// Few and middling rows (ring.hip): which tile of its family, and in how many parts of K, an [M, K] x [K, ncols]
// product runs, and what it should take (us, with the merge of its parts).  tile < 0: not for these kernels.
struct RingPlan {
  int tile, ksplit;
  float us;
};
constexpr int kRingMaxRows = 1100;  // the range that the cost model was fitted over, and some more
// ... and that of products with so few large tiles, each with so much to sum, that these leave most of the chip idle
// (ring_wins in gemm.hip)
constexpr int kRingMaxRowsNarrow = 8192, kRingMaxColsNarrow = 1 << 16, kRingMinKNarrow = 2048;
// ncols: weight columns (gate and up, or q, k and v, together).  Tiles must be a multiple of `unit` wide (whole heads; 1
// otherwise) and at least min_bn.  ws_bytes: fp32 workspace for partial results, ksplit * M * ncols * 4 bytes (1: none).
// merge_us: what the merge of parts takes beside its bytes.
constexpr float kRingMergeUs = 3.5f;
RingPlan ring_plan(int M, int K, int ncols, int unit, int min_bn, int64_t ws_bytes, float merge_us = kRingMergeUs);
// a Q/K/V projection's ring plan gives way to 32-row tiles in one round where they are cheaper
bool ring_fine_plan(int M, int K, int ncols, RingPlan& plan);
int launch_ring_gemm(const GemmArgs& a, const RingPlan& plan, hipStream_t stream);
// whether launch_gemm runs such a product by its ring plan (else by large tiles)
bool gemm_plan(int M, int K, int N, int epi, bool kcontig, int64_t ws_bytes, RingPlan& plan);
// ... and launch_qkv_proj a projection (head: QKNorm, tiles of whole heads of that width; 0: any)
bool qkv_ring_plan(int S, int K, int ncols, int head, bool kcontig, int64_t ws_bytes, bool deferred, RingPlan& plan);
// few rows over K-contiguous weights in one part (strip.hip): what it should take (us; 1e30: not for it), and the launch
float strip_us(const GemmArgs& a);
int launch_strip(const GemmArgs& a, hipStream_t stream);
bool ring_gemm_in_place(const GemmArgs& a);  // out overlaps x, and the workspace holds the one part it takes to allow that
// workspace that lets launch_gemm take its best plan for [M, K] x [K, ncols] (0: no plan in parts)
int64_t gemm_workspace_bytes(int M, int K, int ncols);
// the same for the Q/K/V projection; unit as in ring_plan; deferred: the attention kernel merges the parts
int64_t qkv_workspace_bytes(int S, int K, int ncols, int unit, bool deferred);

// [Q | K | V] = X . [Wq | Wk | Wv], optional per-head RMSNorm of Q and K,
// scattered to q [S, Hq*D] and the head-major k/v buffers.
struct QkvProjArgs {
  const half_t* x;
  int64_t ldx;
  const half_t *wq, *wk, *wv;
  int64_t ldwq, ldwk, ldwv;
  half_t* q;  // [S, Hq*D]
  int64_t ldq;
  half_t *k, *v;            // element (h, row, d) at h*stride_h + row*stride_r + d
  int64_t k_sh, k_sr, v_sh, v_sr;
  int S, K, Hq, Hkv, D, P;
  int qknorm;
  float eps;
  float* ws;  // nullable: fp32 workspace for plans that cut K into parts (qkv_workspace_bytes)
  int64_t ws_bytes;
  int n_big, big_cols;  // tile plan (filled in by launch_qkv_proj)
  int w_kcontig;        // the three weight matrices are K-contiguous (ldwq / ldwk / ldwv: strides between columns)
  // nullable: fp8 caches that the merge of partial results appends the new k / v rows to (rows [append_row,
  // append_row + S)) in place of k / v, as launch_kv_quant_append would from there
  uint8_t *k8, *v8;
  int64_t k8_sh, k8_sr, v8_sh, v8_sr;
  int append_row;
  float k_scale, v_scale;
};
// deferred_ksplit (nullable): when given and the projection runs in parts, its merge kernel is left out - q, k and v
// stay fp32 partial results ws [ksplit][S][(Hq + 2 Hkv) * D] for the attention kernel to merge - and the number of
// parts is stored there; 0 is stored when the projection finished the job itself.
// appended (nullable): whether the new rows went to k8 / v8 instead of k / v.
int launch_ring_qkv(const QkvProjArgs& a, const RingPlan& plan, hipStream_t stream, int* deferred_ksplit, bool* appended);
int launch_qkv_proj(const QkvProjArgs& a, hipStream_t stream, int* deferred_ksplit = nullptr, bool* appended = nullptr);

struct AttnArgs {
  const half_t* q;  // [S, Hq*D]
  int64_t ldq;
  const half_t *k, *v;  // head-major, rows [0, P+S)
  int64_t k_sh, k_sr, v_sh, v_sr;
  half_t* out;  // [S, Hq*D]
  int64_t ldo;
  float* lse;       // nullable [Hq, S], natural log
  float* lse_pert;  // nullable [Hq, S]: logsumexp of the perturbed logits (KeyFormer)
  const half_t* noise;  // nullable [Hq, S, P+S]
  int S, P, Hq, Hkv, D;
  float scale, tau;
  int causal;
  uint64_t seed;
  float* ws;  // nullable: workspace of the few-query path (few_attn_workspace_bytes)
  int64_t ws_bytes;
  float out_scale;  // multiplies the normalised output (v_scale of an fp8 cache; 1 otherwise)
  // fp8 (e4m3) caches read directly - by the few-query and key-split kernels, without log-sum-exps; k / v are then unused.  Strides in elements = bytes.
  const uint8_t *k8, *v8;
  int64_t k8_sh, k8_sr, v8_sh, v8_sr;
  // Few-query paths fused with the merge of a split-K projection (pj != nullptr): q and
  // the S new rows of k / v are not read from memory but summed from the projection's partial results
  // pj [pj_ksplit][S][pj_ntot] (columns [q heads | k heads | v heads]), rounded, RMS-normalised per head when
  // qknorm (q and k), and stored to q_w and to rows [P, P+S) of k_w / v_w (the buffers k / v point to) on the way.
  int split_runs;  // set by launch_attention for its long-prefix variant: runs the key tiles are dealt out to
  const float* pj;
  int pj_ksplit, pj_ntot, qknorm;
  float eps;
  half_t *q_w, *k_w, *v_w;
};
// merge_parts (nullable): when given, the few-query kernel may leave its partial results in a.ws for the score kernel to
// merge (ScoreArgs::part); their number, or 0 when out and the log-sum-exp are finished, is stored there.
int launch_attention(const AttnArgs& a, hipStream_t stream, int* merge_parts = nullptr);

// With at most kFewMaxQueries queries attention is bound by reading the K/V cache once; it then runs split
// over the key axis (partial results in the workspace) followed by a merge kernel.
constexpr int kFewMaxQueries = 32;
constexpr int kFewKeysPerWg = 256;  // keys per workgroup
int64_t few_attn_workspace_bytes(int S, int Hq, int D, int Ltot);
int launch_attention_few(const AttnArgs& a, hipStream_t stream, int* merge_parts = nullptr);
int launch_attention_few_combine(const AttnArgs& a, int nsplit, hipStream_t stream);  // the merge kernel alone
// workspace of launch_attention's long-prefix variant for a call (0 when it does not take it): for all the runs it would
// cut the key axis into, or (least) for the fewest it works with - given less than the former it takes fewer runs
int64_t split_attn_workspace_bytes(int S, int Hq, int Hkv, int D, int Ltot, bool least);
// the kernel of calls that neither the key-split nor the few-query kernels take: four waves on 32 queries each; eight waves on two
// tiles of keys at a time, within a round of workgroups (causal: a late and an early half block of queries) or beyond it
// (whole blocks); eight query groups; four waves on 64 queries each
enum PrefillForm { kPrefillFourWaves, kPrefillTwoWays, kPrefillTwoWaysWhole, kPrefillEightGroups, kPrefillWide };
int prefill_form(int S, int P, int Hq, int D, bool causal, int kf);  // (kf: 0 plain and RoCo, 1 KeyFormer, 2 with seeded noise)
bool split_attn_takes(int S, int Hq, int Hkv, int D, int Ltot, int64_t ws_bytes);  // the key-split kernel runs, with that workspace
// its form for a call with room for all runs (-1: not taken): four waves on 32 stacked rows each; two query groups whose waves take the
// two halves of a tile; eight waves on two tiles at a time
enum SplitForm { kSplitFourWaves, kSplitHalves, kSplitPairs };
int split_attn_form(int S, int Hq, int Hkv, int Ltot, bool fp8);
// From this many keys on, plain attention for few new tokens leaves the one-tile-per-wave kernel for one that
// loops over its keys with the query heads of a KV head stacked along the query axis (launch_attention decides).
// 16 tokens: at 1040 keys the two are level, at 2064 keys the looping kernel is 2-5 us ahead, at 32784 keys
// 2.3x (8 KV heads, head dimension 128) to 3x (1 KV head, 64) on the whole block.
constexpr int kSplitMinKeys = 2048;
// Most tokens, and rows (heads of a group x tokens), whose projection's partial sums that kernel adds up itself; most
// tokens of 128-wide heads for the one-tile-per-wave kernel, and where it has more than kFewFusedWorkgroups (two a CU)
// workgroups (attn_may_merge_proj has the measurements).
constexpr int kSplitFusedRows = 8, kSplitFusedTokens = 4, kFewFusedTokens = 8, kFewFusedTokensMany = 4, kFewFusedWorkgroups = 512;

// fp8 (OCP e4m3) KV caches, value = scale * fp8: append of the new rows, and 16-bit copies (without the scale)
// for the kernels that read 16-bit K / V tiles.
struct KvQuantArgs {
  const half_t *k, *v;  // new rows [Hkv][S][D] as written by the projection
  int64_t k_sh, k_sr, v_sh, v_sr;
  uint8_t *kc, *vc;  // caches; rows [P, P+S) are written
  int64_t kc_sh, kc_sr, vc_sh, vc_sr;
  int S, P, Hkv, D;
  float k_scale, v_scale;
};
int launch_kv_quant_append(const KvQuantArgs& a, hipStream_t stream);
struct KvDequantArgs {
  const uint8_t *kc, *vc;
  int64_t kc_sh, kc_sr, vc_sh, vc_sr;
  half_t *k, *v;  // [Hkv][rows][D] contiguous
  int rows, Hkv, D;
};
int launch_kv_dequant(const KvDequantArgs& a, hipStream_t stream);

// Per-key accumulators over queries.  mode 0: RoCo (o1 = sum p, o2 = sum p^2,
// or mean / variance when mean_var); mode 1: KeyFormer (o1 = sum p_perturbed).
struct ScoreArgs {
  const half_t* q;
  int64_t ldq;
  const half_t* k;
  int64_t k_sh, k_sr;
  const float* lse;  // [Hq, S]: plain (mode 0) or perturbed (mode 1)
  const half_t* noise;
  float *o1, *o2;  // [Hq, P+S]
  int64_t ldo1, ldo2;
  int S, P, Hq, Hkv, D;
  float scale, tau;
  int causal, mode, mean_var;
  uint64_t seed;
  // few queries: attention left part_n (at most eight) partial results in `part`, in the few-query kernel's layout; lse
  // is then not read, and the scores' kernel also writes out = the merged rows * out_scale
  const float* part;
  int part_n;
  half_t* out;
  int64_t ldo;
  float out_scale;
};
int launch_scores(const ScoreArgs& a, hipStream_t stream);
// what a workgroup of launch_scores takes (more than kFewMaxQueries tokens): a block of 128 keys, two of them, a block of 64 keys, two
enum ScoreForm { kScoreBlock, kScoreBlockPair, kScoreHalfBlock, kScoreHalfBlockPair };
int score_form(int S, int P, int Hq, bool causal);
int launch_scores_few(const ScoreArgs& a, hipStream_t stream);  // S <= kFewMaxQueries; 1 = not applicable

}  // namespace tri

#endif  // once per element type
