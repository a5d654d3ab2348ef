// Host-side interface between the C ABI (abi.hip) and the kernel files.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace swvr {

// Kernel kinds, for the launch timing record.
enum KernelKind {
  kKindFwdTile = 0,
  kKindFwdCombine,
  kKindBwdDelta,
  kKindBwdScores,
  kKindBwdGemm,
  kKindBwdReduce,
  kKindFill,
  kKindPack,
  kKindBwdExpand,
  kKindLoss,
  kKindQuant,
  kKindF64,
  kKindProbe,
  kNumKinds
};

// Timing hooks (abi.hip): bracket one launch when timing is enabled.
void timing_begin(int kind, hipStream_t stream);
void timing_end(int kind, hipStream_t stream);

// ---------------------------------------------------------------- forward
struct FwdParams {
  const void* h;
  int64_t ldh;
  const void* W;
  int64_t ldw;
  const void* E;
  int64_t lde;
  const float* bias;  // fp32 [V] or null
  float scale;
  int N, K, V, D;
  int n_tb, n_split, n_vt;
  float* part_m;       // [n_part][N]
  float* part_l;       // [n_part][N]
  float* part_acc;     // [n_part][DP][N]
  const void* Ep;      // packed E^T tiles [n_vt][DP][BV], compute dtype
  const float* biasp;  // packed bias [V_pad], -inf past V
  const void* hp;      // h packed in its tiles' LDS image (pack_rows_tiled_kernel)
  const void* Wp;      // W packed the same way, [V_pad] rows
  int hS;              // reduction slices of both
  int h_f32, w_f32;    // h / W stored in fp32 (rounded to the compute dtype as they are packed)
  const float* h_scale;  // e4m3 forward: [1] dequantisation scale of h, else null
  const float* w_scale;  // e4m3 forward: [V] dequantisation scales of W's rows, else null
  // Active-token forward: [0] the count of active tokens, whose rows are packed
  // in position order (hp), [3] / [4] the token blocks and vocabulary splits
  // (fwd_active_grid_kernel), all on the device; null: every token, at its own row.
  const int* n_act;
};

constexpr int kFwdRound = 256;

// Model of a forward whose n_tb x s workgroups hold a CU each and run 256 at a time, in units of about
// 1.5 us: a workgroup takes n_vt / s vocabulary tiles on average, `tile` each, and 5 for its ring fill
// and partial stores; a single round ends with its longest workgroup, several even out half of that; the
// merge reads every workgroup's partials, `part` each (0.3 us per MB).
struct FwdCost {
  double tile, part;
};
inline FwdCost fwd_cost(int64_t K, int DP, int BM, int WV) {
  return {((double)K + DP) / 32 * 0.3 * (BM / 128.0), 0.2e-6 * 4 * WV * BM * DP};
}
__host__ __device__ inline double fwd_span(int64_t n_tb, int64_t n_vt, int64_t s, FwdCost c) {
  const int64_t rounds = (n_tb * s + kFwdRound - 1) / kFwdRound;
  const double avg = (double)n_vt / s, rest = (double)((n_vt + s - 1) / s) - avg;
  return rounds * (avg * c.tile + 5.0) + rest * c.tile * (rounds > 1 ? 0.5 : 1.0) + n_tb * s * c.part;
}

// Vocabulary splits an active-token forward of tb token blocks may take: at least two vocabulary
// tiles each, and no more workgroups than twice the all-token tiling's n_tb_max x n_split0, which is
// what the launch and the partial buffers hold.
__host__ __device__ inline int active_splits_max(int tb, int n_tb_max, int n_split0, int n_vt) {
  const int cap = n_vt / 2 > 1 ? n_vt / 2 : 1;
  const int64_t fit = 2 * (int64_t)n_tb_max * n_split0 / (tb > 0 ? tb : 1);
  return fit < cap ? (int)fit : cap;
}

struct FwdPlan {
  int BV, BM, DP;
  int DS, n_dslices;     // embedding columns per pass, passes (D > DS runs in slices of E's columns)
  int n_tb, n_vt, n_split, n_part;
  int V_pad;
  int64_t N_pad;         // token rows of the packed h
  int hS;                // reduction slices of the packed h and W
  size_t off_m, off_l, off_acc, off_Ep, off_bias, off_hp, off_Wp, ws_bytes;
  // active-token forward: per-token flags, positions, the count and the
  // non-finite parameter flag (ws_bytes includes them only when planned so)
  bool active;
  int WV;
  size_t off_flag, off_idx, off_inv, off_nact;
  // the last pass of a D in several passes, when it is narrow enough for a narrower kernel (rem_DP > 0)
  int rem_DP, rem_BM, rem_tb, rem_split, rem_part;
  // few tokens (fwd_few.hip): tile, split and workspace of that path; few = false: not taken
  bool few;
  int few_DP, few_NB, few_tb, few_split, few_wgs;  // few_wgs: workgroups the partials hold
  size_t few_m, few_l, few_acc, few_hp, few_E;
};

// fwd_plan / fwd_launch dtype of the e4m3 forward (h, W in e4m3; E in bf16).
constexpr int kFwdFP8 = 3;

// Tile shape, split count and workspace for a forward call; ok=false if the
// dtype / D combination is unsupported.
bool fwd_plan(int dtype, int64_t N, int64_t K, int64_t V, int64_t D, FwdPlan* plan, bool active = false);
// O / lse, or with m_out / l_out set the merged partial softmax (m, l, and the
// unnormalised acc in O) of the vocabulary rows given.
hipError_t fwd_launch(int dtype, const FwdPlan& plan, FwdParams p, char* ws, float* O, float* lse, float* m_out,
                      float* l_out, hipStream_t stream);
// The forward of the tokens with a non-zero weight (weight: fp32 [N]); O rows
// and lse of the others are 0.  A zero-weight token whose h row holds an
// infinity or a NaN stays active, and so does every token when W, E or the
// bias holds a NaN or +inf or when every bias entry is -inf: the rows whose
// loss the reference makes NaN (0 * NaN) are computed.  With few tokens every token is computed, and
// the finite values of a zero-weight one written as 0.  Plan with active set.
hipError_t fwd_launch_active(int dtype, const FwdPlan& plan, FwdParams p, const float* weight, char* ws, float* O,
                             float* lse, hipStream_t stream);
// ---- few tokens (fwd_few.hip): W and E read as the caller stores them
struct FwdFewParams {
  const void* hp;      // h packed in its tiles' LDS image (pack_rows_tiled_kernel), hS slices
  int hS;
  const void* W;       // [V][ldw]: the compute dtype, or fp32 (w_f32) under a 2-byte one
  int64_t ldw;
  int w_f32;
  const void* E;       // [V][lde], 16-byte aligned rows of D columns, D a multiple of the 16-byte chunk
  int64_t lde;
  const float* bias;   // [V] or null
  float scale;
  int N, K, V, D;
  int DP, NB;          // padded D (32 fp32 only, 64, 128, 256), 32-token blocks per workgroup (1, 2, 4)
  int n_tb, n_split;   // token blocks, vocabulary runs
  int n_wg;            // workgroups to launch (n_tb x n_split, or with n_act as many as may be needed)
  // active tokens only: hp holds their rows in position order, [3] / [4] of this device block the token
  // blocks and runs (few_runs); null: every token at its own row
  const int* n_act;
  float* part_m;       // [n_split][N] (with n_act, rows of [3] x 32 NB positions)
  float* part_l;
  float* part_acc;     // [n_split][DP][N]
};

// Vocabulary runs of the few-token forward for n_tb token blocks over grp 32-row groups, when one
// workgroup runs per CU: the count that ends soonest, each workgroup taking its longest run and about
// one group's time more for its ring fill and partial stores, over at most kFewRounds rounds of the CUs.
constexpr int kFewRounds = 4;
__host__ __device__ inline int64_t few_span(int64_t n_tb, int64_t grp, int64_t s) {
  return (n_tb * s + kFwdRound - 1) / kFwdRound * ((grp + s - 1) / s + 1);
}
__host__ __device__ inline int few_runs_max(int64_t n_tb, int64_t grp) {
  const int64_t m = kFewRounds * kFwdRound / (n_tb > 0 ? n_tb : 1), c = m < grp ? m : grp;
  return c < 1 ? 1 : (int)c;
}
// Within a number of rounds the span falls with the length of the longest run alone, so the candidates are
// the most runs that each number of rounds holds, brought down to the fewest with the same longest run (all
// counts tried one by one took the host 5 us of a one-token call, twice).
__host__ __device__ inline int few_runs(int64_t n_tb, int64_t grp) {
  const int64_t most = few_runs_max(n_tb, grp);
  int best = 1;
  for (int64_t r = 1; r <= kFewRounds; ++r) {
    const int64_t fit = r * kFwdRound / (n_tb > 0 ? n_tb : 1), s = fit < most ? fit : most;
    if (s < 1 || grp < 1) continue;
    const int64_t run = (grp + s - 1) / s;
    const int64_t fewest = (grp + run - 1) / run;
    if (few_span(n_tb, grp, fewest) < few_span(n_tb, grp, best)) best = (int)fewest;
  }
  return best;
}
hipError_t fwd_few_launch(int dtype, const FwdFewParams& p, hipStream_t stream);

// Order-preserving compaction of flagged tokens (flag[n] != 0): idx[q] = token
// of position q, inv[n] = position of token n or -1, n_act[0] = count.
hipError_t compact_tokens(const int* flag, int N, int* idx, int* inv, int* n_act, hipStream_t stream);
// Merge S vocabulary shards' partials (m, l: [S][N]; acc: [S][N][D]) in shard order.
hipError_t shard_combine(int S, int N, int D, const float* m, const float* l, const float* acc, float* O, float* lse,
                         hipStream_t stream);

// ---------------------------------------------------------------- backward
struct BwdPlan {
  int DP;
  int BM, BV;            // dS kernel tile: BM tokens x BV vocabulary
  int GM, GN;            // gradient GEMM tile
  int n_tb;              // token blocks of the dS kernel
  int64_t N_pad;         // token stride of the dS stage
  int64_t C;             // vocabulary rows per chunk (multiple of BV)
  int n_chunks;
  int G;                 // token groups of the dS kernel (a full chunk)
  int wgs;               // workgroups the dS kernel's tiling fills the chip with (G per chunk from it)
  int n_gpart;           // dE / db partials per chunk
  int kind;              // scores kernel: kScoresGeneral, kScoresRing (narrow), kScoresWide
  bool dh_acc;           // dh accumulates in fp32 (over the active tokens), then expands into gh
  int V_pad;             // vocabulary rows of the packed E / bias
  int hS;                // reduction slices of the packed h and W
  size_t off_stage, off_pe, off_pb, off_dh, off_gO, off_gOt, off_lsed, off_Ep, off_bias, off_hp, off_Wp;
  size_t off_flag, off_idx, off_inv, off_nact, off_delta, off_hc, off_Wc, ws_bytes;
  int hS8;               // e4m3 scores: reduction slices of the packed e4m3 h and W (K8 / 2 pairs)
  size_t off_hqc, off_mult;
  size_t off_pstage;     // P stage (wide scores kernel), the dS stage's layout
  // vocabulary runs each dh tile's reduction is split over (dh_split_of), beside dW tiles and alone
  int dh_split_w, dh_split_h;
};

// Scores kernels of the backward (BwdPlan::kind).
enum { kScoresGeneral = 0, kScoresRing = 1, kScoresWide = 2 };
// With the wide scores kernel, dE^T = gO^T P is formed by the gradient GEMM launch as up to this
// many partial sums over equal runs of the positions (fixed-order sum after the launch): one run
// per 2048 token rows (64 reduction slices), 1 to kDeSplit (de_split).
constexpr int kDeSplit = 8;
inline int de_split(int64_t n_pad) {
  const int64_t s = n_pad / 2048;
  return s < 1 ? 1 : s > kDeSplit ? kDeSplit : (int)s;
}

// Runs of a chunk's vocabulary rows that each dh tile is split over, every run a piece of the
// gradient GEMM launch with an fp32 accumulator of its own (summed in run order when gh is
// written).  A launch has n_dw dW tiles of s_dw reduction slices and n_dh dh tiles of s_dh; with
// few tokens the dh tiles are few and long (8 tiles of 256 slices beside 128 of 16 at 512 tokens,
// K = 1024), and the launch waits for them with most CUs idle.  The split minimises the launch's
// duration when `slots` workgroups run at a time, dW tiles dealt first, with o_dw / o_dh slices'
// worth of time per tile for its prologue and stores: a run that ends in a read-modify-write of
// its accumulator costs more than a dW tile.  Runs keep at least 8 slices, the accumulators beyond
// the first (acc_bytes each) stay within `room` (two dS stages and kDhSplitBytes), and a split must
// gain 5%.
// Measured, the whole call, whole tiles against split: N = 2048, K = 1024, V = 151936, gh alone (32 dh
// tiles per chunk, 8 runs) 4.65 -> 2.63 ms; N = 500, K = 1024, V = 32000, every gradient (8 dh and 128
// dW tiles, 16 runs) 1.02 -> 0.53 ms; N = 2048, K = 2048, V = 65536 (64 and 256, 4 runs) 3.48 -> 2.95.
constexpr int64_t kDhSplitBytes = (int64_t)64 << 20;
inline int dh_split_of(int64_t n_dw, int64_t s_dw, int64_t n_dh, int64_t s_dh, int slots, int o_dw, int o_dh,
                       int64_t acc_bytes, int64_t room) {
  if (n_dh <= 0) return 1;
  const int64_t a = s_dw + o_dw, q = n_dw / slots, r = n_dw % slots;
  auto span = [&](int64_t s) {
    const int64_t jobs = n_dh * s, b = (s_dh + s - 1) / s + o_dh;
    // r slots are free at (q + 1) a, the others at q a: the earliest end of all jobs of length b
    auto fits = [&](int64_t t) {
      const int64_t x = t >= (q + 1) * a ? (t - (q + 1) * a) / b : 0, y = t >= q * a ? (t - q * a) / b : 0;
      return r * x + (slots - r) * y >= jobs;
    };
    const int64_t lo = (q + 1) * a, rounds = jobs / slots + 2;
    int64_t best = INT64_MAX;
    for (int64_t i = 0; i <= rounds; ++i) {
      const int64_t t0 = q * a + i * b, t1 = (q + 1) * a + i * b;
      if (fits(t0) && t0 < best) best = t0;
      if (fits(t1) && t1 < best) best = t1;
    }
    return r > 0 && best < lo ? lo : best;
  };
  int64_t best = span(1) * 95 / 100;
  int split = 1;
  for (int s = 2; s <= 64 && s_dh / s >= 8 && (s - 1) * acc_bytes <= room; s *= 2) {
    const int64_t t = span(s);
    if (t < best) {
      best = t;
      split = s;
    }
  }
  return split;
}

// w_f32: W is stored in fp32 and needs a row-major copy in the compute dtype
// (the dh product reads W rows directly).
// K8 > 0: the scores are recomputed from e4m3 h and W of K8 bytes per row.
bool bwd_plan(int dtype, int64_t N, int64_t K, int64_t V, int64_t D, int64_t chunk, bool need_gh,
              BwdPlan* plan, bool w_f32 = false, int64_t K8 = 0);
// Vocabulary rows to stage at a time when the caller names no chunk.
int64_t bwd_default_chunk(int dtype, int64_t N, int64_t K, int64_t V, int64_t D, bool need_gh, bool w_f32, int64_t K8);

struct BwdParams {
  const void* h;
  int64_t ldh;
  const void* W;
  int64_t ldw;
  const void* E;
  int64_t lde;
  const float* bias;
  float scale;
  int N, K, V, D;
  const float* O;
  const float* lse;
  const float* gO;
  const float* glse;
  void* gh;
  int gh_dtype;
  void* gW;
  int gW_dtype;
  void* gE;
  int gE_dtype;
  float* gb;
  char* ws;
  int h_f32, w_f32;    // h / W stored in fp32 (rounded to the compute dtype as they are read)
  // e4m3 scores (null hq: the compute dtype's): h and W as e4m3 bytes, K8 per
  // row, leading dims in bytes, with the forward's dequantisation scales
  const void* hq;
  int64_t ldhq;
  const void* Wq;
  int64_t ldwq;
  const float* h_scale;
  const float* w_scale;
  int K8;
};

hipError_t bwd_launch(int dtype, const BwdPlan& plan, const BwdParams& p, hipStream_t stream);

// ---------------------------------------------------------------- MSE loss
struct MseParams {
  const float* O;       // [N][D] fp32
  const float* lse;     // [N] fp32
  const void* target;   // [N][ldt], target_dtype (0 bf16, 1 f16, 2 f32)
  int64_t ldt;
  int target_dtype;
  const float* weight;  // [N] fp32 or null
  int N, D;
  float z;              // z-loss weight
  int reduce;           // 0 none, 1 sum, 2 mean
  float* per_tok;       // [N] (reduce == 0) or null
  float* out;           // [1] (reduce != 0)
  float* scale;         // [1] (reduce != 0): the c of the loss
  float* gO;            // [N][D] or null
  float* glse;          // [N] or null (with gO)
};
size_t mse_workspace_bytes(int N);
// Largest N of the allocation-free loss entry point, whose partial sums live in
// a fixed device array (loss.hip) instead of the caller's workspace.
constexpr int kMseNoAllocMaxTokens = 1 << 22;
// Address of that array on the device of `stream` (the current device for the
// null stream), looked up once per device.
hipError_t mse_noalloc_scratch(hipStream_t stream, void** ptr);

// ---------------------------------------------------------------- e4m3 quantisation
struct QuantParams {
  const void* x;   // [R][ld], x_dtype (0 bf16, 1 f16, 2 f32)
  int64_t ld;
  int x_dtype;
  int R, K, Kp;    // rows, columns, output columns (zero past K)
  int per_row;     // scales per row ([R]) or one for the matrix ([1])
  void* out;       // e4m3 bytes [R][ldo]
  int64_t ldo;
  float* scale;
  float* amax;     // per-tensor: [R] row amaxes (workspace)
};
hipError_t quant_launch(const QuantParams& q, hipStream_t stream);

// ---------------------------------------------------------------- fp64
struct F64Params {
  const double* h;
  int64_t ldh;
  const double* W;
  int64_t ldw;
  const double* E;
  int64_t lde;
  const double* bias;  // [V] or null
  double scale;
  int N, K, V, D;
  int64_t chunk;
  double* O;            // forward: [N][D]; backward: the forward's O (read)
  double* lse;          // forward: [N]; backward: the forward's lse (read)
  const double* gO;     // backward: [N][D]
  const double* glse;   // backward: [N]
  double* gh;           // [N][K] or null
  double* gW;           // [V][K] or null
  double* gE;           // [V][D] or null
  double* gb;           // [V] or null
  char* ws;
};
// Vocabulary rows per chunk and workspace bytes of the fp64 forward / backward.
void f64_plan(int64_t N, int64_t V, int64_t D, int64_t chunk, int64_t* C, size_t* fwd_bytes, size_t* bwd_bytes);
hipError_t f64_fwd(const F64Params& p, hipStream_t stream);
hipError_t f64_bwd(const F64Params& p, hipStream_t stream);

// Matrix-core throughput probe (probe.hip): workgroups of 8 waves, iters k16 steps of
// 8 MFMAs per wave; out receives workgroups * 512 floats.
hipError_t probe_mfma(int workgroups, int iters, int mode, float* out, hipStream_t stream);
hipError_t mse_launch(const MseParams& p, void* ws, hipStream_t stream);

}  // namespace swvr
