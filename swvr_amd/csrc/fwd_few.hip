// Forward that streams W as it is stored: O = softmax(s * h W^T + b) E and LSE of
// few tokens, bound by reading W once and not by matrix work, and of any number
// in fp32.
//
// The general forward (fwd.hip) packs W into its tiles' LDS image first, which
// pays where many token blocks read it but moves W's bytes three times, and its
// tiles of 128 or 256 tokens are mostly padding here.  In fp32, where a matrix
// instruction takes 16 times as long and the operand traffic hardly counts, this
// kernel's 128 x 128 tile of 8 waves is the faster one at any size: 8192 tokens on
// V = 32000, K = 2560, D = 64 13.3 -> 10.7 ms (129 TF/s).  This kernel streams W's
// rows as the caller stores them (rounding an fp32 W to the compute dtype at
// the operand read), E's rows likewise, and the bias:
//   * a workgroup owns a run of vocabulary rows (whole 32-row groups; one
//     workgroup per CU, so the runs are equal to 32 rows) and a block of 32, 64
//     or 128 tokens; it walks its run 128 rows at a time.  4 waves of 32 rows, or
//     twice those, half the tokens each, so that the accumulators of a wider
//     block stay within the 256 registers of two waves per SIMD;
//   * W arrives in 128-byte row pieces through an LDS ring as deep as the 160 KB
//     allow, so 48 to 100 KB of W are in flight per CU: the loop is bound by HBM.
//     Rows past the run are not loaded;
//   * the online softmax and acc^T += E^T P^T run as in the general forward,
//     the tile of 128 rows being each wave's own 32, to whose maximum P is relative in
//     the 2-byte types, times a power of two (tile_shift): its largest P stays exact (O of
//     1000 tokens on V = 151936 at a logit spread of 3: 5.8e-5 from 64 bits in bf16, 1.3e-4
//     with running maxima).
//     The E^T operand is read from the row-major E tile with transposing LDS reads;
//   * the waves' partial softmaxes are merged in LDS, so a workgroup writes one
//     partial; fwd_combine_kernel merges those in a fixed order.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace swvr {

namespace {

constexpr int kFewBV = 128, kFewWV = 4;  // vocabulary rows per tile, waves along them
constexpr int kLdsBytes = 160 * 1024;

// Tile of E rows [128][DP] in LDS as the caller stores them, 16-byte chunks swizzled so that the
// transposing reads (4 rows x 64 bytes per 32 lanes) fall on all 64 banks.
template <class T, int DP, int NT>
struct FewETile {
  static constexpr int CE = 16 / (int)sizeof(T);
  static constexpr int ROWB = DP * (int)sizeof(T);
  static constexpr int BYTES = kFewBV * ROWB;
  static constexpr int NI = BYTES / (NT * 16);
  static_assert(ROWB >= 128 && BYTES % (NT * 16) == 0, "whole loads, at least 8 chunks per row");
  __device__ static __forceinline__ int swz(int row) {
    return sizeof(T) == 4 ? 0 : ROWB == 128 ? 4 * ((row >> 1) & 1) : 4 * (row & 3);
  }
  // Rows 0 .. rows - 1 of E (row stride ldb bytes), columns 0 .. D - 1; zeros elsewhere.
  __device__ static __forceinline__ void issue(const T* E, int64_t ldb, int rows, int D, uint32_t lds) {
    const rsrc_t r = make_rsrc(E);
    const int tid = (int)threadIdx.x + opaque_zero();  // offsets computed here, not kept across the walk
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int lin = (i * NT + tid) * 16;
      const int row = lin / ROWB, c = ((lin % ROWB) / 16) ^ swz(lin / ROWB);
      const uint32_t off = row < rows && c * CE < D ? (uint32_t)(row * ldb + c * 16) : kOOB;
      dma_batch1(r, off, lds + i * NT * 16 + wave_id() * 1024);
    }
  }
  // Operand of columns d0 .. d0 + 31 (this lane: d0 + lane % 32) over the 8 rows of k16 step c of a
  // 32-row block: row0 + 16 c + 8 (t / 4) + 4 (lane / 32) + t % 4, the order of the score registers.
  __device__ static __forceinline__ typename Vec8<T>::type read(const char* s, int row0, int c, int d0, int lane) {
    typedef typename Vec8<T>::type V8;
    const int hi = lane >> 5;
    V8 out;
    if constexpr (sizeof(T) == 2) {
      const int g = (lane >> 4) & 1, a = (lane & 15) >> 2, q = lane & 3;
      const int d = d0 + 16 * g + 4 * q;
      s16x4_t v[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = row0 + 16 * c + 8 * h + 4 * hi + a;
        const char* p = s + row * ROWB + (((d / CE) ^ swz(row)) * 16) + (d % CE) * 2;
        v[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
      }
      const s16x8_t both = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
      __builtin_memcpy(&out, &both, 16);
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t)
        out[t] = *reinterpret_cast<const float*>(s + (row0 + 16 * c + 8 * (t >> 2) + 4 * hi + (t & 3)) * ROWB +
                                                 (d0 + (lane & 31)) * 4);
    }
    return out;
  }
};

// T: compute dtype; WS: storage of W (T, or float for a 2-byte T); FT: 32-token blocks per wave; WT:
// waves along the tokens.
template <class T, class WS, int DP, int FT, int WT>
struct FewCfg {
  static constexpr int NT = 64 * kFewWV * WT, NB = FT * WT;  // threads, 32-token blocks
  static constexpr int BK = 128 / (int)sizeof(WS);  // reduction elements per stage: 128-byte pieces of W's rows
  static constexpr int HK = SliceK<T>::value;       // reduction elements of a packed slice of h
  static constexpr int HS = BK / HK;                // such slices per stage
  static_assert(BK % HK == 0 && HS >= 1, "whole slices of h");
  typedef KTile<WS, kFewBV, BK, NT> TW;
  typedef KTile<T, 32 * NB, HK, NT> TH;         // layout of one slice of h
  static constexpr int HBYTES = HS * TH::BYTES;
  static constexpr int NIH = HBYTES / (NT * 16);
  static constexpr bool HPART = HBYTES < NT * 16;  // h of a stage is less than one load per thread
  static constexpr int SB = TW::BYTES + HBYTES;
  static constexpr int L = TW::NI + NIH;            // loads a thread issues per stage (at least)
  typedef FewETile<T, DP, NT> TE;
  static constexpr int FIT = (kLdsBytes - TE::BYTES) / SB;
  static constexpr int NS = FIT < 8 ? FIT : 8;
  static_assert(NS >= 2 && (NS - 2) * L < 64, "ring depth");
  static constexpr int LDS = NS * SB + TE::BYTES;
  // the merge of the waves' partials reuses the LDS: 4 x [DP][32] floats, then 4 x [32 NB] of two
  static_assert(kFewWV * (DP * 32 + 2 * 32 * NB) * 4 <= LDS, "merge fits");
};

// At most min(ahead, MAX) stages of L loads may stay outstanding.
template <int L, int MAX>
__device__ __forceinline__ void wait_ahead(int ahead) {
  if constexpr (MAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (ahead >= MAX)
      wait_vmcnt<MAX * L>();
    else
      wait_ahead<L, MAX - 1>(ahead);
  }
}

template <class T, class WS, int DP, int FT, int WT>
__global__ __launch_bounds__((FewCfg<T, WS, DP, FT, WT>::NT)) void fwd_few_kernel(FwdFewParams p) {
  typedef FewCfg<T, WS, DP, FT, WT> C;
  constexpr int NT = C::NT, NB = C::NB;
  typedef typename C::TW TW;
  typedef typename C::TH TH;
  typedef typename C::TE TE;
  typedef typename Vec8<T>::type V8;
  constexpr int BK = C::BK, HS = C::HS, NS = C::NS, SB = C::SB, L = C::L, DB = DP / 32;
  constexpr int J = C::HK / 16;  // k16 steps per slice of h
  __shared__ __attribute__((aligned(1024))) char smem[C::LDS];
  char* const sE = smem + NS * SB;

  const int lane = lane_id(), w = wave_id(), wv = w % kFewWV, wt = w / kFewWV;
  // an XCD works through a contiguous range of runs, a run's token blocks side by side: they share W in its L2
  int n_tb = p.n_tb, n_split = p.n_split, ntok = p.N;  // ntok: token rows of a partial
  if (p.n_act) {
    n_tb = p.n_act[3];
    n_split = p.n_act[4];
    if ((int)blockIdx.x >= n_tb * n_split) return;
    ntok = n_tb * 32 * NB;
  }
  const int t = xcd_swizzle(blockIdx.x, n_tb * n_split);
  const int split = t / n_tb, n0 = (t % n_tb) * 32 * NB;
  const int n_grp = (p.V + 31) / 32;
  const int v_begin = (int)((int64_t)split * n_grp / n_split) * 32;
  const int v_end = min(p.V, (int)((int64_t)(split + 1) * n_grp / n_split) * 32);
  const int n_tiles = v_end > v_begin ? (v_end - v_begin + kFewBV - 1) / kFewBV : 0;
  const int nk = max(1, (p.K + BK - 1) / BK);  // K = 0: one all-zero slice (bias-only scores)
  const int total = n_tiles * nk;
  const uint32_t lds0 = lds_addr(smem), ldsE = lds0 + NS * SB;

  TW tw;
  tw.setup(static_cast<const WS*>(p.W) + (int64_t)v_begin * p.ldw, p.ldw, v_end - v_begin, p.K);
  // h of a stage: HS slices of FT 32-row groups, 2 KB pieces of the packed h
  constexpr int GROUP = 32 * C::HK * (int)sizeof(T);
  constexpr int NIH = C::HPART ? 1 : C::NIH;
  const char* const hb = static_cast<const char*>(p.hp) + (int64_t)(n0 >> 5) * p.hS * GROUP;
  uint32_t hoff[NIH];
#pragma unroll
  for (int i = 0; i < NIH; ++i) {
    const int lin = (i * NT + (int)threadIdx.x) * 16;
    hoff[i] = (uint32_t)((lin / TH::BYTES) * GROUP + (lin % TH::BYTES) / GROUP * p.hS * GROUP + lin % GROUP);
  }
  int issued = 0, is_tile = 0, is_kt = 0, is_slot = 0;
  auto issue_next = [&]() {
    if (issued >= total) return;
    const uint32_t st = lds0 + is_slot * SB;
    if (is_kt == 0) {
      const int v0 = v_begin + is_tile * kFewBV;
      tw.rebase(static_cast<const WS*>(p.W) + (int64_t)v0 * p.ldw, v_end - v0, (int)threadIdx.x + opaque_zero());
    }
    tw.issue(st, is_kt * BK);
    if (!C::HPART || (int)threadIdx.x * 16 < C::HBYTES) {
      const rsrc_t r = make_rsrc(hb + (int64_t)is_kt * HS * GROUP);
      uint32_t v[NIH];
#pragma unroll
      for (int i = 0; i < NIH; ++i) {
        const int sub = ((i * NT + (int)threadIdx.x) * 16) / TH::BYTES;
        v[i] = is_kt * HS + sub < p.hS ? hoff[i] : kOOB;  // slices past the packed h are zero
      }
#pragma unroll
      for (int i = 0; i < NIH; ++i) dma_batch1(r, v[i], st + TW::BYTES + i * NT * 16 + w * 1024);
    }
    ++issued;
    if (++is_kt == nk) {
      is_kt = 0;
      ++is_tile;
    }
    is_slot = is_slot == NS - 1 ? 0 : is_slot + 1;
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue_next();

  // fp32 keeps the running maximum: it does not round P, and a shift per tile would round l and acc at every
  // tile instead (8192 tokens on V = 151936: l 3.4e-7 from 64 bits then, 8.4e-8 so)
  constexpr bool TS = sizeof(T) == 2;
  float m[FT], sh[FT], l[FT];  // running maximum, which l is relative to; the shift acc is relative to
  f32x16_t oacc[DB][FT], sacc[FT];
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    m[ft] = sh[ft] = kNegInf;
    l[ft] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db][ft] = zero16();
  }
  OpOffsets<TH, FT, J> ho;
  ho.init(wt * 32 * FT);
  // byte offsets of this lane's W operand of k16 step j of a stage: row 32 wv + lane % 32, elements
  // 16 j + 8 (lane / 32) .. + 7
  uint32_t wo[BK / 16];
#pragma unroll
  for (int j = 0; j < BK / 16; ++j) wo[j] = TW::elem(32 * wv + (lane & 31), 16 * j + 8 * (lane >> 5));

  int cur = -1, slot = NS - 1;
  for (int tile = 0; tile < n_tiles; ++tile) {
    const int v0 = v_begin + tile * kFewBV;
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) sacc[ft] = zero16();
    for (int kt = 0; kt < nk; ++kt) {
      ++cur;
      wait_ahead<L, NS - 2>(issued - 1 - cur);
      stage_barrier();
      slot = slot == NS - 1 ? 0 : slot + 1;
      // every wave has finished the stage before this one, whose slot the next load takes, and with
      // a tile's first stage the previous tile's epilogue, so its E tile can be replaced
      if (kt == 0)
        TE::issue(static_cast<const T*>(p.E) + (int64_t)v0 * p.lde, p.lde * (int64_t)sizeof(T), v_end - v0, p.D, ldsE);
      issue_next();
      const char* st = smem + slot * SB;
#pragma unroll
      for (int s = 0; s < HS; ++s)
#pragma unroll
        for (int j = 0; j < J; ++j) {
          V8 a;
          if constexpr (sizeof(WS) == sizeof(T) && sizeof(T) == 2) {
            a = *reinterpret_cast<const V8*>(st + wo[s * J + j]);
          } else {
            // 8 fp32 values in the chunks at o and o ^ 16 (8 elements: an even chunk and the next)
            const float4 lo = *reinterpret_cast<const float4*>(st + wo[s * J + j]);
            const float4 hi = *reinterpret_cast<const float4*>(st + (wo[s * J + j] ^ 16u));
            a[0] = from_float<T>(lo.x); a[1] = from_float<T>(lo.y); a[2] = from_float<T>(lo.z); a[3] = from_float<T>(lo.w);
            a[4] = from_float<T>(hi.x); a[5] = from_float<T>(hi.y); a[6] = from_float<T>(hi.z); a[7] = from_float<T>(hi.w);
          }
#pragma unroll
          for (int ft = 0; ft < FT; ++ft) mfma_k16(sacc[ft], a, ho.read(st + TW::BYTES + s * TH::BYTES, j, ft));
        }
    }
    // the E tile: covered by the stage waits after it unless the walk is short
    if (nk < NS) {
      wait_vmcnt<0>();
      stage_barrier();
    }

    // ---- scores -> running softmax of this wave's 32 rows
    float bb[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int v = v0 + 32 * wv + c_row(r, lane);
      bb[r] = v < v_end ? (p.bias ? p.bias[v] : 0.f) : kNegInf;
    }
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      float mx = kNegInf;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = fmaf(sacc[ft][r], p.scale, bb[r]);  // rounded as the backward rounds it
        sacc[ft][r] = x;
        mx = fmaxf(mx, x);
      }
      mx = wave_max32(mx);
      const float mnew = fmaxf(m[ft], mx);
      const float snew = TS ? tile_shift(mx, mnew) : mnew;
      // a column whose scores so far are all -inf keeps -inf; shift it by 0
      // (swvr/chunked.py:98-99)
      const float shift = snew == kNegInf ? 0.f : snew;
      const float alpha = fast_exp(sh[ft] - shift);
      sh[ft] = snew;
      float rs = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = fast_exp(sacc[ft][r] - shift);
        sacc[ft][r] = pv;
        rs += pv;
      }
      rs = wave_sum32(rs);
      l[ft] = TS ? shifted_sum(l[ft], m[ft], rs, shift, mnew) : l[ft] * alpha + rs;
      m[ft] = mnew;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][ft][r] *= alpha;
    }
    // ---- acc^T[d][token] += E^T[d][v] P^T[v][token]
    const int ln = lane + opaque_zero();
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      V8 bv[FT];
#pragma unroll
      for (int ft = 0; ft < FT; ++ft)
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) bv[ft][tt] = from_float<T>(sacc[ft][8 * c + tt]);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const V8 av = TE::read(sE, 32 * wv, c, db * 32, ln);
#pragma unroll
        for (int ft = 0; ft < FT; ++ft) mfma_k16(oacc[db][ft], av, bv[ft]);
      }
    }
  }

  // ---- merge the waves' partials through LDS: one (m, l, acc) per workgroup
  wait_vmcnt<0>();
  stage_barrier();
  float* const sA = reinterpret_cast<float*>(smem);  // [4][DP][32]
  float* const sM = sA + kFewWV * DP * 32;           // [4][32 NB]
  float* const sL = sM + kFewWV * 32 * NB;           // [4][32 NB]
#pragma unroll
  for (int ft = 0; ft < FT; ++ft)
    if (lane < 32) {
      const int c = (wt * FT + ft) * 32 + lane;
      sM[wv * 32 * NB + c] = m[ft];
      sL[wv * 32 * NB + c] = l[ft];
    }
  __syncthreads();
  for (int bt = 0; bt < WT; ++bt)
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      const int c = (bt * FT + ft) * 32 + (lane & 31);
      float M = kNegInf;
#pragma unroll
      for (int j = 0; j < kFewWV; ++j) M = fmaxf(M, sM[j * 32 * NB + c]);
      const float shift = M == kNegInf ? 0.f : M;
      if (wt == bt) {
        const float f = expf(sh[ft] - shift);  // exp(-inf) = 0: a wave of masked rows adds nothing
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            sA[(wv * DP + db * 32 + c_row(r, lane)) * 32 + (lane & 31)] = oacc[db][ft][r] * f;
      }
      __syncthreads();
      for (int e = threadIdx.x; e < DP * 32; e += NT) {
        const int n = n0 + (bt * FT + ft) * 32 + (e & 31);
        const float a = ((sA[e] + sA[DP * 32 + e]) + sA[2 * DP * 32 + e]) + sA[3 * DP * 32 + e];
        if (n < ntok) p.part_acc[((int64_t)split * DP + (e >> 5)) * ntok + n] = a;
      }
      if (w == 0 && lane < 32 && n0 + c < ntok) {
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < kFewWV; ++j) sum += sL[j * 32 * NB + c] * expf(sM[j * 32 * NB + c] - shift);
        p.part_m[(int64_t)split * ntok + n0 + c] = M;
        p.part_l[(int64_t)split * ntok + n0 + c] = sum;
      }
      __syncthreads();
    }
}

template <class T, class WS, int DP, int FT, int WT>
hipError_t launch(const FwdFewParams& p, hipStream_t stream) {
  if (p.n_tb * 32 * FT * WT < p.N) return hipErrorInvalidValue;
  timing_begin(kKindFwdTile, stream);
  fwd_few_kernel<T, WS, DP, FT, WT><<<p.n_wg, FewCfg<T, WS, DP, FT, WT>::NT, 0, stream>>>(p);
  timing_end(kKindFwdTile, stream);
  return hipGetLastError();
}

template <class T, class WS, int DP>
hipError_t dispatch_nb(const FwdFewParams& p, hipStream_t stream) {
  switch (p.NB) {
    case 1: return launch<T, WS, DP, 1, 1>(p, stream);
    case 2: return launch<T, WS, DP, 1, 2>(p, stream);
    case 4:
      if constexpr (DP <= 128) return launch<T, WS, DP, 2, 2>(p, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

template <class T, class WS>
hipError_t dispatch_dp(const FwdFewParams& p, hipStream_t stream) {
  switch (p.DP) {
    case 32:
      if constexpr (sizeof(T) == 4) return dispatch_nb<T, WS, 32>(p, stream);
      return hipErrorInvalidValue;
    case 64: return dispatch_nb<T, WS, 64>(p, stream);
    case 128: return dispatch_nb<T, WS, 128>(p, stream);
    case 256:
      if constexpr (sizeof(T) == 2) return dispatch_nb<T, WS, 256>(p, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t fwd_few_launch(int dtype, const FwdFewParams& p, hipStream_t stream) {
  switch (dtype) {
    case kBF16: return p.w_f32 ? dispatch_dp<bf16_t, float>(p, stream) : dispatch_dp<bf16_t, bf16_t>(p, stream);
    case kF16: return p.w_f32 ? dispatch_dp<f16_t, float>(p, stream) : dispatch_dp<f16_t, f16_t>(p, stream);
    case kF32: return dispatch_dp<float, float>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace swvr
