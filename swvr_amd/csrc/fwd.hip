// Fused forward: O = softmax(s * h W^T + b) E and LSE, without writing scores.
//
// Algorithm: the online softmax of swvr/chunked.py:82-105 (docs/DESIGN.md:12-24),
// reorganised for the GPU:
//   * a workgroup owns BM tokens and one of n_split contiguous vocabulary
//     ranges; it walks that range BV rows at a time;
//   * per vocabulary tile it forms S^T = W_tile h_tile^T (BV x BM) with MFMA
//     over the whole hidden size K, streaming K slices of the packed W and h
//     through an NS-slot LDS ring (3 slots beside the pinned E^T tile for
//     2-byte dtypes with D <= 64, 4 for fp32; for 2-byte D of 128 and 256
//     E^T travels through the ring instead, 3 stages of two slices each,
//     fwd_stream_kernel);
//   * the waves form a WV (vocabulary) x WT (tokens) grid: at D <= 64, 8 waves
//     of 128 vocabulary rows x 64 tokens (2 x 4) over a 256 x 256 tile.  In
//     the S^T layout each lane holds one token column, so the softmax max/sum
//     over the vocabulary is a register reduction plus one lane swap;
//   * every wave keeps its own running (m, l, acc) over its half of each tile
//     (an independent partial softmax), and P, rounded to the compute dtype as
//     the reference rounds it (swvr/chunked.py:103, triton_kernels.py:69),
//     feeds acc^T += E^T P^T straight from the score registers;
//     P is relative to the tile's own maximum times a power of two (tile_shift), not
//     to the running maximum: the maximum's row has a P of 1, 1/2, 1/4 ..., which no
//     rounding changes, so most rows that dominate a peaked softmax stay exact (O of 3000
//     tokens on V = 151936 at a logit spread of 3: 1.0e-4 from 64 bits in bf16,
//     1.7e-4 with the running maximum), whatever the number of splits;
//   * partials (m, l, acc) of all waves and splits are merged by
//     fwd_combine_kernel in a fixed order (deterministic).
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace swvr {

namespace {

// Tile shape per (dtype, padded D): BV vocabulary rows x BM tokens per
// workgroup of WV x WT waves (two waves per SIMD for bf16 / f16); the
// per-wave score block and acc^T block share the register file, NS K-slices
// of W and h plus the E^T tile and the bias share LDS (160 KB).  For the
// narrow embeddings (DP <= 64) each wave owns 128 vocabulary rows x 64
// tokens: 0.75 operand reads per MFMA.
template <class T, int DP>
struct FwdTile {
  static constexpr bool wide = sizeof(T) == 2;
  static constexpr bool narrow = wide && DP <= 64;
  // D = 128 and 256 (2-byte dtypes): E^T streamed through the ring in D-slices (fwd_stream_kernel)
  static constexpr bool stream_e = wide && (DP == 256 || DP == 128);
  // 2-byte dtypes: 128 x 64 waves (D <= 64), 128 x 32 (D = 128 and 256, E^T streamed): the widest
  // whose score and acc^T accumulators fit beside the operands at D = 256; at D = 128 they run
  // 2% faster than 64 x 64 waves with E^T pinned
  static constexpr int BV = wide ? 256 : 128;
  static constexpr int BM = narrow ? 256 : wide ? 128 : 64;
  static constexpr int WV = 2;
  static constexpr int WT = narrow ? 4 : wide ? 4 : 2;
  static constexpr int NT = 64 * WV * WT;
  static constexpr int NS = narrow ? 3 : kStages;  // LDS ring depth of fwd_tile_kernel (160 KB with E^T)
};

// The e4m3 forward (h and W in OCP e4m3, E and P in bf16): one k64 MFMA per
// 64-byte slice takes 32 operand bytes per lane, twice the bf16 k16 step's, so
// the 128 x 64 wave of the bf16 tile would not fit its accumulators and
// operands in 256 registers.  D <= 64: waves of 64 x 64 (one operand read per
// MFMA), a 4-deep ring of 24 KB slices and the software-pipelined reduction
// (two operand sets).  D = 128 (wider E^T tile and accumulators): 128 x 32
// waves, 3 slices, one operand set.
static_assert(kFP8 == kFwdFP8, "one dtype code for the e4m3 forward");

template <int DP>
struct FwdTileF8 {
  static constexpr bool pipe = DP <= 64;
  static constexpr int BV = 256, BM = 128, WV = pipe ? 4 : 2, WT = pipe ? 2 : 4;
  static constexpr int NT = 64 * WV * WT;
  static constexpr int NS = pipe ? 4 : 3;
};

template <class T, int DP, bool F8>
using FwdCfg = typename std::conditional<F8, FwdTileF8<DP>, FwdTile<T, DP>>::type;

// Vocabulary operands of the forward, packed once per call: E^T per
// vocabulary tile as [n_vt][DP][BV] (compute dtype; column p of tile vt is
// row vt * BV + pe_row(p) of E; zero past D and V) and the bias as fp32
// [V_pad] (-inf past V: padding rows drop out of the softmax).
// With w_scale set (the e4m3 forward) the bias goes out as (bias, multiplier)
// pairs, multiplier = logit_scale * h_scale * w_scale[v] (0 past V): the
// factor that turns the e4m3 dot product into a score.
// One workgroup per 32 columns of a tile: E's rows are read along d (64-byte
// runs, any alignment of E), E^T rows written as whole 16-byte chunks.  Bound by
// its traffic (E in, E^T out); one thread per element, which read E a row per
// lane, took 53 us at V = 151936, D = 64 and this 15 us.
template <class T, int BV>
__global__ __launch_bounds__(256) void pack_et_kernel(const T* __restrict__ E, int64_t lde,
                                                      const float* __restrict__ bias, int V, int D, int V_pad,
                                                      int DP, T* __restrict__ Et, float* __restrict__ biasp,
                                                      const float* __restrict__ h_scale,
                                                      const float* __restrict__ w_scale, float logit_scale) {
  constexpr int CE = 16 / (int)sizeof(T);
  constexpr int LS = 32 + 4 / (int)sizeof(T);  // elements per LDS row (one 4-byte word of padding)
  __shared__ T tile[BV * LS];
  const int ndb = DP / 32;
  const int vt = blockIdx.x / ndb, d0 = (blockIdx.x % ndb) * 32, v0 = vt * BV;
  const int t = threadIdx.x;
  {
    const int d = d0 + t % 32;
    T x[BV / 8];  // every load issued before the first is used
#pragma unroll
    for (int i = 0; i < BV / 8; ++i) {
      const int v = v0 + i * 8 + t / 32;
      x[i] = v < V && d < D ? E[(int64_t)v * lde + d] : (T)0.f;
    }
#pragma unroll
    for (int i = 0; i < BV / 8; ++i) tile[(i * 8 + t / 32) * LS + t % 32] = x[i];
  }
  __syncthreads();
  T* out = Et + ((int64_t)vt * DP + d0) * BV;
#pragma unroll
  for (int i = 0; i < BV * 32 / CE / 256; ++i) {
    const int c = i * 256 + t;  // 16-byte chunk of the 32 rows
    const int d = c / (BV / CE), p = (c % (BV / CE)) * CE;
    T q[CE];
#pragma unroll
    for (int j = 0; j < CE; ++j) q[j] = tile[pe_row(p + j) * LS + d];
    uint4 u;
    __builtin_memcpy(&u, q, 16);
    *reinterpret_cast<uint4*>(out + (int64_t)c * CE) = u;
  }
  if (d0 == 0)
    for (int i = t; i < BV; i += 256) {
      const int e = v0 + i;
      const float b = e < V ? (bias ? bias[e] : 0.f) : kNegInf;
      if (w_scale) {
        biasp[2 * (int64_t)e] = b;
        biasp[2 * (int64_t)e + 1] = e < V ? logit_scale * h_scale[0] * w_scale[e] : 0.f;
      } else {
        biasp[e] = b;
      }
    }
}

template <class T, int DP, bool F8 = false>
__global__ __launch_bounds__((FwdCfg<T, DP, F8>::NT)) void fwd_tile_kernel(FwdParams p) {
  typedef FwdCfg<T, DP, F8> C;
  typedef typename Vec8<T>::type V8;
  constexpr int kBK = SliceK<T>::value;
  constexpr int BV = C::BV, BM = C::BM, NT = C::NT;
  constexpr int WVR = BV / C::WV, WTR = BM / C::WT;  // rows per wave
  typedef PackedKLoader<T, BV, kBK, NT> TA;  // W rows of the vocabulary tile (packed)
  typedef PackedKLoader<T, BM, kBK, NT> TB;  // h rows of the token block (packed)
  typedef KTile<T, DP, BV, NT> TE;   // E^T tile [DP][BV] in pe_row order, swizzled like an operand tile
  constexpr int SB = TA::BYTES + TB::BYTES;
  constexpr int L = TA::NI_MIN + TB::NI_MIN;  // conservative for partial tiles
  constexpr int FV = WVR / 32, FT = WTR / 32;  // 32x32 blocks per wave
  constexpr int DB = DP / 32;
  constexpr int EBYTES = TE::BYTES;
  constexpr int BBYTES = BV * 4 * (F8 ? 2 : 1);  // bias, or (bias, multiplier) pairs

  constexpr int NS = C::NS;
  __shared__ __attribute__((aligned(1024))) char smem[NS * SB + EBYTES + BBYTES];
  char* const sE = smem + NS * SB;
  const float* const sBias = reinterpret_cast<const float*>(sE + EBYTES);

  const int lane = lane_id(), w = (int)(threadIdx.x >> 6);
  const int wv = w / C::WT, wt = w % C::WT;
  int n_tb = p.n_tb, n_split = p.n_split, ntok = p.N;  // ntok: token rows of a partial
  if (p.n_act) {
    n_tb = p.n_act[3];
    n_split = p.n_act[4];
    if ((int)blockIdx.x >= n_tb * n_split) return;
    ntok = n_tb * BM;
  }
  int split, tb;
  grouped_tile(blockIdx.x, n_split, n_tb, &split, &tb);
  const int n0 = tb * BM;
  const int vt_begin = (int)((int64_t)split * p.n_vt / n_split);
  const int vt_end = (int)((int64_t)(split + 1) * p.n_vt / n_split);
  const T* Ep = static_cast<const T*>(p.Ep);

  // P relative to its tile's maximum: not in fp32, which does not round it, nor in the e4m3 forward, whose
  // operands are rounded far more coarsely (0.8% faster there)
  constexpr bool TS = !F8 && sizeof(T) == 2;
  float m[FT], sh[FT], l[FT];  // running maximum, which l is relative to; the shift acc is relative to
  f32x16_t oacc[DB][FT];
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    m[ft] = sh[ft] = kNegInf;
    l[ft] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db][ft] = zero16();
  }

  const int nk = max(1, (p.K + kBK - 1) / kBK);  // K = 0: one all-zero slice (bias-only scores)
  const int n_tiles = vt_end - vt_begin;
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t ldsE = lds0 + NS * SB, ldsB = ldsE + EBYTES;
  TA ta;
  ta.setup(p.Wp, vt_begin * BV, p.hS);
  TB tbh;
  tbh.setup(p.hp, n0, p.hS);
  // issue cursor: the next stage to load (NS - 1 ahead of the compute)
  int is_tile = 0, is_kt = 0, is_slot = 0;
  auto issue_next = [&]() {
    if (is_tile >= n_tiles) return;
    if (is_kt == 0) {
      const int v0 = (vt_begin + is_tile) * BV;
      ta.rebase(v0);
    }
    const uint32_t st = lds0 + is_slot * SB;
    ta.issue(st, is_kt * kBK);
    tbh.issue(st + TA::BYTES, is_kt * kBK);
    if (++is_kt == nk) {
      is_kt = 0;
      ++is_tile;
    }
    is_slot = is_slot == NS - 1 ? 0 : is_slot + 1;
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue_next();

  f32x16_t sacc[FV][FT];
  Ring<NS> ring{NS - 1, n_tiles * nk};  // the first publish_next() moves to stage 0, slot 0
  for (int tile = 0; tile < n_tiles; ++tile) {
    const int v0 = (vt_begin + tile) * BV;
    // first stage of the tile; every wave has also finished the previous
    // tile's epilogue, so the E and bias tiles can be replaced
    ring.template publish_next<L>();
    {
      TE te;
      te.setup(Ep + (int64_t)v0 * DP, BV, DP, BV);
      te.issue(ldsE, 0);
      if ((int)threadIdx.x * 16 < BBYTES)
        dma_batch1(make_rsrc(p.biasp + (int64_t)v0 * (F8 ? 2 : 1)), (uint32_t)threadIdx.x * 16, ldsB + w * 1024);
    }
#pragma unroll
    for (int fv = 0; fv < FV; ++fv)
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) sacc[fv][ft] = zero16();
    if constexpr (F8)
      tile_reduce_f8<L, FwdTileF8<DP>::pipe>(sacc, ta, tbh, smem, SB, ring, nk, wv * WVR, wt * WTR, issue_next);
    else
      tile_reduce<T, kBK, L>(sacc, ta, tbh, smem, SB, ring, nk, wv * WVR, wt * WTR, issue_next);
    if (nk < NS) {
      // short reduction: the E / bias loads may still be in flight
      wait_vmcnt<0>();
      stage_barrier();
    }

    // ---- scores -> running softmax of this wave's slice of the tile
    float mx[FT];
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) mx[ft] = kNegInf;
#pragma unroll
    for (int fv = 0; fv < FV; ++fv)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        // registers 4g..4g+3 hold rows 8g + 4(lane/32) + 0..3 of the block
        const int row = wv * WVR + fv * 32 + 8 * g + (lane >> 5) * 4;
        float bb[4], mm[4];
        if constexpr (F8) {
          const float4 x0 = *reinterpret_cast<const float4*>(sBias + 2 * row);
          const float4 x1 = *reinterpret_cast<const float4*>(sBias + 2 * row + 4);
          bb[0] = x0.x; mm[0] = x0.y; bb[1] = x0.z; mm[1] = x0.w;
          bb[2] = x1.x; mm[2] = x1.y; bb[3] = x1.z; mm[3] = x1.w;
        } else {
          const float4 b4 = *reinterpret_cast<const float4*>(sBias + row);
          bb[0] = b4.x; bb[1] = b4.y; bb[2] = b4.z; bb[3] = b4.w;
          mm[0] = mm[1] = mm[2] = mm[3] = p.scale;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int ft = 0; ft < FT; ++ft) {
            const float x = fmaf(sacc[fv][ft][4 * g + i], mm[i], bb[i]);  // rounded as the backward rounds it
            sacc[fv][ft][4 * g + i] = x;
            mx[ft] = fmaxf(mx[ft], x);
          }
      }
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      const float mt = wave_max32(mx[ft]), mnew = fmaxf(m[ft], mt);
      const float snew = TS ? tile_shift(mt, mnew) : mnew;
      // a column whose scores so far are all -inf keeps -inf; shift it by 0
      // (swvr/chunked.py:98-99)
      const float shift = snew == kNegInf ? 0.f : snew;
      const float alpha = fast_exp((TS ? sh[ft] : m[ft]) - shift);
      float rs = 0.f;
#pragma unroll
      for (int fv = 0; fv < FV; ++fv)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pv = fast_exp(sacc[fv][ft][r] - shift);
          sacc[fv][ft][r] = pv;
          rs += pv;
        }
      rs = wave_sum32(rs);
      l[ft] = TS ? shifted_sum(l[ft], m[ft], rs, shift, mnew) : l[ft] * alpha + rs;
      m[ft] = mnew;
      if (TS) sh[ft] = snew;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][ft][r] *= alpha;
    }

    // ---- acc^T[d][token] += E^T[d][v] P^T[v][token]
    // Score registers 8c..8c+7 of a block are the B operand of one k16 step;
    // they hold vocabulary rows 16c + 8(t/4) + 4(lane/32) + t%4, t = 0..7,
    // which the packed E^T tile stores contiguously (pe_row): one read per
    // operand.
    const char* sEe = sE + opaque_zero();  // read base, recomputed per tile
#pragma unroll
    for (int fv = 0; fv < FV; ++fv)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        V8 av[DB];
        const int p0 = wv * WVR + fv * 32 + 8 * (2 * c + (lane >> 5));
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const int d = db * 32 + (lane & 31);
          if constexpr (sizeof(T) == 2) {
            av[db] = *reinterpret_cast<const V8*>(sEe + TE::elem(d, p0));
          } else {
            const float4 lo = *reinterpret_cast<const float4*>(sEe + TE::elem(d, p0));
            const float4 hi = *reinterpret_cast<const float4*>(sEe + TE::elem(d, p0 + 4));
            av[db][0] = lo.x; av[db][1] = lo.y; av[db][2] = lo.z; av[db][3] = lo.w;
            av[db][4] = hi.x; av[db][5] = hi.y; av[db][6] = hi.z; av[db][7] = hi.w;
          }
        }
#pragma unroll
        for (int ft = 0; ft < FT; ++ft) {
          V8 bv;
#pragma unroll
          for (int tt = 0; tt < 8; ++tt) bv[tt] = from_float<T>(sacc[fv][ft][8 * c + tt]);
#pragma unroll
          for (int db = 0; db < DB; ++db) mfma_k16(oacc[db][ft], av[db], bv);
        }
      }
  }

  // ---- partial (m, l, acc) of this wave's vocabulary slice of this split
  // (lane offsets from an opaque lane: computed here, not kept live through the loop)
  const int part = split * C::WV + wv;
  const int ln = lane + opaque_zero();
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    const int n = n0 + wt * WTR + ft * 32 + (ln & 31);
    // to the running maximum; no score yet: 0
    const float f = !TS ? 1.f : m[ft] == kNegInf ? 0.f : fast_exp(sh[ft] - m[ft]);
    if (n < ntok) {
      if (ln < 32) {
        p.part_m[(int64_t)part * ntok + n] = m[ft];
        p.part_l[(int64_t)part * ntok + n] = l[ft];
      }
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int d = db * 32 + c_row(r, ln);
          p.part_acc[((int64_t)part * DP + d) * ntok + n] = oacc[db][ft][r] * f;
        }
    }
  }
}

// Forward for D = 128 and 256 (2-byte dtypes): E^T is not pinned in LDS.  Per
// vocabulary tile the ring carries the K-slices of W and h (-> S^T), then the
// DP / 32 D-slices of the tile's packed E^T (32 x BV each, 16 KB), so the LDS
// holds only the ring: 256 vocabulary rows x 128 tokens per workgroup of 8
// waves (2 vocabulary halves x 4 token quarters, 128 x 32 each); at D = 256
// that is twice the tile a pinned E^T tile would leave room for (85 flop per
// byte of operand traffic instead of 64).  Each of the ring's 3 stages holds two slices (48 KB: two
// K-slices, or two D-slices), so the wait + barrier that publishes a stage
// comes once per 128 MFMAs of the workgroup, as in the 256 x 256 tile of the
// narrow forward.  The bias of a tile is loaded with its first K-slices into a
// double-buffered strip.
template <class T, int DP>
__global__ __launch_bounds__((FwdTile<T, DP>::NT)) void fwd_stream_kernel(FwdParams p) {
  typedef FwdTile<T, DP> C;
  typedef typename Vec8<T>::type V8;
  constexpr int kBK = SliceK<T>::value;
  constexpr int BV = C::BV, BM = C::BM, NT = C::NT;
  constexpr int NS = 3, P = 2;  // ring stages, slices per stage
  constexpr int WVR = BV / C::WV, WTR = BM / C::WT;  // rows per wave
  typedef PackedKLoader<T, BV, kBK, NT> TA;  // W rows of the vocabulary tile (packed)
  typedef PackedKLoader<T, BM, kBK, NT> TB;  // h rows of the token block (packed)
  constexpr int DS = 32;                     // E^T rows (embedding columns) per D-slice
  typedef KTile<T, DS, BV, NT> TE;           // one D-slice of the packed E^T tile, pe_row order
  constexpr int SB1 = TA::BYTES + TB::BYTES; // one slice
  constexpr int SB = P * SB1;                // one stage
  constexpr int L1 = TA::NI + TB::NI;        // loads per thread per slice (E^T slices padded to it)
  constexpr int L = P * L1;                  // per stage
  static_assert(sizeof(T) == 2 && DP % (DS * P) == 0 && TE::BYTES <= SB1 && TE::NI <= L1, "E^T slices fit");
  static_assert(L1 * NT * 16 == SB1, "a slice's loads fill its bytes");
  static_assert(!TA::PARTIAL && !TB::PARTIAL && !TE::PARTIAL, "whole loads");
  constexpr int FV = WVR / 32, FT = WTR / 32;  // 32x32 blocks per wave
  constexpr int DB = DP / 32, ND = DP / DS, NE = ND / P;

  __shared__ __attribute__((aligned(1024))) char smem[NS * SB + 2 * BV * 4];
  const float* const sBias = reinterpret_cast<const float*>(smem + NS * SB);  // [2][BV]

  const int lane = lane_id(), w = wave_id();
  const int wv = w / C::WT, wt = w % C::WT;
  int n_tb = p.n_tb, n_split = p.n_split, ntok = p.N;  // ntok: token rows of a partial
  if (p.n_act) {
    n_tb = p.n_act[3];
    n_split = p.n_act[4];
    if ((int)blockIdx.x >= n_tb * n_split) return;
    ntok = n_tb * BM;
  }
  int split, tb;
  // per XCD, 2 vocabulary splits x 16 token blocks at D = 256, 1 x 32 at D = 128 (each 1-2% faster
  // than the other there)
  grouped_tile<DP == 128 ? 1 : 2>(blockIdx.x, n_split, n_tb, &split, &tb);
  const int n0 = tb * BM;
  const int vt_begin = (int)((int64_t)split * p.n_vt / n_split);
  const int vt_end = (int)((int64_t)(split + 1) * p.n_vt / n_split);
  const T* Ep = static_cast<const T*>(p.Ep);

  float m[FT], sh[FT], l[FT];  // running maximum, which l is relative to; the shift acc is relative to
  f32x16_t oacc[DB][FT];
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    m[ft] = sh[ft] = kNegInf;
    l[ft] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db][ft] = zero16();
  }

  const int nk = max(1, (p.K + kBK - 1) / kBK);  // K = 0: one all-zero slice (bias-only scores)
  const int nkst = (nk + P - 1) / P;             // K-stages per tile; an odd nk leaves a zero slice
  const int n_tiles = vt_end - vt_begin;
  const int per_tile = nkst + NE;
  const int total = n_tiles * per_tile;
  const uint32_t lds0 = lds_addr(smem);
  const uint32_t ldsB = lds0 + NS * SB;
  TA ta;
  ta.setup(p.Wp, vt_begin * BV, p.hS);
  TB tbh;
  tbh.setup(p.hp, n0, p.hS);
  TE te;
  te.setup(Ep, BV, DS, BV);
  const rsrc_t r_none = make_rsrc(nullptr);
  auto zero_fill = [&](int from, uint32_t st) {  // zero-filling loads from..L1-1 of a slice
#pragma unroll
    for (int i = 0; i < L1; ++i)
      if (i >= from) dma_batch1(r_none, kOOB, st + i * NT * 16 + w * 1024);
  };
  // issue cursor over the walk: stage `issued` is (tile is_tile, sub-stage
  // is_sub) into slot is_slot; sub-stages 0..nkst-1 hold K-slices 2 sub and
  // 2 sub + 1, nkst.. D-slices 2 e and 2 e + 1 of the tile's E^T
  int issued = 0, is_tile = 0, is_sub = 0, is_slot = 0;
  auto issue_next = [&]() {
    if (issued >= total) return;
    const uint32_t st = lds0 + is_slot * SB;
    const int v0 = (vt_begin + is_tile) * BV;
    if (is_sub < nkst) {
      if (is_sub == 0) {
        ta.rebase(v0);
        // the tile's bias into strip (tile & 1), ahead of its slices (wave 0)
        if ((int)threadIdx.x * 16 < BV * 4)
          dma_batch1(make_rsrc(p.biasp + v0), (uint32_t)threadIdx.x * 16, ldsB + (is_tile & 1) * (BV * 4) + w * 1024);
      }
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const int k = P * is_sub + s;
        const uint32_t ss = st + s * SB1;
        if (k < nk) {
          ta.issue(ss, k * kBK);
          tbh.issue(ss + TA::BYTES, k * kBK);
        } else {
          zero_fill(0, ss);
        }
      }
    } else {
      // rows d0 .. d0 + 31 of the tile's E^T [DP][BV]: one contiguous run per D-slice
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const int ds = P * (is_sub - nkst) + s;
        const uint32_t ss = st + s * SB1;
        te.base = reinterpret_cast<const char*>(Ep + ((int64_t)v0 * DP + (int64_t)ds * DS * BV));
        te.issue(ss, 0);
        zero_fill(TE::NI, ss);
      }
    }
    ++issued;
    if (++is_sub == per_tile) {
      is_sub = 0;
      ++is_tile;
    }
    is_slot = is_slot == NS - 1 ? 0 : is_slot + 1;
  };
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue_next();

  f32x16_t sacc[FV][FT];
  Ring<NS> ring{NS - 1, total};  // the first publish_next() moves to stage 0, slot 0
  for (int tile = 0; tile < n_tiles; ++tile) {
    // first K-stage of the tile; every wave has also finished the previous
    // tile's E^T slices, and its bias strip is free again
    ring.template publish_next<L>();
#pragma unroll
    for (int fv = 0; fv < FV; ++fv)
#pragma unroll
      for (int ft = 0; ft < FT; ++ft) sacc[fv][ft] = zero16();
    tile_reduce_multi<T, kBK, P, L>(sacc, ta, tbh, smem, SB, SB1, ring, nkst, wv * WVR, wt * WTR, issue_next);

    // ---- scores -> running softmax of this wave's slice of the tile
    const float* sB = sBias + (tile & 1) * BV + opaque_zero();
    float mx[FT];
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) mx[ft] = kNegInf;
#pragma unroll
    for (int fv = 0; fv < FV; ++fv)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        // registers 4g..4g+3 hold rows 8g + 4(lane/32) + 0..3 of the block
        const int row = wv * WVR + fv * 32 + 8 * g + (lane >> 5) * 4;
        const float4 b4 = *reinterpret_cast<const float4*>(sB + row);
        const float bb[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int ft = 0; ft < FT; ++ft) {
            const float x = fmaf(sacc[fv][ft][4 * g + i], p.scale, bb[i]);  // rounded as the backward rounds it
            sacc[fv][ft][4 * g + i] = x;
            mx[ft] = fmaxf(mx[ft], x);
          }
      }
#pragma unroll
    for (int ft = 0; ft < FT; ++ft) {
      const float mt = wave_max32(mx[ft]), mnew = fmaxf(m[ft], mt);
      const float snew = tile_shift(mt, mnew);
      // a column whose scores so far are all -inf keeps -inf; shift it by 0
      // (swvr/chunked.py:98-99)
      const float shift = snew == kNegInf ? 0.f : snew;
      const float alpha = fast_exp(sh[ft] - shift);
      sh[ft] = snew;
      float rs = 0.f;
#pragma unroll
      for (int fv = 0; fv < FV; ++fv)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float pv = fast_exp(sacc[fv][ft][r] - shift);
          sacc[fv][ft][r] = pv;
          rs += pv;
        }
      l[ft] = shifted_sum(l[ft], m[ft], wave_sum32(rs), shift, mnew);
      m[ft] = mnew;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][ft][r] *= alpha;
    }

    // ---- acc^T[d][token] += E^T[d][v] P^T[v][token], two D-slices per stage.
    // Score registers 8c..8c+7 of a block are the B operand of one k16 step;
    // they hold vocabulary rows 16c + 8(t/4) + 4(lane/32) + t%4, which the
    // packed E^T stores contiguously (pe_row): one read per operand.
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      ring.template publish_next<L>();
      issue_next();
      const int d = lane & 31;
#pragma unroll
      for (int s = 0; s < P; ++s) {
        const char* sEe = smem + ring.slot * SB + s * SB1 + opaque_zero();
#pragma unroll
        for (int fv = 0; fv < FV; ++fv)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const int p0 = wv * WVR + fv * 32 + 8 * (2 * c + (lane >> 5));
            const V8 av = *reinterpret_cast<const V8*>(sEe + TE::elem(d, p0));
#pragma unroll
            for (int ft = 0; ft < FT; ++ft) {
              V8 bv;
#pragma unroll
              for (int tt = 0; tt < 8; ++tt) bv[tt] = from_float<T>(sacc[fv][ft][8 * c + tt]);
              mfma_k16(oacc[P * e + s][ft], av, bv);
            }
          }
      }
    }
  }

  // ---- partial (m, l, acc) of this wave's vocabulary slice of this split
  const int part = split * C::WV + wv;
  const int ln = lane + opaque_zero();
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) {
    const int n = n0 + wt * WTR + ft * 32 + (ln & 31);
    const float f = m[ft] == kNegInf ? 0.f : fast_exp(sh[ft] - m[ft]);  // to the running maximum; no score yet: 0
    if (n < ntok) {
      if (ln < 32) {
        p.part_m[(int64_t)part * ntok + n] = m[ft];
        p.part_l[(int64_t)part * ntok + n] = l[ft];
      }
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int d = db * 32 + c_row(r, ln);
          p.part_acc[((int64_t)part * DP + d) * ntok + n] = oacc[db][ft][r] * f;
        }
    }
  }
}

// Merge partial softmaxes in a fixed order (O rows ldo apart): O = sum_p acc_p e^(m_p - M) /
// sum_p l_p e^(m_p - M), LSE = M + log(...).  A row with every score -inf ends
// with M = -inf, L = 0: O = NaN and LSE = -inf, as swvr/chunked.py:105 gives.
// Partial p of (row n, column d) of acc sits at p * sp + d * sd + n * sn, so
// one kernel merges the forward's own partials ([n_part][DP][N], token
// fastest) and vocabulary shards' ([S][N][D]).  With m_out set, it writes the
// merged partial (M, L and the unnormalised acc, [N][D]) instead of O / LSE.
// A thread merges DT consecutive columns of a row (n fastest over the threads), so the row's m and l
// are read and exponentiated once per DT columns; the d = 0 threads also write their row's LSE (or M, L).
//
// Merge over n_part partials by a workgroup of G thread rows x 256 / G columns (G = 32: x 32): m / l
// of partial q at pm[q * sml] / pl[q * sml], its acc of column i at pa[q * sp + i * sd] (i < nd).  Each
// thread row merges a contiguous run of the partials, loads going out in batches of 8 ahead of the
// arithmetic, and the runs' sums are added in run order, so the result has a fixed order.
//   G = 32, DT = 1: few elements and many partials, where the merge is bound by the latency of a
//   run's loads: one token's 594 partials take 11 us (102 us in one run per element).
//   G = 4, DT = 4: many partials, many elements: 2048 tokens, D = 128, 128 partials 74 us (G = 1: 96).
//   G = 1, DT = 4: few partials: bound by their bytes.  16384 tokens, D = 64, 32 partials 50 us
//   (G = 4: 55; one column per thread, with four loads of m and l for each of acc: 79).
template <int G>
struct MergeWidth {
  static constexpr int value = G == 32 ? 32 : 256 / G;
};

template <int G, int DT>
__device__ __forceinline__ void merge_partials(const float* __restrict__ pm, const float* __restrict__ pl,
                                               const float* __restrict__ pa, int n_part, int64_t sml, int64_t sp,
                                               int64_t sd, bool live, int nd, float* M_, float* L_, float (&a_)[DT]) {
  constexpr int B = 8, CW = MergeWidth<G>::value;
  __shared__ float sm[G][CW], sl[G][CW], sa[DT][G][CW];
  const int g = threadIdx.x / CW, c = threadIdx.x % CW;
  const int run = (n_part + G - 1) / G;
  const int q_begin = min(n_part, g * run), q_end = live ? min(n_part, q_begin + run) : q_begin;
  float M = kNegInf;
  for (int q0 = q_begin; q0 < q_end; q0 += B) {
    float x[B];
#pragma unroll
    for (int u = 0; u < B; ++u) x[u] = q0 + u < q_end ? pm[(q0 + u) * sml] : kNegInf;
#pragma unroll
    for (int u = 0; u < B; ++u) M = fmaxf(M, x[u]);
  }
  if constexpr (G > 1) {
    sm[g][c] = M;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < G; ++i) M = fmaxf(M, sm[i][c]);
  }
  const float shift = M == kNegInf ? 0.f : M;
  float L = 0.f;
#pragma unroll
  for (int i = 0; i < DT; ++i) a_[i] = 0.f;
  for (int q0 = q_begin; q0 < q_end; q0 += B) {
    float xm[B], xl[B], xa[B][DT];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const bool in = q0 + u < q_end;
      xm[u] = in ? pm[(q0 + u) * sml] : 0.f;
      xl[u] = in ? pl[(q0 + u) * sml] : 0.f;
#pragma unroll
      for (int i = 0; i < DT; ++i) xa[u][i] = in && i < nd ? pa[(q0 + u) * sp + i * sd] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (q0 + u < q_end) {
        const float wq = expf(xm[u] - shift);
        L += xl[u] * wq;
#pragma unroll
        for (int i = 0; i < DT; ++i) a_[i] += xa[u][i] * wq;
      }
  }
  if constexpr (G > 1) {
    sl[g][c] = L;
#pragma unroll
    for (int i = 0; i < DT; ++i) sa[i][g][c] = a_[i];
    __syncthreads();
    L = 0.f;
#pragma unroll
    for (int j = 0; j < G; ++j) L += sl[j][c];
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      a_[i] = 0.f;
#pragma unroll
      for (int j = 0; j < G; ++j) a_[i] += sa[i][j][c];
    }
  }
  *M_ = M;
  *L_ = L;
}

// Thread rows G of a merge (DT = 1 with 32, else 4).  4 also for 16 to 63 partials whose one-row merge
// would leave CUs without a workgroup (1100 tokens, D = 100, 48 partials: the call 142 -> 135 us; 2500
// tokens, D = 300, whose last pass merges 44 columns: 572 -> 564; 2000 tokens, D = 200 is past the line).
int combine_rows(int64_t elements, int n_part) {
  if (n_part < 16) return 1;
  return elements <= 65536 ? 32 : n_part >= 64 || elements <= 4 * 256 * 256 ? 4 : 1;
}

template <int G, int DT>
__global__ __launch_bounds__(G * MergeWidth<G>::value) void fwd_combine_kernel(
    const float* __restrict__ part_m, const float* __restrict__ part_l, const float* __restrict__ part_acc, int n_part,
    int N, int D, int64_t sp, int64_t sd, int64_t sn, float* __restrict__ O, int64_t ldo, float* __restrict__ lse,
    float* __restrict__ m_out, float* __restrict__ l_out, const float* __restrict__ weight) {
  constexpr int CW = MergeWidth<G>::value;
  const int64_t e = (int64_t)blockIdx.x * CW + threadIdx.x % CW;
  const int nb = D > 0 ? (D + DT - 1) / DT : 1;
  const bool live = e < (int64_t)N * nb;
  const int d = live ? (int)(e / N) * DT : 0, n = live ? (int)(e % N) : 0;
  float M, L, a[DT];
  merge_partials<G, DT>(part_m + n, part_l + n, part_acc + d * sd + n * sn, n_part, N, sp, sd, live, D - d, &M, &L, a);
  if (!live || threadIdx.x >= CW) return;
  const bool zero = weight && weight[n] == 0.f;  // finite values of a zero-weight token: 0
#pragma unroll
  for (int i = 0; i < DT; ++i)
    if (d + i < D) {
      const float o = m_out ? a[i] : a[i] / L;
      O[(int64_t)n * ldo + d + i] = zero && __builtin_isfinite(o) ? 0.f : o;
    }
  if (d == 0) {
    if (m_out) {
      m_out[n] = M;
      l_out[n] = L;
    } else {
      const float x = M + logf(L);
      lse[n] = zero && __builtin_isfinite(x) ? 0.f : x;
    }
  }
}

// fwd_combine_kernel of the active-token forward: token n merges the partials
// of its position inv[n] (WV x n_split partials of n_tb x BM rows each, n_tb and
// n_split at n_act[3], n_act[4]); a token outside the active set gets an O row
// of 0 and LSE 0.
template <int G, int DT>
__global__ __launch_bounds__(G * MergeWidth<G>::value) void fwd_combine_active_kernel(
    const float* __restrict__ part_m, const float* __restrict__ part_l, const float* __restrict__ part_acc,
    const int* __restrict__ inv, const int* __restrict__ n_act, int BM, int WV, int N, int D, int DP,
    float* __restrict__ O, int64_t ldo, float* __restrict__ lse) {
  constexpr int CW = MergeWidth<G>::value;
  const int64_t e = (int64_t)blockIdx.x * CW + threadIdx.x % CW;
  const int nb = D > 0 ? (D + DT - 1) / DT : 1;
  const bool in = e < (int64_t)N * nb;
  const int d = in ? (int)(e / N) * DT : 0, n = in ? (int)(e % N) : 0;
  const int q = in ? inv[n] : -1, qc = q < 0 ? 0 : q;
  const int tb = n_act[3], sp = n_act[4];
  const int64_t rows = (int64_t)tb * BM;
  float M, L, a[DT];
  merge_partials<G, DT>(part_m + qc, part_l + qc, part_acc + d * rows + qc, WV * sp, rows, (int64_t)DP * rows, rows,
                        q >= 0, D - d, &M, &L, a);
  if (!in || threadIdx.x >= CW) return;
#pragma unroll
  for (int i = 0; i < DT; ++i)
    if (d + i < D) O[(int64_t)n * ldo + d + i] = q >= 0 ? a[i] / L : 0.f;
  if (d == 0) lse[n] = q >= 0 ? M + logf(L) : 0.f;
}

// Workgroups of a merge of N rows x D columns.
template <int G, int DT>
unsigned combine_blocks(int N, int D) {
  constexpr int CW = MergeWidth<G>::value;
  return (unsigned)(((int64_t)N * (D > 0 ? (D + DT - 1) / DT : 1) + CW - 1) / CW);
}

template <class F>
void dispatch_combine(int64_t elements, int n_part, F&& go) {
  switch (combine_rows(elements, n_part)) {
    case 1: go(std::integral_constant<int, 1>(), std::integral_constant<int, 4>()); break;
    case 4: go(std::integral_constant<int, 4>(), std::integral_constant<int, 4>()); break;
    default: go(std::integral_constant<int, 32>(), std::integral_constant<int, 1>()); break;
  }
}

// Merge launch over n_part partials of N rows x D columns (see fwd_combine_kernel).
hipError_t launch_combine(const float* m, const float* l, const float* acc, int n_part, int N, int D, int64_t sp,
                          int64_t sd, int64_t sn, float* O, int64_t ldo, float* lse, float* m_out, float* l_out,
                          const float* weight, hipStream_t stream) {
  if (N == 0) return hipSuccess;
  timing_begin(kKindFwdCombine, stream);
  auto go = [&](auto g, auto dt) {
    constexpr int G = decltype(g)::value, DT = decltype(dt)::value;
    fwd_combine_kernel<G, DT><<<combine_blocks<G, DT>(N, D), G * MergeWidth<G>::value, 0, stream>>>(
        m, l, acc, n_part, N, D, sp, sd, sn, O, ldo, lse, m_out, l_out, weight);
  };
  dispatch_combine((int64_t)N * D, n_part, go);
  timing_end(kKindFwdCombine, stream);
  return hipGetLastError();
}

// The active-token forward's token blocks and vocabulary splits from the count, into n_act[3],
// n_act[4]: once per call, so every kernel uses the same values and the host needs no copy of them.
// The launch has room for twice the all-token tiling's workgroups, of which the first n_tb x n_split
// work; the split is the one fwd_span ends soonest with (the smaller on a tie).  One wave, a candidate
// per lane.
__global__ __launch_bounds__(64) void fwd_active_grid_kernel(int* __restrict__ n_act, int BM, int n_tb_max,
                                                             int n_split0, int n_vt, FwdCost cost) {
  int tb = (n_act[0] + BM - 1) / BM, pick = 1;
  if (tb > n_tb_max) tb = n_tb_max;
  double best = 1e300;
  if (tb > 0) {
    const int hi = active_splits_max(tb, n_tb_max, n_split0, n_vt);
    for (int s = 1 + (int)threadIdx.x; s <= hi; s += 64) {
      const double t = fwd_span(tb, n_vt, s, cost);
      if (t < best) {
        best = t;
        pick = s;
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double t = __shfl_xor(best, o);
    const int q = __shfl_xor(pick, o);
    if (t < best || (t == best && q < pick)) {
      best = t;
      pick = q;
    }
  }
  if (threadIdx.x == 0) {
    n_act[3] = tb;
    n_act[4] = pick;
  }
}

// Flags of the active-token forward's parameter checks, bad[0..1]:
// bad[0] = 1 when the logit scale is not finite, E holds an infinity or a NaN
// or the bias a NaN or +inf (W is checked as it is packed); bad[1] starts at 1
// when there is a bias (or no vocabulary) and drops to 0 once a bias entry
// above -inf is seen (every entry -inf makes every score -inf).
__global__ __launch_bounds__(64) void fwd_flags_init_kernel(int* __restrict__ bad, int scale_bad, int bias_all_neg) {
  if (threadIdx.x == 0) {
    bad[0] = scale_bad;
    bad[1] = bias_all_neg;
  }
}

// Grid-stride scan of E's V x D elements and the bias for fwd_flags_init_kernel's
// words.  Every store writes the same value, so the words end the same
// whatever the order of the stores.
template <class T>
__global__ __launch_bounds__(256) void fwd_param_scan_kernel(const T* __restrict__ E, int64_t lde, int V, int D,
                                                             const float* __restrict__ bias, int* __restrict__ bad) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool nf = false, live = false;
  if (D > 0)
    for (int64_t e = t0; e < (int64_t)V * D; e += stride) {
      const int64_t v = e / D;
      nf |= !__builtin_isfinite((float)E[v * lde + (e - v * D)]);
    }
  if (bias)
    for (int64_t v = t0; v < V; v += stride) {
      const float b = bias[v];
      nf |= b != b || b == kPosInf;
      live |= b > kNegInf;
    }
  if (__syncthreads_or(nf) && threadIdx.x == 0) bad[0] = 1;
  if (__syncthreads_or(live) && threadIdx.x == 0) bad[1] = 0;
}

// flag[n] = 1 for a token of the active-token forward: a non-zero (or NaN)
// weight, an h row holding an infinity or a NaN (in the compute dtype), or a
// flagged parameter (bad[0] or bad[1]: then every token).  One wave per token;
// only a zero-weight token's row is read, in 16-byte chunks.
template <class Src, class T>
__global__ __launch_bounds__(256) void fwd_active_flag_kernel(const float* __restrict__ weight,
                                                              const Src* __restrict__ h, int64_t ldh, int N, int K,
                                                              const int* __restrict__ bad, int* __restrict__ flag) {
  const int n = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (n >= N) return;
  const int lane = lane_id();
  bool act = weight[n] != 0.f || bad[0] != 0 || bad[1] != 0;  // NaN != 0
  if (!act) {  // uniform over the wave
    constexpr int CE = 16 / (int)sizeof(T);
    bool nf = false;
    for (int c = lane; c < K / CE; c += 64)
      nf |= chunk_nonfinite<T>(load_chunk<Src, T>(h + (int64_t)n * ldh + (int64_t)c * CE));
    act = __ballot(nf) != 0;
  }
  if (lane == 0) flag[n] = act ? 1 : 0;
}

template <class T, int DP, bool F8 = false>
hipError_t launch_tile(const FwdPlan& plan, const FwdParams& p, hipStream_t stream) {
  typedef FwdCfg<T, DP, F8> C;
  if (plan.BV != C::BV || plan.BM != C::BM) return hipErrorInvalidValue;
  // the active-token forward may use up to twice the all-token grid (active_splits_max); the rest exit at once
  const int blocks = plan.n_tb * plan.n_split * (p.n_act ? 2 : 1);
  timing_begin(kKindFwdTile, stream);
  if constexpr (!F8 && FwdTile<T, DP>::stream_e)
    fwd_stream_kernel<T, DP><<<blocks, C::NT, 0, stream>>>(p);
  else
    fwd_tile_kernel<T, DP, F8><<<blocks, C::NT, 0, stream>>>(p);
  timing_end(kKindFwdTile, stream);
  return hipGetLastError();
}

template <class T>
hipError_t dispatch_dp(const FwdPlan& plan, const FwdParams& p, hipStream_t stream) {
  switch (plan.DP) {
    case 32: return launch_tile<T, 32>(plan, p, stream);
    case 64: return launch_tile<T, 64>(plan, p, stream);
    case 128: return launch_tile<T, 128>(plan, p, stream);
    case 256:
      if constexpr (sizeof(T) == 2) return launch_tile<T, 256>(plan, p, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

hipError_t dispatch_dp_f8(const FwdPlan& plan, const FwdParams& p, hipStream_t stream) {
  switch (plan.DP) {
    case 32: return launch_tile<bf16_t, 32, true>(plan, p, stream);
    case 64: return launch_tile<bf16_t, 64, true>(plan, p, stream);
    case 128: return launch_tile<bf16_t, 128, true>(plan, p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <class T, int DP>
void tile_get(int* BV, int* BM, int* WV) {
  *BV = FwdTile<T, DP>::BV;
  *BM = FwdTile<T, DP>::BM;
  *WV = FwdTile<T, DP>::WV;
}

template <class T>
void tile_of(int DP, int* BV, int* BM, int* WV) {
  switch (DP) {
    case 32: tile_get<T, 32>(BV, BM, WV); break;
    case 64: tile_get<T, 64>(BV, BM, WV); break;
    case 128: tile_get<T, 128>(BV, BM, WV); break;
    default: tile_get<T, 256>(BV, BM, WV); break;
  }
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// E^T tiles and the bias of one D-slice (p.E, p.D: the slice's columns).
template <class T>
hipError_t pack_et(const FwdParams& p, const FwdPlan& plan, hipStream_t stream) {
  constexpr int BV = FwdTile<T, 32>::BV;  // one per dtype
  if (plan.BV != BV) return hipErrorInvalidValue;
  const int64_t blocks = (int64_t)plan.n_vt * (plan.DP / 32);
  if (blocks == 0) return hipSuccess;
  timing_begin(kKindPack, stream);
  pack_et_kernel<T, BV><<<(unsigned)blocks, 256, 0, stream>>>(
      static_cast<const T*>(p.E), p.lde, p.bias, p.V, p.D, plan.V_pad, plan.DP,
      const_cast<T*>(static_cast<const T*>(p.Ep)), const_cast<float*>(p.biasp), p.h_scale, p.w_scale, p.scale);
  timing_end(kKindPack, stream);
  return hipGetLastError();
}

// h and W in their tiles' LDS image, once per call.
template <class T>
hipError_t pack(const FwdParams& p, const FwdPlan& plan, hipStream_t stream) {
  timing_begin(kKindPack, stream);
  hipError_t e = hipSuccess;
  T* const hp = const_cast<T*>(static_cast<const T*>(p.hp));
  T* const Wp = const_cast<T*>(static_cast<const T*>(p.Wp));
  if (e == hipSuccess)
    e = pack_src<T>(p.h, p.h_f32, p.ldh, p.N, p.K, plan.hS, plan.N_pad, hp, stream);
  if (e == hipSuccess)
    e = pack_src<T>(p.W, p.w_f32, p.ldw, p.V, p.K, plan.hS, plan.V_pad, Wp, stream);
  timing_end(kKindPack, stream);
  return e;
}

}  // namespace

namespace {

// Vocabulary splits of a forward whose workgroups hold a CU each, from the rule's n_split: the split
// that fwd_span ends soonest with, if that is 3% sooner.
// 2500 tokens on V = 50021, K = 768, D = 256 (20 token blocks): 52 splits are 1040 workgroups, a fifth
// round for 16 of them, and the pass took 436 us; 25 make 2 whole rounds, 356 us.
int balanced_split(int64_t n_tb, int64_t n_vt, int n_split, int s_min, FwdCost cost) {
  auto span = [&](int64_t s) { return fwd_span(n_tb, n_vt, s, cost); };
  double best = 0.97 * span(n_split);
  const int64_t cap = n_vt / 2 > 1 ? n_vt / 2 : 1, hi = 6 * (int64_t)kFwdRound / n_tb;
  int pick = n_split;
  for (int64_t s = s_min; s <= hi && s <= cap; ++s)
    if (span(s) < best) {
      best = span(s);
      pick = (int)s;
    }
  return pick;
}

// The few-token forward (fwd_few.hip) serves calls of up to this many tokens.  Measured, the whole
// call in us, general forward -> few-token forward (K, V, D):
//            N =       64         256         512         1024
//   bf16 2560, 151936, 64    552 -> 168  569 -> 315   700 -> 570  1080 -> 1062
//   bf16 1024, 32000, 64     106 -> 54   108 -> 54    114 -> 75    137 -> 120
//   bf16 4096, 128256, 128   666 -> 228  784 -> 409  1049 -> 748  1471 -> 1414
//   bf16 768, 50021, 256      91 -> 54   118 -> 96    159 -> 133   271 -> 224
//   fp32 2560, 32000, 64     333 -> 145  543 -> 401   966 -> 786  1792 -> 1541
//   autocast 2048, 65536, 128 254 -> 146 269 -> 194   346 -> 308   493 -> 545
// Towards 1024 tokens W is read by enough token blocks for the packing to pay, under autocast before
// that (an fp32 W's operands are rounded at every read); one line for both, so that an fp32 W gives the
// bits of one cast beforehand.  fp32 calls take it at any size (8192 tokens: 13.3 -> 10.7 ms).
constexpr int64_t kFewTokens = 768;
// A weighted loss's forward of up to this many tokens computes all of them, zero weight or not: the
// one pass over W costs no more than the passes that find the active ones do with W to be searched for
// non-finite values first.  Past it the few-token kernel runs over the active tokens' positions.
constexpr int64_t kFewTokensActive = 512, kFewTokensActiveF32 = 128;

// Whether a call is planned for the few-token forward.
bool takes_few(int dtype, int64_t N) { return dtype != kFP8 && (dtype == kF32 || N <= kFewTokens); }

// Tile, split and workspace (from offset off on) of the few-token forward for one pass of Dw columns:
// vocabulary runs of whole 32-row groups.
void few_plan(int dtype, int64_t N, int64_t V, int64_t Dw, bool active, size_t off, FwdPlan* plan) {
  plan->few = takes_few(dtype, N);
  if (!plan->few) return;
  const bool two = dtype != kF32;
  plan->few_DP = !two && Dw <= 32 ? 32 : Dw <= 64 ? 64 : Dw <= 128 ? 128 : 256;
  const int nb_max = plan->few_DP <= 128 ? 4 : 2;
  plan->few_NB = N <= 32 ? 1 : N <= 64 || nb_max == 2 ? 2 : 4;
  plan->few_tb = (int)((N + 32 * plan->few_NB - 1) / (32 * plan->few_NB));
  const int64_t grp = (V + 31) / 32;
  plan->few_split = few_runs(plan->few_tb, grp);
  // with the active tokens counted on the device: any smaller number of token blocks, in at most
  // kFewRounds rounds or one run each
  const int64_t wgs = active ? (plan->few_tb > kFewRounds * kFwdRound ? plan->few_tb : kFewRounds * kFwdRound)
                             : (int64_t)plan->few_tb * plan->few_split;
  const int64_t cap = (int64_t)plan->few_tb * few_runs_max(1, grp);
  plan->few_wgs = (int)(wgs < cap ? wgs : cap);
  const size_t part = (size_t)plan->few_wgs * 32 * plan->few_NB * 4;
  const size_t tb = two ? 2 : 4;
  const int sk = two ? SliceK<bf16_t>::value : SliceK<float>::value;
  plan->few_m = off;
  off += align256(part);
  plan->few_l = off;
  off += align256(part);
  plan->few_acc = off;
  off += align256(part * plan->few_DP);
  plan->few_hp = off;
  off += align256((size_t)plan->N_pad * plan->hS * sk * tb);
  plan->few_E = off;  // aligned copy of E's rows, for a caller's E that is not
  off += align256((size_t)plan->V_pad * plan->few_DP * tb);
  if (off > plan->ws_bytes) plan->ws_bytes = off;
}

// Whether the call takes the few-token forward: planned so, and 32-bit offsets reach 128 rows of W and E.
// Rows 16 MB and more apart go to the general kernels, whatever the type and the number of tokens; the
// workspace, sized before the strides are known, holds either route.
bool few_fits(const FwdPlan& plan, const FwdParams& p, int dtype) {
  const int64_t esz = dtype == kF32 ? 4 : 2, wsz = p.w_f32 ? 4 : esz, lim = (int64_t)1 << 31;
  return plan.few && p.ldw * wsz * 128 < lim && p.lde * esz * 128 < lim;
}

// Workspace pointers and sizes of the few-token kernel's parameters.
FwdFewParams few_params(const FwdPlan& plan, const FwdParams& p, char* ws) {
  FwdFewParams q{};
  q.hp = ws + plan.few_hp;
  q.hS = plan.hS;
  q.W = p.W;
  q.ldw = p.ldw;
  q.w_f32 = p.w_f32;
  q.bias = p.bias;
  q.scale = p.scale;
  q.N = p.N;
  q.K = p.K;
  q.V = p.V;
  q.DP = plan.few_DP;
  q.NB = plan.few_NB;
  q.n_tb = plan.few_tb;
  q.n_split = plan.few_split;
  q.n_wg = plan.few_tb * plan.few_split;
  q.part_m = reinterpret_cast<float*>(ws + plan.few_m);
  q.part_l = reinterpret_cast<float*>(ws + plan.few_l);
  q.part_acc = reinterpret_cast<float*>(ws + plan.few_acc);
  return q;
}

// One pass of the few-token kernel over E's columns from d0 on (E's rows as 16-byte chunks: the
// caller's, or an aligned copy).
template <class T>
hipError_t few_pass(int dtype, const FwdPlan& plan, const FwdParams& p, int d0, FwdFewParams q, char* ws,
                    hipStream_t stream) {
  const T* E = static_cast<const T*>(p.E) + d0;
  q.D = p.D - d0 < plan.DS ? p.D - d0 : plan.DS;
  q.E = E;
  q.lde = p.lde;
  if (p.V > 0 && q.D > 0 && !(rows_vec16(E, p.lde) && q.D % (16 / (int)sizeof(T)) == 0)) {
    T* const Ep = reinterpret_cast<T*>(ws + plan.few_E);
    const int64_t n = (int64_t)p.V * (plan.few_DP / 8);
    timing_begin(kKindPack, stream);
    pack_vocab_kernel<T><<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(
        E, p.lde, nullptr, p.V, q.D, p.V, plan.few_DP, rows_vec16(E, p.lde), Ep, nullptr);
    timing_end(kKindPack, stream);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    q.E = Ep;
    q.lde = plan.few_DP;
    q.D = plan.few_DP;
  }
  return fwd_few_launch(dtype, q, stream);
}

// With weight set (a weighted loss), a finite O element or LSE of a zero-weight token is written as 0.
template <class T>
hipError_t fwd_few_typed(int dtype, const FwdPlan& plan, const FwdParams& p, const float* weight, char* ws, float* O,
                         float* lse, float* m_out, float* l_out, hipStream_t stream) {
  const FwdFewParams q = few_params(plan, p, ws);
  timing_begin(kKindPack, stream);
  hipError_t e = pack_src<T>(p.h, p.h_f32, p.ldh, p.N, p.K, plan.hS, plan.N_pad, reinterpret_cast<T*>(ws + plan.few_hp),
                             stream);
  timing_end(kKindPack, stream);
  for (int d0 = 0; e == hipSuccess && d0 < (p.D > 0 ? p.D : 1); d0 += plan.DS) {
    if ((e = few_pass<T>(dtype, plan, p, d0, q, ws, stream)) != hipSuccess) return e;
    const int D = p.D - d0 < plan.DS ? p.D - d0 : plan.DS;
    e = launch_combine(q.part_m, q.part_l, q.part_acc, q.n_split, p.N, D, (int64_t)plan.few_DP * p.N, p.N, 1,
                       O ? O + d0 : nullptr, p.D, lse, m_out, l_out, weight, stream);
  }
  return e;
}

hipError_t fwd_few(int dtype, const FwdPlan& plan, const FwdParams& p, const float* weight, char* ws, float* O,
                   float* lse, float* m_out, float* l_out, hipStream_t stream) {
  switch (dtype) {
    case kBF16: return fwd_few_typed<bf16_t>(dtype, plan, p, weight, ws, O, lse, m_out, l_out, stream);
    case kF16: return fwd_few_typed<f16_t>(dtype, plan, p, weight, ws, O, lse, m_out, l_out, stream);
    default: return fwd_few_typed<float>(dtype, plan, p, weight, ws, O, lse, m_out, l_out, stream);
  }
}

}  // namespace

bool fwd_plan(int dtype, int64_t N, int64_t K, int64_t V, int64_t D, FwdPlan* plan, bool active) {
  (void)K;
  if (active && dtype == kFP8) return false;
  plan->active = active;
  // Widest embedding slice of one pass: 256 (2-byte dtypes), 128 (fp32, e4m3).  A wider D runs
  // in slices of that width, each pass recomputing the same scores for its columns of E.
  const int DS = dtype == kBF16 || dtype == kF16 ? 256 : 128;
  if (dtype == kFP8 && D > DS) return false;
  const int64_t Dw = D < DS ? D : DS;
  const int DP = Dw <= 32 ? 32 : Dw <= 64 ? 64 : Dw <= 128 ? 128 : 256;
  plan->DS = DS;
  plan->n_dslices = D > DS ? (int)((D + DS - 1) / DS) : 1;
  int BV, BM, WV;
  size_t tbytes;
  if (dtype == kF32) {
    if (DP > 128) return false;
    tile_of<float>(DP, &BV, &BM, &WV);
    tbytes = 4;
  } else if (dtype == kBF16 || dtype == kF16) {
    tile_of<bf16_t>(DP, &BV, &BM, &WV);
    tbytes = 2;
  } else if (dtype == kFP8) {
    // K counts byte pairs: the e4m3 rows are packed as bf16 rows of K / 2 elements
    if (DP > 128) return false;
    static_assert(FwdTileF8<128>::BV == FwdTileF8<64>::BV && FwdTileF8<128>::BM == FwdTileF8<64>::BM, "one tile");
    BV = FwdTileF8<64>::BV;
    BM = FwdTileF8<64>::BM;
    WV = DP <= 64 ? FwdTileF8<64>::WV : FwdTileF8<128>::WV;
    tbytes = 2;
  } else {
    return false;
  }
  plan->BV = BV;
  plan->BM = BM;
  plan->DP = DP;
  plan->n_tb = (int)((N + BM - 1) / BM);
  plan->n_vt = (int)((V + BV - 1) / BV);
  plan->V_pad = plan->n_vt * BV;
  // Enough workgroups (one per CU) to fill 256 CUs several times over, at
  // least two vocabulary tiles per split.
  int n_split = 1;
  if (plan->n_tb > 0) {
    // (a call planned for the few-token forward comes here for rows too far apart for it alone: one round)
    const int target = takes_few(dtype, N) ? kFwdRound : 1024;
    n_split = (target + plan->n_tb - 1) / plan->n_tb;
    const int max_split = plan->n_vt / 2 > 1 ? plan->n_vt / 2 : 1;
    if (n_split > max_split) n_split = max_split;
    if (n_split < 1) n_split = 1;
    // (the e4m3 forward's P is relative to the running maximum, so it keeps at least the rule's splits)
    if (!active && tbytes == 2 && !takes_few(dtype, N))
      n_split = balanced_split(plan->n_tb, plan->n_vt, n_split, dtype == kFP8 ? n_split : 1,
                               fwd_cost(K, DP, BM, WV));
  }
  plan->n_split = n_split;
  plan->n_part = WV * n_split;
  plan->WV = WV;
  plan->rem_DP = 0;
  int64_t parts = plan->n_part;  // partials, and partials x columns, the buffers hold: the larger of the passes'
  int64_t part_cols = (int64_t)plan->n_part * DP;
  if (!active && plan->n_dslices > 1 && N > 0) {
    FwdPlan rem;
    fwd_plan(dtype, N, K, V, D - (int64_t)(plan->n_dslices - 1) * DS, &rem);
    if (rem.DP < DP && rem.BV == BV) {
      plan->rem_DP = rem.DP;
      plan->rem_BM = rem.BM;
      plan->rem_tb = rem.n_tb;
      plan->rem_split = rem.n_split;
      plan->rem_part = rem.n_part;
      if (rem.n_part > parts) parts = rem.n_part;
      if ((int64_t)rem.n_part * rem.DP > part_cols) part_cols = (int64_t)rem.n_part * rem.DP;
    }
  }
  // token rows of a partial: N; the active-token forward's partials hold up to
  // 2 x n_tb x n_split workgroups' n_tb x BM positions each (active_splits_max)
  const int64_t NR = active ? 2 * (int64_t)plan->n_tb * BM : N;
  size_t off = 0;
  plan->off_flag = plan->off_idx = plan->off_inv = plan->off_nact = 0;
  if (active) {
    plan->off_flag = off;
    off += align256((size_t)N * 4);
    plan->off_idx = off;
    off += align256((size_t)N * 4);
    plan->off_inv = off;
    off += align256((size_t)N * 4);
    plan->off_nact = off;  // [0] count, [1..2] parameter flags
    off += 256;
  }
  const size_t base = off;  // the general and the few-token forward's buffers, one or the other, follow
  plan->off_m = off;
  off += align256((size_t)parts * NR * 4);
  plan->off_l = off;
  off += align256((size_t)parts * NR * 4);
  plan->off_acc = off;
  off += align256((size_t)part_cols * NR * 4);
  plan->off_Ep = off;
  off += align256((size_t)plan->V_pad * DP * tbytes);
  plan->off_bias = off;
  off += align256((size_t)plan->V_pad * 4 * (dtype == kFP8 ? 2 : 1));
  plan->N_pad = ((N + 255) / 256) * 256;
  plan->hS = packed_slices(K, tbytes == 4 ? SliceK<float>::value : SliceK<bf16_t>::value);
  plan->off_hp = off;
  off += align256((size_t)plan->N_pad * plan->hS * (tbytes == 4 ? SliceK<float>::value : SliceK<bf16_t>::value) * tbytes);
  plan->off_Wp = off;
  off += align256((size_t)plan->V_pad * plan->hS * (tbytes == 4 ? SliceK<float>::value : SliceK<bf16_t>::value) * tbytes);
  plan->ws_bytes = off;
  few_plan(dtype, N, V, Dw, active, base, plan);
  return true;
}

hipError_t fwd_launch(int dtype, const FwdPlan& plan, FwdParams p, char* ws, float* O, float* lse, float* m_out,
                      float* l_out, hipStream_t stream) {
  if (p.N == 0) return hipSuccess;
  if (few_fits(plan, p, dtype)) return fwd_few(dtype, plan, p, nullptr, ws, O, lse, m_out, l_out, stream);
  p.n_tb = plan.n_tb;
  p.n_split = plan.n_split;
  p.n_vt = plan.n_vt;
  p.part_m = reinterpret_cast<float*>(ws + plan.off_m);
  p.part_l = reinterpret_cast<float*>(ws + plan.off_l);
  p.part_acc = reinterpret_cast<float*>(ws + plan.off_acc);
  p.Ep = ws + plan.off_Ep;
  p.biasp = reinterpret_cast<const float*>(ws + plan.off_bias);
  p.hp = ws + plan.off_hp;
  p.Wp = ws + plan.off_Wp;
  p.hS = plan.hS;
  hipError_t e;
  switch (dtype) {
    case kBF16: e = pack<bf16_t>(p, plan, stream); break;
    case kF16: e = pack<f16_t>(p, plan, stream); break;
    case kF32: e = pack<float>(p, plan, stream); break;
    case kFP8: e = pack<bf16_t>(p, plan, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess) return e;
  // one pass per slice of E's columns (one pass unless D exceeds the slice width)
  const int64_t esz = dtype == kF32 ? 4 : 2;
  const int D = p.D;
  for (int d0 = 0; d0 < (D > 0 ? D : 1); d0 += plan.DS) {
    FwdParams q = p;
    q.E = static_cast<const char*>(p.E) + d0 * esz;
    q.D = D - d0 < plan.DS ? D - d0 : plan.DS;
    FwdPlan pass = plan;
    if (plan.rem_DP > 0 && d0 + plan.DS >= D) {  // the last, narrower pass: its own kernel, tiles and split
      pass.DP = plan.rem_DP;
      pass.BM = plan.rem_BM;
      pass.n_tb = q.n_tb = plan.rem_tb;
      pass.n_split = q.n_split = plan.rem_split;
      pass.n_part = plan.rem_part;
    }
    switch (dtype) {
      case kBF16: e = pack_et<bf16_t>(q, pass, stream); if (e == hipSuccess) e = dispatch_dp<bf16_t>(pass, q, stream); break;
      case kF16: e = pack_et<f16_t>(q, pass, stream); if (e == hipSuccess) e = dispatch_dp<f16_t>(pass, q, stream); break;
      case kF32: e = pack_et<float>(q, pass, stream); if (e == hipSuccess) e = dispatch_dp<float>(pass, q, stream); break;
      default: e = pack_et<bf16_t>(q, pass, stream); if (e == hipSuccess) e = dispatch_dp_f8(pass, q, stream); break;
    }
    if (e != hipSuccess) return e;
    // every pass computes the same scores, so each writes the same lse (m, l); O gets its columns
    e = launch_combine(p.part_m, p.part_l, p.part_acc, pass.n_part, p.N, q.D, (int64_t)pass.DP * p.N, p.N, 1,
                       O ? O + d0 : nullptr, D, lse, m_out, l_out, nullptr, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

namespace {

// Whether W (rows of 16-byte chunks, K a multiple of 8) holds an infinity or a NaN in the compute
// dtype, for a forward that does not pack it: bad[0] = 1 (as fwd_param_scan_kernel).
template <class Src, class T>
__global__ __launch_bounds__(256) void fwd_w_scan_kernel(const Src* __restrict__ W, int64_t ldw, int V, int K,
                                                         int* __restrict__ bad) {
  constexpr int CE = 16 / (int)sizeof(T);
  bool nf = false;
  for (int v = blockIdx.x; v < V; v += gridDim.x)
    for (int c = threadIdx.x; c < K / CE; c += 256)
      nf |= chunk_nonfinite<T>(load_chunk<Src, T>(W + (int64_t)v * ldw + (int64_t)c * CE));
  if (__syncthreads_or(nf) && threadIdx.x == 0) bad[0] = 1;
}

// The few-token forward's token blocks and vocabulary runs (few_runs) for the count, into n_act[3],
// n_act[4].
__global__ __launch_bounds__(64) void fwd_few_grid_kernel(int* __restrict__ n_act, int BM, int grp) {
  if (threadIdx.x != 0) return;
  const int tb = (n_act[0] + BM - 1) / BM;
  n_act[3] = tb;
  n_act[4] = few_runs(tb, grp);
}

// Everything of the active-token forward before its passes: the parameter flags (bad[0..1], set
// while W is packed, or with few by a scan of it, and by the E / bias scan), the per-token flags and their compaction into
// positions (idx, inv, n_act[0]), the device-side token blocks and splits (n_act[3..4]), and the
// active tokens' h rows packed in position order.  n_act points at the count block:
// [0] count, [1..2] parameter flags, [3..4] token blocks and splits.
template <class T>
hipError_t active_setup(const FwdPlan& plan, const FwdParams& p, const float* weight, int* flag, int* idx, int* inv,
                        int* n_act, int* bad, bool few, T* hp, hipStream_t stream) {
  timing_begin(kKindPack, stream);
  const bool scale_bad = !std::isfinite(p.scale);
  fwd_flags_init_kernel<<<1, 64, 0, stream>>>(bad, scale_bad ? 1 : 0, (p.bias || p.V == 0) ? 1 : 0);
  hipError_t e = hipGetLastError();
  // W once (as fwd_launch packs it), checked for non-finite values on the way
  PackExtra wx;
  wx.nonfinite = bad;
  T* const Wp = const_cast<T*>(static_cast<const T*>(p.Wp));
  if (few) {
    if (e == hipSuccess && p.V > 0 && p.K > 0) {
      const unsigned blocks = p.V < 2048 ? p.V : 2048;
      if (sizeof(T) == 2 && p.w_f32)
        fwd_w_scan_kernel<float, T><<<blocks, 256, 0, stream>>>(static_cast<const float*>(p.W), p.ldw, p.V, p.K, bad);
      else
        fwd_w_scan_kernel<T, T><<<blocks, 256, 0, stream>>>(static_cast<const T*>(p.W), p.ldw, p.V, p.K, bad);
      e = hipGetLastError();
    }
  } else if (e == hipSuccess) {
    e = pack_src<T>(p.W, p.w_f32, p.ldw, p.V, p.K, plan.hS, plan.V_pad, Wp, stream, nullptr, wx);
  }
  const int64_t work = (int64_t)p.V * (p.D > 0 ? p.D : 1);
  if (e == hipSuccess && work > 0 && (p.D > 0 || p.bias)) {
    const int blocks = (int)((work + 255) / 256 < 2048 ? (work + 255) / 256 : 2048);
    fwd_param_scan_kernel<T><<<blocks, 256, 0, stream>>>(static_cast<const T*>(p.E), p.lde, p.V, p.D, p.bias, bad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) {
    const unsigned blocks = (unsigned)((p.N + 3) / 4);
    if (sizeof(T) == 2 && p.h_f32)
      fwd_active_flag_kernel<float, T><<<blocks, 256, 0, stream>>>(weight, static_cast<const float*>(p.h), p.ldh,
                                                                   p.N, p.K, bad, flag);
    else
      fwd_active_flag_kernel<T, T><<<blocks, 256, 0, stream>>>(weight, static_cast<const T*>(p.h), p.ldh, p.N, p.K,
                                                               bad, flag);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = compact_tokens(flag, p.N, idx, inv, n_act, stream);
  if (e == hipSuccess) {
    if (few)
      fwd_few_grid_kernel<<<1, 64, 0, stream>>>(n_act, 32 * plan.few_NB, (p.V + 31) / 32);
    else
      fwd_active_grid_kernel<<<1, 64, 0, stream>>>(n_act, plan.BM, plan.n_tb, plan.n_split, plan.n_vt,
                                                   fwd_cost(p.K, plan.DP, plan.BM, plan.WV));
    e = hipGetLastError();
  }
  // h rows of the active tokens in position order, zeros past them
  PackExtra hx;
  hx.rows = idx;
  hx.n_rows = n_act;
  if (e == hipSuccess) e = pack_src<T>(p.h, p.h_f32, p.ldh, p.N, p.K, plan.hS, plan.N_pad, hp, stream, nullptr, hx);
  timing_end(kKindPack, stream);
  return e;
}

}  // namespace

hipError_t fwd_launch_active(int dtype, const FwdPlan& plan, FwdParams p, const float* weight, char* ws, float* O,
                             float* lse, hipStream_t stream) {
  if (p.N == 0) return hipSuccess;
  if (!plan.active || dtype == kFP8) return hipErrorInvalidValue;
  const bool few = few_fits(plan, p, dtype);
  if (few && p.N <= (dtype == kF32 ? kFewTokensActiveF32 : kFewTokensActive))
    return fwd_few(dtype, plan, p, weight, ws, O, lse, nullptr, nullptr, stream);
  p.n_tb = plan.n_tb;
  p.n_split = plan.n_split;
  p.n_vt = plan.n_vt;
  p.part_m = reinterpret_cast<float*>(ws + plan.off_m);
  p.part_l = reinterpret_cast<float*>(ws + plan.off_l);
  p.part_acc = reinterpret_cast<float*>(ws + plan.off_acc);
  p.Ep = ws + plan.off_Ep;
  p.biasp = reinterpret_cast<const float*>(ws + plan.off_bias);
  p.hp = ws + plan.off_hp;
  p.Wp = ws + plan.off_Wp;
  p.hS = plan.hS;
  int* flag = reinterpret_cast<int*>(ws + plan.off_flag);
  int* idx = reinterpret_cast<int*>(ws + plan.off_idx);
  int* inv = reinterpret_cast<int*>(ws + plan.off_inv);
  int* n_act = reinterpret_cast<int*>(ws + plan.off_nact);
  p.n_act = n_act;
  FwdFewParams fq = few_params(plan, p, ws);
  fq.n_act = n_act;
  fq.n_wg = plan.few_wgs;
  void* const hp = few ? ws + plan.few_hp : ws + plan.off_hp;
  hipError_t e;
  switch (dtype) {
    case kBF16: e = active_setup<bf16_t>(plan, p, weight, flag, idx, inv, n_act, n_act + 1, few, static_cast<bf16_t*>(hp), stream); break;
    case kF16: e = active_setup<f16_t>(plan, p, weight, flag, idx, inv, n_act, n_act + 1, few, static_cast<f16_t*>(hp), stream); break;
    case kF32: e = active_setup<float>(plan, p, weight, flag, idx, inv, n_act, n_act + 1, few, static_cast<float*>(hp), stream); break;
    default: return hipErrorInvalidValue;
  }
  if (e != hipSuccess) return e;
  const int64_t esz = dtype == kF32 ? 4 : 2;
  const int D = p.D;
  for (int d0 = 0; d0 < (D > 0 ? D : 1); d0 += plan.DS) {
    FwdParams q = p;
    q.E = static_cast<const char*>(p.E) + d0 * esz;
    q.D = D - d0 < plan.DS ? D - d0 : plan.DS;
    switch (few ? 4 + dtype : dtype) {
      case kBF16: e = pack_et<bf16_t>(q, plan, stream); if (e == hipSuccess) e = dispatch_dp<bf16_t>(plan, q, stream); break;
      case kF16: e = pack_et<f16_t>(q, plan, stream); if (e == hipSuccess) e = dispatch_dp<f16_t>(plan, q, stream); break;
      case kF32: e = pack_et<float>(q, plan, stream); if (e == hipSuccess) e = dispatch_dp<float>(plan, q, stream); break;
      case 4 + kBF16: e = few_pass<bf16_t>(dtype, plan, p, d0, fq, ws, stream); break;
      case 4 + kF16: e = few_pass<f16_t>(dtype, plan, p, d0, fq, ws, stream); break;
      default: e = few_pass<float>(dtype, plan, p, d0, fq, ws, stream); break;
    }
    if (e != hipSuccess) return e;
    const float* const cm = few ? fq.part_m : p.part_m;
    const float* const cl = few ? fq.part_l : p.part_l;
    const float* const ca = few ? fq.part_acc : p.part_acc;
    const int cBM = few ? 32 * plan.few_NB : plan.BM, cWV = few ? 1 : plan.WV, cDP = few ? plan.few_DP : plan.DP;
    timing_begin(kKindFwdCombine, stream);
    auto go = [&](auto g, auto dt) {
      constexpr int G = decltype(g)::value, DT = decltype(dt)::value;
      fwd_combine_active_kernel<G, DT><<<combine_blocks<G, DT>(p.N, q.D), G * MergeWidth<G>::value, 0, stream>>>(
          cm, cl, ca, inv, n_act, cBM, cWV, p.N, q.D, cDP, O + d0, D, lse);
    };
    dispatch_combine((int64_t)p.N * q.D, few ? plan.few_split : plan.n_part, go);
    timing_end(kKindFwdCombine, stream);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t shard_combine(int S, int N, int D, const float* m, const float* l, const float* acc, float* O, float* lse,
                         hipStream_t stream) {
  return launch_combine(m, l, acc, S, N, D, (int64_t)N * D, 1, D, O, D, lse, nullptr, nullptr, nullptr,
                        stream);
}

}  // namespace swvr
