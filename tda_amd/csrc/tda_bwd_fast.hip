// tda_bwd_fast.hip -- bf16 backward of threshold attention for gfx950, driven by the forward's
// tile-occupancy bitmask.
//
// Reference semantics: snap-research/TDA triton_threshold_attention.py backward kernels
// (TTA:118-324) and host backward (TTA:406-469); the normalize / clamp / combine gradients
// follow torch autograd of TTA:505-517; dbeta is new (the reference returns None, TTA:469).
// The formulas are listed at the top of tda_bwd.hip.
//
// Layout of the work.  With the forward's pair lists (the non-zero weights of each (branch,
// query tile), see tda_params.hpp) the backward touches only the rows those weights name:
//   * bwd_dq_pairs: one wave per (branch, query tile) whose list fit; whole-row vector work per
//     pair, the tile's other gradient rows stored as zeros.
//   * bwd_dkv_pairs: one wave per key tile whose bitmask column has only lists that fit; whole-
//     row vector work per key row its pairs name, with the dk weight of each pair stored by
//     bwd_dq_pairs (no V, no matrix cores), the tile's other gradient rows stored as zeros.
// Gradient rows are streaming (non-temporal) stores: nothing reads them back soon.
// The block tile passes take the rest (lists past the cap, or no lists at all), driven by the
// bitmask: four consecutive tiles of one head per workgroup, one wave each, sharing every streamed
// tile's rows through LDS:
//   * bwd_dq_blk: four query tiles of one (branch, head); walks the set bits of their bitmask
//     rows, so only key tiles with a non-zero score are touched; dq_br is finished (F.normalize
//     backward) at the end.
//   * bwd_dkv_blk: four key tiles of one head; walks the set bits of the bitmask columns of each
//     branch; dv accumulates over both branches (A1 - lam A2), dk_br is finished per branch.
//   * bwd_tiles: both in one launch over the blocks that the key-major pair pass queued (with
//     normalisation, where usually every list fits and the queue is empty).
// dbeta / dlambda partials: one pair per (branch, query tile), summed in a fixed order by
// bwd_finish.
#include "tda_common.hpp"
#include "tda_params.hpp"
#include "tda_pos.hpp"

namespace tda {


// Descriptor of one tile's rows: loads past `bytes` read as zeros (its range check).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
// Lane-distributed pair list: lane e < n holds entry e (key, query row in the tile, x).
struct PairLanes {
  int key, row;
  float x;
  uint32_t slot;  // the pair's column-bucket slot (kNoSlot: none)
};
__device__ __forceinline__ PairLanes load_pairs(const uint32_t* ent, uint32_t n) {
  const int l = lane_id();
  u32x4 e = u32x4{0u, 0u, 0u, 0u};
  if ((uint32_t)l < n) e = *reinterpret_cast<const u32x4*>(ent + 4 * l);
  // x through a bit cast of the whole vector: hipcc compiled __builtin_bit_cast(float, e[2])
  // to element 0 (the key index)
  const f32x4 ef = __builtin_bit_cast(f32x4, e);
  return PairLanes{(int)e[0], (int)e[1], ef[2], e[3]};
}

// Row fragment t of a swizzled tile: lane (m, g) gets elements 16t + 8g .. +7 of row m.
template <int D>
__device__ __forceinline__ bf16x8 tile_row_frag(const bf16* tile, int t) {
  const int l = lane_id(), m = l & 31, g = l >> 5;
  return *reinterpret_cast<const bf16x8*>(tile + m * D + 8 * ((2 * t + g) ^ bswz<D>(m)));
}
// Load this lane's 16 values of a 32-float row table at C rows crow(r, g).
__device__ __forceinline__ void crow_vals(const float* tab, float (&v)[16]) {
  const int g = lane_id() >> 5;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(tab + 8 * u + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * u + e] = x[e];
  }
}

// This lane's elements of NC input columns in the transposed C layout of a gradient tile
// (elements 32c + 8u + 4g .. +3), for the F.normalize backward.
template <int NC>
struct GradRow {
  bf16x4 x[NC / 32][4];
};
template <int NC>
__device__ __forceinline__ void load_grad_row(const bf16* xrow, GradRow<NC>& r) {
  const int g = lane_id() >> 5;
#pragma unroll
  for (int c = 0; c < NC / 32; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u) r.x[c][u] = *reinterpret_cast<const bf16x4*>(xrow + 32 * c + 8 * u + 4 * g);
}

// The row dot x^ . acc over the NC columns of a gradient tile in the transposed C layout (lane =
// row, value r of column block c = element 32c + crow(r, g)), the same in both lanes of the row.
template <int NC>
__device__ __forceinline__ float grad_row_dot(const f32x16 (&acc)[NC / 32], const GradRow<NC>& xr, float rinv) {
  float dot = 0.f;
#pragma unroll
  for (int c = 0; c < NC / 32; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) dot = __builtin_fmaf((float)xr.x[c][u][e] * rinv, acc[c][4 * u + e], dot);
  return dot + __shfl_xor(dot, 32);
}
// Apply the F.normalize backward (see finish_rows in tda_bwd.hip) to scale times the tile and store
// it; xr, rinv, dot: the input row, its inverse norm and the whole row's x^ . acc (NORM only).
template <int NC, bool NORM>
__device__ __forceinline__ void store_grad_rows(const f32x16 (&acc)[NC / 32], const GradRow<NC>& xr, bf16* grow,
                                                float rinv, float dot, float scale) {
  const int g = lane_id() >> 5;
  const bool clamped = NORM && rinv >= 1.0f / kNormEps;
  const float rs = rinv * scale;
#pragma unroll
  for (int c = 0; c < NC / 32; ++c)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = acc[c][4 * u + e];
        if constexpr (NORM) o[e] = clamped ? a * rs : (a - (float)xr.x[c][u][e] * rinv * dot) * rs;
        else o[e] = a * scale;
      }
      store4(grow + 32 * c + 8 * u + 4 * g, o[0], o[1], o[2], o[3]);
    }
}

// ------------------------------------------------------------------ query-major pass, pairs
// One wave per (branch, query tile) whose pair list fit.  A list holds a few non-zero weights,
// so the wave works on whole rows, D / 64 elements per lane: the tile's gradient rows that no
// pair names are stored as zeros (16-byte stores), and for each named row i, in increasing
// order, dq_i = sum over its pairs, in list order, of dS k_j (times the key's inverse norm with
// normalisation), dS = coef p x^(p-1) (do_i . v_j) with x the forward's exact value; then the
// normalize backward of the row.  Each pair's dk weight, dS (times rq_i with normalisation),
// goes to the workspace slot of its list entry and to its column-bucket entry for
// bwd_dkv_pairs.  No LDS, no matrix cores: per pair two row loads and one wave-wide dot product.
template <int D>
struct RowVec {
  static constexpr int E = D / 64;  // elements per lane
  float v[E];
};
template <int D>
__device__ __forceinline__ RowVec<D> load_rowvec(const bf16* row) {
  RowVec<D> r;
  const int l = lane_id();
  if constexpr (D == 128) {
    const bf16x2 x = *reinterpret_cast<const bf16x2*>(row + 2 * l);
    r.v[0] = (float)x[0];
    r.v[1] = (float)x[1];
  } else {
    r.v[0] = (float)row[l];
  }
  return r;
}
template <int D>
__device__ __forceinline__ RowVec<D> load_rowvec(const float* row) {
  RowVec<D> r;
  const int l = lane_id();
  if constexpr (D == 128) {
    const float2 x = *reinterpret_cast<const float2*>(row + 2 * l);
    r.v[0] = x.x;
    r.v[1] = x.y;
  } else {
    r.v[0] = row[l];
  }
  return r;
}
// The lane's D/64 elements of a row as loaded (bf16: the bits, element 2l in the low half for
// D = 128, one register per row while loads are in flight; fp32: the values).
template <int D, class T>
struct RowRaw;
template <int D>
struct RowRaw<D, bf16> {
  uint32_t u;
};
template <int D>
struct RowRaw<D, float> {
  float v[D / 64];
};
template <int D>
__device__ __forceinline__ RowRaw<D, bf16> load_rowraw(const bf16* row) {
  const int l = lane_id();
  if constexpr (D == 128) return RowRaw<D, bf16>{*reinterpret_cast<const uint32_t*>(row + 2 * l)};
  else return RowRaw<D, bf16>{(uint32_t)*reinterpret_cast<const uint16_t*>(row + l)};
}
template <int D>
__device__ __forceinline__ RowRaw<D, float> load_rowraw(const float* row) {
  RowRaw<D, float> r;
  const RowVec<D> v = load_rowvec<D>(row);
#pragma unroll
  for (int e = 0; e < D / 64; ++e) r.v[e] = v.v[e];
  return r;
}
template <int D>
__device__ __forceinline__ RowVec<D> unpack(RowRaw<D, bf16> r) {
  RowVec<D> v;
  v.v[0] = __uint_as_float(r.u << 16);
  if constexpr (D == 128) v.v[1] = __uint_as_float(r.u & 0xffff0000u);
  return v;
}
template <int D>
__device__ __forceinline__ RowVec<D> unpack(RowRaw<D, float> r) {
  RowVec<D> v;
#pragma unroll
  for (int e = 0; e < D / 64; ++e) v.v[e] = r.v[e];
  return v;
}
template <int D>
__device__ __forceinline__ void store_rowvec(bf16* row, const RowVec<D>& r) {
  const int l = lane_id();
  if constexpr (D == 128)
    __builtin_nontemporal_store(__builtin_bit_cast(uint32_t, bf16x2{(bf16)r.v[0], (bf16)r.v[1]}),
                                reinterpret_cast<uint32_t*>(row + 2 * l));
  else row[l] = (bf16)r.v[0];
}
template <int D>
__device__ __forceinline__ void store_rowvec(float* row, const RowVec<D>& r) {
  const int l = lane_id();
  if constexpr (D == 128)
    __builtin_nontemporal_store(__builtin_bit_cast(uint64_t, float2{r.v[0], r.v[1]}),
                                reinterpret_cast<uint64_t*>(row + 2 * l));
  else __builtin_nontemporal_store(r.v[0], row + l);
}
template <int D>
__device__ __forceinline__ float row_dot(const RowVec<D>& a, const RowVec<D>& b) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < RowVec<D>::E; ++e) s = __builtin_fmaf(a.v[e], b.v[e], s);
  return wave_sum(s);
}
// The F.normalize backward of one row (see store_grad_rows): x the input row, rinv its inverse norm.
template <int D, bool NORM>
__device__ __forceinline__ RowVec<D> normalize_back(const RowVec<D>& g, const RowVec<D>& x, float rinv) {
  if constexpr (!NORM) return g;
  RowVec<D> xh, o;
#pragma unroll
  for (int e = 0; e < RowVec<D>::E; ++e) xh.v[e] = x.v[e] * rinv;
  const float dot = row_dot<D>(xh, g);
  const bool clamped = rinv >= 1.0f / kNormEps;
#pragma unroll
  for (int e = 0; e < RowVec<D>::E; ++e) o.v[e] = clamped ? g.v[e] * rinv : (g.v[e] - xh.v[e] * dot) * rinv;
  return o;
}
// Zero rows 0..nrows-1 of a 32-row tile except those in `keep` (16 bytes per lane and store).
template <int D, class T>
__device__ __forceinline__ void zero_rows(T* tile0, int64_t st, int nrows, uint32_t keep) {
  constexpr int EPC = 16 / sizeof(T), CH = D / EPC, RPI = 64 / CH;  // elements per chunk, chunks per row
  const int l = lane_id();
#pragma unroll
  for (int u = 0; u < 32 / RPI; ++u) {
    const int r = u * RPI + l / CH;
    if (r < nrows && !((keep >> r) & 1u))  // streaming stores: nothing reads them soon
      __builtin_nontemporal_store(u32x4{0u, 0u, 0u, 0u},
                                  reinterpret_cast<u32x4*>(tile0 + (int64_t)r * st + EPC * (l % CH)));
  }
}

// Tiles per workgroup of the block tile passes.
constexpr int kBwdBlk = 4;

// The tile-pass queue (P.dkvq, bf16 with normalisation), u32 words: [0] key blocks queued, [1]
// query blocks queued, [2] tickets taken, up to kTileqHead; one mask per key block (head, key
// tile / kBwdBlk): its key tiles that the pair pass left; the queued key blocks (as many as there
// are); the queued query blocks (of BR B H ceil(nqt / kBwdBlk)).  Head and masks are zeroed by the
// query-major pair pass, the rest filled by the key-major one.  It fits where nkt <= 64 nqt:
// 2 ceil(nkt / 4) + 2 ceil(nqt / 4) <= 64 nqt words per head.
constexpr int kTileqHead = 64;

// Pairs whose row loads the pair passes keep in flight together: the query-major pass 4 (64
// VGPRs, eight waves per SIMD: 23.6 us against 24.8 with 8 at B4 H16 N4096 d128), the
// key-major pass 8.
constexpr int kRowBatch = 4;
constexpr int kColBatch = 8;

// A pair list sorted by query row, then list order: lane s < n holds the entry of rank s, and
// e = its index in the list; lanes past n hold their own slot (a permutation of the lanes, so
// the forward permutes below write every lane once).
struct SortedPairs {
  int key, row, e;
  float x;
};
__device__ __forceinline__ SortedPairs sort_pairs(const PairLanes& PL, uint32_t n) {
  const int l = lane_id();
  int rank = l;
  if ((uint32_t)l < n) {
    rank = 0;
    for (uint32_t f = 0; f < n; ++f) {
      const int rf = __builtin_amdgcn_readlane(PL.row, (int)f);
      rank += rf < PL.row || (rf == PL.row && (int)f < l) ? 1 : 0;
    }
  }
  SortedPairs S;
  S.key = __builtin_amdgcn_ds_permute(4 * rank, PL.key);
  S.row = __builtin_amdgcn_ds_permute(4 * rank, PL.row);
  S.e = __builtin_amdgcn_ds_permute(4 * rank, l);
  S.x = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(4 * rank, __builtin_bit_cast(int, PL.x)));
  return S;
}

template <int D, int BR, int PK, bool NORM, class T = bf16>
__global__ void __launch_bounds__(64) bwd_dq_pairs(BwdParams P) {
  const int l = lane_id();
  const int BH = P.B * P.H;
  // (query tile, head, branch), query tiles ascending: the early rows' thresholds are the
  // lowest, their lists the longest
  const int64_t item = blockIdx.x;
  if (item >= (int64_t)BR * BH * P.nqt) return;
  const int br = BR == 2 ? (int)(item & 1) : 0;
  const int64_t rest = BR == 2 ? item >> 1 : item;
  const int qt = (int)(rest / BH);
  const int bh = (int)(rest % BH);
  const int b = bh / P.H, h = bh % P.H;
  const int64_t lidx = ((int64_t)br * BH + bh) * P.nqt + qt;
  // the count and every entry slot at once (slots past the count are never used)
  const PairLanes PL = load_pairs(P.pairs + lidx * (4 * kPairCap), (uint32_t)kPairCap);
  const uint32_t npairs = P.pairs[pair_lists(BR, BH, P.nqt) * 4 * kPairCap + lidx];
  if (P.dkvq) {  // the key-major pair pass fills the queue later
    if (item == 0 && l < kTileqHead) P.dkvq[l] = 0u;
    if constexpr (sizeof(T) == 2) {  // the key blocks' masks
      const int64_t nkb = (int64_t)BH * ((P.nkt + kBwdBlk - 1) / kBwdBlk);
      for (int64_t x = item * 64 + l; x < nkb; x += (int64_t)BR * BH * P.nqt * 64) P.dkvq[kTileqHead + x] = 0u;
    }
  }
  if (npairs > (uint32_t)kPairCap) return;  // the block tile pass walks the tiles

  auto base = [&](int slot) {
    return (const T*)P.in[slot] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };
  const int qslot = br == 0 ? B_Q1 : B_Q2, kslot = br == 0 ? B_K1 : B_K2, gslot = br == 0 ? B_DQ1 : B_DQ2;
  const int64_t sq = P.s[qslot][2], sk = P.s[kslot][2], sv = P.s[B_V][2], sdo = P.s[B_DO][2], sg = P.s[gslot][2];
  const T* qb = base(qslot);
  const T* kb = base(kslot);
  const T* vb = base(B_V);
  const T* dob = base(B_DO);
  T* gb = (T*)P.grad[br == 0 ? 0 : 2] + (int64_t)b * P.s[gslot][0] + (int64_t)h * P.s[gslot][1];
  const float* nq = NORM ? P.norms + norm_base(P, br == 0 ? N_Q1 : N_Q2, bh) : nullptr;
  const float* nk = NORM ? P.norms + norm_base(P, br == 0 ? N_K1 : N_K2, bh) : nullptr;
  const float pw = P.p;
  float coef = 1.f;
  if constexpr (BR == 2) coef = br == 0 ? 1.f : -clamp01(*P.lam);
  const bool want_l = BR == 2 && br == 1;  // dlambda comes from branch 2 alone

  uint32_t used = 0u;  // rows (within the tile) some pair names
  unsigned tiles = 0;
  int last_kt = -1;
  for (uint32_t e = 0; e < npairs; ++e) {
    used |= 1u << __builtin_amdgcn_readlane(PL.row, (int)e);
    const int kt = __builtin_amdgcn_readlane(PL.key, (int)e) >> 5;
    tiles += kt != last_kt ? 1u : 0u;  // pairs of one key tile are consecutive
    last_kt = kt;
  }
  const int q0 = 32 * qt;
  if (!P.grads_zeroed) zero_rows<D>(gb + (int64_t)q0 * sg, sg, min(32, P.Nq - q0), used);

  // The pairs sorted by query row, then list order: lane s gets the pair of rank s (lanes past
  // the count keep their own slot, so the ranks form a permutation of the lanes).
  const SortedPairs SP = sort_pairs(PL, npairs);

  // Rows in increasing order, each row's pairs in list order; the loads of kRowBatch pairs at a
  // time are in flight together, a row is finished when the next pair names another.
  float pb = 0.f, pl = 0.f;  // dbeta, dlambda partials (the same in every lane)
  float wks = 0.f;           // lane s: the dk weight of sorted pair s
  int cur = -1;              // row being accumulated
  RowVec<D> acc = {}, cur_x = {};
  float cur_r = 1.f;
  auto finish = [&]() {
    if (cur >= 0) store_rowvec<D>(gb + (int64_t)(q0 + cur) * sg, normalize_back<D, NORM>(acc, cur_x, cur_r));
  };
  for (uint32_t s0 = 0; s0 < npairs; s0 += kRowBatch) {
    int il[kRowBatch], jj[kRowBatch];
    float rq[kRowBatch], rk[kRowBatch];
    RowRaw<D, T> dor[kRowBatch], qr[kRowBatch], kr[kRowBatch], vr[kRowBatch];
#pragma unroll
    for (int u = 0; u < kRowBatch; ++u) {
      const int s = (int)s0 + u;
      if ((uint32_t)s >= npairs) continue;
      il[u] = __builtin_amdgcn_readlane(SP.row, s);
      jj[u] = __builtin_amdgcn_readlane(SP.key, s);
      const int i = q0 + il[u];
      dor[u] = load_rowraw<D>(dob + (int64_t)i * sdo);
      kr[u] = load_rowraw<D>(kb + (int64_t)jj[u] * sk);
      vr[u] = load_rowraw<D>(vb + (int64_t)jj[u] * sv);
      qr[u] = RowRaw<D, T>{};
      rq[u] = rk[u] = 1.f;
      if constexpr (NORM) {
        qr[u] = load_rowraw<D>(qb + (int64_t)i * sq);
        rq[u] = nq[i];
        rk[u] = nk[jj[u]];
      }
    }
#pragma unroll
    for (int u = 0; u < kRowBatch; ++u) {
      const int s = (int)s0 + u;
      if ((uint32_t)s >= npairs) continue;
      if (il[u] != cur) {
        finish();
        acc = RowVec<D>{};
        cur = il[u];
        cur_x = unpack<D>(qr[u]);
        cur_r = rq[u];
      }
      const float xx = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, SP.x), s));
      const float ci = tau_coeff(P.qoff + q0 + il[u], P.inv_d);
      const float dp = row_dot<D>(unpack<D>(dor[u]), unpack<D>(vr[u]));
      const float ds = coef * dpow_p<PK>(xx, pw) * dp;
      pb = __builtin_fmaf(-ci, ds, pb);
      if (want_l) pl = __builtin_fmaf(-pow_p<PK>(xx, pw), dp, pl);
      const float w = NORM ? ds * rk[u] : ds;
      wks = l == s ? (NORM ? ds * rq[u] : ds) : wks;
      const RowVec<D> kv = unpack<D>(kr[u]);
#pragma unroll
      for (int c = 0; c < RowVec<D>::E; ++c) acc.v[c] = __builtin_fmaf(w, kv.v[c], acc.v[c]);
    }
  }
  finish();
  // back to list order: lane s sends its weight to the lane of its list entry
  const float wkl = __builtin_bit_cast(float, __builtin_amdgcn_ds_permute(4 * SP.e, __builtin_bit_cast(int, wks)));
  if ((uint32_t)l < npairs) {
    P.pws[lidx * kPairCap + l] = wkl;
    if (P.colbuf && PL.slot < (uint32_t)kColCap)  // the dk weight of the pair's column-bucket entry
      P.colbuf[(((int64_t)bh * P.nkt + (PL.key >> 5)) * kColCap + PL.slot) * 4 + 3] = __builtin_bit_cast(uint32_t, wkl);
  }
  if (l == 0) {
    P.ws[2 * lidx + 0] = pb;  // slot of (branch, head, query tile), whichever pass takes it
    P.ws[2 * lidx + 1] = pl;
    if (P.stats) {
      atomicAdd(P.stats + 0, (unsigned long long)tiles);
      atomicAdd(P.stats + 1, (unsigned long long)tiles);
    }
  }
}

// ------------------------------------------------------------------ key-major pass, pairs
// LDS slots of the key-major pair pass: pairs of one column gathered at once.
constexpr int kColPairs = 64;
static_assert(kColCap == kColPairs && kColCap == 64, "a column bucket: one entry per lane, as many as the slots");
// List-load rounds of one walk step of the key-major pair pass (two lists per round).
constexpr int kWalkRounds = 4;

// One entry of a column's pair list as seen by one lane of the key-major pair pass.
struct ColEntry {
  bool valid;  // the lane holds an entry
  int br;      // branch of the lane's list
  int key;     // key index j
  int i;       // query row
  float x;     // exact forward value
  float wk;    // dk weight from the query-major pair pass
};

// Query block j of a head's BR ceil(nqt / kBwdBlk), from the last query tiles (the longest rows), the
// branches adjacent: the list count of its tile `lane` (0 past the block).
template <int BR>
__device__ __forceinline__ uint32_t query_block_count(const BwdParams& P, const uint32_t* counts, int bh, int j) {
  const int nqt = P.nqt, l = lane_id(), nqb = (nqt + kBwdBlk - 1) / kBwdBlk;
  if (j >= BR * nqb) return 0u;
  const int br = BR == 2 ? j & 1 : 0, qt = kBwdBlk * (nqb - 1 - (BR == 2 ? j >> 1 : j)) + l;
  return l < kBwdBlk && qt < nqt ? counts[((int64_t)br * (P.B * P.H) + bh) * nqt + qt] : 0u;
}

// One wave per key tile whose column has only lists that fit.  Its pairs come from the column's
// bucket when the forward filled one with all of them (every entry with its dk weight: one round
// of loads), else it walks the column's lists (both branches, query-tile chunks of 64, two lists
// per step: lanes 0-31 and 32-63) and keeps the pairs with a key in this tile.  For each key row j that some pair names, in increasing
// order, whole-row vector work over its pairs:
//   dv_j  += coef A_ij do_i          A_ij = x^p (x the forward's exact value)
//   dk_j  += w_ij q_i                w_ij = coef p x^(p-1) (do_i . v_j) (times rq_i with
//                                    normalisation), stored by the query-major pair pass
// then the normalize backward of dk_j; the tile's other gradient rows are stored as zeros.
// Pairs of a row meet its accumulators in walk order (chunk, branch, query tile, list entry),
// or, from a bucket, in the order (branch, query row).
// Up to kColPairs pairs are gathered into LDS slots in one walk; a column with more walks its
// lists once per named row.  No matrix cores and no V: per pair two row loads.
template <int D, int BR, int PK, bool NORM, class T = bf16>
__global__ void __launch_bounds__(64) bwd_dkv_pairs(BwdParams P) {
  __shared__ int ps_i[kColPairs];    // query row, branch in bit 31
  __shared__ int ps_jl[kColPairs];   // key row within the tile
  __shared__ float ps_x[kColPairs];  // exact forward value x
  __shared__ float ps_w[kColPairs];  // dk weight

  const int l = lane_id();
  const int BH = P.B * P.H;
  const int64_t item = blockIdx.x;  // (key tile, head), the first key tiles (most queries) first
  if (item >= (int64_t)BH * P.nkt) return;
  const int kt = (int)(item / BH), bh = (int)(item % BH);
  const int b = bh / P.H, h = bh % P.H;
  const int qtf = qt_first(kt, P.qoff);

  auto base = [&](int slot) {
    return (const T*)P.in[slot] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };
  auto gbase = [&](int slot, int gi) {
    return (T*)P.grad[gi] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };
  const uint32_t* counts = P.pairs + pair_lists(BR, BH, P.nqt) * 4 * kPairCap;
  const float pw = P.p;
  float lam = 0.f;
  if constexpr (BR == 2) lam = clamp01(*P.lam);
  // query block kt of the head (and every nkt-th after it) goes to the tile-pass queue when one of
  // its tiles' lists did not fit; its counts are loaded here and tested once the bucket has arrived
  const bool queue = sizeof(T) == 2 && NORM && P.dkvq;
  uint32_t qcount = 0u;
  if (queue) qcount = query_block_count<BR>(P, counts, bh, kt);

  // Walk the column's lists in the order (query-tile chunk of 64, branch, query tile): the
  // bitmask bits and counts of 128 query tiles per load round, then 2 kWalkRounds lists per
  // step, all loaded before the first is used (lanes 0-31 and 32-63 take one list each per
  // round); body(entry) once per round.  Returns false, before any body call of that chunk pair, when a
  // list of the column did not fit (the same test as bwd_dkv_blk's: the tile pass takes the
  // key tile); the caller has then written nothing.
  auto walk = [&](auto&& body) -> bool {
    for (int q0c = qtf; q0c < P.nqt; q0c += 128) {
      uint64_t mask[2 * BR];  // [chunk * BR + branch]
      uint32_t cnt_l[2 * BR];
      bool ovf = false;
#pragma unroll
      for (int k = 0; k < 2 * BR; ++k) {
        const int c = k / BR, br = k % BR;
        const int qtl = q0c + 64 * c + l;
        const bool in = qtl < P.nqt;
        const int64_t row = ((int64_t)br * BH + bh) * P.nqt + (in ? qtl : P.nqt - 1);
        const uint32_t w = P.occ[row * P.occ_w + (kt >> 5)];
        cnt_l[k] = counts[row];
        const bool has = in && ((w >> (kt & 31)) & 1u);
        ovf = ovf || (has && cnt_l[k] > (uint32_t)kPairCap);
        mask[k] = wave_ballot(has);
      }
      if (wave_ballot(ovf) != 0ull) return false;
      while (true) {
        int ix[2 * kWalkRounds], sx[2 * kWalkRounds];
        uint32_t cx[2 * kWalkRounds];
#pragma unroll
        for (int u = 0; u < 2 * kWalkRounds; ++u) {  // next lists
          ix[u] = -1;
          sx[u] = 0;
          cx[u] = 0u;
          bool found = false;
#pragma unroll
          for (int k = 0; k < 2 * BR; ++k)
            if (!found && mask[k]) {
              found = true;
              ix[u] = k;
              sx[u] = __builtin_ctzll(mask[k]);
              mask[k] &= mask[k] - 1ull;
              cx[u] = (uint32_t)__builtin_amdgcn_readlane((int)cnt_l[k], sx[u]);
            }
        }
        if (ix[0] < 0) break;
        u32x4 ent[kWalkRounds];
        float wk[kWalkRounds];
        int brl[kWalkRounds], qtl[kWalkRounds];
        bool valid[kWalkRounds];
#pragma unroll
        for (int r = 0; r < kWalkRounds; ++r) {
          const int idx = l < 32 ? ix[2 * r] : ix[2 * r + 1];
          const int sel = l < 32 ? sx[2 * r] : sx[2 * r + 1];
          const uint32_t cnt = l < 32 ? cx[2 * r] : cx[2 * r + 1];
          const int e = l & 31;
          brl[r] = idx >= 0 ? idx % BR : 0;
          qtl[r] = q0c + 64 * (idx >= 0 ? idx / BR : 0) + sel;
          valid[r] = idx >= 0 && (uint32_t)e < cnt;
          const int64_t lidx = ((int64_t)brl[r] * BH + bh) * P.nqt + qtl[r];
          ent[r] = u32x4{0u, 0u, 0u, 0u};
          wk[r] = 0.f;
          if (valid[r]) {
            ent[r] = *reinterpret_cast<const u32x4*>(P.pairs + lidx * (4 * kPairCap) + 4 * e);
            wk[r] = P.pws[lidx * kPairCap + e];
          }
        }
#pragma unroll
        for (int r = 0; r < kWalkRounds; ++r) {
          if (ix[2 * r] < 0) break;
          // x through a bit cast of the whole vector (see load_pairs)
          const f32x4 ef = __builtin_bit_cast(f32x4, ent[r]);
          ColEntry c;
          c.valid = valid[r];
          c.br = brl[r];
          c.key = (int)ent[r][0];
          c.i = 32 * qtl[r] + (int)ent[r][1];
          c.x = ef[2];
          c.wk = wk[r];
          body(c);
        }
      }
    }
    return true;
  };

  uint32_t np = 0;
  unsigned visited = 0;
  uint32_t used[BR];  // key rows named by a pair, per branch
#pragma unroll
  for (int br = 0; br < BR; ++br) used[br] = 0u;
  // lane s < np: pair s {query row | branch << 31, key row in the tile, x, dk weight}, and the
  // second key of the order the pairs are taken in (after the key row)
  int pi_l = 0, pjl_l = 0;
  float px_l = 0.f, pw_l = 0.f;
  uint32_t k2_l = (uint32_t)l;

  // ---- the column's bucket, when the forward filled it with every pair of the column (one
  // round of loads; the pairs are then taken in the order (key row, branch, query row))
  bool from_bucket = false;
  if (P.colcnt) {
    const int64_t col = (int64_t)bh * P.nkt + kt;
    const uint32_t cc = (uint32_t)__builtin_amdgcn_readfirstlane((int)P.colcnt[col]);
    const u32x4 be = *reinterpret_cast<const u32x4*>(P.colbuf + (col * kColCap + l) * 4);
    if (!(cc & kColTaint) && cc <= (uint32_t)kColCap) {
      from_bucket = true;
      np = cc;
      const bool in = (uint32_t)l < np;
      const f32x4 bf = __builtin_bit_cast(f32x4, be);  // x, w: a bit cast of the whole vector (see load_pairs)
      pi_l = in ? (int)be[0] : 0;
      pjl_l = in ? (int)be[1] : 0;
      px_l = in ? bf[2] : 0.f;
      pw_l = in ? bf[3] : 0.f;
      k2_l = (uint32_t)pi_l;
#pragma unroll
      for (int br = 0; br < BR; ++br)
        used[br] = wave_or(in && (int)(((uint32_t)pi_l >> 31) & 1u) == br ? 1u << pjl_l : 0u);
      if (P.stats) {  // the counters as the walk counts them: (branch, query tile) lists in the column
        const int lk = (int)(((uint32_t)pi_l >> 31) << 30) | ((pi_l & 0x7fffffff) >> 5);
        bool dup = false;
        for (int f = 0; f < (int)np; ++f) dup = dup || (f < l && __builtin_amdgcn_readlane(lk, f) == lk);
        visited = (unsigned)__builtin_popcountll(wave_ballot(in && !dup));
      }
    }
  }

  if (queue) {
    // up to 64 blocks at a time, one addition to the counter for all of them (additions to one
    // counter come 11 ns apart: 24576 blocks of 8192 heads 281 us)
    const int nb = BR * ((P.nqt + kBwdBlk - 1) / kBwdBlk);
    for (int j0 = kt; j0 < nb; j0 += 64 * P.nkt) {
      uint64_t hit = 0ull;
      for (int it = 0; it < 64 && j0 + it * P.nkt < nb; ++it) {
        const int j = j0 + it * P.nkt;
        if (j != kt) qcount = query_block_count<BR>(P, counts, bh, j);
        if (wave_ballot(qcount > (uint32_t)kPairCap) != 0ull) hit |= 1ull << it;
      }
      if (hit == 0ull) continue;
      uint32_t at = 0u;
      if (l == 0) at = atomicAdd(P.dkvq + 1, (uint32_t)__builtin_popcountll(hit));
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      const int64_t nkb = (int64_t)BH * ((P.nkt + kBwdBlk - 1) / kBwdBlk);
      if ((hit >> l) & 1ull)
        P.dkvq[kTileqHead + 2 * nkb + at + (uint32_t)__builtin_popcountll(hit & ((1ull << l) - 1ull))] = (uint32_t)(bh * nb + j0 + l * P.nkt);
    }
  }

  // ---- else the first walk: rows named, pairs into the slots while they fit
  const bool fits = from_bucket || walk([&](const ColEntry& c) {
    const bool match = c.valid && (c.key >> 5) == kt;
    const uint64_t mm = wave_ballot(match);
    visited += ((mm & 0xffffffffull) ? 1u : 0u) + ((mm >> 32) ? 1u : 0u);
    const uint32_t slot = np + __builtin_amdgcn_mbcnt_hi((uint32_t)(mm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mm, 0u));
    if (match && slot < (uint32_t)kColPairs) {
      ps_i[slot] = c.i | (c.br ? (int)0x80000000u : 0);
      ps_jl[slot] = c.key & 31;
      ps_x[slot] = c.x;
      ps_w[slot] = c.wk;
    }
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      uint32_t ub = match && c.br == br ? 1u << (c.key & 31) : 0u;
      ub = wave_or(ub);
      used[br] |= ub;
    }
    np += (uint32_t)__builtin_popcountll(mm);
  });
  if (!fits) {  // the tile pass takes the key tile
    if (P.dkvq && l == 0) {
      if constexpr (sizeof(T) == 2) {  // its block of key tiles, queued by the first of them
        const int64_t nkb = (P.nkt + kBwdBlk - 1) / kBwdBlk, blk = (int64_t)bh * nkb + kt / kBwdBlk;
        uint32_t* masks = P.dkvq + kTileqHead;
        if (atomicOr(masks + blk, 1u << (kt % kBwdBlk)) == 0u) masks[BH * nkb + atomicAdd(P.dkvq, 1u)] = (uint32_t)blk;
      } else {
        P.dkvq[1 + atomicAdd(P.dkvq, 1u)] = (uint32_t)item;
      }
    }
    return;
  }
  wave_lds_sync();  // slots written by other lanes
  const bool slotted = np <= (uint32_t)kColPairs;

  // ---- rows: zeros for the rows no pair names, then each named key row
  const int nrows = min(32, P.Nk - 32 * kt);
  const uint32_t uall = BR == 2 ? used[0] | used[BR - 1] : used[0];
  T* dvb = gbase(B_DV, 4);
  const int64_t sdv = P.s[B_DV][2];
  if (!P.grads_zeroed) {
    zero_rows<D>(dvb + (int64_t)(32 * kt) * sdv, sdv, nrows, uall);
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      const int gslot = br == 0 ? B_DK1 : B_DK2;
      zero_rows<D>(gbase(gslot, br == 0 ? 1 : 3) + (int64_t)(32 * kt) * P.s[gslot][2], P.s[gslot][2], nrows, used[br]);
    }
  }
  const T* dob = base(B_DO);
  const int64_t sdo = P.s[B_DO][2];
  // key row jl's finished rows: dv, and dk of each branch whose pairs name it (the others were
  // stored as zeros above)
  auto store_key_row = [&](int jl, const RowVec<D>& av, const RowVec<D>(&ak)[BR], const RowVec<D>(&kx)[BR],
                           const float(&rk)[BR]) {
    const int j = 32 * kt + jl;
    store_rowvec<D>(dvb + (int64_t)j * sdv, av);
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      if (!((used[br] >> jl) & 1u)) continue;
      const int gslot = br == 0 ? B_DK1 : B_DK2;
      store_rowvec<D>(gbase(gslot, br == 0 ? 1 : 3) + (int64_t)j * P.s[gslot][2],
                      normalize_back<D, NORM>(ak[br], kx[br], rk[br]));
    }
  };
  // the same, packed (rows zero, norms 1 where not needed)
  auto load_key_raw = [&](int jl, RowRaw<D, T>(&kx)[BR], float(&rk)[BR]) {
    const int j = 32 * kt + jl;
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      kx[br] = RowRaw<D, T>{};
      rk[br] = 1.f;
      if constexpr (NORM)
        if ((used[br] >> jl) & 1u) {
          const int kslot = br == 0 ? B_K1 : B_K2;
          kx[br] = load_rowraw<D>(base(kslot) + (int64_t)j * P.s[kslot][2]);
          rk[br] = P.norms[norm_base(P, br == 0 ? N_K1 : N_K2, bh) + j];
        }
    }
  };
  // the key rows and inverse norms of key row jl for the normalize backward
  auto load_key_rows = [&](int jl, RowVec<D>(&kx)[BR], float(&rk)[BR]) {
    const int j = 32 * kt + jl;
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      kx[br] = RowVec<D>{};
      rk[br] = 1.f;
      if constexpr (NORM)
        if ((used[br] >> jl) & 1u) {
          const int kslot = br == 0 ? B_K1 : B_K2;
          kx[br] = load_rowvec<D>(base(kslot) + (int64_t)j * P.s[kslot][2]);
          rk[br] = P.norms[norm_base(P, br == 0 ? N_K1 : N_K2, bh) + j];
        }
    }
  };

  if (slotted) {
    // The pairs sorted by key row, then the second key (walk: slot order; bucket: branch and
    // query row): lane s gets the pair of rank s (lanes past np keep their own slot).  Then the
    // pairs in that order, the loads of kColBatch at a time in flight together; a key row is
    // finished when the next pair names another.
    if (!from_bucket) {
      const int sl = (uint32_t)l < np ? l : 0;
      pi_l = ps_i[sl];
      pjl_l = ps_jl[sl];
      px_l = ps_x[sl];
      pw_l = ps_w[sl];
    }
    int rank = l;
    if ((uint32_t)l < np) {
      rank = 0;
      for (uint32_t f = 0; f < np; ++f) {
        const int jf = __builtin_amdgcn_readlane(pjl_l, (int)f);
        const uint32_t kf = (uint32_t)__builtin_amdgcn_readlane((int)k2_l, (int)f);
        rank += jf < pjl_l || (jf == pjl_l && kf < k2_l) ? 1 : 0;
      }
    }
    const int s_i = __builtin_amdgcn_ds_permute(4 * rank, pi_l);
    const int s_jl = __builtin_amdgcn_ds_permute(4 * rank, pjl_l);
    const int s_x = __builtin_amdgcn_ds_permute(4 * rank, __builtin_bit_cast(int, px_l));
    const int s_w = __builtin_amdgcn_ds_permute(4 * rank, __builtin_bit_cast(int, pw_l));
    int cur = -1;
    RowVec<D> av = {}, ak[BR], kx[BR];
    float rk[BR];
#pragma unroll
    for (int br = 0; br < BR; ++br) {
      ak[br] = kx[br] = RowVec<D>{};
      rk[br] = 1.f;
    }
    for (uint32_t s0 = 0; s0 < np; s0 += kColBatch) {
      int jl[kColBatch], ibr[kColBatch];
      RowRaw<D, T> dor[kColBatch], qr[kColBatch], kxu[kColBatch][BR];
      float rku[kColBatch][BR];
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) {
        const int s = (int)s0 + u;
        ibr[u] = 0;
        if ((uint32_t)s >= np) continue;
        jl[u] = __builtin_amdgcn_readlane(s_jl, s);
        const int pi = __builtin_amdgcn_readlane(s_i, s);
        const int i = pi & 0x7fffffff;
        ibr[u] = (pi >> 31) & 1;
        const int qslot = ibr[u] ? B_Q2 : B_Q1;
        dor[u] = load_rowraw<D>(dob + (int64_t)i * sdo);
        qr[u] = load_rowraw<D>(base(qslot) + (int64_t)i * P.s[qslot][2]);
        load_key_raw(jl[u], kxu[u], rku[u]);
      }
#pragma unroll
      for (int u = 0; u < kColBatch; ++u) {
        const int s = (int)s0 + u;
        if ((uint32_t)s >= np) continue;
        if (jl[u] != cur) {
          if (cur >= 0) store_key_row(cur, av, ak, kx, rk);
          cur = jl[u];
          av = RowVec<D>{};
#pragma unroll
          for (int br = 0; br < BR; ++br) {
            ak[br] = RowVec<D>{};
            kx[br] = unpack<D>(kxu[u][br]);
            rk[br] = rku[u][br];
          }
        }
        const float x = __builtin_bit_cast(float, __builtin_amdgcn_readlane(s_x, s));
        const float wk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(s_w, s));
        const float wa = (ibr[u] ? -lam : 1.f) * pow_p<PK>(x, pw);
        const RowVec<D> dv_ = unpack<D>(dor[u]), qv = unpack<D>(qr[u]);
#pragma unroll
        for (int c = 0; c < RowVec<D>::E; ++c) av.v[c] = __builtin_fmaf(wa, dv_.v[c], av.v[c]);
#pragma unroll
        for (int br = 0; br < BR; ++br)
          if (ibr[u] == br)
#pragma unroll
            for (int c = 0; c < RowVec<D>::E; ++c) ak[br].v[c] = __builtin_fmaf(wk, qv.v[c], ak[br].v[c]);
      }
    }
    if (cur >= 0) store_key_row(cur, av, ak, kx, rk);
  } else {
    // more pairs than slots: each named key row walks the lists for its own pairs (lane order
    // within a step), up to four row pairs in flight
    for (uint32_t um = uall; um; um &= um - 1u) {
      const int jl = __builtin_ctz(um), j = 32 * kt + jl;
      RowVec<D> kx[BR];
      float rk[BR];
      load_key_rows(jl, kx, rk);
      RowVec<D> av = {}, ak[BR];
#pragma unroll
      for (int br = 0; br < BR; ++br) ak[br] = RowVec<D>{};
      walk([&](const ColEntry& c) {
        uint64_t pm = wave_ballot(c.valid && c.key == j);
        while (pm) {
          int e[4], ibr[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            e[u] = pm ? __builtin_ctzll(pm) : -1;
            if (pm) pm &= pm - 1ull;
          }
          RowVec<D> dor[4], qr[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            ibr[u] = 0;
            if (e[u] < 0) continue;
            const int i = __builtin_amdgcn_readlane(c.i, e[u]);
            ibr[u] = __builtin_amdgcn_readlane(c.br, e[u]);
            const int qslot = ibr[u] ? B_Q2 : B_Q1;
            dor[u] = load_rowvec<D>(dob + (int64_t)i * sdo);
            qr[u] = load_rowvec<D>(base(qslot) + (int64_t)i * P.s[qslot][2]);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (e[u] < 0) continue;
            const float x = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c.x), e[u]));
            const float wk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c.wk), e[u]));
            const float wa = (ibr[u] ? -lam : 1.f) * pow_p<PK>(x, pw);
#pragma unroll
            for (int cc = 0; cc < RowVec<D>::E; ++cc) av.v[cc] = __builtin_fmaf(wa, dor[u].v[cc], av.v[cc]);
#pragma unroll
            for (int br = 0; br < BR; ++br)
              if (ibr[u] == br)
#pragma unroll
                for (int cc = 0; cc < RowVec<D>::E; ++cc) ak[br].v[cc] = __builtin_fmaf(wk, qr[u].v[cc], ak[br].v[cc]);
          }
        }
      });
      store_key_row(jl, av, ak, kx, rk);
    }
  }
  if (P.stats && l == 0) {
    atomicAdd(P.stats + 0, (unsigned long long)visited);
    atomicAdd(P.stats + 1, (unsigned long long)visited);
  }
}

// ------------------------------------------------------------------ block tile passes
// kBwdBlk consecutive tiles of one head per workgroup, one wave each, walking the union of their
// bitmask tiles in step; each streamed tile's rows are loaded once per workgroup (each wave a
// quarter, one or two tiles ahead into registers) into a two-stage LDS ring of chunk-swizzled tiles
// (tile_row_frag / tile_tr_frag read them), one fence-free barrier per tile.  A wave computes only
// its own tiles, the masks branch-free and only on the tiles that need them.  The per-element work
// sets the pace, so what is the same for a whole branch stays out of it: dS = coef p x^(p-1) dP is
// accumulated without coef and, at p = 2, without the factor 2 (ds_scale times it, exactly, in
// the epilogue and in the dbeta sum), and the branch that counts -lambda in dv runs first, its sum
// scaled before the other's is added.
// At d = 256 a tile's row fragments and accumulators do not fit one wave's registers, so two waves
// share each tile (kSplit): wave 0 forms the scores and wave 1 dP, each in one chain over the row (the
// forward's bits, so the same weights), they exchange them through LDS, and each owns half of the
// gradient columns; the normalize backward's row dots are added through LDS in half order.  There the
// weights and dS carry their coefficients (-lambda, 2) before their rounding to bf16, and the
// key-major pass (bwd_dkv_wide) combines both branches' weights in fp32, rounded once for dv.
template <int D>
constexpr int kSplit = D > 128 ? 2 : 1;
template <int D, int W>
constexpr int kQryThreads = 64 * W * kSplit<D>;

// A wave's 16 values through LDS: give writes them, take (after a barrier) reads some wave's.
__device__ __forceinline__ void give16(f32x4 (*x)[64], const f32x16& v) {
#pragma unroll
  for (int u = 0; u < 4; ++u) x[u][lane_id()] = f32x4{v[4 * u], v[4 * u + 1], v[4 * u + 2], v[4 * u + 3]};
}
__device__ __forceinline__ f32x16 take16(const f32x4 (*x)[64]) {
  f32x16 o;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const f32x4 v = x[u][lane_id()];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[4 * u + e] = v[e];
  }
  return o;
}

// max(x, 0) of 16 values on their bits: a float is > 0 iff its bits as an int32 are.
__device__ __forceinline__ f32x16 relu_bits(const f32x16& x) {
  typedef int i32x16_ __attribute__((ext_vector_type(16)));
  i32x16_ b = __builtin_bit_cast(i32x16_, x);
#pragma unroll
  for (int r = 0; r < 16; ++r) b[r] = max(b[r], 0);
  return __builtin_bit_cast(f32x16, b);
}
// The same with a NaN taken to 0: with normalisation a score of a non-finite row has no weight.
template <bool NORM>
__device__ __forceinline__ f32x16 relu16(f32x16 x) {
  if constexpr (!NORM) return relu_bits(x);
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = fmaxf(x[r], 0.f);
  return x;
}

// dP as the p = 2 passes multiply it by t = relu(x): with normalisation 0 at a pair without a weight where
// dP is not finite (a value row that no weight meets).  Only a tile that has such a value pays for the
// selection: bwd_tiles, TDA (2, 16, 1500, 64) at beta 0.5, 162 us so, 166 with it on every tile.
template <bool NORM>
__device__ __forceinline__ f32x16 finite_dp(f32x16 dp, const f32x16& t) {
  if constexpr (NORM) {
    auto m3 = [](float a, float b, float c) {  // NaN if any is
      return __builtin_elementwise_maximum(__builtin_elementwise_maximum(fabsf(a), fabsf(b)), fabsf(c));
    };
    const float a = m3(dp[0], dp[1], dp[2]), b = m3(dp[3], dp[4], dp[5]), c = m3(dp[6], dp[7], dp[8]);
    const float d = m3(dp[9], dp[10], dp[11]), e = m3(dp[12], dp[13], dp[14]);
    if (wave_ballot(!(m3(m3(a, b, c), m3(d, e, dp[15]), dp[15]) < INFINITY)) != 0ull) {
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] = t[r] > 0.f ? dp[r] : 0.f;
    }
  }
  return dp;
}

// This wave's share (of NW waves) of a 32-row tile of D columns: rows RPI (LPW wv + i) + l / CH,
// chunk l % CH.
template <int D, int NW>
struct BlkRows {
  static constexpr int CH = D / 8, RPI = 64 / CH, LPW = 32 / RPI / NW;
  static_assert(LPW >= 1 && LPW * RPI * NW == 32, "tile rows split evenly over the waves");
  u32x4 v[LPW];
  __device__ __forceinline__ void load(const bf16* rows, int64_t st, int r0, int n, int wv) {
    const int l = lane_id();
    const int nr = min(32, n - r0);
    const __amdgpu_buffer_rsrc_t rs = rows_rsrc(rows + (int64_t)r0 * st, (uint32_t)(((int64_t)(nr - 1) * st + D) * 2));
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int r = RPI * (LPW * wv + i) + l / CH;
      v[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)(((int64_t)r * st + 8 * (l % CH)) * 2), 0, 0);
    }
  }
  __device__ __forceinline__ void store(bf16* tile, int wv) const {
    const int l = lane_id();
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int r = RPI * (LPW * wv + i) + l / CH;
      *reinterpret_cast<u32x4*>(tile + r * D + 8 * ((l % CH) ^ bswz<D>(r))) = v[i];
    }
  }
};

// Query-major: W query tiles (kBwdBlk, or fewer where no head has more) of one (branch, head), streaming K, V and the key norms.  The
// block takes its tiles whose lists did not fit (or all, without lists).
//
// The block functions' LDS, arrays of the kernel.
template <int D, int W>
struct BlkLds {
  bf16* ring;             // two stages of two tiles of D columns
  float (*vals)[2][32];   // [stage]: key norms; query norms and tau values
  bf16 (*rows)[32 * D];   // key-major, one wave per tile: each wave's key rows (swizzled)
  f32x4 (*xch)[4][64];    // a split tile's waves: its scores, its dP
  float (*dots)[2][32];   // and row dots
};
// Their declaration: W tiles; ROWS as above.
#define TDA_BLK_LDS(D, W, ROWS)                                                               \
  __shared__ __attribute__((aligned(16))) bf16 lds_ring[2 * 2 * 32 * D];                      \
  __shared__ __attribute__((aligned(16))) float lds_vals[2][2][32];                           \
  __shared__ __attribute__((aligned(16))) bf16 lds_rows[(ROWS) && kSplit<D> == 1 ? W : 1][(ROWS) && kSplit<D> == 1 ? 32 * D : 8]; \
  __shared__ __attribute__((aligned(16))) f32x4 lds_xch[kSplit<D> == 2 ? 2 * W : 1][kSplit<D> == 2 ? 4 * 64 : 1]; \
  __shared__ float lds_dots[W][kSplit<D> == 2 ? 64 : 1];                                      \
  const BlkLds<D, W> L{lds_ring, lds_vals, reinterpret_cast<bf16(*)[32 * D]>(&lds_rows[0][0]),             \
                       reinterpret_cast<f32x4(*)[4][64]>(&lds_xch[0][0]), reinterpret_cast<float(*)[2][32]>(&lds_dots[0][0])}
template <int D, int BR, int PK, bool NORM, int W>
__device__ __forceinline__ void dq_block(const BwdParams& P, const BlkLds<D, W>& L, int jb, int br, int bh) {
  constexpr int SP = kSplit<D>, NT = D / 16, ND = D / 32 / SP;
  constexpr int STAGE = 2 * 32 * D;  // K tile, V tile
  bf16* ring = L.ring;
  const int l = lane_id(), n32 = l & 31, g = l >> 5;
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wv = wid / SP, hh = wid % SP;  // the wave's tile of the block, its half of the columns
  const int BH = P.B * P.H, nqt = P.nqt, Nq = P.Nq, Nk = P.Nk, qoff = P.qoff;
  const int b = bh / P.H, h = bh % P.H;
  const uint32_t* counts = P.pairs ? P.pairs + pair_lists(BR, BH, nqt) * 4 * kPairCap : nullptr;
  const int64_t lrow0 = ((int64_t)br * BH + bh) * nqt + W * jb;  // list / bitmask row of the block's first tile
  // the tiles whose lists did not fit (or all, without lists): the same for every wave
  uint32_t needm = 0u;
#pragma unroll
  for (int r = 0; r < W; ++r) {
    const int q = W * jb + r;
    const bool nd = q < nqt && (!counts || (uint32_t)__builtin_amdgcn_readfirstlane((int)counts[lrow0 + r]) > (uint32_t)kPairCap);
    needm |= nd ? 1u << r : 0u;
  }
  if (!needm) return;
  const int qt = W * jb + wv;
  const bool need = (needm >> wv) & 1u;
  const int qtc = min(qt, nqt - 1);
  const int i = 32 * qt + n32;
  const bool qvalid = need && i < Nq;
  const int ic = min(32 * qtc + n32, Nq - 1);
  const int pq = qoff + i;
  const bool rowpad = 32 * qt + 31 >= Nq;
  auto base = [&](int slot) {
    return (const bf16*)P.in[slot] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };
  const int qslot = br == 0 ? B_Q1 : B_Q2, kslot = br == 0 ? B_K1 : B_K2;
  bf16x8 DO[SP == 1 ? NT : 1], Q[NT];  // (a split tile: Q holds the wave's operand, wave 1's is dO)
  {
    const bf16* r = base(B_DO) + (int64_t)ic * P.s[B_DO][2];
    const bf16* rq_ = SP == 2 && hh ? r : base(qslot) + (int64_t)ic * P.s[qslot][2];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (SP == 1) DO[t] = *reinterpret_cast<const bf16x8*>(r + 16 * t + 8 * g);
      Q[t] = *reinterpret_cast<const bf16x8*>(rq_ + 16 * t + 8 * g);
    }
  }
  const float rq = NORM ? P.norms[norm_base(P, br == 0 ? N_Q1 : N_Q2, bh) + ic] : 1.f;
  const float ci = tau_coeff(pq, P.inv_d);
  const float tau = (*P.beta) * ci;
  const float pw = P.p;
  float coef = 1.f;
  if constexpr (BR == 2) coef = br == 0 ? 1.f : -clamp01(*P.lam);
  const float ds_scale = SP == 2 ? 1.f : PK == 2 ? 2.f * coef : coef;
  const bool want_l = BR == 2 && br == 1;  // dlambda comes from branch 2 alone
  const bf16* vb = base(B_V);
  const int64_t sv = P.s[B_V][2];
  const bf16* kb = base(kslot);
  const int64_t sk = P.s[kslot][2];
  const float* nk = nullptr;
  if constexpr (NORM) nk = P.norms + norm_base(P, br == 0 ? N_K1 : N_K2, bh);
  // dbeta / dlambda sums: a tile's in fp32, over the tiles in fp64 (terms of both signs: the sums'
  // own rounding was the larger part of the scalars' error)
  double bsum = 0., lsum = 0.;
  unsigned visited = 0, computed = 0;

  f32x16 A[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c) A[c] = f32x16{};

  // word w of the block's row r, masked to the key tiles the row sees (uniform); every causal
  // tile without a bitmask
  const int klast_b = kt_last(min(W * jb + W - 1, nqt - 1), qoff, P.nkt);
  auto row_word = [&](int r, int w) -> uint32_t {
    if (!((needm >> r) & 1u)) return 0u;
    const int kl = kt_last(W * jb + r, qoff, P.nkt);
    if (w > (kl >> 5)) return 0u;
    uint32_t x = P.occ ? (uint32_t)__builtin_amdgcn_readfirstlane((int)P.occ[(lrow0 + r) * P.occ_w + w]) : 0xffffffffu;
    if (w == (kl >> 5) && (kl & 31) != 31) x &= (2u << (kl & 31)) - 1u;
    return x;
  };
  int sw = -1;
  uint32_t ub = 0u, sown = 0u;
  auto next_tile = [&](uint32_t& own_out) -> int {
    while (ub == 0u) {
      if (++sw > (klast_b >> 5)) return -1;
      uint32_t u = 0u, o = 0u;
#pragma unroll
      for (int r = 0; r < W; ++r) {
        const uint32_t x = row_word(r, sw);
        u |= x;
        o = r == wv ? x : o;
      }
      ub = u;
      sown = o;
    }
    const int kt = 32 * sw + __builtin_ctz(ub);
    ub &= ub - 1u;
    own_out = sown;
    return kt;
  };
  constexpr int AHEAD = D <= 64 && W > 2 ? 2 : 1;  // tiles in flight past the one being worked on
  struct Pre {  // a tile's share in flight: its rows and norms, index and the own row's word
    BlkRows<D, W * SP> kr, vr;
    f32x4 nr;
    int kt;
    uint32_t own;
  };
  auto fetch = [&](Pre& p) {
    p.kt = next_tile(p.own);
    const int kt = max(p.kt, 0);  // loads on every path: the waits then count them exactly
    p.kr.load(kb, sk, 32 * kt, Nk, wid);
    p.vr.load(vb, sv, 32 * kt, Nk, wid);
    if (NORM && wid == 0 && l < 8)
      p.nr = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                          rows_rsrc(nk + 32 * kt, (uint32_t)(min(32, Nk - 32 * kt) * 4)), 16u * (uint32_t)l, 0, 0));
  };
  int it = 0;
  auto step = [&](Pre& p) {
    const int kt = p.kt;
    const uint32_t cown = p.own;
    bf16* kst = ring + (it & 1) * STAGE;
    bf16* vst = kst + 32 * D;
    float* nst = L.vals[it & 1][0];
    p.kr.store(kst, wid);
    p.vr.store(vst, wid);
    if (NORM && wid == 0 && l < 8) *reinterpret_cast<f32x4*>(nst + 4 * l) = p.nr;
    fetch(p);  // the tile AHEAD steps on, in flight during this tile's work
    lds_barrier();
    ++it;
    auto tile = [&](const f32x16& S, const f32x16& Dp) {
      ++visited;
      const int k0 = 32 * kt;
      bool anyw = true;  // without a bitmask the counters count the tiles with a weight
      float rk[16];
      if constexpr (NORM) crow_vals(nst, rk);
      // exact x, branch-free; keys after the query's position, padding keys and rows past Nq
      // set to -1 (only on the tiles that have any)
      f32x16 X;
#pragma unroll
      for (int r = 0; r < 16; ++r) X[r] = __builtin_fmaf(NORM ? S[r] * rk[r] : S[r], rq, -tau);
      if (k0 + 31 > min(qoff + 32 * qt, Nk - 1) || rowpad) {
        // key crow(r, g) = c_r + 4 g (c_r = 8 (r / 4) + r % 4) is visible iff c_r <= lim: one
        // comparison per value
        const int lim = (qvalid ? min(pq, Nk - 1) - k0 : -1) - 4 * g;
#pragma unroll
        for (int r = 0; r < 16; ++r) X[r] = 8 * (r >> 2) + (r & 3) <= lim ? X[r] : -1.f;
      }
      f32x16 E;
      float bt = 0.f, lt = 0.f;
      if constexpr (SP == 2) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool pos = X[r] > 0.f;
          const float ds = pos ? coef * dpow_p<PK>(X[r], pw) * Dp[r] : 0.f;
          bt += ds;
          if (want_l) lt = pos ? __builtin_fmaf(pow_p<PK>(X[r], pw), Dp[r], lt) : lt;
          E[r] = NORM ? ds * rk[r] : ds;
        }
      } else if constexpr (PK == 2) {
        // relu on the bits (a float is > 0 iff its bits as an int32 are): t = max(x, 0) with no
        // comparison per value; t and t^2 vanish with t.  (Whole-vector bit casts: hipcc
        // compiled a bit cast of one element of an ext_vector to element 0.)
        const f32x16 T = relu16<NORM>(X), dP = finite_dp<NORM>(Dp, T);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float ds = T[r] * dP[r];
          bt += ds;
          if (want_l) lt = __builtin_fmaf(T[r], ds, lt);
          E[r] = NORM ? ds * rk[r] : ds;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool pos = X[r] > 0.f;
          const float ds = pos ? dpow_p<PK>(X[r], pw) * Dp[r] : 0.f;
          bt += ds;
          if (want_l) lt = pos ? __builtin_fmaf(pow_p<PK>(X[r], pw), Dp[r], lt) : lt;
          E[r] = NORM ? ds * rk[r] : ds;
        }
      }
      bsum += (double)bt;
      if (want_l) lsum += (double)lt;
      if (!P.occ) {
        float xm = X[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) xm = fmaxf(xm, X[r]);
        anyw = wave_ballot(xm > 0.f) != 0ull;
      }
      computed += anyw ? 1u : 0u;
      const bf16x8 E0 = PolBF16::pack_c(E, 0), E1 = PolBF16::pack_c(E, 1);
#pragma unroll
      for (int c = 0; c < ND; ++c) {
        A[c] = PolBF16::mma(tile_tr_frag<D>(kst, 0, c + ND * hh), E0, A[c]);
        A[c] = PolBF16::mma(tile_tr_frag<D>(kst, 1, c + ND * hh), E1, A[c]);
      }
    };
    const bool own = (cown >> (kt & 31)) & 1u;
    if constexpr (SP == 1) {
      if (own) {
        f32x16 S = f32x16{}, Dp = f32x16{};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          S = PolBF16::mma(tile_row_frag<D>(kst, t), Q[t], S);
          Dp = PolBF16::mma(tile_row_frag<D>(vst, t), DO[t], Dp);
        }
        tile(S, Dp);
      }
    } else {  // the waves of a tile agree on `own`; every wave takes the barrier
      if (own) {
        const bf16* src = hh ? vst : kst;
        f32x16 acc = f32x16{};
#pragma unroll
        for (int t = 0; t < NT; ++t) acc = PolBF16::mma(tile_row_frag<D>(src, t), Q[t], acc);
        give16(L.xch[wid], acc);
      }
      lds_barrier();
      if (own) tile(take16(L.xch[2 * wv]), take16(L.xch[2 * wv + 1]));
    }
  };
  Pre pa;
  fetch(pa);
  if constexpr (AHEAD == 2) {
    Pre pb;
    fetch(pb);
    while (pa.kt >= 0) {
      step(pa);
      if (pb.kt < 0) break;
      step(pb);
    }
  } else {
    while (pa.kt >= 0) step(pa);
  }
  float dot = 0.f;  // the query row's x^ . dq^
  if constexpr (NORM && SP == 2) {
    if (need) {
      GradRow<32 * ND> XR;
      load_grad_row<32 * ND>(base(qslot) + (int64_t)ic * P.s[qslot][2] + 32 * ND * hh, XR);
      dot = grad_row_dot<32 * ND>(A, XR, rq);
    }
    if (g == 0) L.dots[wv][hh][n32] = dot;
    lds_barrier();
    dot = L.dots[wv][0][n32] + L.dots[wv][1][n32];
  }
  if (!need) return;
  if (qvalid) {
    GradRow<32 * ND> XR;  // the query row's columns for the normalize backward
    if constexpr (NORM) {
      load_grad_row<32 * ND>(base(qslot) + (int64_t)ic * P.s[qslot][2] + 32 * ND * hh, XR);
      if constexpr (SP == 1) dot = grad_row_dot<32 * ND>(A, XR, rq);
    }
    const int gslot = br == 0 ? B_DQ1 : B_DQ2;
    bf16* grow = (bf16*)P.grad[br == 0 ? 0 : 2] + (int64_t)b * P.s[gslot][0] + (int64_t)h * P.s[gslot][1] +
                 (int64_t)i * P.s[gslot][2] + 32 * ND * hh;
    store_grad_rows<32 * ND, NORM>(A, XR, grow, rq, dot, ds_scale);
  }
  if (hh != 0) return;
  const float pb = (float)wave_sum(-(double)ci * (double)ds_scale * bsum);
  const float pl = (float)wave_sum(-lsum);
  if (l == 0) {
    const int64_t lidx = lrow0 + wv;
    P.ws[2 * lidx + 0] = pb;  // slot of (branch, head, query tile), whichever pass takes it
    P.ws[2 * lidx + 1] = pl;
    if (P.stats) {
      atomicAdd(P.stats + 0, (unsigned long long)visited);
      atomicAdd(P.stats + 1, (unsigned long long)computed);
    }
  }
}

// Key-major: W consecutive key tiles (kBwdBlk, or fewer where no head has more) of one head (aligned: one
// bitmask word holds their bits), streaming per branch the query tiles' Q and dO rows, query norms and tau values.  needm:
// the block's key tiles to take (at least one).
template <int D, int BR, int PK, bool NORM, int W>
__device__ __forceinline__ void dkv_block(const BwdParams& P, const BlkLds<D, W>& L, int jb, int bh, uint32_t needm) {
  constexpr int NT = D / 16, ND = D / 32;
  constexpr int STAGE = 2 * 32 * D;  // Q tile, dO tile
  bf16* ring = L.ring;
  const int l = lane_id(), n32 = l & 31, g = l >> 5;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int BH = P.B * P.H, nqt = P.nqt, nkt = P.nkt, Nq = P.Nq, Nk = P.Nk, qoff = P.qoff;
  const int b = bh / P.H, h = bh % P.H;
  const int kt0 = W * jb, kt = kt0 + wv;
  const int qtf_b = qt_first(kt0, qoff);  // first query tile of the block
  const bool need = (needm >> wv) & 1u;
  const int j = 32 * kt + n32;
  const bool kvalid = need && j < Nk;
  const int jc = min(j, Nk - 1);
  const int qtf_w = qt_first(kt, qoff);  // first query tile that sees this wave's key tile
  auto base = [&](int slot) {
    return (const bf16*)P.in[slot] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };

  bf16x8 V[NT];
  {
    const bf16* r = base(B_V) + (int64_t)jc * P.s[B_V][2];
#pragma unroll
    for (int t = 0; t < NT; ++t) V[t] = *reinterpret_cast<const bf16x8*>(r + 16 * t + 8 * g);
  }
  const float beta = *P.beta;
  const float pw = P.p;
  float lam = 0.f;
  if constexpr (BR == 2) lam = clamp01(*P.lam);
  const bf16* dob = base(B_DO);
  const int64_t sdo = P.s[B_DO][2];
  f32x16 AV[ND];
#pragma unroll
  for (int c = 0; c < ND; ++c) AV[c] = f32x16{};
  unsigned visited = 0, computed = 0;
  int it = 0;  // ring position, continued across the branches
  bf16* kti = L.rows[wv];

#pragma unroll
  for (int bi = 0; bi < BR; ++bi) {
    const int br = BR - 1 - bi;  // the second branch first: dv = dO^T A1 - lambda dO^T A2
    const int qslot = br == 0 ? B_Q1 : B_Q2, kslot = br == 0 ? B_K1 : B_K2;
    const bf16* qb = base(qslot);
    const int64_t sq = P.s[qslot][2];
    const float rk = NORM ? P.norms[norm_base(P, br == 0 ? N_K1 : N_K2, bh) + jc] : 1.f;
    const float* nq = nullptr;
    if constexpr (NORM) nq = P.norms + norm_base(P, br == 0 ? N_Q1 : N_Q2, bh);
    const float ds_scale = (PK == 2 ? 2.f : 1.f) * (br == 0 ? 1.f : -lam);
    // the wave's key rows (swizzled tile; rows past Nk read as zeros), read as score operands
    {
      BlkRows<D, W> kr4[W];
#pragma unroll
      for (int s4 = 0; s4 < W; ++s4) kr4[s4].load(base(kslot), P.s[kslot][2], 32 * min(kt, nkt - 1), Nk, s4);
#pragma unroll
      for (int s4 = 0; s4 < W; ++s4) kr4[s4].store(kti, s4);
    }
    f32x16 AK[ND];
#pragma unroll
    for (int c = 0; c < ND; ++c) AK[c] = f32x16{};
    const int64_t row0 = ((int64_t)br * BH + bh) * nqt;  // bitmask / list row of query tile 0

    // union walk over query tiles qtf_b .. nqt-1, 64 per round: lane q tests query tile q0c + q
    int q0c = qtf_b - 64;
    uint64_t um = 0ull, om = 0ull;
    auto next_tile = [&](bool& own_out) -> int {
      while (um == 0ull) {
        q0c += 64;
        if (q0c >= nqt) return -1;
        const int qtl = q0c + l;
        const bool in = qtl < nqt;
        const uint32_t w = !in ? 0u : P.occ ? P.occ[(row0 + qtl) * P.occ_w + (kt0 >> 5)] : 0xffffffffu;
        uint32_t bits = (w >> (kt0 & 31)) & needm;
        // causal: key tile kt0 + r is seen from query tile qt_first(kt0 + r) on
#pragma unroll
        for (int r = 0; r < W; ++r)
          if (qtl < qt_first(kt0 + r, qoff)) bits &= ~(1u << r);
        um = wave_ballot(bits != 0u);
        om = wave_ballot((bits >> wv) & 1u);
      }
      const int q = __builtin_ctzll(um);
      um &= um - 1ull;
      own_out = (om >> q) & 1ull;
      return q0c + q;
    };
    constexpr int AHEAD = D <= 64 && W > 2 ? 2 : 1;  // tiles in flight past the one being worked on
    struct Pre {  // a tile's share in flight: its rows, norms and thresholds, index, and whether it is the wave's
      BlkRows<D, W> qr, dr;
      float vrq, vtq;
      int qt;
      bool own;
    };
    auto fetch = [&](Pre& p) {
      p.qt = next_tile(p.own);
      const int qt = max(p.qt, 0);  // loads on every path: the waits then count them exactly
      p.qr.load(qb, sq, 32 * qt, Nq, wv);
      p.dr.load(dob, sdo, 32 * qt, Nq, wv);
      if (wv == 0 && l < 32) {
        const int qi = min(32 * qt + l, Nq - 1);
        p.vrq = NORM ? nq[qi] : 1.f;
        p.vtq = beta * tau_coeff(qoff + 32 * qt + l, P.inv_d);
      }
    };
    auto step = [&](Pre& p) {
      const int qt = p.qt;
      const bool cown = p.own;
      bf16* qst = ring + (it & 1) * STAGE;
      bf16* dst = qst + 32 * D;
      float* rqs = L.vals[it & 1][0];
      float* tqs = L.vals[it & 1][1];
      p.qr.store(qst, wv);
      p.dr.store(dst, wv);
      if (wv == 0 && l < 32) {
        rqs[l] = p.vrq;
        tqs[l] = p.vtq;
      }
      fetch(p);  // the tile AHEAD steps on, in flight during this tile's work
      lds_barrier();
      ++it;
      if (cown) {
        ++visited;
        const int q0 = 32 * qt;
        f32x16 S = f32x16{}, Dp = f32x16{};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          S = PolBF16::mma(tile_row_frag<D>(qst, t), tile_row_frag<D>(kti, t), S);
          Dp = PolBF16::mma(tile_row_frag<D>(dst, t), V[t], Dp);
        }
        float rq[16], tq[16];
        if constexpr (NORM) crow_vals(rqs, rq);
        crow_vals(tqs, tq);
        f32x16 X;
#pragma unroll
        for (int r = 0; r < 16; ++r) X[r] = __builtin_fmaf(NORM ? S[r] * rk : S[r], NORM ? rq[r] : 1.f, -tq[r]);
        // masks only on the tiles that need them: queries before the key (the diagonal), rows
        // past Nq, keys past Nk
        if (32 * kt + 31 > qoff + q0 || q0 + 31 >= Nq || 32 * kt + 31 >= Nk) {
          // query row crow(r, g) = c_r + 4 g (c_r = 8 (r / 4) + r % 4) sees the key iff
          // lo <= c_r <= lo + span: one unsigned comparison per value (an empty range: lo past
          // every c_r)
          const int lo0 = j - qoff - q0 - 4 * g, hi0 = Nq - 1 - q0 - 4 * g;
          const bool some = kvalid && hi0 >= lo0;
          const int lo = some ? lo0 : 64;
          const uint32_t span = some ? (uint32_t)(hi0 - lo0) : 0u;
#pragma unroll
          for (int r = 0; r < 16; ++r) X[r] = (uint32_t)(8 * (r >> 2) + (r & 3) - lo) <= span ? X[r] : -1.f;
        }
        f32x16 EV, EK;
        if constexpr (PK == 2) {  // relu on the bits, as in bwd_dq_blk
          const f32x16 T = relu16<NORM>(X), dP = finite_dp<NORM>(Dp, T);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            EV[r] = T[r] * T[r];
            const float ds = T[r] * dP[r];
            EK[r] = NORM ? ds * rq[r] : ds;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool pos = X[r] > 0.f;
            EV[r] = pos ? pow_p<PK>(X[r], pw) : 0.f;
            const float ds = pos ? dpow_p<PK>(X[r], pw) * Dp[r] : 0.f;
            EK[r] = NORM ? ds * rq[r] : ds;
          }
        }
        bool anyw = true;  // without a bitmask the counters count the tiles with a weight
        if (!P.occ) {
          float xm = X[0];
#pragma unroll
          for (int r = 1; r < 16; ++r) xm = fmaxf(xm, X[r]);
          anyw = wave_ballot(xm > 0.f) != 0ull;
        }
        computed += anyw ? 1u : 0u;
        const bf16x8 V0 = PolBF16::pack_c(EV, 0), V1 = PolBF16::pack_c(EV, 1);
        const bf16x8 K0 = PolBF16::pack_c(EK, 0), K1 = PolBF16::pack_c(EK, 1);
#pragma unroll
        for (int c = 0; c < ND; ++c) {
          AV[c] = PolBF16::mma(tile_tr_frag<D>(dst, 0, c), V0, AV[c]);
          AV[c] = PolBF16::mma(tile_tr_frag<D>(dst, 1, c), V1, AV[c]);
          AK[c] = PolBF16::mma(tile_tr_frag<D>(qst, 0, c), K0, AK[c]);
          AK[c] = PolBF16::mma(tile_tr_frag<D>(qst, 1, c), K1, AK[c]);
        }
      }
    };
    Pre pa;
    fetch(pa);
    if constexpr (AHEAD == 2) {
      Pre pb;
      fetch(pb);
      while (pa.qt >= 0) {
        step(pa);
        if (pb.qt < 0) break;
        step(pb);
      }
    } else {
      while (pa.qt >= 0) step(pa);
    }
    if (kvalid) {
      GradRow<D> XR;  // the key row for the normalize backward
      float dot = 0.f;
      if constexpr (NORM) {
        load_grad_row<D>(base(kslot) + (int64_t)jc * P.s[kslot][2], XR);
        dot = grad_row_dot<D>(AK, XR, rk);
      }
      const int gslot = br == 0 ? B_DK1 : B_DK2;
      bf16* grow = (bf16*)P.grad[br == 0 ? 1 : 3] + (int64_t)b * P.s[gslot][0] + (int64_t)h * P.s[gslot][1] +
                   (int64_t)j * P.s[gslot][2];
      store_grad_rows<D, NORM>(AK, XR, grow, rk, dot, ds_scale);
    }
    if (BR == 2 && bi == 0) {
#pragma unroll
      for (int c = 0; c < ND; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) AV[c][r] *= -lam;
    }
    lds_barrier();  // every wave is done with its key tile before the next branch's rows
  }
  if (kvalid) {
    bf16* vrow = (bf16*)P.grad[4] + (int64_t)b * P.s[B_DV][0] + (int64_t)h * P.s[B_DV][1] + (int64_t)j * P.s[B_DV][2];
    store_grad_rows<D, false>(AV, GradRow<D>{}, vrow, 1.f, 0.f, 1.f);
  }
  if (P.stats && l == 0 && need) {
    atomicAdd(P.stats + 0, (unsigned long long)visited);
    atomicAdd(P.stats + 1, (unsigned long long)computed);
  }
}

// One workgroup per block of query tiles: longest blocks (last query tiles) of every (head,
// branch) first, the branches adjacent.
template <int D, int BR, int PK, bool NORM, int W>
__global__ void __launch_bounds__((kQryThreads<D, W>)) __attribute__((amdgpu_waves_per_eu(2))) bwd_dq_blk(BwdParams P) {
  TDA_BLK_LDS(D, W, false);
  const int BH = P.B * P.H, nqb = (P.nqt + W - 1) / W;
  if (D > 128 && blockIdx.y && grid_bid<kQryThreads<D, W>>() >= (uint32_t)(BR * BH) * (uint32_t)nqb) return;
  const int bid = D > 128 ? (int)grid_bid<kQryThreads<D, W>>() : blockIdx.x, jb = nqb - 1 - bid / (BR * BH), rem = bid % (BR * BH);
  dq_block<D, BR, PK, NORM>(P, L, jb, BR == 2 ? rem & 1 : 0, BR == 2 ? rem >> 1 : rem);
}

// Waves per SIMD that the key-major pass is compiled for: the most without spills at d = 64 (three
// with one branch spill 9 VGPRs: 92 against 86.7 us at (4, 16, 2048, 64)); at d = 128 one, two with
// one branch and no normalisation (19 VGPRs spilled, yet a dense step (4, 16, 2048, 128) of 473
// against 539 us).
template <int D, int BR, bool NORM>
constexpr int dkv_waves() {
  return D <= 64 || (BR == 1 && !NORM) ? 2 : 1;
}

// One workgroup per block of key tiles: longest blocks (first key tiles) of every head first.  A
// key tile takes this pass when a list of its column did not fit (the test bwd_dkv_pairs leaves
// it by; it writes nothing for such a key tile), or always without lists.
template <int D, int BR, int PK, bool NORM, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(dkv_waves<D, BR, NORM>()))) bwd_dkv_blk(BwdParams P) {
  TDA_BLK_LDS(D, W, true);
  __shared__ uint32_t needs[W];
  const int l = lane_id();
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int BH = P.B * P.H, nqt = P.nqt;
  const int bid = blockIdx.x, jb = bid / BH, bh = bid % BH, kt = W * jb + wv;
  const uint32_t* counts = P.pairs ? P.pairs + pair_lists(BR, BH, nqt) * 4 * kPairCap : nullptr;
  // this wave's key tile: does a list of its column not fit (every branch, query tiles from
  // the first that sees it)?
  {
    bool nd = kt < P.nkt;
    if (nd && counts) {
      const int qtf = qt_first(kt, P.qoff);
      bool ovf = false;
      for (int q0c = qtf; q0c < nqt && !ovf; q0c += 64) {
        bool o = false;
#pragma unroll
        for (int br = 0; br < BR; ++br) {
          const int qtl = q0c + l;
          const bool in = qtl < nqt;
          const int64_t row = ((int64_t)br * BH + bh) * nqt + (in ? qtl : nqt - 1);
          const uint32_t w = P.occ ? P.occ[row * P.occ_w + (kt >> 5)] : 0xffffffffu;
          o = o || (in && ((w >> (kt & 31)) & 1u) && counts[row] > (uint32_t)kPairCap);
        }
        ovf = wave_ballot(o) != 0ull;
      }
      nd = ovf;
    }
    if (l == 0) needs[wv] = nd ? 1u : 0u;
  }
  __syncthreads();
  uint32_t needm = 0u;
#pragma unroll
  for (int r = 0; r < W; ++r) needm |= needs[r] ? 1u << r : 0u;
  needm = (uint32_t)__builtin_amdgcn_readfirstlane((int)needm);
  if (needm) dkv_block<D, BR, PK, NORM>(P, L, jb, bh, needm);
}

// Key-major at head_dim 256: kWideKeys key tiles of one head, 2 BR waves each (branch br, half hh),
// walking the query tiles that any of them has in either branch (their bitmask bits, or every causal
// one) and staging the Q rows of every branch and dO, one tile ahead.  Wave (br, 0) of a tile forms
// branch br's scores, wave (0, 1) dP; all take them from LDS, and wave (br, hh) owns half of dk_br's
// columns and a share of dv's.  At most 256 registers with two branches: accumulators past those live in
// the accumulation registers, and a branch around them copies them all (B2 H8 N1000: 83 us so, 166 with
// one wave per half, both branches in it; the query-major pass 46).
constexpr int kWideKeys = 2;

// tile_row_frag<256> and tile_tr_frag<256> from one byte offset per lane each: with rows of 512 bytes the
// swizzle's exclusive or with a step's chunk is one of the offset with a constant.  keep_here makes the
// offsets values of the loop's body (held as loop invariants, one register per step, they spill).
struct WideTile {
  int row, tr;
  __device__ __forceinline__ WideTile() {
    const int l = lane_id(), m = l & 31, g = l >> 5, j = l & 15, r = 4 * (l >> 5) + (j >> 2);
    row = 512 * m + 16 * (g ^ bswz<256>(m));
    tr = 512 * r + 16 * ((2 * ((l >> 4) & 1) + ((j & 3) >> 1)) ^ bswz<256>(r)) + 8 * (j & 1);
  }
  __device__ __forceinline__ void keep_here() { asm volatile("" : "+v"(row), "+v"(tr)); }
  __device__ __forceinline__ bf16x8 row_frag(const bf16* tile, int t) const {
    return *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(tile) + (row ^ (32 * (t & 7))) + 256 * (t >> 3));
  }
  __device__ __forceinline__ bf16x8 tr_frag(const bf16* tile, int st, int dsub) const {
    bf16x8 out;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const char* p = reinterpret_cast<const char*>(tile) + (tr ^ (16 * ((4 * (dsub & 3)) ^ (8 * u)))) + 8192 * st + 4096 * u + 256 * (dsub >> 2);
      const bf16x4 w = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p)));
#pragma unroll
      for (int e = 0; e < 4; ++e) out[4 * u + e] = w[e];
    }
    return out;
  }
};

template <int BR, int PK, bool NORM>
__global__ void __launch_bounds__(128 * BR * kWideKeys) __attribute__((amdgpu_waves_per_eu(BR))) bwd_dkv_wide(BwdParams P) {
  constexpr int D = 256, W = kWideKeys, NT = D / 16, NW = 2 * BR;  // NW: waves per key tile
  constexpr int NDK = D / 64, NDV = D / 32 / NW;                   // a wave's column blocks of dk, of dv
  constexpr int TILE = 32 * D, STAGE = (BR + 1) * TILE;            // Q of every branch, dO
  constexpr int RT = BR == 2 ? NT - 6 : NT;                        // steps of the resident operand in registers
  __shared__ __attribute__((aligned(16))) bf16 ring[2 * STAGE];
  __shared__ __attribute__((aligned(16))) float vals[2][BR + 1][32];  // [stage]: query norms per branch, tau values
  __shared__ __attribute__((aligned(16))) f32x4 xch[W][BR + 1][4][64];  // a tile's scores per branch, its dP
  __shared__ float dots[W][BR][2][32];                                 // the halves' row dots
  __shared__ __attribute__((aligned(16))) bf16x8 rest[BR == 2 ? W * (BR + 1) : 1][BR == 2 ? NT - RT : 1][64];
  const int l = lane_id(), n32 = l & 31, g = l >> 5;
  const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int wv = wid / NW, sub = wid % NW, br = sub >> 1, hh = sub & 1;
  const int BH = P.B * P.H, nqt = P.nqt, nkt = P.nkt, Nq = P.Nq, Nk = P.Nk, qoff = P.qoff;
  // longest blocks (first key tiles) of every head first
  if (blockIdx.y && grid_bid<64 * W * NW>() >= (uint32_t)BH * (uint32_t)((nkt + W - 1) / W)) return;
  const int bid = (int)grid_bid<64 * W * NW>(), kt0 = W * (bid / BH), bh = bid % BH, kt = kt0 + wv;
  const int b = bh / P.H, h = bh % P.H;
  const int j = 32 * kt + n32, jc = min(j, Nk - 1);
  const bool kvalid = j < Nk;
  const int qtf_b = qt_first(kt0, qoff);  // first query tile of the block
  const uint32_t actm = nkt - kt0 >= W ? (1u << W) - 1u : (1u << (nkt - kt0)) - 1u;  // key tiles there are
  auto base = [&](int slot) {
    return (const bf16*)P.in[slot] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1];
  };
  const int kslot = br == 0 ? B_K1 : B_K2;
  // this wave's resident operand: its branch's K rows, or (wave (0, 1)) the V rows; with two branches
  // its last steps wait in LDS (in registers they spill)
  bf16x8 R[RT];
  const int chain = (BR + 1) * wv + (hh ? BR : br);  // (wave (1, 1) has none: wave (0, 1)'s, the same values)
  {
    const int slot = hh ? B_V : kslot;
    const bf16* r = base(slot) + (int64_t)jc * P.s[slot][2] + 8 * g;
#pragma unroll
    for (int t = 0; t < RT; ++t) R[t] = *reinterpret_cast<const bf16x8*>(r + 16 * t);
#pragma unroll
    for (int t = RT; t < NT; ++t) rest[chain][t - RT][l] = *reinterpret_cast<const bf16x8*>(r + 16 * t);
  }
  float rk[BR];
#pragma unroll
  for (int b2 = 0; b2 < BR; ++b2) rk[b2] = NORM ? P.norms[norm_base(P, b2 == 0 ? N_K1 : N_K2, bh) + jc] : 1.f;
  const float beta = *P.beta;
  const float pw = P.p;
  float lam = 0.f;
  if constexpr (BR == 2) lam = clamp01(*P.lam);
  const float coef = br == 0 ? 1.f : -lam;
  f32x16 AV[NDV], AK[NDK];
#pragma unroll
  for (int c = 0; c < NDV; ++c) AV[c] = f32x16{};
#pragma unroll
  for (int c = 0; c < NDK; ++c) AK[c] = f32x16{};
  unsigned visited = 0, computed = 0;

  // union walk over query tiles qtf_b .. nqt - 1, 64 per round: lane q tests query tile q0c + q
  int q0c = qtf_b - 64;
  uint64_t um = 0ull, om[BR];
  auto next_tile = [&](uint32_t& own) -> int {  // own: bit b2, the wave's key tile in branch b2
    own = 0u;
    while (um == 0ull) {
      q0c += 64;
      if (q0c >= nqt) return -1;
      const int qtl = q0c + l;
      uint32_t any = 0u;
#pragma unroll
      for (int b2 = 0; b2 < BR; ++b2) {
        const int64_t row = ((int64_t)b2 * BH + bh) * nqt + qtl;
        uint32_t bits = qtl >= nqt ? 0u : P.occ ? P.occ[row * P.occ_w + (kt0 >> 5)] >> (kt0 & 31) : 0xffffffffu;
        bits &= actm;
        // causal: key tile kt0 + r is seen from query tile qt_first(kt0 + r) on
#pragma unroll
        for (int r = 0; r < W; ++r)
          if (qtl < qt_first(kt0 + r, qoff)) bits &= ~(1u << r);
        om[b2] = wave_ballot((bits >> wv) & 1u);
        any |= bits;
      }
      um = wave_ballot(any != 0u);
    }
    const int q = __builtin_ctzll(um);
    um &= um - 1ull;
#pragma unroll
    for (int b2 = 0; b2 < BR; ++b2) own |= (uint32_t)((om[b2] >> q) & 1ull) << b2;
    return q0c + q;
  };
  BlkRows<D, W * NW> qr[BR], dr;  // the wave's share of the tile in flight
  float vrq[BR], vtq = 0.f;
  int qt;
  uint32_t own;
  auto fetch = [&]() {
    qt = next_tile(own);
    const int q0 = 32 * max(qt, 0);  // loads on every path: the waits then count them exactly
#pragma unroll
    for (int b2 = 0; b2 < BR; ++b2) {
      const int slot = b2 == 0 ? B_Q1 : B_Q2;
      qr[b2].load(base(slot), P.s[slot][2], q0, Nq, wid);
      if (NORM && wid == 0 && l < 32) vrq[b2] = P.norms[norm_base(P, b2 == 0 ? N_Q1 : N_Q2, bh) + min(q0 + l, Nq - 1)];
    }
    dr.load(base(B_DO), P.s[B_DO][2], q0, Nq, wid);
    if (wid == 0 && l < 32) vtq = beta * tau_coeff(qoff + q0 + l, P.inv_d);
  };
  WideTile wt;
  fetch();
#pragma unroll 1
  for (int it = 0; qt >= 0; ++it) {
    const int q0 = 32 * qt;
    const uint32_t cown = own;
    bf16* st = ring + (it & 1) * STAGE;
    bf16* dst = st + BR * TILE;
    float (*vs)[32] = vals[it & 1];
#pragma unroll
    for (int b2 = 0; b2 < BR; ++b2) {
      qr[b2].store(st + b2 * TILE, wid);
      if (NORM && wid == 0 && l < 32) vs[b2][l] = vrq[b2];
    }
    dr.store(dst, wid);
    if (wid == 0 && l < 32) vs[BR][l] = vtq;
    fetch();  // the next tile, in flight during this one's work
    lds_barrier();
    wt.keep_here();
    if (hh ? br == 0 && cown : (cown >> br) & 1u) {
      const bf16* src = hh ? dst : st + br * TILE;
      give16(xch[wv][hh ? BR : br], mma_chain<NT>([&](int t) { return wt.row_frag(src, t); }, [&](int t) { return t < RT ? R[t] : rest[chain][t - RT][l]; }));
    }
    lds_barrier();
    if (!cown) continue;  // (the waves of a tile agree)
    ++visited;
    const bool edge = 32 * kt + 31 > qoff + q0 || q0 + 31 >= Nq || 32 * kt + 31 >= Nk;
    // query crow(r, g) sees the key iff c_r >= lo and exists iff c_r < hi (c_r = 8 (r / 4) + r % 4)
    const int lo = (kvalid ? j - qoff - q0 : 64) - 4 * g, hi = Nq - q0 - 4 * g;
    f32x16 EV = f32x16{}, E = f32x16{};
    bool any = false;
#pragma unroll
    for (int b2 = 0; b2 < BR; ++b2) {
      if (!((cown >> b2) & 1u)) continue;
#pragma unroll
      for (int u = 0; u < 4; ++u) {  // four values at a time: all sixteen's operands at once spill
        const f32x4 S = xch[wv][b2][u][l], Dp = xch[wv][BR][u][l];
        const f32x4 tq = *reinterpret_cast<const f32x4*>(vs[BR] + 8 * u + 4 * g);
        f32x4 rq = {1.f, 1.f, 1.f, 1.f};
        if constexpr (NORM) rq = *reinterpret_cast<const f32x4*>(vs[b2] + 8 * u + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = 8 * u + e, r = 4 * u + e;
          float x = __builtin_fmaf(NORM ? S[e] * rk[b2] : S[e], rq[e], -tq[e]);
          if (edge) x = c >= lo && c < hi ? x : -1.f;
          const bool pos = x > 0.f;
          const float w = pos ? pow_p<PK>(x, pw) : 0.f;
          EV[r] = b2 == 0 ? w : __builtin_fmaf(-lam, w, EV[r]);
          any |= pos;
          if (BR == 1 || b2 == br) {
            const float ds = pos ? coef * dpow_p<PK>(x, pw) * Dp[e] : 0.f;
            E[r] = NORM ? ds * rq[e] : ds;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!P.occ && wave_ballot(any) == 0ull) continue;  // the same decision in every wave of the tile
    ++computed;
    const bf16x8 V0 = PolBF16::pack_c(EV, 0), V1 = PolBF16::pack_c(EV, 1);
#pragma unroll
    for (int c = 0; c < NDV; ++c) {
      AV[c] = PolBF16::mma(wt.tr_frag(dst, 0, c + NDV * sub), V0, AV[c]);
      AV[c] = PolBF16::mma(wt.tr_frag(dst, 1, c + NDV * sub), V1, AV[c]);
    }
    if ((cown >> br) & 1u) {
      const bf16x8 K0 = PolBF16::pack_c(E, 0), K1 = PolBF16::pack_c(E, 1);
      const bf16* src = st + br * TILE;
#pragma unroll
      for (int c = 0; c < NDK; ++c) {
        AK[c] = PolBF16::mma(wt.tr_frag(src, 0, c + NDK * hh), K0, AK[c]);
        AK[c] = PolBF16::mma(wt.tr_frag(src, 1, c + NDK * hh), K1, AK[c]);
      }
    }
  }
  const float rkb = br == 0 ? rk[0] : rk[BR - 1];
  GradRow<32 * NDK> XR;  // the key row's columns for the normalize backward
  if constexpr (NORM) {
    load_grad_row<32 * NDK>(base(kslot) + (int64_t)jc * P.s[kslot][2] + 32 * NDK * hh, XR);
    const float part = grad_row_dot<32 * NDK>(AK, XR, rkb);
    if (g == 0) dots[wv][br][hh][n32] = part;
    lds_barrier();
  }
  if (kvalid) {
    auto grow = [&](int gi, int slot) {
      return (bf16*)P.grad[gi] + (int64_t)b * P.s[slot][0] + (int64_t)h * P.s[slot][1] + (int64_t)j * P.s[slot][2];
    };
    store_grad_rows<32 * NDV, false>(AV, GradRow<32 * NDV>{}, grow(4, B_DV) + 32 * NDV * sub, 1.f, 0.f, 1.f);
    store_grad_rows<32 * NDK, NORM>(AK, XR, grow(br == 0 ? 1 : 3, br == 0 ? B_DK1 : B_DK2) + 32 * NDK * hh, rkb,
                                    NORM ? dots[wv][br][0][n32] + dots[wv][br][1][n32] : 0.f, 1.f);
  }
  if (P.stats && l == 0 && sub == 0) {
    atomicAdd(P.stats + 0, (unsigned long long)visited);
    atomicAdd(P.stats + 1, (unsigned long long)computed);
  }
}

// Both block passes over the queue of the key-major pair pass, in one launch: the workgroups
// take tickets, the key blocks (the longer ones) first, each kind longest blocks first as nearly as
// the queue's order has it.  With every list fitting the queue is empty and a workgroup leaves
// after one load (4.6 us); at a threshold scale of 0.5 nearly every block is queued
// (TDA (2, 16, 1500, 64): 162 us, 2632 us with one wave per query or key tile fetching
// its own rows).
// W = 1 or 2 where no head has more query or key tiles: the other waves of four would have no tile, and
// hold the registers of a block that has.  Its blocks are of one length and are taken in turn: the
// tickets of one counter come 11 ns apart.  With the pair passes, 8192 heads of 32 rows at a threshold
// scale of 0.4: TRA d = 64 280 us, d = 128 433 (with four waves 403, 690); TDA 404 and 691 (732, 1281).
template <int D, int BR, int PK, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(dkv_waves<D, BR, true>()))) bwd_tiles(BwdParams P) {
  TDA_BLK_LDS(D, W, true);
  __shared__ uint32_t ticket;
  const uint32_t nk = P.dkvq[0], total = nk + P.dkvq[1];
  if (total == 0u) return;
  const int BH = P.B * P.H, nqb = (P.nqt + kBwdBlk - 1) / kBwdBlk, nkb = (P.nkt + kBwdBlk - 1) / kBwdBlk;
  const uint32_t* masks = P.dkvq + kTileqHead;
  for (uint32_t turn = blockIdx.x;; turn += gridDim.x) {
    uint32_t t = turn;
    __syncthreads();  // every wave is done with the previous block's LDS and ticket
    if constexpr (W == kBwdBlk) {
      if (threadIdx.x == 0) ticket = atomicAdd(P.dkvq + 2, 1u);
      __syncthreads();
      t = (uint32_t)__builtin_amdgcn_readfirstlane((int)ticket);
    }
    if (t >= total) return;
    if (t < nk) {
      const uint32_t blk = (uint32_t)__builtin_amdgcn_readfirstlane((int)masks[(int64_t)BH * nkb + t]);
      dkv_block<D, BR, PK, true>(P, L, (int)(blk % nkb), (int)(blk / nkb),
                                 (uint32_t)__builtin_amdgcn_readfirstlane((int)masks[blk]));
    } else {
      const uint32_t k = (uint32_t)__builtin_amdgcn_readfirstlane((int)masks[2 * (int64_t)BH * nkb + (t - nk)]);
      const int j = (int)(k % (uint32_t)(BR * nqb));
      dq_block<D, BR, PK, true>(P, L, nqb - 1 - (BR == 2 ? j >> 1 : j), BR == 2 ? j & 1 : 0, (int)(k / (uint32_t)(BR * nqb)));
    }
  }
}

// ------------------------------------------------------------------ dispatch
// With pair lists the pair passes take the lists that fit, then the block tile passes the rest,
// then the sum.  With normalisation most calls leave nothing, so the block passes run from a queue
// in one launch (when the workspace holds it); without, nearly every list is past its cap and each
// pass launches a workgroup per block.
template <int D, int BR, int PK, bool NORM>
static int launch_t(const BwdParams& p, void* stream) {
  const int64_t qitems = (int64_t)BR * p.B * p.H * p.nqt, kitems = (int64_t)p.B * p.H * p.nkt;
  hipStream_t s = (hipStream_t)stream;
  BwdParams q = p;
  if (!NORM) q.dkvq = nullptr;
  if constexpr (D <= 128) {
    if (q.pairs) {
      hipLaunchKernelGGL((bwd_dq_pairs<D, BR, PK, NORM>), dim3((unsigned)qitems), dim3(64), 0, s, q);
      launched(s, "bwd_dq_pairs");
      hipLaunchKernelGGL((bwd_dkv_pairs<D, BR, PK, NORM>), dim3((unsigned)kitems), dim3(64), 0, s, q);
      launched(s, "bwd_dkv_pairs");
    }
  }
  const int BH = q.B * q.H;
  const unsigned qblocks = (unsigned)(BR * BH * ((q.nqt + kBwdBlk - 1) / kBwdBlk));  // (one block of one tile too)
  constexpr int KB = D <= 128 ? kBwdBlk : kWideKeys;
  const unsigned kblocks = (unsigned)(BH * ((q.nkt + KB - 1) / KB));
  bool queued = false;
  if constexpr (NORM && D <= 128) {
    if (q.pairs && q.dkvq) {
      // as many workgroups as the GPU's 256 CUs hold at dkv_waves waves per SIMD
      const int tiles = q.nqt > q.nkt ? q.nqt : q.nkt, W = tiles == 1 ? 1 : tiles == 2 ? 2 : kBwdBlk;
      // (of W = 1 as many as its 21 and 41 KB of LDS let in: more would wait for the first ones' whole share)
      const unsigned most = 256u * (W == 1 ? (D <= 64 ? 7 : 3) : dkv_waves<D, BR, true>() * (kBwdBlk / W)), blocks = qblocks + kblocks;
      const dim3 grid(blocks < most ? blocks : most);
      if (W == 1)
        hipLaunchKernelGGL((bwd_tiles<D, BR, PK, 1>), grid, dim3(64), 0, s, q);
      else if (W == 2)
        hipLaunchKernelGGL((bwd_tiles<D, BR, PK, 2>), grid, dim3(128), 0, s, q);
      else
        hipLaunchKernelGGL((bwd_tiles<D, BR, PK, kBwdBlk>), grid, dim3(64 * kBwdBlk), 0, s, q);
      launched(s, "bwd_tiles");
      queued = true;
    }
  }
  if (!queued) {
    bool one = false;  // a head's only tile: a block of one, as in bwd_tiles
    if constexpr (!NORM && D <= 64) {  // (d = 128: 189 us in blocks of four, 228 so, 8192 heads of 16 rows)
      one = q.nqt == 1;
      if (one) hipLaunchKernelGGL((bwd_dq_blk<D, BR, PK, NORM, 1>), dim3(qblocks), dim3(kQryThreads<D, 1>), 0, s, q);
    }
    const dim3 qgrid = D > 128 ? grid_of<kQryThreads<D, kBwdBlk>>(qblocks) : dim3(qblocks);
    if (!one) hipLaunchKernelGGL((bwd_dq_blk<D, BR, PK, NORM, kBwdBlk>), qgrid, dim3(kQryThreads<D, kBwdBlk>), 0, s, q);
    launched(s, "bwd_dq_blk");
    one = false;
    if constexpr (!NORM && D <= 128) {
      one = q.nkt == 1;
      if (one) hipLaunchKernelGGL((bwd_dkv_blk<D, BR, PK, NORM, 1>), dim3(kblocks), dim3(64), 0, s, q);
    }
    if constexpr (D <= 128) {
      if (!one) hipLaunchKernelGGL((bwd_dkv_blk<D, BR, PK, NORM, kBwdBlk>), dim3(kblocks), dim3(64 * kBwdBlk), 0, s, q);
    } else {
      hipLaunchKernelGGL((bwd_dkv_wide<BR, PK, NORM>), grid_of<128 * BR * kWideKeys>(kblocks), dim3(128 * BR * kWideKeys), 0, s, q);
    }
    launched(s, "bwd_dkv_blk");
  }
  const int e = (int)hipGetLastError();
  return e ? e : launch_bwd_finish(q, BR, qitems, stream);
}
template <int D, int BR, int PK>
static int sel_norm(const BwdParams& p, const KernelKey& k, void* s) {
  return k.normalize ? launch_t<D, BR, PK, true>(p, s) : launch_t<D, BR, PK, false>(p, s);
}
template <int D, int BR>
static int sel_pk(const BwdParams& p, const KernelKey& k, void* s) {
  switch (k.pkind) {
    case 2: return sel_norm<D, BR, 2>(p, k, s);
    case 1: return sel_norm<D, BR, 1>(p, k, s);
    default: return sel_norm<D, BR, 0>(p, k, s);
  }
}
template <int D>
static int sel_br(const BwdParams& p, const KernelKey& k, void* s) {
  return k.branches == 2 ? sel_pk<D, 2>(p, k, s) : sel_pk<D, 1>(p, k, s);
}

int launch_bwd_fast(const BwdParams& p, const KernelKey& k, void* stream) {
  return k.d == 128 ? sel_br<128>(p, k, stream) : sel_br<64>(p, k, stream);
}

// head_dim 256 has no pair lists: the block passes over the bitmask (or every causal tile).
int launch_bwd_blk256(const BwdParams& p0, const KernelKey& k, void* stream) {
  BwdParams p = p0;
  p.pairs = nullptr;
  p.dkvq = nullptr;
  return sel_br<256>(p, k, stream);
}

// The pair passes on fp32 rows (the fp32 backward's launcher in tda_bwd.hip runs the tile passes
// for what they leave).
template <int D, int BR, int PK, bool NORM>
static int pairs_f32_t(const BwdParams& p, hipStream_t s) {
  const int64_t qitems = (int64_t)BR * p.B * p.H * p.nqt, kitems = (int64_t)p.B * p.H * p.nkt;
  hipLaunchKernelGGL((bwd_dq_pairs<D, BR, PK, NORM, float>), dim3((unsigned)qitems), dim3(64), 0, s, p);
  launched(s, "bwd_dq_pairs");
  hipLaunchKernelGGL((bwd_dkv_pairs<D, BR, PK, NORM, float>), dim3((unsigned)kitems), dim3(64), 0, s, p);
  launched(s, "bwd_dkv_pairs");
  return (int)hipGetLastError();
}
template <int D, int BR, int PK>
static int pairs_f32_norm(const BwdParams& p, const KernelKey& k, hipStream_t s) {
  return k.normalize ? pairs_f32_t<D, BR, PK, true>(p, s) : pairs_f32_t<D, BR, PK, false>(p, s);
}
template <int D, int BR>
static int pairs_f32_pk(const BwdParams& p, const KernelKey& k, hipStream_t s) {
  switch (k.pkind) {
    case 2: return pairs_f32_norm<D, BR, 2>(p, k, s);
    case 1: return pairs_f32_norm<D, BR, 1>(p, k, s);
    default: return pairs_f32_norm<D, BR, 0>(p, k, s);
  }
}
template <int D>
static int pairs_f32_br(const BwdParams& p, const KernelKey& k, hipStream_t s) {
  return k.branches == 2 ? pairs_f32_pk<D, 2>(p, k, s) : pairs_f32_pk<D, 1>(p, k, s);
}
int launch_bwd_pairs_f32(const BwdParams& p, const KernelKey& k, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  return k.d == 128 ? pairs_f32_br<128>(p, k, s) : pairs_f32_br<64>(p, k, s);
}

}  // namespace tda
