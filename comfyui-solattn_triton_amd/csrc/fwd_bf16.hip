// BF16 Sol-Attn forward on gfx950 MFMA.
//
// One workgroup per (batch, head, query block of BLK rows); each wave owns 32
// query rows, two waves share a SIMD. Work is a list of 64-key tiles staged in
// LDS by global -> LDS copies (no VGPR staging):
//   pooled tiles  64 pooled keys kc_j / values vc_j, masked to the approximate
//                 blocks of this query block, softmax weight x len_j
//                 (/root/reference/_tri_fwd.py:288-308);
//   exact tiles   64 tokens of an exact block (/root/reference/_tri_fwd.py:310-340).
// All tiles feed one online softmax per query row, which is exact under any
// tile order (up to fp32 rounding), through a software pipeline of half tiles
// (32 keys): step n computes S(n+1) = K(n+1) Q^T, O += P(n-1) V(n-1) and the
// softmax of S(n) in one instruction stream, hand-ordered from inline-asm MFMAs
// and softmax exp pairs (fwd_common.hpp), which the compiler's own schedule did
// not give.
//
// MFMA dataflow (v_mfma_f32_32x32x16_bf16): S^T = K . Q^T puts one query row
// per lane column, so row max / sum need one cross-lane step (lanes 32 apart,
// v_permlane32_swap) and the S accumulator converts in place into the B
// operand of O^T += V^T . P^T. V stays row-major in LDS and ds_read_b64_tr_b16
// delivers it transposed as the MFMA A operand. XOR-swizzled 16-byte chunks
// keep the LDS reads conflict free (fwd_common.hpp).
#include "common.hpp"
#include "fwd_common.hpp"

namespace solattn {
namespace bf16fwd {

// Three-stage step over half tiles of 32 keys: S(n+1) = K(n+1) Q^T (8 MFMAs),
// O += P(n-1) V(n-1) (8 MFMAs) and the softmax of S(n) (8 pairs of exps) in one
// hand-ordered stream: slot i issues score MFMA i, the exps of P(n) word i, then
// P.V MFMA i; the K and V operands of slot i + 2 are read at the top of slot i
// (the empty asm with a memory clobber keeps the reads there). O is rescaled to
// the new running max after the P(n-1) V(n-1) products. HH: the half of its tile
// that n is. psum: this lane's sum of the tile's P, started by half 0 and carried
// on by half 1 (POOLED, the keys of n are pooled keys: of the fp32 p). kl, vl:
// this lane's operand addresses in K(n+1) and V(n-1). Returns the factor that the
// row sum so far takes with a new running max.
// Lazy tile max: the exps use the running max as it stands, and the tile's max
// is taken only when a lane's row sum exceeds 255. No sum above 255 means every
// p <= 255, i.e. every score is below the running max + log2(255.5) <
// kMaxSlack, so the tile would not have moved the max: the running max evolves
// as with the max taken every step.
// Raised wave priority for the step's stream: the issue arbiter then prefers a
// wave inside its MFMAs over one at its copies or barrier (without it, 6%
// slower at block 64 and 32760 tokens).
// 64 channels halve the MFMAs: one of each product per two slots.
template <int D, bool POOLED, int HH>
__device__ __forceinline__ float half_step(SoftmaxStateOf<D / 32>& st, const f32x16& sc, f32x16& sn,
                                          const bf16x8 (&pp)[2], bf16x8 (&pn)[2], uint32_t kl,
                                          uint32_t vl, const bf16x8 (&q)[D / 16], float c, float& psum) {
  static_assert(kMaxSlack >= 8.f, "the lazy test relies on 255 < 2^kMaxSlack");
  constexpr int ND = D / 32, NM = D / 16;  // MFMAs of each product
  constexpr int SLOTS = 8 / NM;            // slots per MFMA of each
  bf16x8 ka[3], va[3];
  uint32_t pw[2][4];
  const float before = HH == 0 ? 0.f : psum;
  if constexpr (HH == 0) psum = 0.f;
  const float neg = -st.m;
  ka[0] = k_op_x<D>(kl, 0, 0);
  ka[1] = k_op_x<D>(kl, 0, 1);
  va[0] = v_op_x<D>(vl, 0, 0);
  va[1] = v_op_x<D>(vl, 0, 1);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = i / SLOTS;  // MFMA j of each product: scores first, P.V after the slots' exps
    if (i % SLOTS == 0) {
      if (j + 2 < NM) {
        ka[(j + 2) % 3] = k_op_x<D>(kl, 0, j + 2);
        va[(j + 2) % 3] = v_op_x<D>(vl, (j + 2) / ND, (j + 2) % ND);
        asm volatile("" ::: "memory");
      }
      if (j == 0)
        mfma_v0(sn, ka[0], q[0]);
      else
        mfma_v(sn, ka[j % 3], q[j]);
    }
    pw[i >> 2][i & 3] = POOLED ? exp_pair_f32sum(sc[2 * i], sc[2 * i + 1], c, neg, psum)
                               : exp_pair(sc[2 * i], sc[2 * i + 1], c, neg, psum);
    if (i % SLOTS == SLOTS - 1) {
      if (j == 0)
        mfma_v_first(st.acc[0], va[0], pp[0]);
      else if (j == NM - 1)
        mfma_v_tie(st.acc[ND - 1], va[j % 3], pp[1], sn);
      else
        mfma_v(st.acc[j % ND], va[j % 3], pp[j / ND]);
    }
    if (i == 0) __builtin_amdgcn_s_setprio(1);
  }
  __builtin_amdgcn_s_setprio(0);
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    pn[ks] = __builtin_bit_cast(bf16x8, make_uint4(pw[ks][0], pw[ks][1], pw[ks][2], pw[ks][3]));
  float alpha = 1.f;
  if (__any(!(psum <= 255.f))) {  // (also catches inf / NaN)
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[r]);
    const float m_new = new_max(st.m, xhalf_max(mx) * c, alpha);
    if (__any(m_new != st.m)) {  // lanes whose max stays recompute the same P
      st.m = m_new;
      psum = before * alpha;
      if constexpr (POOLED) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sc[r], c, -m_new));
          pn[r >> 3][r & 7] = static_cast<__bf16>(p);
          psum += p;
        }
      } else {
        psum = exp8<0>(sc, c, -m_new, pn[0], psum);
        psum = exp8<8>(sc, c, -m_new, pn[1], psum);
      }
      mfma_fence(st.acc);  // the rescale reads O
      rescale(st, alpha);
    }
  }
  return alpha;
}

// The score of key `key` (of the 32 of s) in the lanes that hold it, -inf elsewhere.
__device__ __forceinline__ float score_of_key(const f32x16& s, int key, int half) {
  float x = -INFINITY;
#pragma unroll
  for (int r = 0; r < 16; ++r) x = 8 * (r >> 2) + 4 * half + (r & 3) == key ? s[r] : x;
  return x;
}

// The forward. Workgroups of 2 waves at block 64 (four per CU), 4 at block 128
// (two per CU): two waves per SIMD. K and V hold two half tiles of 32 keys each
// (32 KiB). Every tile takes two half steps of the pipeline, in the order pooled,
// ragged exact (the short last block's, its rows past T masked), full exact at
// block 64, and full exact, ragged exact, pooled at block 128. The pooled key of
// a short last block weighs its own length.
//
// Bound: at 32760 tokens the MFMAs at the power-limited clock and the tile
// copies (block 64: without them, results wrong by construction, the two-stage
// form of this kernel ran 19% faster; with all of them hitting L2, 8%); at 4096
// tokens (1.5 workgroups a slot at block 64) the workgroup's own latency.
// Half tiles against a two-stage step over whole tiles at block 64 (K copied
// behind 16 bare P.V MFMAs, V behind QK and the exps): every copy gets a whole
// step, the MFMAs of both products hide the exps, and the scores take 32
// registers less, so the pooled tiles fit the pipeline. Calls: 32760 tokens 2835
// -> 2737 us, 12133 packed 623 -> 606, 4096 91.2 -> 87.4. At block 128 against a
// three-stage step over whole tiles, double buffered in 64 KiB, with plain
// pooled tiles: 32760 tokens 2370 -> 2325 us, 75600 tokens 21.2 -> 21.0 ms; four
// half buffers with copies two steps ahead were slower (2400 us).
// The order of the tiles, the max of the whole first tile and the row sums of whole
// tiles are those of that whole-tile step, and so are the results, but for rows whose
// max a later tile moves. Against a max of 32 keys and the short last block's tile
// first, on a plain path: 32760 tokens 2744 -> 2742 us at block 64 and 2379 -> 2384
// at block 128, 4096 tokens 81.9 -> 82.0, 1000 tokens 29.35 -> 29.8.
template <int BLK, int D>
__global__ void __launch_bounds__(BLK * 2) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2)))
fwd_bf16_kernel(const uint16_t* __restrict__ q, int64_t sq_b, int64_t sq_t, int64_t sq_h,
                const uint16_t* __restrict__ k, int64_t sk_b, int64_t sk_t, int64_t sk_h,
                const uint16_t* __restrict__ v, int64_t sv_b, int64_t sv_t, int64_t sv_h,
                const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, int64_t npad,
                const int32_t* __restrict__ counts, const uint32_t* __restrict__ mask, int T, int H, int NT, int W, float c,
                uint16_t* __restrict__ o, int64_t so_b, int64_t so_t, int64_t so_h) {
  constexpr int NTHREADS = BLK * 2;
  constexpr uint32_t kHalfBytes = kKeys * D;  // half a tile: 32 rows of 2 D bytes
  __shared__ __align__(256) uint16_t kbuf[kKeys * D];
  __shared__ __align__(256) uint16_t vbuf[kKeys * D];
  __shared__ TileList tl;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, half = lane >> 5;
  int bh, qb;
  tile_coords_lpt<kLptTokens / BLK>(counts, NT, bh, qb);
  const int b = bh / H, h = bh % H;
  const int64_t row = static_cast<int64_t>(bh) * NT + qb;

  const int ntiles = build_tile_list<BLK>(tl, mask, row, NT, W, T);
  if (ntiles == 0) return;  // cannot happen for routed masks: the diagonal is exact
  // (the lists' sizes made scalar: the loops and branches over tiles are uniform)
  const int npool = __builtin_amdgcn_readfirstlane(tl.npool);
  const int nrag = __builtin_amdgcn_readfirstlane(ragged_tiles(tl, NT, T));
  const int nfull = __builtin_amdgcn_readfirstlane(tl.nexact) - nrag;
  // the order: tile t is pooled from pool0 on, ragged at rag0 (if there is one),
  // full exact from full0 on
  constexpr bool kPoolFirst = BLK == 64;
  const int pool0 = kPoolFirst ? 0 : nfull + nrag, rag0 = kPoolFirst ? npool : nfull;
  const int full0 = kPoolFirst ? npool + nrag : 0, last = npool + nrag + nfull - 1;

  const KVSource src{k + b * sk_b + h * sk_h, sk_t, v + b * sv_b + h * sv_h, sv_t,
                     kc + (static_cast<int64_t>(b) * npad * H + h) * D,
                     static_cast<int64_t>(H) * D, vc + (static_cast<int64_t>(b) * npad * H + h) * D};
  CopyOffsets<NTHREADS, D> off;
  off.init(sk_t, sv_t);
  const uint32_t kb = lds_addr(kbuf), vb = lds_addr(vbuf);  // LDS byte addresses
  const uint32_t kl = k_lane<D>(kb, col, half), vl = v_lane<D>(vb, lane);  // this lane's operands
  // Half hh of a tile into K or V half buffer hh. (The lambdas are always_inline: one
  // that is called in several places would take its captures through memory.)
  const auto full_first = [&](int e) __attribute__((always_inline)) { return exact_first<BLK>(tl, e); };
  const auto issue_k_at = [&](int first, int hh) __attribute__((always_inline)) {
    issue_half<NTHREADS, D>(kb + hh * kHalfBytes, src.k + static_cast<int64_t>(first + 32 * hh) * src.sk,
                         src.sk, off.k);
  };
  const auto issue_v_at = [&](int first, int hh) __attribute__((always_inline)) {
    issue_half<NTHREADS, D>(vb + hh * kHalfBytes, src.v + static_cast<int64_t>(first + 32 * hh) * src.sv,
                         src.sv, off.v);
  };
  const auto issue_pooled = [&](int p, int kv, int hh) __attribute__((always_inline)) {
    issue_clamped_half<NTHREADS, D>((kv == 0 ? kb : vb) + hh * kHalfBytes, kv, pooled_desc(tl, p, NT), hh, src);
  };
  const auto issue_ragged = [&](int kv, int hh) __attribute__((always_inline)) {
    issue_clamped_half<NTHREADS, D>((kv == 0 ? kb : vb) + hh * kHalfBytes, kv,
                                    exact_desc<BLK>(tl, tl.nexact - 1, T, NT), hh, src);
  };
  const auto issue_any_k = [&](int t, int hh) __attribute__((always_inline)) {
    if (nrag && t == rag0)
      issue_ragged(0, hh);
    else if (t >= pool0 && t < pool0 + npool)
      issue_pooled(t - pool0, 0, hh);
    else
      issue_k_at(full_first(t - full0), hh);
  };
  const bool first_pooled = npool && pool0 == 0, first_ragged = nrag && rag0 == 0;
  issue_any_k(0, 0);
  issue_any_k(0, 1);
  if (first_pooled)
    issue_pooled(0, 1, 0);
  else if (first_ragged)
    issue_ragged(1, 0);
  else
    issue_v_at(full_first(0), 0);

  // This wave's 32 query rows as the B operand of S^T = K Q^T (rows past T
  // repeat row T - 1 and are not stored).
  const int qrow = qb * BLK + wave * 32 + col;
  bf16x8 qreg[D / 16];
  {
    const uint16_t* qp = q + b * sq_b + static_cast<int64_t>(min(qrow, T - 1)) * sq_t + h * sq_h + half * 8;
#pragma unroll
    for (int cc = 0; cc < D / 16; ++cc)
      qreg[cc] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + cc * 16));
  }

  SoftmaxStateOf<D / 32> st;
  st.init();

  // The tiles by half tiles n = 2t, 2t + 1. On entry to step n: S(n) and P(n-1)
  // in registers, K(n+1) and V(n-1) in LDS; the step copies K(n+2) over K(n) and
  // V(n) over V(n-2), so a copy has a whole step to land. K of the tile past the
  // last is clamped to it: a redundant copy that nothing reads.
  f32x16 sa, sb;  // scores of the halves 0 and 1
  bf16x8 pa[2], pb[2];
  float psum = 0.f;
  const uint32_t kl1 = kl + kHalfBytes, vl1 = vl + kHalfBytes;
  const auto land = [&]() __attribute__((always_inline)) {
    wait_tile_copies();
    __syncthreads();
  };
  // The pooled tile with a short last block's key, that key's score (-inf in the
  // lanes without it), and the weight it lacks of BLK.
  const int klast = npool ? NT - 1 - tl.pchunk[npool - 1] * kKeys : kKeys;
  const int pshort = T % BLK != 0 && klast < kKeys ? npool - 1 : -1;
  float slast = -INFINITY;

  // Step 0, without a stream: the running max comes from the whole first tile, so
  // both halves' scores come first. (P is rounded relative to that max, and the
  // keys at it round to nothing: with a max over the first 32 keys the result was
  // 0.02-0.45% further from the exact one at block 64.)
  land();
  {
    const uint64_t keep = first_pooled ? tl.pmask[0] : first_ragged ? exact_desc<BLK>(tl, tl.nexact - 1, T, NT).amask : ~0ull;
    f32x16 s[2];
    const f32x16 zero = {};
#pragma unroll
    for (int cc = 0; cc < D / 16; ++cc) s[0] = mfma_bf16(k_op_x<D>(kl, 0, cc), qreg[cc], cc == 0 ? zero : s[0]);
    __syncthreads();  // every wave is done with K(0)
    issue_any_k(min(1, last), 0);
#pragma unroll
    for (int cc = 0; cc < D / 16; ++cc) s[1] = mfma_bf16(k_op_x<D>(kl1, 0, cc), qreg[cc], cc == 0 ? zero : s[1]);
    mask_scores(s, keep);
    float mx = -INFINITY;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[m][r]);
    st.m = xhalf_max(mx) * c;
    if (first_pooled) {
      if (pshort == 0) slast = score_of_key(s[0], klast, half);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[0][r], c, -st.m));
        pa[r >> 3][r & 7] = static_cast<__bf16>(p);
        psum += p;
      }
    } else {
      psum = exp8<0>(s[0], c, -st.m, pa[0], psum);
      psum = exp8<8>(s[0], c, -st.m, pa[1], psum);
    }
    sb = s[1];
  }
  mfma_fence(st.acc);  // O's zeros are in their registers before the asm MFMAs that add to them
  land();

  // The half steps of the three kinds of tiles.
  const auto pooled_next_k = [&](int p, int hh) __attribute__((always_inline)) {
    if (!kPoolFirst || p + 1 < npool)
      issue_pooled(min(p + 1, npool - 1), 0, hh);
    else
      issue_any_k(min(npool, last), hh);
  };
  const auto pooled_half0 = [&](int p) __attribute__((always_inline)) {
    pooled_next_k(p, 0);
    issue_pooled(p, 1, 0);
    mask_scores(sa, static_cast<uint32_t>(tl.pmask[p]));
    if (p == pshort) slast = score_of_key(sa, klast, half);
    st.l *= half_step<D, true, 0>(st, sa, sb, pb, pa, kl1, vl1, qreg, c, psum);
    land();
  };
  const auto pooled_half1 = [&](int p) __attribute__((always_inline)) {
    pooled_next_k(p, 1);
    issue_pooled(p, 1, 1);
    mask_scores(sb, static_cast<uint32_t>(tl.pmask[p] >> 32));
    if (p == pshort) slast = fmaxf(slast, score_of_key(sb, klast - 32, half));
    const float alpha = half_step<D, true, 1>(st, sb, sa, pa, pb, kl, vl, qreg, c, psum);
    psum *= static_cast<float>(BLK);
    if (p == pshort)
      psum = fmaf(__builtin_amdgcn_exp2f(fmaf(slast, c, -st.m)), static_cast<float>(T - NT * BLK), psum);
    st.l = fmaf(st.l, alpha, psum);
    land();
  };
  const auto ragged_half0 = [&]() __attribute__((always_inline)) {
    issue_any_k(min(rag0 + 1, last), 0);
    issue_ragged(1, 0);
    mask_scores(sa, static_cast<uint32_t>(exact_desc<BLK>(tl, tl.nexact - 1, T, NT).amask));
    st.l *= half_step<D, false, 0>(st, sa, sb, pb, pa, kl1, vl1, qreg, c, psum);
    land();
  };
  const auto ragged_half1 = [&]() __attribute__((always_inline)) {
    issue_any_k(min(rag0 + 1, last), 1);
    issue_ragged(1, 1);
    mask_scores(sb, static_cast<uint32_t>(exact_desc<BLK>(tl, tl.nexact - 1, T, NT).amask >> 32));
    const float alpha = half_step<D, false, 1>(st, sb, sa, pa, pb, kl, vl, qreg, c, psum);
    st.l = fmaf(st.l, alpha, psum);
    land();
  };
  // f0, f1: the first token rows of full tiles e and e + 1, read from the LDS list
  // an iteration ahead, so no copy waits on an LDS read
  int f0 = 0, f1 = 0;
  // (behind: K of the tile behind the last full one comes next)
  const auto full_next_k = [&](int hh, bool behind) __attribute__((always_inline)) {
    if (behind)
      issue_any_k(min(nfull, last), hh);
    else
      issue_k_at(f1, hh);
  };
  const auto full_half0 = [&](bool behind) __attribute__((always_inline)) {
    full_next_k(0, behind);
    issue_v_at(f0, 0);
    st.l *= half_step<D, false, 0>(st, sa, sb, pb, pa, kl1, vl1, qreg, c, psum);
    land();
  };
  const auto full_half1 = [&](int e, bool behind) __attribute__((always_inline)) {
    full_next_k(1, behind);
    issue_v_at(f0, 1);
    const float alpha = half_step<D, false, 1>(st, sb, sa, pa, pb, kl, vl, qreg, c, psum);
    st.l = fmaf(st.l, alpha, psum);
    asm volatile("" ::: "memory");  // the list read stays behind the MFMA stream
    f0 = f1;
    f1 = full_first(min(e + 2, nfull - 1));
    land();
  };

  // The tiles in order; half 0 of the first one is step 0.
  const auto pooled_tiles = [&]() __attribute__((always_inline)) {
    if (npool == 0) return;
    int p = 0;
    if constexpr (kPoolFirst) pooled_half1(p++);
    for (; p < npool; ++p) {
      if (kPoolFirst || pool0 + p > 0) pooled_half0(p);
      pooled_half1(p);
    }
  };
  const auto ragged_tile = [&]() __attribute__((always_inline)) {
    if (nrag == 0) return;
    if (rag0 > 0) ragged_half0();
    ragged_half1();
  };
  const auto full_tiles = [&]() __attribute__((always_inline)) {
    if (nfull == 0) return;
    f0 = full_first(0);
    f1 = full_first(min(1, nfull - 1));
    if constexpr (kPoolFirst) {
      for (int e = 0; e < nfull; ++e) {
        if (full0 + e > 0) full_half0(false);
        full_half1(e, false);
      }
    } else {
      int e = 0;
      if (nfull > 1) {
        full_half1(e++, false);
        for (; e < nfull - 1; ++e) {
          full_half0(false);
          full_half1(e, false);
        }
        full_half0(true);
      }
      full_half1(e, true);
    }
  };
  if constexpr (kPoolFirst) {
    pooled_tiles();
    ragged_tile();
    full_tiles();
  } else {
    full_tiles();
    ragged_tile();
    pooled_tiles();
  }
  // P.V of the last half tile
  mfma_fence(st.acc);
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const int ks = i / (D / 32), dt = i % (D / 32);
    st.acc[dt] = mfma_bf16(v_op_x<D>(vl1, ks, dt), pb[ks], st.acc[dt]);
  }
  wait_tile_copies();

  store_rows(st, o + b * so_b + h * so_h, so_t, qrow, T, half);
}

}  // namespace bf16fwd
}  // namespace solattn

using namespace solattn;

namespace solattn {

int fwd_bf16(const uint16_t* q, int64_t sq_b, int64_t sq_t, int64_t sq_h, const uint16_t* k,
             int64_t sk_b, int64_t sk_t, int64_t sk_h, const uint16_t* v, int64_t sv_b, int64_t sv_t,
             int64_t sv_h, const uint16_t* kc, const uint16_t* vc, int64_t npad, const int32_t* counts,
             const uint32_t* mask, int64_t B, int64_t T, int64_t H, int64_t D, int64_t block,
             float scale, uint16_t* o, int64_t so_b, int64_t so_t, int64_t so_h, hipStream_t s) {
  SOLATTN_REQUIRE(D == 64 || D == kD, SOLATTN_EUNSUPPORTED, "fwd_bf16: head_dim %lld", (long long)D);
  if (int rc = check_fwd_args(q, sq_b, sq_t, sq_h, k, sk_b, sk_t, sk_h, v, sv_b, sv_t, sv_h, kc,
                              vc, npad, counts, mask, B, T, H, block, o, so_b, so_t, so_h, "fwd_bf16"))
    return rc;
  const int64_t NT = cdiv(T, block);
  const int W = static_cast<int>(cdiv(NT, 32));
  const float c = scale * kLog2e;
  const uint32_t grid = static_cast<uint32_t>(B * H * NT);
  const auto kern = D == 64 ? (block == 128 ? bf16fwd::fwd_bf16_kernel<128, 64> : bf16fwd::fwd_bf16_kernel<64, 64>)
                            : (block == 128 ? bf16fwd::fwd_bf16_kernel<128, 128> : bf16fwd::fwd_bf16_kernel<64, 128>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(static_cast<uint32_t>(block) * 2), blist_lds_bytes(NT), s, q,
                     sq_b, sq_t, sq_h, k, sk_b, sk_t, sk_h, v, sv_b, sv_t, sv_h, kc, vc, npad, counts,
                     mask, static_cast<int>(T), static_cast<int>(H), static_cast<int>(NT), W, c, o, so_b,
                     so_t, so_h);
  return check_launch("fwd_bf16");
}

}  // namespace solattn

extern "C" int solattn_fwd_bf16(const uint16_t* q, int64_t sq_b, int64_t sq_t, int64_t sq_h,
                                const uint16_t* k, int64_t sk_b, int64_t sk_t, int64_t sk_h,
                                const uint16_t* v, int64_t sv_b, int64_t sv_t, int64_t sv_h,
                                const uint16_t* kc, const uint16_t* vc, int64_t npad,
                                const int32_t* counts, const uint32_t* mask, int64_t B, int64_t T, int64_t H, int64_t D,
                                int64_t block, float scale, uint16_t* o, int64_t so_b,
                                int64_t so_t, int64_t so_h, solattn_stream_t stream) {
  clear_error();
  SOLATTN_REQUIRE(D == kD, SOLATTN_EUNSUPPORTED, "fwd_bf16: head_dim %lld != 128", (long long)D);
  return fwd_bf16(q, sq_b, sq_t, sq_h, k, sk_b, sk_t, sk_h, v, sv_b, sv_t, sv_h, kc, vc, npad, counts,
                  mask, B, T, H, D, block, scale, o, so_b, so_t, so_h, reinterpret_cast<hipStream_t>(stream));
}
