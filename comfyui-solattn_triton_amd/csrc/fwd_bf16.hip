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
// tile order (up to fp32 rounding). The pooled and the full exact tiles run
// through a software pipeline of half tiles (32 keys): step n computes S(n+1) =
// K(n+1) Q^T, O += P(n-1) V(n-1) and the softmax of S(n) in one instruction
// stream, hand-ordered from inline-asm MFMAs and softmax exp pairs
// (fwd_common.hpp), which the compiler's own schedule did not give. The tile of
// a short last block goes through a plain path first.
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
// the new running max after the P(n-1) V(n-1) products. PV = false: the first
// half tile, which has no value product to add. POOLED: the keys of n are
// pooled keys of whole blocks (masked scores -inf), each weighing BLK in the row
// sum, which adds the fp32 p. kl, vl: this lane's operand addresses in K(n+1)
// and V(n-1).
// Lazy tile max: the exps use the running max as it stands, and the tile's max
// is taken only when a lane's row sum exceeds 255. No sum above 255 means every
// p <= 255, i.e. every score is below the running max + log2(255.5) <
// kMaxSlack, so the tile would not have moved the max: the running max evolves
// as with the max taken every step. The first tile of a workgroup (running max
// -inf, p = inf or NaN) always takes that path.
// Raised wave priority for the step's stream: the issue arbiter then prefers a
// wave inside its MFMAs over one at its copies or barrier (without it, 6%
// slower at block 64 and 32760 tokens).
// 64 channels halve the MFMAs: one of each product per two slots.
template <int BLK, int D, bool POOLED, bool PV>
__device__ __forceinline__ void half_step(SoftmaxStateOf<D / 32>& st, const f32x16& sc, f32x16& sn,
                                          const bf16x8 (&pp)[2], bf16x8 (&pn)[2], uint32_t kl,
                                          uint32_t vl, const bf16x8 (&q)[D / 16], float c) {
  static_assert(kMaxSlack >= 8.f, "the lazy test relies on 255 < 2^kMaxSlack");
  constexpr int ND = D / 32, NM = D / 16;  // MFMAs of each product
  constexpr int SLOTS = 8 / NM;            // slots per MFMA of each
  bf16x8 ka[3], va[3];
  uint32_t pw[2][4];
  float psum = 0.f;
  const float neg = -st.m;
  ka[0] = k_op_x<D>(kl, 0, 0);
  ka[1] = k_op_x<D>(kl, 0, 1);
  if constexpr (PV) {
    va[0] = v_op_x<D>(vl, 0, 0);
    va[1] = v_op_x<D>(vl, 0, 1);
  }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int j = i / SLOTS;  // MFMA j of each product: scores first, P.V after the slots' exps
    if (i % SLOTS == 0) {
      if (j + 2 < NM) {
        ka[(j + 2) % 3] = k_op_x<D>(kl, 0, j + 2);
        if constexpr (PV) va[(j + 2) % 3] = v_op_x<D>(vl, (j + 2) / ND, (j + 2) % ND);
        asm volatile("" ::: "memory");
      }
      if (j == 0)
        mfma_v0(sn, ka[0], q[0]);
      else
        mfma_v(sn, ka[j % 3], q[j]);
    }
    pw[i >> 2][i & 3] = POOLED ? exp_pair_f32sum(sc[2 * i], sc[2 * i + 1], c, neg, psum)
                               : exp_pair(sc[2 * i], sc[2 * i + 1], c, neg, psum);
    if constexpr (PV) {
      if (i % SLOTS == SLOTS - 1) {
        if (j == 0)
          mfma_v_first(st.acc[0], va[0], pp[0]);
        else if (j == NM - 1)
          mfma_v_tie(st.acc[ND - 1], va[j % 3], pp[1], sn);
        else
          mfma_v(st.acc[j % ND], va[j % 3], pp[j / ND]);
      }
    }
    if (i == 0) __builtin_amdgcn_s_setprio(1);
  }
  __builtin_amdgcn_s_setprio(0);
  if constexpr (!PV) mfma_fence(sn);
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    pn[ks] = __builtin_bit_cast(bf16x8, make_uint4(pw[ks][0], pw[ks][1], pw[ks][2], pw[ks][3]));
  float alpha = 1.f;
  if (__any(!(psum <= 255.f))) {  // (also catches inf / NaN)
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[r]);
    const float m_new = new_max(st.m, xhalf_max(mx) * c, alpha);
    // A first half tile without a single unmasked pooled key (its 32 blocks all
    // exact) leaves the max at -inf: its P are 0, not exp2(-inf + inf).
    const bool none = POOLED && m_new == -INFINITY;
    if (__any(m_new != st.m || none)) {  // lanes whose max stays recompute the same P
      st.m = m_new;
      psum = 0.f;
      if constexpr (POOLED) {
        const float neg_new = none ? 0.f : -m_new;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sc[r], c, neg_new));
          pn[r >> 3][r & 7] = static_cast<__bf16>(p);
          psum += p;
        }
      } else {
        psum = exp8<0>(sc, c, -m_new, pn[0], psum);
        psum = exp8<8>(sc, c, -m_new, pn[1], psum);
      }
      if constexpr (PV) mfma_fence(st.acc);  // the rescale reads O
      rescale(st, alpha);
    }
  }
  st.l = fmaf(st.l, alpha, POOLED ? psum * static_cast<float>(BLK) : psum);
}

// The forward. Workgroups of 2 waves at block 64 (four per CU), 4 at block 128
// (two per CU): two waves per SIMD. K and V hold two half tiles of 32 keys each
// (32 KiB). Tile order: the tile of a short last block, if any, through the
// plain path (as a ragged exact tile, or inside its pooled tile, where it weighs
// its own length); then the pooled and the full exact tiles through the
// pipeline, two half steps a tile.
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
  // The plain tile: a ragged exact one, or the pooled tile of a short last block.
  const bool rag = ragged_tiles(tl, NT, T) != 0;
  const bool tail = T % BLK != 0 && tl.last != NT - 1;
  const int nplain = rag || tail ? 1 : 0;
  const int npool = tl.npool - (tail ? 1 : 0);  // pipelined pooled tiles, first in order
  const int npipe = ntiles - nplain;

  const KVSource src{k + b * sk_b + h * sk_h, sk_t, v + b * sv_b + h * sv_h, sv_t,
                     kc + (static_cast<int64_t>(b) * npad * H + h) * D,
                     static_cast<int64_t>(H) * D, vc + (static_cast<int64_t>(b) * npad * H + h) * D};
  CopyOffsets<NTHREADS, D> off;
  off.init(sk_t, sv_t);
  const uint32_t kb = lds_addr(kbuf), vb = lds_addr(vbuf);  // LDS byte addresses
  const uint32_t kl = k_lane<D>(kb, col, half), vl = v_lane<D>(vb, lane);  // this lane's operands
  // Half hh of pipelined tile t (pooled tiles, then the full exact tiles) into
  // K or V half buffer hh.
  const auto first_of = [&](int t) { return exact_first<BLK>(tl, max(t - npool, 0)); };
  const auto issue_k_at = [&](int first, int hh) {
    issue_half<NTHREADS, D>(kb + hh * kHalfBytes, src.k + static_cast<int64_t>(first + 32 * hh) * src.sk,
                         src.sk, off.k);
  };
  const auto issue_v_at = [&](int first, int hh) {
    issue_half<NTHREADS, D>(vb + hh * kHalfBytes, src.v + static_cast<int64_t>(first + 32 * hh) * src.sv,
                         src.sv, off.v);
  };
  const auto issue_any = [&](int t, int kv, int hh) {
    if (t >= npool) {
      if (kv == 0) issue_k_at(first_of(t), hh); else issue_v_at(first_of(t), hh);
    } else {
      issue_pooled_half<NTHREADS, D>((kv == 0 ? kb : vb) + hh * kHalfBytes, kv, pooled_desc(tl, t, NT), hh, src);
    }
  };
  const auto issue_start = [&] {  // what the first half steps need
    issue_any(0, 0, 0);
    issue_any(0, 0, 1);
    issue_any(0, 1, 0);
  };
  const auto plain_desc = [&] {
    return rag ? exact_desc<BLK>(tl, tl.nexact - 1, T, NT) : pooled_desc(tl, tl.npool - 1, NT);
  };
  if (nplain) {
    issue_generic<NTHREADS, D>(kb, 0, plain_desc(), src);
    issue_generic<NTHREADS, D>(vb, 1, plain_desc(), src);
  } else {
    issue_start();
  }

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

  // ---- the short last block's tile
  if (nplain) {
    wait_tile_copies();
    __syncthreads();
    f32x16 s[2];
    qk_tile<D>(kl, qreg, s);
    finish_tile<BLK>(st, s, vl, plain_desc(), c, lane, NT, T);
    __syncthreads();  // every wave is done with K and V
    if (npipe > 0) issue_start();
  }

  // ---- pooled and full exact tiles, pipelined by half tiles n = 2t, 2t + 1. On
  // entry to step n: S(n) and P(n-1) in registers, K(n+1) and V(n-1) in LDS; the
  // step copies K(n+2) over K(n) and V(n) over V(n-2), so a copy has a whole step
  // to land. K of the tile past the last is clamped to it: a redundant copy that
  // nothing reads.
  if (npipe > 0) {
    f32x16 sa, sb;
    bf16x8 pa[2], pb[2];
    wait_tile_copies();
    __syncthreads();
    {
      const f32x16 zero = {};
#pragma unroll
      for (int cc = 0; cc < D / 16; ++cc) sa = mfma_bf16(k_op_x<D>(kl, 0, cc), qreg[cc], cc == 0 ? zero : sa);
    }
    mfma_fence(sa);   // the steps read the scores through asm
    __syncthreads();  // every wave is done with K(0)
    const uint32_t kl1 = kl + kHalfBytes, vl1 = vl + kHalfBytes;
    const int last = npipe - 1;
    int t = 0;
    const auto land = [&] {
      wait_tile_copies();
      __syncthreads();
    };
    // half steps 0 (its V came with the first copies) and 1
    if (npool > 0) {
      issue_any(min(1, last), 0, 0);
      mask_scores(sa, static_cast<uint32_t>(tl.pmask[0]));
      half_step<BLK, D, true, false>(st, sa, sb, pb, pa, kl1, 0u, qreg, c);
      land();
      issue_any(min(1, last), 0, 1);
      issue_any(0, 1, 1);
      mask_scores(sb, static_cast<uint32_t>(tl.pmask[0] >> 32));
      half_step<BLK, D, true, true>(st, sb, sa, pa, pb, kl, vl, qreg, c);
      land();
      for (t = 1; t < npool; ++t) {
        issue_any(min(t + 1, last), 0, 0);
        issue_any(t, 1, 0);
        mask_scores(sa, static_cast<uint32_t>(tl.pmask[t]));
        half_step<BLK, D, true, true>(st, sa, sb, pb, pa, kl1, vl1, qreg, c);
        land();
        issue_any(min(t + 1, last), 0, 1);
        issue_any(t, 1, 1);
        mask_scores(sb, static_cast<uint32_t>(tl.pmask[t] >> 32));
        half_step<BLK, D, true, true>(st, sb, sa, pa, pb, kl, vl, qreg, c);
        land();
      }
    }
    // The first token rows of tiles t and t + 1 are read from the LDS list an
    // iteration ahead, so no copy waits on an LDS read.
    int f0 = first_of(min(t, last)), f1 = first_of(min(t + 1, last));
    if (npool == 0) {
      issue_k_at(f1, 0);
      half_step<BLK, D, false, false>(st, sa, sb, pb, pa, kl1, 0u, qreg, c);
      land();
      issue_k_at(f1, 1);
      issue_v_at(f0, 1);
      half_step<BLK, D, false, true>(st, sb, sa, pa, pb, kl, vl, qreg, c);
      f0 = f1;
      f1 = first_of(min(2, last));
      land();
      t = 1;
    }
    for (; t < npipe; ++t) {
      issue_k_at(f1, 0);
      issue_v_at(f0, 0);
      half_step<BLK, D, false, true>(st, sa, sb, pb, pa, kl1, vl1, qreg, c);
      asm volatile("" ::: "memory");  // the list read stays behind the MFMA stream
      const int f2 = first_of(min(t + 2, last));
      land();
      issue_k_at(f1, 1);
      issue_v_at(f0, 1);
      half_step<BLK, D, false, true>(st, sb, sa, pa, pb, kl, vl, qreg, c);
      land();
      f0 = f1;
      f1 = f2;
    }
    // P.V of the last half tile
    mfma_fence(st.acc);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
      const int ks = i / (D / 32), dt = i % (D / 32);
      st.acc[dt] = mfma_bf16(v_op_x<D>(vl1, ks, dt), pb[ks], st.acc[dt]);
    }
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
