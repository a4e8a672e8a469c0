"""GPU parity: every HIP kernel against the CPU oracle on seeded inputs.

Integer/byte results (pooled keys, thresholds, routing lists, INT8 codes and
scales, permutations) must match bit for bit; forward outputs must agree with
the oracle's restatement of the reference loop within max-abs 2e-2 and cosine
>= 0.9995 (BF16) / cosine >= 0.999 (INT8).
"""

import importlib

import numpy as np
import pytest
import torch

import oracle
from _util import bits, check_int8_blocks, compare_rows, cosine, mask_bits, randn_bf16, u32

pytestmark = pytest.mark.gpu

BF16_MAXABS, BF16_COS, INT8_COS = 2e-2, 0.9995, 0.999


def _mods(pkg):
    import importlib
    n = pkg.__name__
    return (importlib.import_module(f"{n}._preprocess"), importlib.import_module(f"{n}._tri_fwd"),
            importlib.import_module(f"{n}._int8_fwd"), importlib.import_module(f"{n}._fused_prep"),
            importlib.import_module(f"{n}._fused_quant"), importlib.import_module(f"{n}._morton"))


CASES = [  # (B, T, H, block, tau, sink_kv, sink_q)
    (1, 1000, 2, 64, 0.9, (0, 0), (0, 0)),
    (2, 777, 3, 128, 0.5, (0, 2), (0, 0)),
    (1, 4096, 4, 64, 1.3, (0, 3), (0, 3)),
    (1, 2500, 2, 128, -1e30, (0, 0), (0, 0)),
    # just past the 256 blocks a moments thread holds in registers and a route
    # workgroup scores in one pass (NT 257, ragged; NT 513)
    (1, 256 * 64 + 10, 2, 64, 0.9, (0, 0), (0, 0)),
    (1, 512 * 128 + 50, 1, 128, 0.8, (0, 1), (0, 0)),
    (2, 6000, 2, 64, 0.9, (0, 1), (2, 3)),  # NT 94: the route's two-group form
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("int8", [False, True])
def test_route_bit_exact(pkg, dev, case, int8):
    prep = _mods(pkg)[0]
    B, T, H, block, tau, skv, sq = case
    print(f"[route] case={case} int8={int8}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (10, 11, 12))
    r = prep.route(q.to(dev), k.to(dev), v.to(dev), scale=128 ** -0.5, tau=tau, block=block,
                   int8=int8, v_absmax=int8, sink_blocks=skv, sink_q=sq)
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau, int8=int8,
                         sink_kv=skv, sink_q=sq)
    NT = ref["NT"]
    assert np.array_equal(bits(r.kc), ref["kc"])
    assert np.array_equal(bits(r.vc), ref["vc"])
    assert np.array_equal(r.qbar.cpu().numpy().view(np.uint32), ref["qbar"].view(np.uint32))
    assert np.array_equal(r.kc_mean.cpu().numpy().view(np.uint32), ref["kc_mean"].view(np.uint32))
    assert np.array_equal(r.kc_var.cpu().numpy().view(np.uint32), ref["kc_var"].view(np.uint32))
    assert np.array_equal(r.threshold.cpu().numpy().view(np.uint32), ref["thr"].view(np.uint32))
    assert np.array_equal(r.counts.cpu().numpy(), ref["counts"])
    assert np.array_equal(u32(r.mask), ref["mask"])
    # the forwards build each query block's ascending exact list from its mask row
    ex = mask_bits(u32(r.mask), NT)
    assert np.array_equal(ex.sum(-1), ref["counts"])
    for b in range(B):
        for h in range(H):
            for i in range(NT):
                n = ref["counts"][b, h, i]
                assert np.array_equal(np.nonzero(ex[b, h, i])[0], ref["lists"][b, h, i, :n])
    if int8:
        assert np.array_equal(r.vscale.cpu().numpy().view(np.uint32), ref["vscale"].view(np.uint32))


@pytest.mark.parametrize("shape", [(2, 333, 3), (1, 2048, 8)])
@pytest.mark.parametrize("mean", [False, True])
def test_quant_bit_exact(pkg, dev, mean, shape):
    """Codes and scales bit-exact, including exact ties: rows with scale 1 and
    values k + 0.5 must round away from zero."""
    fq = _mods(pkg)[4]
    B, T, H = shape
    x = randn_bf16((B, T, H, 128), 5, scale=3.0)
    x[0, 7, 1] = 0  # all-zero row: scale floors at 1e-8
    ties = torch.arange(128, dtype=torch.float32) + 0.5
    ties[-1] = 127.0  # row max 127: scale exactly 1
    x[0, 5, 0] = ties.to(torch.bfloat16)
    x[0, 6, H - 1] = (-ties).to(torch.bfloat16)
    m = torch.randn(B, H, 128, generator=torch.Generator().manual_seed(6)) if mean else None
    xi, xs = fq.quantize_bthd(x.to(dev), mean=None if m is None else m.reshape(B * H, 128).to(dev))
    rxi, rxs = oracle.quant_rows(bits(x), None if m is None else m.numpy())
    assert np.array_equal(xi.cpu().numpy(), rxi)
    assert np.array_equal(xs.cpu().numpy().view(np.uint32), rxs.view(np.uint32))
    vi, vsc = fq.quantize_v_per_channel(x.to(dev))
    absmax = np.abs(oracle.bf16_to_f32(bits(x))).max(axis=1)
    rsc = np.maximum(absmax * (np.float32(1) / np.float32(127)), np.float32(1e-8)).astype(np.float32)
    assert np.array_equal(vsc.cpu().numpy().reshape(B, H, 128).view(np.uint32), rsc.view(np.uint32))
    assert np.array_equal(vi.cpu().numpy(), oracle.quant_v(bits(x), rsc))


PV_MODES = {  # name: (int8_pv, pv_codes)
    "int8_pv": (True, "block"), "int8_pv_running": (True, "running"), "bf16_pv": (False, "block")}


@pytest.mark.parametrize("shape,block", [((2, 333, 3), 64), ((1, 2048, 8), 128), ((1, 200, 2), 64)])
def test_quant_blocked_bit_exact(pkg, dev, shape, block):
    """Per-128-token-block Q and smoothed-K scales (the config 3 variant) through
    the INT8 preparation: codes and scales bit-exact against the oracle,
    including a ragged last scale block and a head whose block max is planted
    in one row. The one call folds each tile's shared K scale into the tile's
    score factor (one multiply per tile); the composed call through
    forward_int8 multiplies every score by its key's scale: the two agree up
    to fp32 rounding, and both against the oracle."""
    fp, i8 = _mods(pkg)[3], _mods(pkg)[2]
    B, T, H = shape
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (50, 51, 52))  # unit scale, as the
    q[0, 3, 0, 5] = 6.0  # other INT8 tests' bounds assume; one row holds its block's max
    print(f"[quant_blocked] shape={shape} block={block}", flush=True)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    r, qi, qs, ki, ks, vi = fp.fused_preprocess_routing(qd, kd, vd, tau=0.9, scale=128 ** -0.5,
                                                        block=block, quant_block=128)
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=0.9, int8=True,
                         quant_block=128)
    assert np.array_equal(qi.cpu().numpy(), ref["qi"]) and np.array_equal(ki.cpu().numpy(), ref["ki"])
    assert np.array_equal(qs.cpu().numpy().view(np.uint32), ref["qs"].view(np.uint32))
    assert np.array_equal(ks.cpu().numpy().view(np.uint32), ref["ks"].view(np.uint32))
    assert qs[0, 0, 0].item() == qs[0, min(T, 128) - 1, 0].item()  # one scale per block
    for pv, codes in PV_MODES.values():
        two = i8.forward_int8(qd, vd, r, qi, qs, ki, ks, vi if pv else None, int8_pv=pv,
                              pv_codes=codes)
        one = i8.sol_attn_int8(qd, kd, vd, tau=0.9, block=block, int8_pv=pv, quant_block=128,
                               pv_codes=codes)
        torch.cuda.synchronize()
        diff = (one.float() - two.float()).abs()
        print(f"  pv={pv} {codes}: one call vs composed max|d| {diff.max().item():.3g}, "
              f"{(diff > 0).float().mean().item():.3%} of outputs differ", flush=True)
        if codes == "block":
            assert diff.max().item() <= 1e-2
        if pv:
            assert np.array_equal(vi.cpu().numpy(), ref["vi"])
        refp = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=0.9, int8=True,
                              int8_pv=pv, quant_block=128)
        rows = _rows(B, H, refp["NT"], limit=16)
        # running codes: the one call's tile factor (qs*c*ks, one rounding per
        # tile) and the composed call's per-score scale round the row max
        # differently, so a ceil may land one apart between them; each is held
        # to the oracle instead
        for label, got in (("one call", one), ("composed", two)):
            check_int8_blocks(f"quant_blocked {shape} pv={pv} {codes} {label}",
                              got.float().cpu().numpy(), bits(q), bits(v), refp, rows, pv, block,
                              pv_codes=codes)


def test_reorder_matches_index_select(pkg, dev):
    mort = _mods(pkg)[5]
    x = randn_bf16((2, 21 * 6 * 10, 3 * 128), 7).to(dev)
    perm, inv = mort.morton_perm((21, 6, 10), dev, "3d")
    rperm, rinv = oracle.morton_perm((21, 6, 10), "3d")
    assert np.array_equal(perm.cpu().numpy(), rperm) and np.array_equal(inv.cpu().numpy(), rinv)
    y = mort.reorder_tokens(x, perm, dim=1)
    assert torch.equal(y, x.index_select(1, perm))
    assert torch.equal(mort.reorder_tokens(y, inv, dim=1), x)
    s = randn_bf16((500, 256), 8).to(dev)
    idx = torch.randperm(500, generator=torch.Generator().manual_seed(1)).to(dev)
    assert torch.equal(mort.reorder_tokens(s, idx, dim=0), s[idx])


@pytest.mark.parametrize("chunks", [1, 39, 40, 41, 63, 64, 65, 128, 129, 449, 511, 512, 513, 800, 1000, 1025, 5003])
def test_reorder_row_lengths(pkg, dev, chunks):
    """Rows around the lengths where the copy changes form (40 chunks of 16 bytes,
    one more load per lane, one more piece of 512), strided source rows, a row count that leaves waves idle,
    and an index outside the source (its row is zeroed)."""
    mod, capi = _mods(pkg)[5], importlib.import_module(f"{pkg.__name__}._capi")
    print(f"[reorder rows] chunks={chunks}", flush=True)
    g = torch.Generator().manual_seed(chunks)
    wide = torch.randn(2, 37, chunks * 8 + 8, generator=g).to(torch.bfloat16).to(dev)
    x = wide[..., : chunks * 8]
    idx = torch.randint(0, 37, (41,), generator=g).to(dev)
    assert torch.equal(mod.reorder_tokens(x.contiguous(), idx, dim=1), x[:, idx])
    out = torch.full((2, 41, chunks * 8), 7.0, dtype=torch.bfloat16, device=dev)
    bad = idx.clone()
    bad[3], bad[40] = -1, 37
    capi.call("solattn_reorder_rows", capi.ptr(x), 37, x.stride(0) * 2, x.stride(1) * 2, capi.ptr(out),
              out.stride(0) * 2, out.stride(1) * 2, 2, 41, chunks * 16, capi.ptr(bad), capi.stream(dev))
    want = x[:, idx].clone()
    want[:, [3, 40]] = 0
    assert torch.equal(out, want)


def test_reorder_rows_past_one_launch(pkg, dev):
    """2^26 rows and more, a wave each, are 2^32 threads: more than a launch covers in x.
    Every row is written (rows of 40 chunks of one value, 16 bytes apart in the output)."""
    capi = importlib.import_module(f"{pkg.__name__}._capi")
    rows = (1 << 26) + 5
    print(f"[reorder rows] {rows}", flush=True)
    src = torch.full((320,), 7.0, dtype=torch.bfloat16, device=dev)
    out = torch.zeros(rows * 8 + 312, dtype=torch.bfloat16, device=dev)
    idx = torch.zeros(rows, dtype=torch.int64, device=dev)
    capi.call("solattn_reorder_rows", capi.ptr(src), 1, 0, 0, capi.ptr(out), 0, 16, 1, rows, 640, capi.ptr(idx),
              capi.stream(dev))
    assert bool((out == 7.0).all())


FWD_CASES = [  # (B, T, H, block, tau, sink_kv, sink_q)
    (1, 1000, 2, 64, 0.9, (0, 0), (0, 0)),      # ragged last tile
    (1, 2500, 2, 128, 0.9, (0, 0), (0, 0)),     # block 128: 64-row full tile + 4-row ragged tile
    (2, 777, 3, 128, 0.3, (0, 0), (0, 0)),      # short rows, ragged 9-row tile
    (1, 4096, 2, 64, 1.5, (0, 0), (0, 0)),      # no ragged tile
    (2, 1000, 2, 64, 0.7, (0, 2), (0, 1)),      # sink blocks and sink query blocks
    (1, 3000, 2, 128, 1e30, (0, 0), (0, 0)),    # band only: pooled-heavy, 1-6 exact tiles per block
    (1, 2048, 2, 128, 0.8, (0, 0), (0, 0)),     # block 128, T a multiple of 128: no ragged block
    (1, 2112, 2, 128, 0.8, (0, 1), (0, 0)),     # block 128, last block of exactly 64 keys
    (1, 1536, 2, 64, -1e30, (0, 0), (0, 0)),    # all exact, no ragged or pooled tile: the first
                                                # pipelined tile starts from running max -inf
]


def _rows(B, H, NT, limit=None, seed=0):
    rows = [(b, h, i) for b in range(B) for h in range(H) for i in range(NT)]
    if limit and len(rows) > limit:
        rng = np.random.default_rng(seed)
        rows = [rows[j] for j in sorted(rng.choice(len(rows), limit, replace=False))]
    return rows


@pytest.mark.parametrize("case", FWD_CASES)
def test_fwd_bf16_vs_port(pkg, dev, case):
    tri = _mods(pkg)[1]
    B, T, H, block, tau, skv, sq = case
    print(f"[fwd_bf16] case={case}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (20, 21, 22))
    out = tri.sol_attn(q.to(dev), k.to(dev), v.to(dev), tau=tau, block=block, sink_blocks=skv,
                       sink_q=sq)
    torch.cuda.synchronize()
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau, sink_kv=skv, sink_q=sq)
    rows = _rows(B, H, ref["NT"], limit=24)
    port = oracle.forward_port(bits(q), bits(k), bits(v), ref, rows)
    err, cos = compare_rows(out.float().cpu().numpy(), port, block)
    print(f"[fwd_bf16] max|err|={err:.3e} cos={cos:.6f}", flush=True)
    assert err < BF16_MAXABS and cos >= BF16_COS


@pytest.mark.parametrize("block", [64, 128])
def test_fwd_bf16_all_exact_is_dense(pkg, dev, block):
    """tau = -inf routes every block: the output is dense SDPA."""
    tri = _mods(pkg)[1]
    B, T, H = 1, 1500, 2
    print(f"[fwd_bf16 dense] block={block}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (30, 31, 32))
    out = tri.sol_attn(q.to(dev), k.to(dev), v.to(dev), tau=-1e30, block=block)
    ref = torch.nn.functional.scaled_dot_product_attention(
        *(t.float().transpose(1, 2).to(dev) for t in (q, k, v))).transpose(1, 2)
    err = (out.float() - ref).abs().max().item()
    assert err < BF16_MAXABS
    assert cosine(out.float().cpu().numpy(), ref.cpu().numpy()) >= BF16_COS


@pytest.mark.parametrize("mode", list(PV_MODES))
@pytest.mark.parametrize("case", FWD_CASES)
def test_fwd_int8_vs_port(pkg, dev, case, mode):
    i8 = _mods(pkg)[2]
    B, T, H, block, tau, skv, sq = case
    int8_pv, codes = PV_MODES[mode]
    print(f"[fwd_int8] case={case} mode={mode}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (40, 41, 42))
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = i8.sol_attn_int8(qd, kd, vd, tau=tau, block=block, int8_pv=int8_pv, sink_blocks=skv,
                           sink_q=sq, pv_codes=codes)
    # the one call (Q codes from the pooling pass, heads past H in its last
    # 4-head wave idle) and the composed primitives give the same bits
    r, qi, qs, ki, ks, vi = _mods(pkg)[3].fused_preprocess_routing(
        qd, kd, vd, tau=tau, scale=128 ** -0.5, int8_pv=int8_pv, block=block, sink_blocks=skv,
        sink_q=sq)
    two = i8.forward_int8(qd, vd, r, qi, qs, ki, ks, vi, int8_pv=int8_pv, pv_codes=codes)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), two.view(torch.int16))
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau, int8=True, int8_pv=int8_pv,
                         sink_kv=skv, sink_q=sq)
    rows = _rows(B, H, ref["NT"], limit=16)
    # the ragged last query block of every (b, h) when sampling left it out
    rows = sorted(set(rows) | {(b, h, ref["NT"] - 1) for b in range(B) for h in range(H)})
    check_int8_blocks(f"fwd_int8 {case} {mode}", out.float().cpu().numpy(), bits(q),
                      bits(v), ref, rows, int8_pv, block, pv_codes=codes)


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("mode", ["bf16", "int8_pv", "int8_pv_running", "int8_bf16pv"])
def test_fwd_running_max_moves(pkg, dev, block, mode):
    """Keys scaled up along the sequence (x1 at the start, x8 at the end): a row's
    scores grow with the key index, so its running max moves by more than the
    kernels' slack (8, log2 units) several times inside the pipelined exact
    tiles, and the steps' rare path runs (P recomputed against the new max, O
    rescaled after the step's MFMAs)."""
    B, T, H, tau = 1, 4096, 2, 0.9
    print(f"[fwd max moves] block={block} mode={mode}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (50, 51, 52))
    ramp = (1.0 + 7.0 * torch.arange(T, dtype=torch.float32) / T).view(1, T, 1, 1)
    k = (k.float() * ramp).to(torch.bfloat16)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    if mode == "bf16":
        out = _mods(pkg)[1].sol_attn(qd, kd, vd, tau=tau, block=block)
        torch.cuda.synchronize()
        ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau)
        rows = _rows(B, H, ref["NT"], limit=24)
        port = oracle.forward_port(bits(q), bits(k), bits(v), ref, rows)
        err, cos = compare_rows(out.float().cpu().numpy(), port, block)
        print(f"[fwd max moves] max|err|={err:.3e} cos={cos:.6f}", flush=True)
        assert err < BF16_MAXABS and cos >= BF16_COS
    else:
        int8_pv = mode != "int8_bf16pv"
        codes = "running" if mode == "int8_pv_running" else "block"
        out = _mods(pkg)[2].sol_attn_int8(qd, kd, vd, tau=tau, block=block, int8_pv=int8_pv,
                                          pv_codes=codes)
        torch.cuda.synchronize()
        ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau, int8=True,
                             int8_pv=int8_pv)
        rows = _rows(B, H, ref["NT"], limit=16)
        # Rows here are sharply peaked (few large P codes), so one code of
        # difference where exp2 lands on a rounding boundary moves an output by
        # ~|v| / (sum of codes): the kernel-arithmetic max-abs bound is 3e-2
        # (1.4e-2 measured) instead of the 1e-2 of ordinary inputs; the
        # cosines keep their bounds.
        check_int8_blocks(f"fwd max moves {mode} block={block}", out.float().cpu().numpy(),
                          bits(q), bits(v), ref, rows, int8_pv, block, kernel_maxabs=3e-2,
                          pv_codes=codes)


@pytest.mark.parametrize("block", [64, 128])
def test_fwd_vs_dense_block_mask_diagnostic(pkg, dev, block):
    """Dense SDPA restricted to the same block mask (the pooled term dropped).
    A diagnostic, not the reference's output: the skipped blocks carry real
    mass, so the check is only that the forward sits much closer to its own
    closed form than to the masked dense one; both forwards' gaps are printed."""
    tri, i8 = _mods(pkg)[1], _mods(pkg)[2]
    B, T, H, tau = 1, 2500, 2, 0.9
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (60, 61, 62))
    out = tri.sol_attn(q.to(dev), k.to(dev), v.to(dev), tau=tau, block=block)
    out8 = i8.sol_attn_int8(q.to(dev), k.to(dev), v.to(dev), tau=tau, block=block)
    torch.cuda.synchronize()
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau)
    rows = _rows(B, H, ref["NT"], limit=12)
    masked = oracle.forward_dense_block_mask(bits(q), bits(k), bits(v), ref, rows)
    port = oracle.forward_port(bits(q), bits(k), bits(v), ref, rows)
    e_p, c_p = compare_rows(out.float().cpu().numpy(), port, block)
    e_m, c_m = compare_rows(out.float().cpu().numpy(), masked, block)
    e8, c8 = compare_rows(out8.float().cpu().numpy(), masked, block)
    print(f"[masked dense] block={block} bf16 vs closed form max|err|={e_p:.3e} cos={c_p:.6f}; "
          f"bf16 vs masked dense max|err|={e_m:.3e} cos={c_m:.6f}; int8 vs masked dense "
          f"max|err|={e8:.3e} cos={c8:.6f}", flush=True)
    assert e_p < e_m and c_p > c_m


def test_strided_qkv_view(pkg, dev):
    """An interleaved qkv buffer goes in as strided views, no copies needed."""
    tri = _mods(pkg)[1]
    B, T, H = 1, 900, 2
    qkv = randn_bf16((B, T, 3, H, 128), 50).to(dev)
    q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
    a = tri.sol_attn(q, k, v, tau=0.7, block=64)
    b = tri.sol_attn(q.contiguous(), k.contiguous(), v.contiguous(), tau=0.7, block=64)
    assert torch.equal(a, b)


@pytest.mark.parametrize("block", [64, 128])
def test_strided_views_every_path(pkg, dev, block):
    """Batch 2, q/k/v as views of a fused [B, T, 3, H, 256] buffer narrowed to
    128 channels (token stride 3*H*256, head stride 256): both forwards and
    every INT8 P.V mode give the bits of contiguous copies of the same data."""
    tri, i8 = _mods(pkg)[1], _mods(pkg)[2]
    B, T, H = 2, 1000, 3
    print(f"[strided views] block={block}", flush=True)
    buf = randn_bf16((B, T, 3, H, 256), 51).to(dev)
    q, k, v = (buf[:, :, i, :, :128] for i in range(3))
    assert q.stride(1) == 3 * H * 256 and q.stride(2) == 256
    qc, kc, vc = q.contiguous(), k.contiguous(), v.contiguous()
    assert torch.equal(tri.sol_attn(q, k, v, tau=0.8, block=block),
                       tri.sol_attn(qc, kc, vc, tau=0.8, block=block))
    for pv, codes in PV_MODES.values():
        a = i8.sol_attn_int8(q, k, v, tau=0.8, block=block, int8_pv=pv, pv_codes=codes)
        b = i8.sol_attn_int8(qc, kc, vc, tau=0.8, block=block, int8_pv=pv, pv_codes=codes)
        assert torch.equal(a, b), (pv, codes)


TINY_CASES = [  # (T, block): one partial block, exactly one block, one block + 1 row
    (1, 64), (63, 64), (64, 64), (65, 64), (100, 128), (128, 128), (129, 128),
]


@pytest.mark.parametrize("case", TINY_CASES)
def test_fwd_tiny_sequences(pkg, dev, case):
    """Sequences of one or two blocks, both forwards, against the oracle."""
    tri, i8 = _mods(pkg)[1], _mods(pkg)[2]
    T, block = case
    B, H = 2, 3
    print(f"[fwd tiny] T={T} block={block}", flush=True)
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (60, 61, 62))
    out = tri.sol_attn(q.to(dev), k.to(dev), v.to(dev), tau=0.9, block=block)
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=0.9)
    rows = _rows(B, H, ref["NT"])
    err, cos = compare_rows(out.float().cpu().numpy(), oracle.forward_port(bits(q), bits(k), bits(v), ref, rows), block)
    assert err < BF16_MAXABS and cos >= BF16_COS
    for pv, codes in PV_MODES.values():
        out8 = i8.sol_attn_int8(q.to(dev), k.to(dev), v.to(dev), tau=0.9, block=block, int8_pv=pv,
                                pv_codes=codes)
        ref8 = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=0.9, int8=True, int8_pv=pv)
        check_int8_blocks(f"fwd tiny T={T} block={block} pv={pv} {codes}",
                          out8.float().cpu().numpy(), bits(q), bits(v), ref8, rows, pv, block,
                          pv_codes=codes)


def _block_constant_closed_form(q, kb, vb, T, block, dev, chunk=16384):
    """Exact attention when K and V are constant inside every key block: the
    pooled approximation is then exact for any routing, and the output is a
    softmax over the NT blocks with log(len_j) added to each logit."""
    NT = kb.shape[0]
    lens = torch.tensor([min(block, T - block * j) for j in range(NT)], dtype=torch.float32, device=dev)
    kf, vf = kb.float().to(dev), vb.float().to(dev)
    out = torch.empty((T, 128), dtype=torch.float32, device=dev)
    for t0 in range(0, T, chunk):
        z = (q[t0:t0 + chunk].float().to(dev) @ kf.t()) * 128 ** -0.5 + lens.log()
        out[t0:t0 + chunk] = torch.softmax(z, dim=-1) @ vf
    return out


@pytest.mark.parametrize("block,NT", [(64, 2048), (128, 2048), (64, 16384), (128, 16384)])
def test_fwd_max_blocks_closed_form(pkg, dev, block, NT):
    """Long sequences up to the largest supported (16384 query/key blocks:
    1M tokens at block 64, 2M at block 128; ragged last block) with K and V
    constant inside each block, against the closed form; size-independent, so
    it runs at the full block count."""
    tri, i8 = _mods(pkg)[1], _mods(pkg)[2]
    T = NT * block - 17
    print(f"[fwd max NT] block={block} T={T}", flush=True)
    g = torch.Generator().manual_seed(70)
    kb = torch.randn(NT, 128, generator=g).to(torch.bfloat16)
    vb = torch.randn(NT, 128, generator=g).to(torch.bfloat16)
    q = (torch.randn(T, 128, generator=g) * 2.0).to(torch.bfloat16)
    k = kb.repeat_interleave(block, dim=0)[:T]
    v = vb.repeat_interleave(block, dim=0)[:T]
    ref = _block_constant_closed_form(q, kb, vb, T, block, dev)
    qd, kd, vd = (t.reshape(1, T, 1, 128).to(dev) for t in (q, k, v))
    out = tri.sol_attn(qd, kd, vd, tau=0.9, block=block)[0, :, 0].float()
    err = (out - ref).abs().max().item()
    cos = cosine(out.cpu().numpy(), ref.cpu().numpy())
    print(f"[fwd max NT] bf16 max|err|={err:.3e} cos={cos:.6f}", flush=True)
    assert err < BF16_MAXABS and cos >= BF16_COS
    for pv, codes in PV_MODES.values():
        # running codes: thousands of exact blocks per row, so the running max's
        # forced rise every 256 blocks (the int32 sums' overflow guard) runs
        out8 = i8.sol_attn_int8(qd, kd, vd, tau=0.9, block=block, int8_pv=pv,
                                pv_codes=codes)[0, :, 0].float()
        cos8 = cosine(out8.cpu().numpy(), ref.cpu().numpy())
        print(f"[fwd max NT] int8_pv={pv} {codes} cos={cos8:.6f}", flush=True)
        assert cos8 >= INT8_COS



@pytest.mark.parametrize("curve", ["3d", "2d_frame"])
def test_wan_hooks_neutral_through_gather_kernel(pkg, dev, curve):
    """Morton neutrality on the GPU: a stand-in Wan block stack whose attention
    is the sparse kernel with every block exact (tau = -inf, i.e. dense
    attention) gives the same output with the reorder hooks on and off; the
    hooks permute tokens and the RoPE table through the gather kernel."""
    import importlib
    mort = importlib.import_module(f"{pkg.__name__}._morton")
    tri = importlib.import_module(f"{pkg.__name__}._tri_fwd")
    grid, H = (4, 16, 16), 2
    N = grid[0] * grid[1] * grid[2]

    class Block(torch.nn.Module):
        def forward(self, x, freqs=None, transformer_options=None):
            q = (x * freqs[0]).view(1, N, H, 128)
            out = tri.sol_attn(q, q, x.view(1, N, H, 128), tau=-1e30, block=64)
            return out.reshape(1, N, H * 128)  # no residual: keeps magnitudes near 1

    class Model(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.blocks = torch.nn.ModuleList([Block(), Block()])

        def forward(self, x, freqs, options):
            for blk in self.blocks:
                x = blk(x, freqs=freqs, transformer_options=options)
            return x

    print(f"[wan hooks] grid={grid} curve={curve}", flush=True)
    model = Model()
    mort.install_wan_morton(model)
    x = randn_bf16((1, N, H * 128), 40, scale=0.5).to(dev)  # spread softmax, outputs below 1
    freqs = (torch.rand(1, N, H * 128, generator=torch.Generator().manual_seed(41)) + 0.5).to(
        torch.bfloat16).to(dev)
    plain = model(x, freqs, {"grid_sizes": grid})
    hooked = model(x, freqs, {"grid_sizes": grid, "sol_morton": True, "sol_morton_curve": curve})
    torch.cuda.synchronize()
    err = (hooked.float() - plain.float()).abs().max().item()
    print(f"[wan hooks] max |hooked - plain| = {err:.3e}", flush=True)
    assert err < BF16_MAXABS
    assert cosine(hooked.float().cpu().numpy(), plain.float().cpu().numpy()) >= BF16_COS


@pytest.mark.parametrize("mode", ["bf16", "int8_pv", "int8_pv_running", "int8_bf16pv"])
@pytest.mark.parametrize("case", ["cfg0", "random"])
def test_head_dim_64(pkg, dev, mode, case):
    """Head dim 64 (BASELINE config 0's shape, and a ragged random case): the
    one-call pipelines run the heads zero-padded to 128, so routing and INT8
    codes must equal the oracle's D = 64 computation bit for bit and the
    forward must meet the usual tolerances against the reference loop."""
    import importlib
    import bench
    prep, tri, i8 = _mods(pkg)[0], _mods(pkg)[1], _mods(pkg)[2]
    fp = importlib.import_module(f"{pkg.__name__}._fused_prep")
    if case == "cfg0":
        cfg = bench.CONFIGS[0]
        q, k, v = bench.make_inputs(cfg, "cpu", dtype=torch.float32)
        perm, _ = oracle.morton_perm(cfg["grid"], "3d")
        q, k, v = (t[:, perm].to(torch.bfloat16).contiguous() for t in (q, k, v))
        block, tau = cfg["block"], cfg["tau"]
    else:
        q, k, v = (randn_bf16((2, 1000, 3, 64), s) for s in (80, 81, 82))
        block, tau = 128, 0.7
    B, T, H, D = q.shape
    print(f"[d64] case={case} mode={mode} shape={tuple(q.shape)} block={block}", flush=True)
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    int8 = mode != "bf16"
    pv = mode in ("int8_pv", "int8_pv_running")
    codes = "running" if mode == "int8_pv_running" else "block"
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=tau, int8=int8, int8_pv=pv)
    if int8:
        r, qi, qs, ki, ks, vi = fp.fused_preprocess_routing(qd, kd, vd, tau=tau, scale=D ** -0.5,
                                                            int8_pv=pv, block=block)
        assert np.array_equal(qi.cpu().numpy(), ref["qi"]) and np.array_equal(ki.cpu().numpy(), ref["ki"])
        assert np.array_equal(ks.cpu().numpy().view(np.uint32), ref["ks"].view(np.uint32))
        if pv:
            assert np.array_equal(vi.cpu().numpy(), ref["vi"])
        out = i8.sol_attn_int8(qd, kd, vd, tau=tau, block=block, int8_pv=pv, pv_codes=codes)
    else:
        r = prep.route(qd, kd, vd, scale=D ** -0.5, tau=tau, block=block)
        out = tri.sol_attn(qd, kd, vd, tau=tau, block=block)
    torch.cuda.synchronize()
    assert out.shape == (B, T, H, D)
    NT = ref["NT"]
    assert np.array_equal(bits(r.kc)[:, :NT], ref["kc"][:, :NT])
    assert np.array_equal(r.threshold.cpu().numpy().view(np.uint32), ref["thr"].view(np.uint32))
    assert np.array_equal(u32(r.mask), ref["mask"]) and np.array_equal(r.counts.cpu().numpy(), ref["counts"])
    rows = _rows(B, H, NT, limit=48, seed=3)
    if int8:
        check_int8_blocks(f"d64 {case} {mode}", out.float().cpu().numpy(), bits(q), bits(v), ref,
                          rows, pv, block, pv_codes=codes)
    else:
        port = oracle.forward_port(bits(q), bits(k), bits(v), ref, rows)
        err, cos = compare_rows(out.float().cpu().numpy(), port, block)
        print(f"[d64 {case} bf16] max|err|={err:.3e} cos={cos:.6f}", flush=True)
        assert err < BF16_MAXABS and cos >= BF16_COS


def _check_hand_set_masks(pkg, dev, block, T, exact_rows):
    """The BF16 forward under hand-set exact blocks against float64 over the same pooled rows."""
    prep, tri = _mods(pkg)[0], _mods(pkg)[1]
    q, k, v = (randn_bf16((1, T, 1, 128), s) for s in (90, 91, 92))
    r = prep.route(q.to(dev), k.to(dev), v.to(dev), scale=128 ** -0.5, tau=0.9, block=block)
    NT = r.counts.shape[-1]
    rows = exact_rows(NT)  # [query block, key block]
    j = torch.arange(NT)
    words = torch.zeros(NT, r.mask.shape[-1], dtype=torch.int64)
    words.index_add_(1, j >> 5, rows.long() << (j & 31))
    mask = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32).to(dev)
    r = r._replace(mask=mask.reshape(r.mask.shape).contiguous(),
                   counts=rows.sum(-1).to(torch.int32).to(dev).reshape(r.counts.shape))
    print(f"[hand masks] block={block} T={T}", flush=True)
    out = tri.forward_bf16(q.to(dev), k.to(dev), v.to(dev), r).float().cpu()[0, :, 0]
    lens = torch.full((NT,), float(block), dtype=torch.float64)
    lens[-1] = T - (NT - 1) * block
    qd, kd, vd = (t[0, :, 0].double() for t in (q, k, v))
    kc, vc = (t[0, :NT, 0].double().cpu() for t in (r.kc, r.vc))
    on = rows[torch.arange(T) // block]
    s = (qd @ kd.t() * 128 ** -0.5).masked_fill(~on[:, torch.arange(T) // block], -torch.inf).exp()
    p = (qd @ kc.t() * 128 ** -0.5).masked_fill(on, -torch.inf).exp()
    ref = (s @ vd + p @ vc) / (s.sum(1) + p @ lens)[:, None]
    assert float((out - ref).abs().max()) < BF16_MAXABS
    assert cosine(out.numpy(), ref.numpy()) >= BF16_COS


@pytest.mark.parametrize("block,T", [(64, 64 * 70 + 17), (64, 64 * 64), (128, 128 * 66 + 64), (128, 128 * 65 + 90)])
def test_fwd_bf16_hand_set_masks(pkg, dev, block, T):
    """Tile orders the router never gives: rows with no exact block (pooled tiles
    only, a partial chunk and a short last block among them), with the last block
    alone, with the first alone, with every second block. Against float64: P and
    the outputs are rounded to bf16 (2^-9 each) under values of order 1, far
    inside BF16_MAXABS."""
    def exact_rows(NT):
        exact = torch.zeros(4, NT, dtype=torch.bool)
        exact[1, NT - 1] = exact[2, 0] = True
        exact[3, ::2] = True
        return exact[torch.arange(NT) % 4]

    _check_hand_set_masks(pkg, dev, block, T, exact_rows)


@pytest.mark.parametrize("block,T", [(64, 64 * 70), (128, 128 * 66)])
def test_fwd_bf16_half_chunk_exact(pkg, dev, block, T):
    """The first half tile of pooled keys without a pooled key (its 32 blocks all
    exact, as behind a sink of 32 blocks), alone and with the next one; lengths of
    whole blocks, so that no plain tile comes before it."""
    def exact_rows(NT):
        exact = torch.zeros(3, NT, dtype=torch.bool)
        exact[0, :32] = exact[1, :63] = exact[2, 32:64] = True
        return exact[torch.arange(NT) % 3]

    _check_hand_set_masks(pkg, dev, block, T, exact_rows)


def _rounded_p_model(q, qx, kx, vx, kc, vc, on, lens, first, block):
    """The forward's arithmetic for one head with P rounded to bf16 against the running
    max that its first tile gives (`first`: its keys, exact tokens [T] behind pooled blocks
    [NT] in one row per query block), in float64 otherwise. q scores the pooled keys, qx the exact ones. Rows whose max a later tile
    moves (by more than 8 in log2) are left out: [rows kept, model]."""
    T, D = q.shape
    tok = torch.arange(T, device=q.device) // block
    c = D ** -0.5 * 1.4426950408889634
    s = torch.cat([(q @ kc.t()).masked_fill(on[tok], -torch.inf),
                   (qx @ kx.t()).masked_fill(~on[tok][:, tok], -torch.inf)], 1) * c
    m = s.masked_fill(~first[tok], -torch.inf).amax(1, keepdim=True)
    keep = s.amax(1) <= m[:, 0] + 8
    p = torch.exp2(s - m)
    pr = p.float().to(torch.bfloat16).double()
    NT = kc.shape[0]
    total = (p[:, :NT] * lens).sum(1) + pr[:, NT:].sum(1)  # pooled keys: the fp32 p, exact keys: the packed ones
    return keep, (pr @ torch.cat([vc, vx])) / total[:, None]


@pytest.mark.parametrize("block,T", [(64, 64 * 64), (64, 64 * 70 + 17), (128, 128 * 40), (128, 128 * 33 + 90)])
@pytest.mark.parametrize("path", ["bf16", "int8_bf16pv"])
def test_running_max_of_whole_first_tile(pkg, dev, path, block, T):
    """P is rounded against the max of the whole first 64-key tile: pooled keys (block 64)
    or tokens (block 128, INT8) first, as the order of the tiles is. The bound: fp32 scores
    put one P in some 10^3 on the other side of a bf16 step and leave 1e-5 of the output,
    which puts one output in 10^2 on the other side of its own (2^-9 each): 2e-4 in all
    (measured 6e-5 to 1.1e-4). With the max of 32 keys every P rounds anew: 2e-3 to 3e-3."""
    prep, tri, i8, fp = _mods(pkg)[:4]
    q, k, v = (randn_bf16((1, T, 1, 128), s).to(dev) for s in (101, 102, 103))
    kw = dict(tau=0.9, block=block, scale=128 ** -0.5)
    print(f"[whole first tile] {path} block={block} T={T}", flush=True)
    if path == "bf16":
        r = prep.route(q, k, v, **kw)
        out = tri.forward_bf16(q, k, v, r)
        qx, kx = q[0, :, 0].double(), k[0, :, 0].double()
    else:
        r, qi, qs, ki, ks, _ = fp.fused_preprocess_routing(q, k, v, int8_pv=False, **kw)
        out = i8.forward_int8(q, v, r, qi, qs, ki, ks, None, int8_pv=False)
        qx, kx = (c[0, :, 0].double() * s[0, :, 0, None].double() for c, s in ((qi, qs), (ki, ks)))
    NT = r.counts.shape[-1]
    on = torch.from_numpy(mask_bits(u32(r.mask), NT)[0, 0]).to(dev)
    j = torch.arange(NT, device=dev)
    if block == 64 and path == "bf16":  # the first chunk of pooled keys
        first = torch.cat([(~on) & (j < 64), torch.zeros(NT, T, dtype=torch.bool, device=dev)], 1)
    else:  # the first exact block's first 64 tokens; INT8: the ragged last block's last tile before it
        blk = on.int().argmax(1)
        start = blk * block
        if path != "bf16" and T % 64:
            start = torch.where(on[:, NT - 1], T // 64 * 64, start)
        t = torch.arange(T, device=dev)
        inside = (t >= start[:, None]) & (t < start[:, None] + 64)
        first = torch.cat([torch.zeros(NT, NT, dtype=torch.bool, device=dev), inside], 1)
    lens = torch.full((NT,), float(block), dtype=torch.float64, device=dev)
    lens[-1] = T - (NT - 1) * block
    kc, vc = (t[0, :NT, 0].double() for t in (r.kc, r.vc))
    keep, ref = _rounded_p_model(q[0, :, 0].double(), qx, kx, v[0, :, 0].double(), kc, vc, on, lens, first, block)
    assert keep.float().mean() > 0.9
    ref = ref.to(torch.bfloat16).double()[keep]
    rel = float((out[0, :, 0].double()[keep] - ref).norm() / ref.norm())
    print(f"    rel {rel:.2e}", flush=True)
    assert rel < 4e-4


@pytest.mark.parametrize("block,T", [(64, 64 * 67 + 17), (64, 64 * 66), (128, 128 * 66 + 90), (128, 128 * 65 + 64),
                                     (128, 128 * 65 + 17)])
def test_fwd_int8_bf16pv_hand_set_masks(pkg, dev, block, T):
    """The INT8 forward with bf16 P.V where its pipeline is empty or a tile or two long:
    no exact block, the last alone, the first alone, both, every second block. Against
    float64 over the same codes and scales: P and the outputs are rounded to bf16 (2^-9
    each) under values of order 1, far inside BF16_MAXABS."""
    i8, fp = _mods(pkg)[2:4]
    q, k, v = (randn_bf16((1, T, 1, 128), s) for s in (93, 94, 95))
    r, qi, qs, ki, ks, _ = fp.fused_preprocess_routing(q.to(dev), k.to(dev), v.to(dev), tau=0.9, scale=128 ** -0.5,
                                                       block=block, int8_pv=False)
    NT = r.counts.shape[-1]
    exact = torch.zeros(5, NT, dtype=torch.bool)
    exact[1, NT - 1] = exact[2, 0] = exact[3, 0] = exact[3, NT - 1] = True
    exact[4, ::2] = True
    rows = exact[torch.arange(NT) % 5]  # [query block, key block]
    j = torch.arange(NT)
    words = torch.zeros(NT, r.mask.shape[-1], dtype=torch.int64)
    words.index_add_(1, j >> 5, rows.long() << (j & 31))
    mask = torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32).to(dev)
    r = r._replace(mask=mask.reshape(r.mask.shape).contiguous(),
                   counts=rows.sum(-1).to(torch.int32).to(dev).reshape(r.counts.shape))
    print(f"[int8 bf16pv hand masks] block={block} T={T}", flush=True)
    out = i8.forward_int8(q.to(dev), v.to(dev), r, qi, qs, ki, ks, None, int8_pv=False).float().cpu()[0, :, 0]
    lens = torch.full((NT,), float(block), dtype=torch.float64)
    lens[-1] = T - (NT - 1) * block
    qc, kcode = (c[0, :T, 0].double().cpu() * s[0, :T, 0, None].double().cpu() for c, s in ((qi, qs), (ki, ks)))
    kc, vc = (t[0, :NT, 0].double().cpu() for t in (r.kc, r.vc))
    on = rows[torch.arange(T) // block]
    s = (qc @ kcode.t() * 128 ** -0.5).masked_fill(~on[:, torch.arange(T) // block], -torch.inf).exp()
    p = (q[0, :, 0].double() @ kc.t() * 128 ** -0.5).masked_fill(on, -torch.inf).exp()
    ref = (s @ v[0, :, 0].double() + p @ vc) / (s.sum(1) + p @ lens)[:, None]
    assert float((out - ref).abs().max()) < BF16_MAXABS
    assert cosine(out.numpy(), ref.numpy()) >= BF16_COS


@pytest.mark.parametrize("D", [8, 40, 64])
@pytest.mark.parametrize("shape,block", [((2, 333, 3), 64), ((1, 777, 5), 128), ((1, 64, 1), 64),
                                         ((1, 64 * 65 + 7, 3), 64), ((1, 128 * 20 + 64, 2), 128)])
def test_small_heads_equal_padded_heads(pkg, dev, shape, block, D):
    """Heads of up to 64 channels run on 64-channel kernels (two heads share a
    pooling workgroup, the last of an odd count alone). Zero channels add exact
    zeros to every sum, so the result is that of the heads padded to 128, bit
    for bit; dense tensors and views of a fused qkv buffer."""
    tri = _mods(pkg)[1]
    B, T, H = shape
    print(f"[small heads] D={D} shape={shape} block={block}", flush=True)
    qkv = randn_bf16((B, T, 3, H, D), 95).to(dev)
    views = qkv.unbind(2)
    wide = [torch.nn.functional.pad(t, (0, 128 - D)).contiguous() for t in views]
    want = tri.sol_attn(*wide, tau=0.8, block=block, scale=D ** -0.5)[..., :D]
    for q, k, v in (views, [t.contiguous() for t in views]):
        out = tri.sol_attn(q, k, v, tau=0.8, block=block, scale=D ** -0.5)
        assert out.shape == (B, T, H, D) and torch.equal(out, want)


@pytest.mark.parametrize("NT", [1, 2, 33, 63, 64, 65, 96, 127, 128, 129, 257])
@pytest.mark.parametrize("mode", ["bf16", "int8_pv", "int8_bf16pv"])
def test_one_call_equals_its_stages(pkg, dev, NT, mode):
    """Up to 128 blocks the one calls take the moments inside the routing launch;
    the stage-by-stage path (bit-exact against the oracle above) must give the
    same output bits. Ragged lengths, two batches, an odd head count, sinks."""
    prep, tri, i8, fp = _mods(pkg)[:4]
    block = 64
    B, T, H = 2, (NT - 1) * block + (64 if NT == 64 else 37), 3
    q, k, v = (randn_bf16((B, T, H, 128), s).to(dev) for s in (96, 97, 98))
    k += 0.5  # a mean that centring has to take out
    kw = dict(tau=0.7, block=block, sink_blocks=(0, 1), sink_q=(1, 2))
    print(f"[one call] NT={NT} mode={mode}", flush=True)
    if mode == "bf16":
        one = tri.sol_attn(q, k, v, **kw)
        two = tri.forward_bf16(q, k, v, prep.route(q, k, v, scale=128 ** -0.5, **kw))
    else:
        pv = mode == "int8_pv"
        one = i8.sol_attn_int8(q, k, v, int8_pv=pv, **kw)
        r, *codes = fp.fused_preprocess_routing(q, k, v, scale=128 ** -0.5, int8_pv=pv, **kw)
        two = i8.forward_int8(q, v, r, *codes, int8_pv=pv)
    assert torch.equal(one, two)


@pytest.mark.parametrize("T,block,H,quant_block", [(1, 64, 1, None), (64 * 64, 64, 2, None), (64 * 63 + 9, 64, 3, 128),
                                                   (128 * 65 + 1, 128, 2, None), (777, 128, 3, 128)])
@pytest.mark.parametrize("int8_pv", [True, False])
def test_preprocess_one_call(pkg, dev, T, block, H, quant_block, int8_pv):
    """The INT8 preparation's one call against the oracle, bit for bit; and straight into
    buffers that hold something else, with padding rows behind every length: those of kc
    and vc are zeroed, the other outputs are the same."""
    fp, capi = _mods(pkg)[3], importlib.import_module(f"{pkg.__name__}._capi")
    B = 2
    q, k, v = (randn_bf16((B, T, H, 128), s) for s in (31, 32, 33))
    print(f"[preprocess] T={T} block={block} H={H} quant_block={quant_block} pv={int8_pv}", flush=True)
    r, qi, qs, ki, ks, vi = fp.fused_preprocess_routing(q.to(dev), k.to(dev), v.to(dev), tau=0.8,
                                                        scale=128 ** -0.5, block=block, int8_pv=int8_pv,
                                                        quant_block=quant_block)
    ref = oracle.prepare(bits(q), bits(k), bits(v), block=block, tau=0.8, int8=True, int8_pv=int8_pv,
                         **({"quant_block": 128} if quant_block else {}))
    NT = ref["NT"]
    for name, t in (("kc", r.kc), ("vc", r.vc)):
        assert np.array_equal(bits(t)[:, :NT], ref[name][:, :NT]) and not bits(t)[:, NT:].any()
    f32 = lambda t: t.cpu().numpy().view(np.uint32)  # noqa: E731
    assert np.array_equal(f32(r.threshold), ref["thr"].view(np.uint32))
    assert np.array_equal(u32(r.mask), ref["mask"]) and np.array_equal(r.counts.cpu().numpy(), ref["counts"])
    for name, t in (("qi", qi), ("ki", ki)) + ((("vi", vi),) if int8_pv else ()):
        assert np.array_equal(t.cpu().numpy(), ref[name]), name
    assert np.array_equal(f32(qs), ref["qs"].view(np.uint32)) and np.array_equal(f32(ks), ref["ks"].view(np.uint32))

    npad = (NT // 64 + 1) * 64
    bfs = [torch.full((B, npad, H, 128), 3.0, dtype=torch.bfloat16, device=dev) for _ in range(2)]
    like = lambda t: None if t is None else torch.full_like(t, 5)  # noqa: E731
    outs = [like(t) for t in (r.qbar, r.kc_mean, r.kc_var, r.vamax_part, r.vscale, r.threshold, r.counts, r.mask, qi,
                              qs, ki, ks, vi)]
    dense = [x.to(dev) for x in (q, k, v)]
    args = [n for x in dense for n in (capi.ptr(x), x.stride(0), x.stride(1), x.stride(2))]
    capi.call("solattn_preprocess_int8", *args, B, T, H, 128, block, 128 ** -0.5, 0.8, 0, 0, 0, 0,
              1 if quant_block else 0, capi.ptr(bfs[0]), capi.ptr(bfs[1]), npad, *(capi.ptr(t) for t in outs),
              capi.stream(dev))
    for t, want in zip(bfs, (r.kc, r.vc)):
        assert torch.equal(t[:, :NT], want[:, :NT]) and not bits(t)[:, NT:].any()
    for t, want in zip(outs, (r.qbar, r.kc_mean, r.kc_var, r.vamax_part, r.vscale, r.threshold, r.counts, r.mask, qi, qs,
                              ki, ks, vi)):
        assert (t is None and want is None) or torch.equal(t, want)
