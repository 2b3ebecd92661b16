"""GPU parity: pooling and streaming selection (libfbsa.so) vs the CPU oracle.

Block indices must match bit for bit (ties break to the lower index in both);
pooled values must match exactly (same rounding points)."""
import numpy as np
import pytest
import torch

from oracle import select as osel
from _util import randn, np64

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _say(*a):
    print("[select]", *a, flush=True)


@pytest.mark.parametrize("dtype,H,D,bs", [("f32", 4, 64, 64), ("bf16", 4, 64, 64), ("f16", 4, 64, 64),
                                          ("bf16", 6, 64, 64), ("bf16", 12, 64, 64), ("f16", 13, 64, 64),
                                          ("f32", 1, 64, 64), ("bf16", 1, 64, 64), ("f16", 1, 64, 64),
                                          ("f32", 1, 256, 128), ("bf16", 1, 128, 32), ("f16", 1, 16, 16),
                                          ("bf16", 1, 32, 128)])
def test_pool_mean_tok_then_heads_exact(dtype, H, D, bs):
    """Mean over tokens, then over H heads. A wave takes heads w, w + 4, ... and
    loads two of them together: 6, 12 and 13 heads leave waves with an odd count.
    One head (a plain token mean) runs one block per wave, four per workgroup,
    at every head dim and block size it takes."""
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(0)
    B, N = 2, 1000                               # N % bs != 0: zero-padded tail block
    x = randn(g, (B, H, N, D), dtype)
    _say("pool mean_tok_then_grp", dtype, H)
    got = np64(selection.pool(x.to(DEV), bs, "mean_tok_then_grp", grp=H))
    ref = osel.pool_mean_tok_then_heads(np64(x), bs, dtype)[:, None]
    assert np.array_equal(got, ref), np.abs(got - ref).max()


@pytest.mark.parametrize("op,H,grp,D,bs", [("mean_tok_then_grp", 2, 1, 64, 64), ("mean_tok_then_grp", 4, 4, 64, 32),
                                           ("mean_grp_then_tok", 4, 2, 128, 128), ("minmax", 2, 1, 32, 16)])
def test_pool_l_valid_past_whole_blocks(op, H, grp, D, bs):
    """Tokens at positions >= l_valid count as zeros, also in blocks that lie
    wholly past l_valid (their rows are read at the last valid row's address
    and discarded): the result equals pooling the input with those rows zeroed."""
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(7)
    B, N, lv = 2, 1000, 77                       # blocks from lv // bs + 1 on hold no valid token
    x = randn(g, (B, H, N, D), "bf16")
    xz = x.clone()
    xz[:, :, lv:] = 0
    _say("pool l_valid", op, H, grp, D, bs)
    got = selection.pool(x.to(DEV), bs, op, grp=grp, l_valid=lv)
    if op == "minmax":
        rmin, rmax = osel.pool_minmax(np64(xz), bs)
        assert np.array_equal(np64(got[0]), rmin) and np.array_equal(np64(got[1]), rmax)
        return
    if op == "mean_tok_then_grp":
        ref = np.concatenate([osel.pool_mean_tok_then_heads(np64(xz[:, h0:h0 + grp]), bs, "bf16")[:, None]
                              for h0 in range(0, H, grp)], axis=1)
    else:
        ref = osel.pool_mean_grp_then_tok(np64(xz), H // grp, bs, "bf16")
    assert np.array_equal(np64(got), ref), np.abs(np64(got) - ref).max()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_pool_quest_exact(dtype):
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(1)
    B, Hq, Hkv, N, D, bs = 1, 8, 2, 700, 128, 128
    q = randn(g, (B, Hq, N, D), dtype)
    k = randn(g, (B, Hkv, N, D), dtype)
    _say("pool quest", dtype)
    qp = np64(selection.pool(q.to(DEV), bs, "mean_grp_then_tok", grp=Hq // Hkv))
    kmin, kmax = selection.pool(k.to(DEV), bs, "minmax")
    assert np.array_equal(qp, osel.pool_mean_grp_then_tok(np64(q), Hkv, bs, dtype))
    rmin, rmax = osel.pool_minmax(np64(k), bs)
    assert np.array_equal(np64(kmin), rmin) and np.array_equal(np64(kmax), rmax)


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("bs,D,nblk", [(16, 64, 100), (16, 128, 100), (16, 256, 128), (16, 256, 129), (16, 256, 257),
                                       (32, 64, 100), (32, 128, 128), (32, 128, 129), (32, 256, 256), (32, 256, 257),
                                       (64, 64, 128), (64, 64, 129), (64, 128, 128), (64, 128, 129), (64, 128, 257),
                                       (64, 256, 128), (64, 256, 129), (64, 256, 512), (64, 256, 513),
                                       (128, 64, 128), (128, 64, 129), (128, 128, 64), (128, 128, 65), (128, 256, 32),
                                       (128, 256, 33)])
def test_pool_slices_exact(dtype, bs, D, nblk):
    # group-mean and min / max pooling split a row over workgroups while blocks are few: both
    # sides of every line of launch_pool_op, with a short last block
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(nblk + D)
    x = randn(g, (1, 3, nblk * bs - 5, D), dtype)
    _say("pool slices", dtype, bs, D, nblk)
    got = selection.pool(x.to(DEV), bs, "mean_grp_then_tok", grp=3)
    assert np.array_equal(np64(got), osel.pool_mean_grp_then_tok(np64(x), 1, bs, dtype))
    kmin, kmax = selection.pool(x[:, :1].to(DEV), bs, "minmax")
    rmin, rmax = osel.pool_minmax(np64(x[:, :1]), bs)
    assert np.array_equal(np64(kmin), rmin) and np.array_equal(np64(kmax), rmax)


def _us(run, n=20):
    """Median of five timings of n calls back to back, in us a call."""
    run()
    t = []
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(n):
            run()
        b.record()
        b.synchronize()
        t.append(a.elapsed_time(b) * 1000 / n)
    return sorted(t)[2]


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("op,grp,D,bs,nblk", [("minmax", 1, 256, 32, 1000), ("minmax", 1, 256, 64, 255), ("minmax", 1, 128, 64, 512),
                                              ("mean_grp_then_tok", 2, 256, 16, 1000), ("mean_grp_then_tok", 3, 128, 16, 512),
                                              ("mean_grp_then_tok", 2, 256, 16, 255)])
def test_pool_time_near_the_token_mean(dtype, op, grp, D, bs, nblk):
    # the same bytes as a token mean, whose workgroups always read whole rows: at most twice its
    # time (and a launch) where slices of the rows would be three times behind
    from fbsa_amd import _lib, selection
    x = torch.zeros(1, grp, nblk * bs, D, device=DEV, dtype={"bf16": torch.bfloat16, "f32": torch.float32}[dtype])
    out, out2 = (torch.empty(1, 1, nblk, D, device=DEV, dtype=x.dtype) for _ in range(2))
    lib, s = _lib.load(), torch.cuda.current_stream().cuda_stream

    def call(o):
        d = selection._pool_desc(x, bs, o, grp, None)
        return lambda: _lib.check(lib.fbsa_pool(d, x.data_ptr(), out.data_ptr(), out2.data_ptr(), s), "pool")
    _say("pool time", dtype, op, grp, D, bs, nblk)
    t, ref = _us(call(op)), _us(call("mean_tok_then_grp"))
    assert t <= 2 * ref + 2, (t, ref)


def _check_sel(got, ref, what):
    got = np.asarray(got)
    ref = np.asarray(ref)
    assert got.shape == ref.shape, (got.shape, ref.shape)
    bad = np.argwhere(got != ref)
    assert bad.size == 0, f"{what}: {len(bad)} mismatching slots, first at {bad[:3].tolist()}: " \
                          f"got {got[tuple(bad[0][:-1])]} ref {ref[tuple(bad[0][:-1])]}"


@pytest.mark.parametrize("engine", ["auto", "fp64"])
@pytest.mark.parametrize("dtype,B,H,N,bs,topk,causal", [
    ("f32", 1, 4, 4096, 64, 8, True),      # config 1
    ("bf16", 32, 8, 1024, 32, 4, True),    # config 2
    ("bf16", 1, 2, 8192, 16, 16, True),    # many blocks, small block
    ("bf16", 2, 2, 2048, 64, 5, False),    # non-causal
    ("f16", 1, 2, 2048, 32, 12, True),
])
def test_select_mean_pooled_exact(dtype, B, H, N, bs, topk, causal, engine):
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(2)
    D = 64
    q, k = (randn(g, (B, H, N, D), dtype) for _ in range(2))
    _say("mean-pooled", dtype, B, H, N, bs, topk, causal, engine)
    sel, sc = selection.select_mean_pooled(q.to(DEV), k.to(DEV), bs, topk, causal, need_scores=True, engine=engine)
    ref, raw = osel.select_mean_pooled(np64(q), np64(k), bs, topk, causal, dtype)
    _check_sel(sel.cpu().numpy(), ref, "sel")
    ref_sc = np.take_along_axis(raw, ref, axis=-1)
    assert np.array_equal(sc.cpu().numpy().astype(np.float64), ref_sc)


@pytest.mark.parametrize("dtype,B,Hq,Hk,N,D,bs,topk,scale", [
    ("bf16", 1, 8, 8, 16384, 64, 64, 16, 1.0),     # config 3's shape, shorter
    ("bf16", 2, 4, 2, 3000, 64, 32, 32, 1.0),      # ragged tail block, largest fused budget
    ("bf16", 2, 4, 2, 3000, 64, 32, 48, 1.0),      # past it: pool, pool, fp64 select
    ("f16", 1, 2, 1, 2048, 32, 16, 8, 1.0),
    ("bf16", 1, 2, 2, 4096, 64, 128, 20, 1.0),
    ("bf16", 1, 4, 4, 4096, 64, 64, 49, 1.0),      # budget past the MFMA engine: pool, pool, select
    ("bf16", 1, 2, 2, 4096, 64, 64, 16, 1e19),     # norms past 1e18: every pair takes the exact path
    ("bf16", 1, 2, 2, 4096, 32, 64, 16, 1e-20),    # norms below 2^-40: likewise
    ("bf16", 3, 1, 1, 3000, 64, 32, 16, 1.0),      # one head: plain token means, a block per wave
    ("f16", 1, 1, 1, 4000, 32, 128, 8, 1.0),
    # the shapes above have at most 256 blocks and run select_row_kernel; past that the pooling
    # writes the row norms that the MFMA engine starts from
    ("bf16", 1, 8, 8, 16448, 64, 64, 16, 1.0),     # 257 blocks
    ("bf16", 2, 4, 2, 9000, 64, 32, 32, 1.0),      # ragged tail block, largest fused budget
    ("bf16", 2, 4, 2, 9000, 64, 32, 33, 1.0),      # past it: no norms, fp64 select
    ("f16", 1, 2, 1, 8192, 32, 16, 8, 1.0),
    ("bf16", 1, 2, 2, 8192, 64, 16, 16, 1e19),     # norms past 1e18
    ("bf16", 1, 2, 2, 8192, 32, 16, 16, 1e-20),    # norms below 2^-40
    ("bf16", 3, 1, 1, 9000, 64, 32, 16, 1.0),      # one head: plain token means
    ("f16", 1, 1, 1, 8192, 32, 16, 8, 1.0),
    ("bf16", 40, 2, 1, 4096, 64, 16, 16, 1.0),     # 256 blocks, but more pairs than the row kernel takes
])
def test_select_mean_pooled_fused_equals_separate_calls(dtype, B, Hq, Hk, N, D, bs, topk, scale):
    """fbsa_select_mean_pooled (q and k pooled by one launch that also writes the
    selection's row norms) against fbsa_pool twice + fbsa_select: same blocks,
    same chosen-slot scores."""
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(31)
    q = (randn(g, (B, Hq, N, D), "f32") * scale).to(getattr(torch, {"bf16": "bfloat16", "f16": "float16"}[dtype]))
    k = (randn(g, (B, Hk, N, D), "f32") * scale).to(q.dtype)
    q, k = q.to(DEV), k.to(DEV)
    _say("mean-pooled fused vs separate", dtype, B, Hq, Hk, N, D, bs, topk, scale)
    sel1, sc1 = selection.select_mean_pooled(q, k, bs, topk, True, need_scores=True)
    qp = selection.pool(q, bs, "mean_tok_then_grp", grp=Hq)
    kp = selection.pool(k, bs, "mean_tok_then_grp", grp=Hk)
    sel2, sc2 = selection.select(qp, kp, score="dot", convention="own_first", topk=topk, causal=True,
                                 need_scores=True)
    torch.cuda.synchronize()
    assert torch.equal(sel1, sel2[:, 0])
    assert torch.equal(sc1, sc2[:, 0])


def test_select_config3_full_size_sampled_rows():
    # config 3: B1 H8 N262144 D64 bs64 top-16; q,k ~ N(0,1)/8 in bf16. The oracle
    # pools the full tensors and scores a sample of rows (each row i depends
    # only on qpool[i] and kpool[0..i]).
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(0)
    B, H, N, D, bs, topk = 1, 8, 262144, 64, 64, 16
    q = randn(g, (B, H, N, D), "bf16", scale=0.125)
    k = randn(g, (B, H, N, D), "bf16", scale=0.125)
    _say("config 3 selection")
    sel = selection.select_mean_pooled(q.to(DEV), k.to(DEV), bs, topk, True).cpu().numpy()
    qp = osel.pool_mean_tok_then_heads(np64(q), bs, "bf16")
    kp = osel.pool_mean_tok_then_heads(np64(k), bs, "bf16")
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(4096 - 40, 4096),
                                     np.random.default_rng(0).integers(0, 4096, 200)]))
    raw = osel.scores(qp, kp, "bf16", "dot", rows=rows)
    ref = osel.select_conv_a(raw, topk, True, rows=rows)
    _check_sel(sel[:, rows], ref, "sel (sampled rows)")


@pytest.mark.parametrize("dtype,engine", [("bf16", "auto"), ("bf16", "fp64"), ("f32", "auto")])
def test_select_quest_config4_shape(dtype, engine):
    # config 4 selector: Hq16 Hkv2 D256 bs128 nblk512 top-32 + own + sink
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(3)
    B, Hq, Hkv, N, D, bs, topk = 1, 16, 2, 65536, 256, 128, 32
    q = randn(g, (B, Hq, N, D), dtype)
    k = randn(g, (B, Hkv, N, D), dtype)
    _say("quest config 4", dtype, engine)
    idx = selection.select_quest(q.to(DEV), k.to(DEV), bs, topk, sink=True, engine=engine).cpu().numpy()
    ref, _ = osel.select_quest(np64(q), np64(k), bs, topk, True, dtype)
    _check_sel(idx, ref, "idx")


@pytest.mark.parametrize("D,ties,sink,topk", [(128, False, True, 8), (256, True, True, 62), (128, True, False, 30),
                                               (256, False, False, 16)])
def test_select_quest_wide_rows(D, ties, sink, topk):
    # Quest + _finish at D >= 128 without chosen-slot scores runs on the row-per-
    # workgroup exact kernel; with scores requested, on the streaming fp64 kernel:
    # both must give the oracle's blocks
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(9)
    B, H, nblk = 1, 2, 700
    if ties:
        mk = lambda: torch.randint(-2, 3, (B, H, nblk, D), generator=g).to(torch.bfloat16)  # noqa: E731
    else:
        mk = lambda: randn(g, (B, H, nblk, D), "bf16")  # noqa: E731
    a, b1, b2 = mk(), mk(), mk()
    b1, b2 = torch.maximum(b1, b2), torch.minimum(b1, b2)
    _say("quest wide", D, ties, sink, topk)
    kw = dict(score="quest", convention="sorted_sink", topk=topk, sink=sink)
    sel = selection.select(a.to(DEV), b1.to(DEV), b2.to(DEV), **kw)
    sel2, _ = selection.select(a.to(DEV), b1.to(DEV), b2.to(DEV), need_scores=True, **kw)
    raw = osel.scores(np64(a), np64(b1), "bf16", "quest", b2=np64(b2))
    ref = osel.select_conv_b(raw, topk, sink)
    _check_sel(sel.cpu().numpy(), ref, "sel (row kernel)")
    _check_sel(sel2.cpu().numpy(), ref, "sel (streaming kernel)")


@pytest.mark.parametrize("engine", ["auto", "fp64"])
def test_select_max2_module_scores(engine):
    # BlockSparseSSA._scores: max(sq . sk_mean, sq . sk_max) (src/ssa_model.py:113-119)
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(4)
    B, L, S, bs, topk = 2, 2048, 32, 64, 8
    sq = randn(g, (B, 1, L, S), "bf16")
    sk = randn(g, (B, 1, L, S), "bf16")
    _say("max2")
    a = selection.pool(sq.to(DEV), bs, "mean_tok_then_grp")
    km = selection.pool(sk.to(DEV), bs, "mean_tok_then_grp")
    kx = selection.pool(sk.to(DEV), bs, "max")
    sel, sc = selection.select(a, km, kx, score="max2", topk=topk, causal=True, need_scores=True, engine=engine)
    ra = osel.pool_tok(np64(sq)[:, 0], bs, "bf16", "mean")
    rkm = osel.pool_tok(np64(sk)[:, 0], bs, "bf16", "mean")
    rkx = osel.pool_tok(np64(sk)[:, 0], bs, "bf16", "max")
    raw = osel.scores(ra, rkm, "bf16", "max2", b2=rkx)
    ref = osel.select_conv_a(raw, topk, True)
    _check_sel(sel.cpu().numpy()[:, 0], ref, "sel")
    assert np.array_equal(sc.cpu().numpy()[:, 0].astype(np.float64), np.take_along_axis(raw, ref, -1))


@pytest.mark.parametrize("engine", ["auto", "fp64"])
@pytest.mark.parametrize("nblk,topk,conv", [(1, 4, "own_first"), (3, 8, "own_first"), (5, 0, "own_first"),
                                            (1, 4, "sorted_sink"), (4, 9, "sorted_sink"), (70, 62, "own_first"),
                                            (200, 62, "sorted_sink")])
def test_select_edge_budgets(nblk, topk, conv, engine):
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(5)
    a = randn(g, (1, 2, nblk, 32), "bf16")
    b = randn(g, (1, 2, nblk, 32), "bf16")
    _say("edge", nblk, topk, conv)
    sel = selection.select(a.to(DEV), b.to(DEV), topk=topk, convention=conv, sink=conv == "sorted_sink",
                           engine=engine).cpu().numpy()
    raw = osel.scores(np64(a), np64(b), "bf16", "dot")
    if conv == "own_first":
        ref = np.stack([osel.select_conv_a(raw[:, h], topk, True) for h in range(2)], 1)
    else:
        ref = osel.select_conv_b(raw, topk, True)
    _check_sel(sel, ref, "sel")


@pytest.mark.parametrize("D", [16, 64])
def test_select_ties_break_to_lower_index(D):
    # all-equal scores: every candidate ties; lowest indices must win
    from fbsa_amd import selection
    nblk, topk = 200, 7
    a = torch.ones(1, 1, nblk, D, dtype=torch.bfloat16)
    sel = selection.select(a.to(DEV), a.to(DEV), topk=topk, causal=True).cpu().numpy()[0, 0]
    for i in range(nblk):
        want = [i] + [j for j in range(min(i, topk))] + [i] * max(0, topk - i)
        assert sel[i].tolist() == want, (i, sel[i])


def test_select_config5_prefix_invariance_and_sampled_rows():
    # config 5: B1 H8 D64 N4194304 bs64 (nblk 65536) top-16. The streaming selection
    # on the full sequence must give the 262144-token prefix run's blocks for the
    # first 4096 rows (causal), and the oracle's blocks on sampled later rows.
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(5)
    B, H, N, D, bs, topk = 1, 8, 4194304, 64, 64, 16
    q = randn(g, (B, H, N, D), "bf16")
    k = randn(g, (B, H, N, D), "bf16")
    _say("config 5 selection")
    qd, kd = q.to(DEV), k.to(DEV)
    sel = selection.select_mean_pooled(qd, kd, bs, topk, True).cpu().numpy()
    pre = selection.select_mean_pooled(qd[:, :, :262144].contiguous(), kd[:, :, :262144].contiguous(),
                                       bs, topk, True).cpu().numpy()
    _check_sel(sel[:, :4096], pre, "prefix rows")
    qp = selection.pool(qd, bs, "mean_tok_then_grp", grp=H)[:, 0].float().cpu().numpy().astype(np.float64)
    kp = selection.pool(kd, bs, "mean_tok_then_grp", grp=H)[:, 0].float().cpu().numpy().astype(np.float64)
    rows = np.unique(np.concatenate([np.arange(65536 - 8, 65536),
                                     np.random.default_rng(1).integers(4096, 65536, 40)]))
    raw = osel.scores(qp, kp, "bf16", "dot", rows=rows)
    ref = osel.select_conv_a(raw, topk, True, rows=rows)
    _check_sel(sel[:, rows], ref, "sampled rows")


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("score", ["dot", "max2", "quest"])
@pytest.mark.parametrize("conv,causal,topk", [("own_first", True, 16), ("own_first", False, 16),
                                              ("sorted_sink", True, 16), ("own_first", True, 32),
                                              ("own_first", True, 48)])
@pytest.mark.parametrize("ties,chunk", [(False, 0), (True, 0), (False, 4), (True, 1)])
def test_select_tiled_modes(dtype, D, score, conv, causal, topk, ties, chunk):
    # The MFMA engine over every score mode / convention / width it takes, with
    # nblk = 700 (11 candidate tiles, a ragged last tile). chunk > 0 splits the
    # candidates of a row block over several workgroups (partial lists + merge).
    # ties=True uses small integer operands, so scores are exact integers with
    # many exact ties (tie-break and exact-bracket paths).
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(6)
    B, H, nblk = 1, 2, 700
    if ties:
        mk = lambda: torch.randint(-2, 3, (B, H, nblk, D), generator=g).to(getattr(torch, {"bf16": "bfloat16", "f16": "float16"}[dtype]))
    else:
        mk = lambda: randn(g, (B, H, nblk, D), dtype)
    a, b1, b2 = mk(), mk(), mk()
    if score == "quest":  # kmax >= kmin element-wise, as the pooled operands are
        b1, b2 = torch.maximum(b1, b2), torch.minimum(b1, b2)
    _say("tiled", dtype, D, score, conv, causal, topk, ties, chunk)
    sink = conv == "sorted_sink"
    sel, sc = selection.select(a.to(DEV), b1.to(DEV), b2.to(DEV) if score != "dot" else None, score=score,
                               convention=conv, topk=topk, causal=causal, sink=sink, need_scores=True,
                               chunk_tiles=chunk)
    raw = osel.scores(np64(a), np64(b1), dtype, score, b2=np64(b2))
    if conv == "own_first":
        ref = np.stack([osel.select_conv_a(raw[:, h], topk, causal) for h in range(H)], 1)
    else:
        ref = osel.select_conv_b(raw, topk, sink)
    _check_sel(sel.cpu().numpy(), ref, "sel")
    assert np.array_equal(sc.cpu().numpy().astype(np.float64), np.take_along_axis(raw, ref, -1))


@pytest.mark.parametrize("B,nblk,scale", [(1, 300, 1e19), (1, 300, 1e-20), (33, 256, 1.0), (33, 256, 1e19)])
@pytest.mark.parametrize("D", [32, 64])
def test_select_mfma_engine_equals_fp64(B, nblk, scale, D):
    # past 256 blocks, or with more than 2^21 (row, candidate) pairs, "auto" is the MFMA engine
    # with its exact check of ambiguous pairs (every pair where the norms are past 1e18 or below
    # 2^-40); sampled rows against the oracle as well
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(41)
    a, b = ((torch.randn(B, 1, nblk, D, generator=g) * scale).to(torch.bfloat16) for _ in range(2))
    _say("mfma against fp64", B, nblk, scale, D)
    kw = dict(topk=16, causal=True, need_scores=True)
    sel1, sc1 = selection.select(a.to(DEV), b.to(DEV), engine="auto", **kw)
    sel2, sc2 = selection.select(a.to(DEV), b.to(DEV), engine="fp64", **kw)
    assert torch.equal(sel1, sel2) and torch.equal(sc1, sc2)
    raw = osel.scores(np64(a[:1]), np64(b[:1]), "bf16", "dot")
    _check_sel(sel1[:1, 0].cpu().numpy(), osel.select_conv_a(raw[:, 0], 16, True), "sel")


@pytest.mark.parametrize("dtype,D,score,B,nblk,topk", [
    ("f32", 256, "max2", 32, 256, 8), ("f32", 256, "quest", 8, 256, 8), ("f32", 256, "dot", 32, 256, 8),
    ("f32", 128, "max2", 32, 256, 8), ("f32", 64, "dot", 64, 256, 8), ("f32", 256, "max2", 64, 256, 62),
    ("bf16", 64, "max2", 128, 128, 8), ("bf16", 64, "quest", 32, 256, 8), ("bf16", 64, "dot", 512, 64, 8),
])
def test_select_row_kernel_is_taken_where_it_is_quicker(dtype, D, score, B, nblk, topk):
    # a chunk size rules the row kernel out: the choice made without one takes at most 1.3 times
    # the other engine's time
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(47)
    a, b1, b2 = (randn(g, (B, 1, nblk, D), dtype, device=DEV) for _ in range(3))
    kw = dict(score=score, topk=topk, causal=True, engine="auto")

    def run(chunk):
        return lambda: selection.select(a, b1, None if score == "dot" else b2, chunk_tiles=chunk, **kw)
    assert torch.equal(run(0)(), run(64)())
    t, other = _us(run(0)), _us(run(64))
    _say("choice", dtype, D, score, B, nblk, topk, t, other)
    assert t <= 1.3 * other + 3, (t, other)


@pytest.mark.parametrize("engine", ["auto", "fp64"])
@pytest.mark.parametrize("nblk", [1, 2, 63, 64, 65, 128, 129, 255, 256])
@pytest.mark.parametrize("dtype,D,score,conv,causal,topk,kind", [
    ("bf16", 64, "dot", "own_first", True, 16, "ties"), ("bf16", 32, "dot", "own_first", False, 62, "ties"),
    ("f16", 16, "max2", "own_first", True, 5, "ties"), ("f32", 64, "dot", "own_first", True, 8, "plain"),
    ("f32", 256, "quest", "sorted_sink", True, 30, "ties"), ("bf16", 128, "quest", "sorted_sink", True, 62, "plain"),
    ("f16", 64, "dot", "own_first", True, 16, "special"), ("bf16", 32, "dot", "sorted_sink", True, 62, "special"),
    ("f32", 32, "dot", "own_first", False, 7, "special"), ("bf16", 64, "quest", "sorted_sink", True, 16, "special"),
    ("bf16", 64, "dot", "own_first", True, 0, "plain"),
])
def test_select_row_kernel(dtype, D, score, conv, causal, topk, kind, nblk, engine):
    # one wave per row (up to 256 blocks, budgets up to 62): exact ties, NaN and infinite scores
    # on both sides of the 64th candidate, where ranking by lane reads ends and inserting begins
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(nblk + D)
    B, H = 2, 2
    if kind == "ties":
        dt = randn(g, (1,), dtype).dtype
        mk = lambda: torch.randint(-1, 2, (B, H, nblk, D), generator=g).to(dt)  # noqa: E731
    else:
        mk = lambda: randn(g, (B, H, nblk, D), dtype)  # noqa: E731
    a, b1, b2 = mk(), mk(), mk()
    if score == "quest":
        b1, b2 = torch.maximum(b1, b2), torch.minimum(b1, b2)
    if kind == "special":
        for j, v in ((0, "nan"), (1, "inf"), (62, "nan"), (63, "inf"), (64, "nan"), (65, "-inf"), (66, "inf"), (200, "nan")):
            if j < nblk:
                b1[:, :, j, 3] = float(v)
    _say("row kernel", dtype, D, score, conv, causal, topk, kind, nblk, engine)
    sel, sc = selection.select(a.to(DEV), b1.to(DEV), None if score == "dot" else b2.to(DEV), score=score, convention=conv,
                               topk=topk, causal=causal, sink=conv == "sorted_sink", need_scores=True, engine=engine)
    with np.errstate(invalid="ignore", over="ignore"):
        raw = osel.scores(np64(a), np64(b1), dtype, score, b2=None if score == "dot" else np64(b2))
    if conv == "own_first":
        ref = np.stack([osel.select_conv_a(raw[:, h], topk, causal) for h in range(H)], 1)
    else:
        ref = osel.select_conv_b(raw, topk, True)
    _check_sel(sel.cpu().numpy(), ref, "sel")
    # (a slot that repeats the own block in place of a non-finite pick carries its score)
    assert np.array_equal(sc.cpu().numpy().astype(np.float64), np.take_along_axis(raw, ref, -1), equal_nan=True)


@pytest.mark.parametrize("r0,r1", [(1, 2), (37, 101), (64, 130), (129, 130)])
def test_select_row_kernel_row_range(r0, r1):
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(43)
    B, H, nblk, D, topk = 2, 2, 130, 64, 9
    a, b = (randn(g, (B, H, nblk, D), "bf16") for _ in range(2))
    out = torch.full((B, H, nblk, topk + 1), -7, dtype=torch.int32, device=DEV)
    _say("row kernel rows", r0, r1)
    selection.select(a.to(DEV), b.to(DEV), topk=topk, causal=True, rows=(r0, r1), out=out)
    raw = osel.scores(np64(a), np64(b), "bf16", "dot")
    ref = np.full(out.shape, -7)
    for h in range(H):
        ref[:, h, r0:r1] = osel.select_conv_a(raw[:, h], topk, True)[:, r0:r1]
    _check_sel(out.cpu().numpy(), ref, "sel")


@pytest.mark.parametrize("dtype,score,conv,causal,topk,nblk,ties", [
    ("bf16", "dot", "own_first", True, 64, 900, False),
    ("bf16", "dot", "own_first", True, 128, 900, True),
    ("bf16", "dot", "own_first", False, 63, 300, False),
    ("f32", "dot", "own_first", True, 128, 600, False),
    ("bf16", "max2", "own_first", True, 100, 700, False),
    ("bf16", "dot", "sorted_sink", True, 64, 900, True),
    ("f16", "quest", "sorted_sink", True, 128, 700, False),
    ("bf16", "dot", "sorted_sink", True, 700, 700, False),
    ("bf16", "quest", "sorted_sink", True, 300, 1200, True),
])
def test_select_wide_budgets(dtype, score, conv, causal, topk, nblk, ties):
    # top-k budgets past one wave-wide list (> 62): one workgroup per row with
    # its keys in LDS; blocks and chosen-slot scores bit-exact against the oracle
    # (src/ssa_model.py:158-161 and src/qwen_blocksparse.py:90 take any topk)
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(31)
    B, H, D = 1, 2, 64
    if ties:
        mk = lambda: torch.randint(-2, 3, (B, H, nblk, D), generator=g).to(torch.bfloat16 if dtype == "bf16" else torch.float16 if dtype == "f16" else torch.float32)  # noqa: E731
    else:
        mk = lambda: randn(g, (B, H, nblk, D), dtype)  # noqa: E731
    a, b1, b2 = mk(), mk(), mk()
    if score == "quest":
        b1, b2 = torch.maximum(b1, b2), torch.minimum(b1, b2)
    _say("wide", dtype, score, conv, causal, topk, nblk, ties)
    sel, sc = selection.select(a.to(DEV), b1.to(DEV), None if score == "dot" else b2.to(DEV), score=score,
                               convention=conv, topk=topk, causal=causal, sink=conv == "sorted_sink",
                               need_scores=True)
    raw = osel.scores(np64(a), np64(b1), dtype, score, b2=None if score == "dot" else np64(b2))
    if conv == "own_first":
        ref = np.stack([osel.select_conv_a(raw[:, h], topk, causal) for h in range(H)], 1)
    else:
        ref = osel.select_conv_b(raw, topk, True)
    _check_sel(sel.cpu().numpy(), ref, "sel")
    assert np.array_equal(sc.cpu().numpy().astype(np.float64), np.take_along_axis(raw, ref, -1))


def test_select_quest_topk_100_config4_rows():
    # SelectMax with a budget of 100 at D 256 (the row-per-workgroup Quest kernel)
    from fbsa_amd import selection
    g = torch.Generator().manual_seed(32)
    B, Hq, Hkv, N, D, bs, topk = 1, 4, 2, 128 * 300, 256, 128, 100
    q = randn(g, (B, Hq, N, D), "bf16")
    k = randn(g, (B, Hkv, N, D), "bf16")
    idx = selection.select_quest(q.to(DEV), k.to(DEV), bs, topk, sink=True).cpu().numpy()
    ref, _ = osel.select_quest(np64(q), np64(k), bs, topk, True, "bf16")
    _check_sel(idx, ref, "idx")
