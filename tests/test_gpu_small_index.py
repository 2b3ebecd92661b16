"""GPU test of the one-launch transposed index: against a sorted restatement on the CPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("mask", ["none", "slot", "token"])
@pytest.mark.parametrize("B,hsel,nblk,kk", [(1, 1, 1, 1), (3, 1, 5, 4), (32, 1, 32, 5), (2, 2, 128, 18), (1, 2, 700, 9),
                                            (1, 1, 1024, 16), (5, 1, 33, 99), (1, 1, 1025, 3),
                                            (1, 1, 1024, 9), (1, 1, 16, 512), (3, 2, 65, 8), (3, 2, 65, 9),
                                            (512, 1, 8, 4), (513, 1, 4, 4), (1, 1, 2, 4097)])
def test_transposed_index(mask, B, hsel, nblk, kk):
    # (1025 blocks, 513 groups and walks past 18432 entries take the sort)
    from fbsa_amd import _lib, ops
    g = np.random.default_rng(nblk + kk)
    sel = g.integers(-1, nblk + 1, (B, hsel, nblk, kk)).astype(np.int32)
    sel[..., 0] = np.arange(nblk)
    bs = 16
    L = nblk * bs
    lv = L - 5 if mask != "slot" else L
    m = {"none": ops.MASK_NONE, "slot": ops.MASK_SLOT_CAUSAL, "token": ops.MASK_TOKEN_CAUSAL}[mask]
    q = torch.empty(B, 2, L, 32, device=DEV, dtype=torch.bfloat16)
    st = torch.from_numpy(sel).to(DEV)
    d = ops.make_desc(q, q, q, q, st, mask=m, scale=1.0, l_valid=lv, dout=q)
    d.hsel = hsel
    lib = _lib.load()
    n = lib.fbsa_bwd_workspace_bytes(d)
    ws = torch.zeros(n + 256, dtype=torch.uint8, device=DEV)
    wp = (ws.data_ptr() + 255) // 256 * 256
    print("index", mask, B, hsel, nblk, kk, flush=True)
    _lib.check(lib.fbsa_transpose_index(d, st.data_ptr(), wp, n, torch.cuda.current_stream().cuda_stream), "index")
    host = ws.cpu().numpy()[wp - ws.data_ptr():]
    # reference: valid (segment, i * kk + slot) pairs in stable order
    ref = []
    for b in range(B):
        for hs in range(hsel):
            for i in range(nblk):
                seen = set()
                for s in range(kk):
                    j = int(sel[b, hs, i, s])
                    if not 0 <= j < nblk:
                        continue
                    if mask == "none":
                        ok = j * bs < lv
                    elif mask == "slot":
                        ok = s == 0 or j < i
                    else:
                        ok = j <= i and j * bs < lv and j not in seen
                        seen.add(j)
                    if ok:
                        ref.append(((b * hsel + hs) * nblk + j, i * kk + s))
    ref.sort(key=lambda t: t[0])
    nseg = B * hsel * nblk
    off = np.searchsorted(np.array([t[0] for t in ref], np.int64), np.arange(nseg + 1)).astype(np.int32)
    ent = np.array([t[1] for t in ref], np.int32)
    al = lambda x: (x + 255) // 256 * 256  # noqa: E731
    ne = B * hsel * nblk * kk
    at = al(B * 2 * L * 8)                      # row statistics
    at = al(at + B * 2 * nblk * kk * 4)         # gate-gradient partials
    at += 3 * al(ne * 4)                        # keys in / out, values in
    got_ent = host[at:at + 4 * len(ent)].view(np.int32)
    at += al(ne * 4)
    got_off = host[at:at + 4 * (nseg + 1)].view(np.int32)
    assert np.array_equal(got_off, off)
    assert np.array_equal(got_ent, ent)


def _index(B, hsel, nblk, kk, mask):
    """A call of the index stage over causal picks, and the tensors it reads."""
    from fbsa_amd import _lib, ops
    g = np.random.default_rng(nblk + kk)
    sel = (g.random((B, hsel, nblk, kk)) * (np.arange(nblk)[:, None] + 1)).astype(np.int32)
    st = torch.from_numpy(sel).to(DEV)
    q = torch.empty(B, 2, nblk * 16, 32, device=DEV, dtype=torch.bfloat16)
    d = ops.make_desc(q, q, q, q, st, mask=mask, scale=1.0, l_valid=None, dout=q)
    d.hsel = hsel
    lib = _lib.load()
    n = lib.fbsa_bwd_workspace_bytes(d)
    ws = torch.zeros(n + 256, dtype=torch.uint8, device=DEV)
    wp = (ws.data_ptr() + 255) // 256 * 256
    s = torch.cuda.current_stream().cuda_stream
    return lambda: _lib.check(lib.fbsa_transpose_index(d, st.data_ptr(), wp, n, s), "index"), (st, ws)


def _us(run):
    """Median of seven timings of ten calls back to back, in us a call."""
    for _ in range(3):
        run()
    t = []
    for _ in range(7):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(10):
            run()
        b.record()
        b.synchronize()
        t.append(a.elapsed_time(b) * 100)
    return sorted(t)[3]


@pytest.mark.parametrize("mask", ["slot", "token"])
@pytest.mark.parametrize("B,hsel,nblk,kk", [(1, 2, 128, 18), (1, 1, 512, 16), (1, 1, 1024, 8), (1, 1, 1024, 16), (1, 1, 300, 50)])
def test_index_time_does_not_grow_with_the_blocks(mask, B, hsel, nblk, kk):
    # the longest calls of the one-launch index against the sort's (1025 blocks are past
    # the former's, 15375 entries are the largest both may see): at most half again as long
    from fbsa_amd import ops
    m = ops.MASK_SLOT_CAUSAL if mask == "slot" else ops.MASK_TOKEN_CAUSAL
    print("index time", mask, B, hsel, nblk, kk, flush=True)
    run, keep = _index(B, hsel, nblk, kk, m)
    sort, keep2 = _index(1, 1, 1025, 15, m)
    t, ref = _us(run), _us(sort)
    assert t <= 1.5 * ref, (t, ref)
