"""GPU tests of a short last block without padded copies (FBSA_FLAG_RAGGED): bit for bit
the results of the zero-padded tensors with l_valid, gradients included."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(q, k, v, sel, og, do, gate, mask, L, bs, ragged):
    from fbsa_amd.autograd import block_sparse_attention
    pad = 0 if ragged else -L % bs
    ins = [F.pad(t, (0, 0, 0, pad)).detach().requires_grad_(True) if t is not None else None for t in (q, k, v, og)]
    gt = gate.detach().requires_grad_(True) if gate is not None else None
    kw = {"bs": bs} if ragged else {"l_valid": L}
    o = block_sparse_attention(*ins[:3], sel, mask=mask, gate=gt, out_gate=ins[3], **kw)
    leaves = [t for t in ins if t is not None]
    grads = torch.autograd.grad(o, leaves + ([gt] if gt is not None else []), F.pad(do, (0, 0, 0, pad)))
    cut = [t[..., :L, :] for t in (o.detach(), *grads[:len(leaves)])]
    return cut + list(grads[len(leaves):])


@pytest.mark.parametrize("extra", ["plain", "out_gate", "gate", "dense", "none"])
@pytest.mark.parametrize("dtype,D,bs,nblk,last", [("bf16", 256, 128, 5, 1), ("bf16", 64, 64, 6, 63), ("f16", 128, 128, 3, 65),
                                                  ("f16", 256, 64, 4, 33), ("bf16", 32, 16, 7, 5), ("f32", 64, 64, 5, 17),
                                                  ("f32", 256, 128, 3, 15), ("bf16", 64, 32, 1, 7),
                                                  ("bf16", 128, 64, 5, 7), ("f16", 64, 128, 4, 127), ("f32", 128, 128, 3, 1),
                                                  ("f32", 32, 16, 9, 3)])
def test_ragged_equals_padded(dtype, D, bs, nblk, last, extra):
    from fbsa_amd import ops
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    B, Hq, Hkv, L = 2, 4, 2, (nblk - 1) * bs + last
    g = torch.Generator().manual_seed(D + bs + last)
    q, do, og = (torch.randn(B, Hq, L, D, generator=g).to(dt).to(DEV) for _ in range(3))
    k = torch.randn(B, Hkv, L, D, generator=g).to(dt).to(DEV)
    v = torch.randn(B, L, Hkv, D, generator=g).to(dt).to(DEV).transpose(1, 2)
    kk = min(4, nblk) + 1
    sel = torch.randint(0, nblk, (B, Hkv, nblk, kk), generator=g, dtype=torch.int32)
    sel[..., 0] = torch.arange(nblk)
    gate = torch.randn(B, Hkv, nblk, kk, generator=g).to(DEV) if extra in ("gate", "none") else None
    sel = ops.DenseSelection(B, nblk) if extra == "dense" else sel.to(DEV)
    mask = ops.MASK_NONE if extra == "none" else ops.MASK_TOKEN_CAUSAL
    og = og if extra in ("out_gate", "none") else None
    print("ragged", dtype, D, bs, L, extra, flush=True)
    got = _run(q, k, v, sel, og, do, gate, mask, L, bs, True)
    ref = _run(q, k, v, sel, og, do, gate, mask, L, bs, False)
    assert len(got) == len(ref)
    for n, (x, y) in enumerate(zip(got, ref)):
        assert x.shape == y.shape and torch.equal(x, y), (n, float((x.float() - y.float()).abs().max()))


def test_ragged_rejects():
    from fbsa_amd import ops
    q = torch.randn(1, 2, 100, 64, device=DEV, dtype=torch.bfloat16)
    sel = torch.zeros(1, 1, 2, 1, dtype=torch.int32, device=DEV)
    with pytest.raises(ValueError):   # slot-causal lists have no padding rule
        ops.attention_forward(q, q, q, sel, mask=ops.MASK_SLOT_CAUSAL, bs=64)
    with pytest.raises(ValueError):   # 100 rows are not 2 blocks of 128
        ops.attention_forward(q, q, q, sel, mask=ops.MASK_TOKEN_CAUSAL, bs=128)
    with pytest.raises(ValueError):   # nor, without a block size, an even split into 3
        ops.attention_forward(q, q, q, sel.new_zeros(1, 1, 3, 1), mask=ops.MASK_TOKEN_CAUSAL)
