"""GPU tests of the one-pass block mass: references that move, and walks too long for one launch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _row_mass(q, k, b, h, hk, i, bs, scale):
    """Query block i's masses per key block in float64 (torch, on the GPU): scores
    rounded after the product and after the scale, as the kernel defines them."""
    n = (i + 1) * bs
    qi, kj = q[b, h, i * bs:n].double(), k[b, hk, :n].double()
    s = ((qi @ kj.t()).to(q.dtype).double() * float(np.float32(scale))).to(q.dtype).double()
    t = torch.arange(n, device=q.device)
    s = s.masked_fill(t > t[i * bs:].view(-1, 1), float("-inf"))
    return s.softmax(-1).view(bs, i + 1, bs).sum(-1).mean(0)


def _check(got, ref, smax):
    # every term's exponent is rounded once in fp32 (relative error |S| 2^-24 per term, twice
    # with the reference's), each sum adds at most 2^-24 per level; 4x for the hardware exp2
    tol = 4 * (2 * smax + 16) * 2.0 ** -24
    err = (got.double() - ref).abs() / ref.clamp(min=1e-25)
    assert float(err.max()) <= tol, (float(err.max()), tol)


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("scale", [0.125, 0.11])
@pytest.mark.parametrize("bs,D", [(64, 64), (64, 256), (128, 64), (128, 128), (128, 256)])
def test_mass_with_moving_references(dtype, scale, bs, D):
    # small whole operands: every product is exact, so the rounded scores are the
    # reference's and only the fp32 softmax differs; keys grow with the position, so
    # references move in many blocks, and fall again, so they also stay
    from fbsa_amd import ops
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    nblk = 9
    g = torch.Generator().manual_seed(bs + D)
    q = torch.randint(-1, 2, (2, 4, nblk * bs, D), generator=g).float()
    k = torch.randint(-1, 2, (2, 2, nblk * bs, D), generator=g).float()
    grow = torch.tensor([1.0, 2.0, 4.0, 1.0, 8.0, 2.0, 16.0, 8.0, 0.0]).repeat_interleave(bs)
    q, k = q.to(dt).to(DEV), (k * grow.view(1, 1, -1, 1)).to(dt).to(DEV)
    print("mass", dtype, scale, bs, D, flush=True)
    m = ops.block_mass(q, k, bs, scale)
    smax = float((q.double() @ k.double().repeat_interleave(2, 1).transpose(-1, -2)).abs().max()) * scale
    for b, h in ((0, 0), (1, 3)):
        for i in range(nblk):
            _check(m[b, h, i, :i + 1], _row_mass(q, k, b, h, h // 2, i, bs, scale), smax)
            assert not m[b, h, i, i + 1:].any()


def test_mass_over_several_launches():
    # 2048 key blocks: a workgroup's sums take 786 KB, so 1 GiB holds a third of the workgroups
    from fbsa_amd import ops
    L, D, bs = 131072, 64, 64
    g = torch.Generator(device=DEV).manual_seed(7)
    q, k = (torch.randint(-1, 2, (1, 2, L, D), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    print("mass", L, flush=True)
    m = ops.block_mass(q, k, bs, 0.125)
    nblk = L // bs
    for h in range(2):
        for i in (0, 1, 2, 500, 900, 1023, 1365, 1366, 1700, nblk - 2, nblk - 1):
            _check(m[0, h, i, :i + 1], _row_mass(q, k, 0, h, h, i, bs, 0.125), 8.0)
            assert not m[0, h, i, i + 1:].any()
