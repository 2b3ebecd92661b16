"""CPU tests: rows so far apart that a chunk's copy offsets would not fit 32 bits are copied by the
Python entries and refused by the C ABI."""
import pytest
import torch

from fbsa_amd import _lib, ops
from test_cpu_lib import DUMMY, _desc

FAR = 1 << 28   # bytes: 63 rows of it pass 2^32


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_far_rows_are_copied(dtype):
    es = torch.empty(0, dtype=dtype).element_size()
    for rows, copied in ((64 << 10, False), ((1 << 25) - 16, False), (1 << 25, True), (FAR, True)):
        x = torch.empty_strided((1, 2, 40, 64), (0, 64, rows // es, 1), dtype=dtype, device="meta")
        y = ops._kernel_ready(x)
        assert (y is not x) == copied and y.shape == x.shape
        if copied:
            assert y.is_contiguous()
            # the largest offset a chunk forms from an accepted stride, also where it is signed
        else:
            assert 63 * rows + 256 * es < 1 << 31


@pytest.mark.parametrize("field", ["sk", "sv"])
@pytest.mark.parametrize("flags,l_valid,mask", [(0, 256, _lib.MASK_SLOT_CAUSAL), (_lib.FLAG_RAGGED, 200, _lib.MASK_TOKEN_CAUSAL)])
def test_fwd_refuses_far_rows(field, flags, l_valid, mask):
    lib = _lib.load()
    d = _desc(flags=flags, l_valid=l_valid, mask=mask)
    getattr(d, field)[2] = FAR // 2
    assert lib.fbsa_fwd(d, DUMMY, DUMMY, DUMMY, DUMMY, None, None, DUMMY, None, None) == _lib.EUNSUPPORTED
    assert "row stride" in lib.fbsa_last_error().decode()


@pytest.mark.parametrize("field", ["sq", "sk", "sv", "sdo"])
def test_bwd_refuses_far_rows(field):
    lib = _lib.load()
    d = _desc()
    n = lib.fbsa_bwd_workspace_bytes(d)
    getattr(d, field)[2] = FAR // 2
    st = lib.fbsa_bwd(d, *[DUMMY] * 4, None, None, DUMMY, DUMMY, DUMMY, DUMMY, DUMMY, DUMMY, None, None, DUMMY, n, None)
    assert st == _lib.EUNSUPPORTED and "row stride" in lib.fbsa_last_error().decode()


def test_mass_refuses_far_rows():
    lib = _lib.load()
    d = _desc(mask=_lib.MASK_TOKEN_CAUSAL, kk=1)
    d.sk[2] = (1 << 26) // 2   # 63 rows of 64 MiB pass 2^31, this kernel's signed offsets
    assert lib.fbsa_block_mass(d, DUMMY, DUMMY, DUMMY, DUMMY, None) == _lib.EUNSUPPORTED
    assert "row stride" in lib.fbsa_last_error().decode()
