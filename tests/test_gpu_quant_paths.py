"""The quantizers' and producers' kernels at the sizes and values where each branch can go wrong, against the
CPU oracle (or, for a call that several routes can take, against the general route)."""
import numpy as np
import pytest
import torch

from helpers import FP8_DT, TORCH_DT, f32
from oracle import formats as OF

pytestmark = pytest.mark.gpu


def _u8(t):
    return t.contiguous().view(torch.uint8).cpu().numpy()


def _edge_floats():
    """fp32 values at the fp8 formats' edges: every 16-bit pattern as the upper half, the midpoints between
    neighbouring codes and one ulp to each side, both signs, infinities and NaNs of both signs."""
    top = (np.arange(1 << 16, dtype=np.uint32) << 16)
    mid = top | 0x8000
    parts = [top, top + 1, top - 1, mid, mid + 1, mid - 1, np.array([0x7FC00000, 0xFFC00000, 0x7F800001, 0xFF800001], np.uint32)]
    return np.concatenate(parts).view(np.float32)


@pytest.mark.parametrize("fmt", ["e4m3fn", "e5m2"])
def test_fp8_bytes_of_edge_values(gpu, fmt):
    """base = fp8(k) byte for byte, NaN signs included (the residual of a NaN or an overflow is a NaN whose
    sign the subtraction does not define: compared where the base is finite)."""
    from ffa_mi355x import kfmt_quant as KQ

    x = _edge_floats()
    base, res = KQ.quantize_fp8fp8(torch.from_numpy(x.copy()).to(gpu), FP8_DT[fmt])
    with np.errstate(invalid="ignore", over="ignore"):
        ob, orr = OF.quantize_fp8fp8(x, fmt)
    assert np.array_equal(_u8(base), ob)
    fine = (ob & 0x7F) < (0x7F if fmt == "e4m3fn" else 0x7C)
    assert np.array_equal(_u8(res)[fine], orr[fine])
