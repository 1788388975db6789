"""What vqx_mx_operand_decode refuses: the host checks come before any launch,
so addresses that hold nothing show them without a GPU."""

import pytest

BASE = 1 << 20


# (data, ld, batch stride, scale, scale ld, scale batch stride): one value off
# 16-byte rows each; N-major scales are read in rows of 16 bytes too
@pytest.mark.parametrize("k_major,fields,message", [
    (1, (BASE + 2, 64, 4096, 0, 0, 0), "16-byte aligned"),
    (1, (BASE + 8, 64, 4096, 0, 0, 0), "16-byte aligned"),
    (1, (BASE, 68, 4096, 0, 0, 0), "multiple of 8"),
    (1, (BASE, 64, 4100, 0, 0, 0), "multiple of 8"),
    (0, (BASE, 64, 4096, BASE + 2, 64, 512), "N-major scales"),
    (0, (BASE, 64, 4096, BASE, 68, 544), "N-major scales"),
    (0, (BASE, 64, 4096, BASE, 64, 516), "N-major scales")])
def test_operand_decode_refuses(vqx, k_major, fields, message):
    L = vqx._lib
    data, ld, stride, scale, sld, sstride = fields
    op = L.VqxMxOperand(data, scale or None, None, stride, ld, sstride, sld, k_major, 8 if scale else 0, 0, 0)
    with pytest.raises(ValueError, match=message):
        L.call("vqx_mx_operand_decode", L.ctypes.byref(op), 2, 64, 64, BASE, None)
