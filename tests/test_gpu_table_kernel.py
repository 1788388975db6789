"""GPU: quantize_mx on a caller's 65536-entry table at the sizes where the
table is kept in LDS, bit for bit against the oracle.  The table is random, so
every quotient that rounds to another bf16 pattern shows."""

import pytest
import torch

from oracle import formats as F
from oracle import reference_ops as R
from tests.conftest import assert_bitexact

Q = torch.ops.quantized_ops


def every_pattern(n, seed):
    """bf16 values: all finite patterns, then blocks of mixed magnitudes, with
    zeros, -0, subnormals, NaN and Inf in some blocks."""
    g = torch.Generator().manual_seed(seed)
    bits = torch.randint(0, 65536, (n,), generator=g, dtype=torch.int32)
    bits[:65536] = torch.arange(65536, dtype=torch.int32)
    # most blocks of 128: magnitudes within a few octaves of one exponent
    e = torch.randint(1, 254, (n // 128 + 1,), generator=g, dtype=torch.int32).repeat_interleave(128)[:n]
    near = (e + torch.randint(-6, 1, (n,), generator=g, dtype=torch.int32)).clamp(0, 254) << 7
    near |= torch.randint(0, 128, (n,), generator=g, dtype=torch.int32)
    near |= torch.randint(0, 2, (n,), generator=g, dtype=torch.int32) << 15
    pick = (torch.arange(n) >= 65536) & (torch.arange(n) // 128 % 8 != 0)
    bits = torch.where(pick, near, bits)
    zero = torch.rand(n, generator=g) < 0.02
    bits = torch.where(zero, bits & 0x8000, bits)
    return torch.where(bits >= 32768, bits - 65536, bits).to(torch.int16).view(torch.bfloat16)


def random_table(seed):
    t = torch.randint(0, 0x7F00, (65536,), generator=torch.Generator().manual_seed(seed), dtype=torch.int32)
    # a NaN quotient's payload is not the reference's: every NaN pattern alike, as in its tables
    t[(torch.arange(65536) & 0x7FFF) > 0x7F80] = 0x7FC0
    return t.to(torch.int16).view(torch.bfloat16)


# either side of the size from which the table is kept in LDS, a tail of
# groups past the last whole 1024 elements, every block size, both scales
@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(2049, 1024), (1023, 2048), (1311, 1664), (2303, 1024), (2305, 1024),
                                       (1431, 1664)])
@pytest.mark.parametrize("bs,mode", [(16, "absmax"), (32, "pow2"), (64, "qmap"), (128, "absmax"), (16, "qmap"),
                                     (64, "pow2"), (128, "pow2"), (16, "absmax/1"), (32, "absmax/64"),
                                     (128, "absmax/1")])
def test_table_kernel(vqx, rows, cols, bs, mode):
    print(f"table kernel {rows}x{cols} bs={bs} {mode}", flush=True)
    x = every_pattern(rows * cols, rows + bs).reshape(rows, cols)
    table = random_table(bs)
    smap = R.table_tensor(F.quantization_table("fp8_e5m3")) if mode == "qmap" else None
    qmax = 31.0 if mode != "pow2" else 448.0
    if "/" in mode:
        # the kernel's multiplication in place of the division by a power of
        # two; some whole blocks of subnormal values, whose scales are subnormal
        qmax = float(mode.split("/")[1])
        sub = torch.arange(rows * cols).reshape(rows, cols) // 128 % 16 == 5
        bits = torch.where(sub, x.view(torch.int16) & -32641, x.view(torch.int16))  # exponent bits cleared
        x = bits.view(torch.bfloat16)
    s, q = Q.quantize_mx(x.cuda(), table.cuda(), [-1], bs, qmax, mode == "pow2", None if smap is None else smap.cuda(), None)
    ws, wq = R.quantize_mx(x, table, [-1], bs, qmax, mode == "pow2", smap)
    assert_bitexact(s, ws, "scales")
    assert_bitexact(q, wq, "values")


# Every set of outputs the C entry point can ask of the kernel, against the same
# rows in calls below the size from which the table is kept in LDS
@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["absmax", "absmax/64", "pow2"])
@pytest.mark.parametrize("outputs", ["fq", "values fq"])
def test_table_kernel_fake_quant(vqx, mode, outputs):
    print(f"table kernel {outputs} {mode}", flush=True)
    L, q = vqx._lib, vqx.ops.quantized
    rows, cols, bs = 1431, 1664, 32
    x = every_pattern(rows * cols, 9).reshape(rows, cols).cuda()
    d, keep = q._table_desc(random_table(3).cuda(), x.device)
    qmax, shift = (64.0 if "/" in mode else 31.0), 8

    def call(x):
        n = x.numel()
        out = {k: torch.zeros(n, dtype=torch.bfloat16, device="cuda") for k in outputs.split()}
        scale = torch.zeros(n // bs, dtype=torch.bfloat16, device="cuda")
        scale32 = torch.zeros(n // bs, dtype=torch.float32, device="cuda")
        e8m0 = torch.zeros(n // bs, dtype=torch.uint8, device="cuda") if mode == "pow2" else None
        L.call("vqx_mx_quantize", L.ptr(x), L.BF16, x.shape[0], cols, 1, bs, L.ctypes.byref(d), 0 if mode == "pow2" else 1,
               shift, qmax, None, L.ptr(scale), L.ptr(scale32), L.ptr(e8m0), L.ptr(out.get("values")),
               L.ptr(out.get("fq")), None, 0, L.stream_of(x))
        return [out[k].view(torch.int16) for k in out] + [scale.view(torch.int16), scale32.view(torch.int32)] + (
            [] if e8m0 is None else [e8m0])

    got = call(x)
    parts = [call(x[i:i + 400].contiguous()) for i in range(0, rows, 400)]
    for g, w in zip(got, [torch.cat(p) for p in zip(*parts)]):
        if g.dtype == torch.int16:  # any NaN is as good as another
            f, h = g.view(torch.bfloat16), w.view(torch.bfloat16)
            same = (g == w) | (f.isnan() & h.isnan())
        else:
            same = (g == w) | ((g & 0x7FFFFFFF) > 0x7F800000) & ((w & 0x7FFFFFFF) > 0x7F800000) \
                if g.dtype == torch.int32 else g == w
        assert bool(same.all()), int((~same).sum())
