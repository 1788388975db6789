"""GPU: the decode passes ahead of the products (vqx_mx_operand_rows) and the
products of odd sizes that run on them, against torch.

The decode is bit exact: bf16(code[index] * scale), one fp32 product rounded
once.  The products are compared with float64 products of the decoded
operands within the bound of tests/test_gpu_dense_matmul.py."""

import pytest
import torch

from tests.test_gpu_dense_matmul import close

Q = torch.ops.quantized_ops


def operand(shape, kdim, bs, coded, seed, scaled=True, code_len=16):
    """(values, code, scales) of a convert-format operand blocked along kdim."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    lo, hi = (-code_len, code_len) if coded else (-128, 128)
    x = torch.randint(lo, hi, shape, generator=g, device="cuda").to(torch.bfloat16)
    code = torch.randn(code_len, generator=g, device="cuda").to(torch.bfloat16) if coded else None
    if not scaled:
        return x, code, None
    ss = list(shape)
    ss[kdim] = -(-ss[kdim] // bs)
    return x, code, (torch.rand(ss, generator=g, device="cuda") + 0.25).to(torch.bfloat16)


def decoded(x, code, scale, bs, kdim):
    v = x
    if code is not None:
        K = code.numel()
        i = torch.trunc(x.float())
        ok = (i >= -K) & (i < K)
        v = torch.where(ok, code[torch.where(ok, i, torch.zeros_like(i)).long() % K], torch.full_like(x, float("nan")))
    if scale is None:
        return v
    e = scale.repeat_interleave(bs, kdim).narrow(kdim, 0, x.shape[kdim])
    return (v.float() * e.float()).to(torch.bfloat16)


# tile edges of the 64 x 64 turn, rows of odd length, one value
@pytest.mark.gpu
@pytest.mark.parametrize("R,C", [(1, 1), (64, 64), (65, 63), (7, 200), (200, 7), (130, 129), (128, 4096)])
@pytest.mark.parametrize("kdim", [-1, -2])
@pytest.mark.parametrize("coded,scaled", [(False, True), (True, True), (True, False), (False, False)])
def test_operand_rows(vqx, R, C, kdim, coded, scaled):
    print(f"rows {R}x{C} kdim={kdim} coded={coded} scaled={scaled}", flush=True)
    qops = vqx.ops.quantized
    bs = 8
    x, code, scale = operand((2, R, C), kdim, bs, coded, R * 3 + C, scaled, 13)
    if coded:
        for i, v in enumerate((13.0, -14.0, float("nan"), float("inf"), -13.5, 0.9, 300.0)):
            x.view(-1)[i % x.numel()] = v  # outside the table, and truncated into it
    want = decoded(x, code, scale, bs, kdim)
    for k_last in (True, False):
        rows = want if (kdim == -1) == k_last else want.transpose(-2, -1)
        n = rows.shape[-1]
        turned = (kdim == -1) != k_last
        for ld in {-(-n // 64) * 64, -(-n // 8) * 8} | ({n} if turned or n % 8 == 0 else set()):
            got = qops._mx_rows(x, code, scale, bs, kdim, k_last, ld)
            assert got.shape == (2, rows.shape[-2], ld)
            a, b = got[..., :n], rows
            same = (a.contiguous().view(torch.int16) == b.contiguous().view(torch.int16)) | (a.isnan() & b.isnan())
            assert bool(same.all()), int((~same).sum())
            assert not bool(got[..., n:].count_nonzero())


# every route of a batched product: both decoded ahead, one inside, ragged K
# read in place, odd N, a shared right or left operand, a stored transpose
@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", [((3,), 333, 333, 64), ((2, 2), 333, 128, 333), ((3,), 1300, 64, 77),
                                     ((2,), 5, 1999, 128), ((2,), 1, 128, 1999), ((3,), 700, 66, 130),
                                     ((2,), 40, 33, 9), ((2,), 130, 4, 8), ((1,), 600, 1024, 200), ((2,), 3, 3, 3),
                                     ((2, 2), 4, 65, 513), ((3,), 2, 8, 512), ((1,), 1, 1, 1), ((2,), 4, 100, 4096),
                                     ((2,), 4, 40, 4104), ((1,), 1, 70, 16384), ((2,), 1, 64, 1025)])
@pytest.mark.parametrize("coded", [False, True])
@pytest.mark.parametrize("form", ["plain", "b_shared", "a_shared", "kc", "b_transposed"])
def test_odd_products(vqx, B, M, N, K, coded, form):
    print(f"product B={B} M={M} N={N} K={K} coded={coded} form={form}", flush=True)
    bs = 16
    ab, bb = (() if form == "a_shared" else B), (() if form == "b_shared" else B)
    a, code, sa = operand((*ab, M, K), -1, bs, coded, 1)
    if form == "kc":
        b, _, sb = operand((*bb, N, K), -1, bs, coded, 2)
        bd = decoded(b, code, sb, bs, -1).transpose(-2, -1)
    else:
        b, _, sb = operand((*bb, K, N), -2, bs, coded, 2)
        bd = decoded(b, code, sb, bs, -2)
        if form == "b_transposed":
            b = b.transpose(-2, -1).contiguous().transpose(-2, -1)
    got = Q.matmul_mx(a, b, input_scale=sa, weight_scale=sb, block_size=bs, input_code=code, weight_code=code,
                      weight_layout="kc" if form == "kc" else "ck")
    ad, bd = decoded(a, code, sa, bs, -1).double().expand(*B, M, K), bd.double().expand(*B, K, N)
    want, mag = torch.matmul(ad, bd.contiguous()), torch.matmul(ad.abs(), bd.abs().contiguous())
    assert got.shape == want.shape
    close(got, want, mag, K)


# Every form of the few-row kernel: 64 or 16 columns per workgroup (the first
# where that gives every CU one), an item's workgroups on one XCD (batches of
# eight) or in order
@pytest.mark.gpu
@pytest.mark.parametrize("B,N,K,cols,one_xcd", [(32, 1999, 128, 64, True), (8, 65, 513, 16, True),
                                                (35, 520, 77, 64, False), (32, 128, 1999, 16, True),
                                                (3, 130, 257, 16, False)])
@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("coded", [False, True])
def test_few_rows_forms(vqx, B, N, K, cols, one_xcd, M, coded):
    print(f"few rows B={B} M={M} N={N} K={K} coded={coded}", flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert (B * -(-N // 64) >= cus) == (cols == 64) and (B % 8 == 0) == one_xcd
    bs = 32
    a, code, sa = operand((B, M, K), -1, bs, coded, 3)
    b, _, sb = operand((B, K, N), -2, bs, coded, 4)
    got = vqx.ops.quantized._few_rows_product(a, code, sa, b, code, sb, bs)
    ad, bd = decoded(a, code, sa, bs, -1).double(), decoded(b, code, sb, bs, -2).double()
    close(got, torch.matmul(ad, bd), torch.matmul(ad.abs(), bd.abs()), K)
