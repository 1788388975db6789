"""GPU: vqx_dense_matmul (the product of plain bf16 operands with K
contiguous) and the linears that run on it, against float64.

Tolerance: the inputs are exact, so an output differs from float64 by its
rounding to bf16 (half an ulp: 2^-9 of the value) and by the fp32 sums'
rounding, at most (K + splits) * 2^-24 of sum |a b|.  The bound below doubles
the first for the bias added before the rounding."""

import ctypes

import pytest
import torch

Q = torch.ops.quantized_ops


def close(got, want64, mag64, K):
    err = (got.double() - want64).abs()
    tol = 2.0**-8 * want64.abs() + (K + 16) * 2.0**-24 * mag64 + 1e-30
    bad = err > tol
    assert not bool(bad.any()), (int(bad.sum()), float((err / tol).max()))


def run(vqx, a, b, bias, ws=True):
    L = vqx._lib
    nb, M, K = a.shape
    N = b.shape[1]
    out = torch.full((nb, M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    n = ctypes.c_int64(0)
    L.call("vqx_dense_matmul_workspace_size", nb, M, N, K, ctypes.byref(n))
    w = torch.empty(n.value, dtype=torch.uint8, device="cuda") if ws and n.value else None
    L.call("vqx_dense_matmul", L.ptr(a), K, M * K, L.ptr(b), K, N * K, L.ptr(bias), L.ptr(out), nb, M, N, K, L.ptr(w),
           n.value if w is not None else 0, L.stream_of(a))
    return out, n.value


def plan(M, N, K, nb=1):
    """The tile's columns and the K pieces the product takes on 256 CUs: the
    estimate of plan_dense (vqx_dense_gemm.hip) restated."""
    if K <= 128:
        return ("narrow" if nb * -(-M // 128) * -(-N // 128) <= 256 else "short"), 1
    best = None
    for shape, cols, step, start in (("wide", 256, 0.82, 3.0), ("narrow", 128, 0.45, 2.5)):
        tiles, nk = nb * -(-M // 128) * -(-N // cols), K // 64
        for s in range(1, 17):
            if s == 1 or 4 * s <= nk:
                c = -(-tiles * s // 256) * (step * -(-nk // s) + start)
                c += 4.0 + 0.2 * (128 * cols * 4e-6) * tiles * s if s > 1 else 0.0
                if best is None or c < best[0]:
                    best = (c, shape, s)
    return best[1:]


# (1 to 7 steps of the 64-deep, three-stage ring, with and without a split, row
# bands, odd columns, several items; the narrow and the short shape)
@pytest.mark.gpu
@pytest.mark.parametrize("nb,M,N,K", [(1, 1, 8, 64), (1, 128, 256, 128), (1, 129, 257, 192), (1, 127, 255, 256),
                                      (2, 40, 1000, 320), (1, 1100, 264, 384), (3, 130, 33, 448), (1, 17, 7, 1024),
                                      (1, 333, 512, 4096), (1, 64, 2, 11008), (1, 2300, 4104, 64),
                                      (1, 2048, 2048, 128), (1, 2049, 2048, 128), (5, 1100, 1001, 64),
                                      (5, 1001, 1100, 128)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_dense_matmul(vqx, nb, M, N, K, with_bias):
    print(f"dense nb={nb} M={M} N={N} K={K} bias={with_bias} plan={plan(M, N, K, nb)}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    a = torch.randn(nb, M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(nb, N, K, generator=g, device="cuda").to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16) if with_bias else None
    want = torch.stack([a[i].double() @ b[i].double().t() for i in range(nb)])
    mag = torch.stack([a[i].double().abs() @ b[i].double().abs().t() for i in range(nb)])
    if with_bias:
        want, mag = want + bias.double(), mag + bias.double().abs()
    got, need = run(vqx, a, b, bias)
    close(got, want, mag, K)
    if need:  # the same product without its workspace runs whole tiles
        close(run(vqx, a, b, bias, ws=False)[0], want, mag, K)


# The wide shape: in 5 and 3 pieces of K (its fp32 sums and their reduction),
# and whole with partial row and column tiles, odd N, and 4, 5 and 7 steps.
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,pieces", [(333, 4096, 11008, 5), (640, 4096, 11008, 3), (333, 4093, 11008, 5),
                                          (2047, 11003, 320, 1), (1921, 11009, 256, 1), (2047, 11008, 448, 1)])
def test_dense_matmul_wide(vqx, M, N, K, pieces):
    print(f"dense wide M={M} N={N} K={K} pieces={pieces}", flush=True)
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    assert plan(M, N, K) == ("wide", pieces)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(1, M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(1, N, K, generator=g, device="cuda").to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    want = (a[0].double() @ b[0].double().t() + bias.double())[None]
    mag = (a[0].double().abs() @ b[0].double().abs().t() + bias.double().abs())[None]
    got, need = run(vqx, a, b, bias)
    tiles = -(-M // 128) * -(-N // 256)
    assert need == (tiles * pieces * 128 * 256 * 4 if pieces > 1 else 0)
    close(got, want, mag, K)
    if need:  # the same product without its workspace runs whole tiles
        close(run(vqx, a, b, bias, ws=False)[0], want, mag, K)


# an output that starts inside a 16-byte row, in each of the three shapes (K 64
# short, 200 rows narrow, 2047 rows wide) and with a K split
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2300, 4104, 64), (200, 264, 320), (2047, 11008, 320), (100, 264, 4096)])
@pytest.mark.parametrize("offset", [1, 4])
def test_dense_matmul_output_alignment(vqx, M, N, K, offset):
    print(f"dense output offset {offset} M={M} N={N} K={K}", flush=True)
    L = vqx._lib
    g = torch.Generator(device="cuda").manual_seed(offset)
    a = torch.randint(-2, 3, (M, K), generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randint(-2, 3, (N, K), generator=g, device="cuda").to(torch.bfloat16)
    flat = torch.full((M * N + offset + 8,), 9.0, dtype=torch.bfloat16, device="cuda")
    out = flat[offset:offset + M * N]
    n = ctypes.c_int64(0)
    L.call("vqx_dense_matmul_workspace_size", 1, M, N, K, ctypes.byref(n))
    w = torch.empty(max(n.value, 1), dtype=torch.uint8, device="cuda")
    L.call("vqx_dense_matmul", L.ptr(a), K, 0, L.ptr(b), K, 0, None, L.ptr(out), 1, M, N, K, L.ptr(w), n.value,
           L.stream_of(a))
    assert torch.equal(out.view(M, N), (a.float() @ b.float().t()).to(torch.bfloat16))  # whole numbers: one rounding
    assert bool((flat[:offset] == 9).all()) and bool((flat[offset + M * N:] == 9).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [16, 17, 40])
@pytest.mark.parametrize("fits", [True, False])
def test_nf4_linear_around_the_packed_limit(vqx, monkeypatch, M, fits):
    """Both sides of the row limit between the packed 4-bit weight and its
    cached decode, and the packed way when the decode has no room."""
    print(f"nf4 linear M={M} fits={fits}", flush=True)
    qops = vqx.ops.quantized
    N, K = 384, 320
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(2, M // 2, K, generator=g, device="cuda").to(torch.bfloat16) if M % 2 == 0 else \
        torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    idx = torch.randint(0, 16, (N, K), generator=g, device="cuda").to(torch.bfloat16)
    code = torch.randn(16, generator=g, device="cuda").to(torch.bfloat16)
    scale = (torch.rand(N, K // 64, generator=g, device="cuda") + 0.1).to(torch.bfloat16)
    bias = torch.randn(N, generator=g, device="cuda").to(torch.bfloat16)
    if not fits:
        monkeypatch.setattr(qops, "_DECODED_SHARE", 1 << 60)
    before = dict(qops._DECODED_BYTES)
    y = Q.linear_mx(x, idx, bias, weight_scale=scale, weight_code=code, block_size=64)
    grown = sum(qops._DECODED_BYTES.values()) - sum(before.values())
    assert grown == (2 * N * K if M > 16 and fits else 0)
    w = (code[idx.long()].float() * scale.repeat_interleave(64, 1).float()).to(torch.bfloat16).double()
    want = x.double().reshape(-1, K) @ w.t() + bias.double()
    mag = x.double().abs().reshape(-1, K) @ w.abs().t() + bias.double().abs()
    assert y.shape == (*x.shape[:-1], N)
    close(y.reshape(-1, N), want, mag, K)
    del idx, y
    assert sum(qops._DECODED_BYTES.values()) == sum(before.values())  # given back with the weight
