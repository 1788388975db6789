"""Operands past the sizes a kernel addresses go the way that takes them: the
entry points that calls on FakeTensors of those sizes would launch."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


pytestmark = pytest.mark.filterwarnings("ignore:Accessing the data pointer")


@pytest.fixture
def launches(vqx, monkeypatch):
    """The entry points called, on fake cuda tensors, by name."""
    q = vqx.ops.quantized
    names = []
    monkeypatch.setattr(q._lib, "call", lambda name, *args: names.append(name))
    monkeypatch.setattr(q._lib, "ptr", lambda t: None)
    monkeypatch.setattr(q._lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(q, "_mx_operand", lambda *args: q._lib.VqxMxOperand())
    monkeypatch.setattr(q, "_dense_workspace_bytes", lambda *args: 0)
    monkeypatch.setattr(q, "_aligned16", lambda t: t.contiguous())
    with FakeTensorMode():
        yield q, names


def fake(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="cuda")


# 2^31 values are 4 GiB: past the layout pass that turns the operand
@pytest.mark.parametrize("N,K,scaled,route", [(65536, 32768, True, "vqx_csr_decode_weight"),
                                              (65536, 32768, False, "vqx_csr_decode_weight"),
                                              (65535, 32768, True, "vqx_mx_operand_rows"),
                                              (40000000, 64, True, "vqx_csr_decode_weight"),
                                              (384, 512, False, "vqx_mx_operand_rows")])
def test_spmm_layout(launches, N, K, scaled, route):
    q, names = launches
    rows = 4
    q._spmm(fake(16), fake(16, dtype=torch.int32), fake(rows + 1, dtype=torch.int32), fake(N, K),
            fake(N, K // 64) if scaled else None, None, 64)
    assert names == [route, "vqx_spmm_csr"]


# P V of an odd length: P inside the product, V turned; one item of P is 4 GiB
# from 46341 positions on, and past it the operands decode for the library
# product, as do more items than a launch holds
@pytest.mark.parametrize("shape,route", [
    ((32, 1333, 1333, 128), ["vqx_mx_operand_rows", "vqx_mx_matmul_any"]),
    ((1, 46337, 46337, 128), ["vqx_mx_operand_rows", "vqx_mx_matmul_any"]),
    ((1, 50001, 50001, 128), None),
    ((1, 600, 9000001, 256), None),             # V's item
    ((1 << 22, 600, 9, 4), None),               # the product's launch
    ((32, 1333, 128, 1333), ["vqx_mx_operand_rows", "vqx_mx_operand_rows", "vqx_dense_matmul"]),
    ((1, 16777217, 128, 519), None),            # the left item
    ((1 << 23, 5, 9, 5), None),                 # the dense product's launch
    ((1 << 22, 5, 9, 5), ["vqx_mx_operand_rows", "vqx_mx_operand_rows", "vqx_dense_matmul"])])
def test_batched_products(launches, shape, route):
    q, names = launches
    B, M, K, N = shape
    out = q._mx_product(fake(B, M, K), None, fake(B, M, -(-K // 64)), fake(B, K, N), None, fake(B, -(-K // 64), N), 64,
                        True, None)
    assert (None if out is None else names) == route
    assert route is not None or not names


@pytest.mark.parametrize("B,N,takes", [(32, 1999, True), (1 << 24, 64, False), ((1 << 24) - 1, 64, True),
                                       (1 << 23, 65, False)])
def test_few_rows(launches, B, N, takes):
    q, names = launches
    out = q._few_rows_product(fake(B, 1, 8), None, None, fake(B, 8, N), None, fake(B, 1, N), 8)
    assert (out is not None) == takes and names == ["vqx_mx_few_rows"] * takes


@pytest.mark.parametrize("turned", [False, True])
@pytest.mark.parametrize("batch,R,C,ld,takes", [(1, 65536, 32768, 32768, False), (1, 65535, 32768, 32768, True),
                                                (32768, 65536, 8, 8, None), (1 << 24, 8, 8, 8, None)])
def test_rows_takes(vqx, batch, R, C, ld, takes, turned):
    """takes None: the plain pass's row count, the turned one's launch."""
    got = vqx.ops.quantized._rows_takes(batch, R, C, ld, turned)
    assert got == (takes if takes is not None else not turned and batch * R < 1 << 31)


@pytest.mark.parametrize("batch,M,N,K,coded,eager,graph", [
    (32, 1, 4096, 128, True, True, True), (32, 4, 1999, 128, True, True, True), (32, 4, 2048, 77, True, True, True),
    (32, 2, 2048, 128, True, True, False), (32, 3, 2048, 128, True, False, False),
    (32, 4, 2048, 128, False, True, False), (32, 4, 4096, 128, False, False, False),
    (32, 4, 128, 2048, False, True, True), (1, 2, 11008, 4096, False, False, False),
    (1, 4, 11008, 4096, True, True, True), (256, 2, 128, 1024, False, False, False),
    (96, 2, 128, 1024, False, True, True), (256, 4, 512, 512, False, True, True)])
def test_few_rows_faster(launches, monkeypatch, batch, M, N, K, coded, eager, graph):
    q, names = launches
    for capturing, few in ((False, eager), (True, graph)):
        monkeypatch.setattr(q, "_capturing", lambda device: capturing)
        names.clear()
        code = fake(16) if coded else None
        q.matmul_mx(fake(batch, M, K), fake(batch, K, N), weight_scale=fake(batch, -(-K // 8), N), weight_code=code,
                    block_size=8)
        assert names == (["vqx_mx_few_rows"] if few else ["vqx_mx_matmul"])


# a plain right operand: read in place by up to 512 rows of an item, else turned
@pytest.mark.parametrize("M,N,route", [
    (100, 4096, ["vqx_mx_operand_decode", "vqx_mx_matmul"]), (512, 2048, ["vqx_mx_operand_decode", "vqx_mx_matmul"]),
    (513, 2048, ["vqx_mx_operand_rows", "vqx_mx_operand_rows", "vqx_dense_matmul"]),
    (100, 4095, ["vqx_mx_operand_rows", "vqx_mx_operand_rows", "vqx_dense_matmul"])])
def test_plain_right_operand(launches, M, N, route):
    q, names = launches
    q.matmul_mx(fake(4, M, 1024), fake(4, 1024, N), input_scale=fake(4, M, 16), block_size=64)
    assert names == route


# decode passes ahead of the dense product or of the tiles, either side of each
# line: short K by tiles, long K, a plain left and a plain right operand
@pytest.mark.parametrize("B,M,K,N,coded,dense", [
    (12, 768, 64, 768, "ab", False), (16, 2048, 64, 2048, "ab", True), (12, 640, 128, 640, "ab", False),
    (12, 1024, 128, 1024, "ab", True), (1, 520, 256, 520, "ab", True), (1, 520, 248, 520, "ab", False),
    (31, 1024, 128, 1024, "b", False), (32, 1024, 128, 1024, "b", True), (64, 2048, 64, 2048, "b", False),
    (1, 520, 256, 520, "b", True), (32, 2048, 2048, 128, "b", False), (12, 1024, 1024, 64, "b", True),
    (32, 1024, 128, 1024, "a", False), (16, 2048, 128, 2048, "a", True), (1, 1024, 1024, 1024, "a", True),
    (8, 1024, 512, 1024, "a", False), (1, 1024, 512, 1024, "a", True), (12, 768, 64, 767, "ab", True)])
def test_dense_or_tiles(launches, B, M, K, N, coded, dense):
    q, names = launches
    sa = fake(B, M, -(-K // 8)) if "a" in coded else None
    sb = fake(B, -(-K // 8), N) if "b" in coded else None
    q.matmul_mx(fake(B, M, K), fake(B, K, N), input_scale=sa, weight_scale=sb, block_size=8)
    assert names[-1] == ("vqx_dense_matmul" if dense else "vqx_mx_matmul")


# linears that decode both operands in one launch (the weight ahead above 512
# rows): a short K, at most 512 outputs and one round of tiles, a coded activation
@pytest.mark.parametrize("M,N,K,coded,inside", [
    (512, 512, 1024, False, True), (512, 512, 1088, False, False), (513, 512, 960, False, True),
    (8192, 512, 960, False, True), (8193, 512, 960, False, False), (20, 520, 960, False, False),
    (20, 64, 512, True, True), (20, 64, 576, True, False), (513, 64, 576, True, True)])
def test_small_linear(launches, monkeypatch, M, N, K, coded, inside):
    q, names = launches
    monkeypatch.setattr(q, "_cached_decode", lambda form, deps, *rest: deps[0])
    q.linear_mx(fake(M, K), fake(N, K), None, input_scale=fake(M, K // 8), weight_scale=fake(N, K // 8),
                weight_code=fake(40) if coded else None, block_size=8)
    assert names == (["vqx_mx_matmul"] if inside else ["vqx_mx_operand_rows", "vqx_dense_matmul"])
