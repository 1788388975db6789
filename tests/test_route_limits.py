"""Operands past the sizes a kernel addresses go the way that takes them: the
entry points that calls on FakeTensors of those sizes would launch."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


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
