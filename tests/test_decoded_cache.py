"""The cache of decoded weights: entries dropped while it is being changed, and
entries used on another stream than the one they were made on."""

import threading

import pytest
import torch

Q = torch.ops.quantized_ops


class OnDrop:
    """A decode whose size is asked for while the cache changes: drops another
    entry then, as the finalizer of a weight collected at that point does."""

    device = torch.device("cpu", 7)

    def __init__(self, q, other):
        self.q, self.other = q, other

    def numel(self):
        self.q._release_decoded(self.other)
        return 10

    def element_size(self):
        return 2


def test_entry_dropped_inside_an_update(vqx):
    q = vqx.ops.quantized

    class Plain(OnDrop):
        def numel(self):
            return 3

    def work():
        q._store_decoded("b", ((), (), Plain(q, None), 0))
        q._store_decoded("a", ((), (), OnDrop(q, "b"), 0))

    t = threading.Thread(target=work, daemon=True)
    t.start()
    t.join(20)
    assert not t.is_alive(), "an update waits for itself"
    assert "b" not in q._DECODED and "a" in q._DECODED
    assert q._DECODED_BYTES[7] == 20
    q._release_decoded("a")
    assert q._DECODED_BYTES.pop(7) == 0


@pytest.mark.gpu
def test_decode_outlives_its_weight_on_another_stream(vqx):
    """A product queued on a side stream reads the decode made on the main
    one; the weight goes and its decode's size is allocated again and filled
    before the side stream gets there."""
    print("decoded weight on a side stream", flush=True)
    M, N, K = 64, 1024, 1024
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randint(-3, 4, (M, K), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randint(-3, 4, (N, K), generator=g, device="cuda").to(torch.bfloat16)
    sw = torch.ones(N, K // 32, dtype=torch.bfloat16, device="cuda")
    want = Q.linear_mx(x, w, weight_scale=sw, block_size=32)  # decodes and caches
    ref = x.double() @ w.double().t()
    assert torch.equal(want.double(), ref.to(torch.bfloat16).double())  # small whole numbers: one rounding
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
        y = Q.linear_mx(x, w, weight_scale=sw, block_size=32)
    del w, sw
    again = [torch.full((N, K), 9.0, dtype=torch.bfloat16, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    assert torch.equal(y, want)
    del again
