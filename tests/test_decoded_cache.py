"""The cache of decoded weights: entries dropped while it is being changed."""

import threading

import torch


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
        q._store_decoded("b", ((), (), Plain(q, None)))
        q._store_decoded("a", ((), (), OnDrop(q, "b")))

    t = threading.Thread(target=work, daemon=True)
    t.start()
    t.join(20)
    assert not t.is_alive(), "an update waits for itself"
    assert "b" not in q._DECODED and "a" in q._DECODED
    assert q._DECODED_BYTES[7] == 20
    q._release_decoded("a")
    assert q._DECODED_BYTES.pop(7) == 0
