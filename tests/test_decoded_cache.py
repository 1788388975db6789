"""The cache of decoded weights: entries dropped while it is being changed,
entries used on another stream than the one they were made on, and what a graph
captured after a warm-up reads once its weight has changed."""

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


class HostStream:
    """Counts what the cache asks of a stream."""

    waits, events = 0, 0

    def synchronize(self):
        self.waits += 1

    def wait_event(self, event):
        assert event.recorded is not None and event.recorded is not self
        self.events += 1


class HostEvent:
    recorded = None

    def record(self, stream):
        self.recorded = stream


@pytest.fixture
def host_cache(vqx, monkeypatch):
    """The cache function on CPU tensors, with the current stream and whether
    it is being captured in the returned dict."""
    q = vqx.ops.quantized
    state = {"q": q, "capturing": False, "stream": HostStream()}
    monkeypatch.setattr(q._lib, "stream_of", lambda t: id(state["stream"]))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: state["stream"])
    monkeypatch.setattr(torch.cuda, "Event", HostEvent)
    monkeypatch.setattr(torch._C, "_cuda_isCurrentStreamCapturing", lambda: state["capturing"])
    monkeypatch.setattr(q, "_decoded_fits", lambda nbytes, device: True)
    return state


def cached(state, w):
    """The cached decode of w, here a copy."""
    return state["q"]._cached_decode(("test",), (w, None, None), 4, w.clone)


def test_capture_takes_no_cached_decode(host_cache):
    w = torch.ones(4)
    warm = cached(host_cache, w)
    assert cached(host_cache, w) is warm
    host_cache["capturing"] = True
    inside = cached(host_cache, w)
    assert inside is not warm and cached(host_cache, w) is not inside
    host_cache["capturing"] = False
    assert cached(host_cache, w) is warm  # the entry stays for eager calls


def test_single_use_of_a_wide_weight(host_cache):
    """Where the product that decodes inside is the faster one for a single
    use, the second call with the same operands makes the decode, a capture
    only where that holds for graphs."""
    q, w = host_cache["q"], torch.ones(4)

    def call(inside=True):
        return q._cached_decode(("test",), (w, None, None), 16, w.clone, inside, True)

    assert call() is None
    host_cache["capturing"] = True
    assert call() is None and torch.equal(call(False), w)
    host_cache["capturing"] = False
    kept = call()
    assert torch.equal(kept, w) and call() is kept
    w.add_(1)
    assert call() is None and torch.equal(call(), w)
    key, before = (id(w), ("test",)), q._DECODED_BYTES[None]
    del w, call
    assert key not in q._DECODED and q._DECODED_BYTES[None] == before - 16


@pytest.mark.parametrize("M,N,coded,pays", [
    (128, 12288, False, True), (128, 12289, False, False), (129, 9217, False, False), (256, 9216, False, True),
    (257, 16384, False, True), (512, 16385, False, False), (513, 1 << 20, False, True), (1, 24576, True, True),
    (256, 24577, True, False), (257, 1 << 20, True, True)])
def test_decode_pays_once(vqx, M, N, coded, pays):
    assert vqx.ops.quantized._decode_pays_once(M, N, coded) == pays


def test_no_entry_where_it_does_not_fit(host_cache, monkeypatch):
    q, w = host_cache["q"], torch.ones(4)
    monkeypatch.setattr(q, "_decoded_fits", lambda nbytes, device: False)
    monkeypatch.setattr(q, "_mx_decoded", lambda t, *rest: t.clone())
    assert q._decoded_weight(w, None, None, 32, -1) is None
    assert (id(w), ("dense", 32, -1)) not in q._DECODED


@pytest.mark.parametrize("capturing", [False, True])
def test_no_memory_for_a_decode(host_cache, capturing):
    """The call goes the way that needs none instead of failing."""
    q, w = host_cache["q"], torch.ones(4)
    host_cache["capturing"] = capturing

    def make():
        raise torch.cuda.OutOfMemoryError("out of memory")

    assert q._cached_decode(("test",), (w, None, None), 16, make) is None
    assert (id(w), ("test",)) not in q._DECODED
    host_cache["capturing"] = False
    assert torch.equal(cached(host_cache, w), w)


def test_a_new_decode_waits_on_the_device_only(host_cache, monkeypatch):
    """The host waits for no decode; a call on another stream queues a wait for
    it there, and the stream is recorded on the decode."""
    recorded = []
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda t, stream: recorded.append(stream))
    w, main = torch.ones(4), host_cache["stream"]
    first = cached(host_cache, w)
    assert cached(host_cache, w) is first and (main.waits, main.events) == (0, 0) and not recorded
    side = host_cache["stream"] = HostStream()
    assert cached(host_cache, w) is first
    assert (side.waits, side.events) == (0, 1) and recorded == [side]


def test_writes_that_are_seen(host_cache):
    """Through the tensor itself, and another storage put under it.  (A write
    through .data moves no version counter: such a weight is not rebuilt.)"""
    w = torch.nn.Parameter(torch.ones(4))
    first = cached(host_cache, w)
    with torch.no_grad():
        w.fill_(2.0)
    second = cached(host_cache, w)
    assert second is not first and torch.equal(second, w)
    w.data = torch.full((4,), 3.0)
    assert torch.equal(cached(host_cache, w), w)


@pytest.mark.parametrize("which", [0, 1, 2])
def test_inference_tensors_are_not_cached(host_cache, which):
    """A write in place to a tensor without a version counter is seen, whether
    it is the weight, its code or its scale."""
    q = host_cache["q"]
    deps = [torch.ones(4) for _ in range(3)]
    with torch.inference_mode():
        deps[which] = torch.ones(4)
        for value in (1.0, 2.0):
            deps[which].fill_(value)
            got = q._cached_decode(("test",), tuple(deps), 4, lambda: deps[which].clone())
            assert bool((got == value).all())
    assert (id(deps[0]), ("test",)) not in q._DECODED


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["kc", "ck"])
@pytest.mark.parametrize("rows", [64, 640])
def test_no_entry_past_the_share(vqx, monkeypatch, layout, rows):
    """A weight without a packed form, on either side of the 512 rows up to
    which the product decodes it inside."""
    print(f"full cache, {layout}, {rows} rows", flush=True)
    q = vqx.ops.quantized
    monkeypatch.setattr(q, "_DECODED_SHARE", 1 << 60)
    g = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randint(-3, 4, (rows, 512), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randint(-3, 4, (384, 512), generator=g, device="cuda").to(torch.bfloat16)
    sw = torch.ones(384, 16, dtype=torch.bfloat16, device="cuda")
    want = (x.double() @ w.double().t()).to(torch.bfloat16)
    if layout == "ck":
        w, sw = w.t().contiguous(), sw.t().contiguous()
    before = dict(q._DECODED_BYTES)
    for _ in range(3):
        assert torch.equal(Q.linear_mx(x, w, weight_scale=sw, block_size=32, weight_layout=layout), want)
    assert q._DECODED_BYTES == before


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [64, 640])
def test_inference_weight_written_in_place(vqx, rows):
    print(f"inference-mode weight written in place, {rows} rows", flush=True)
    g = torch.Generator(device="cuda").manual_seed(6)
    with torch.inference_mode():
        x = torch.randint(-3, 4, (rows, 512), generator=g, device="cuda").to(torch.bfloat16)
        w = torch.randint(-3, 4, (384, 512), generator=g, device="cuda").to(torch.bfloat16)
        sw = torch.ones(384, 16, dtype=torch.bfloat16, device="cuda")
        for _ in range(3):
            y = Q.linear_mx(x, w, weight_scale=sw, block_size=32)
            assert torch.equal(y, (x.double() @ w.double().t()).to(torch.bfloat16))
            w.add_(1)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["int8 64 rows", "int8 640 rows", "nf4 40 rows", "outliers", "int8 wide",
                                  "int8 transposed"])
def test_captured_linear_reads_the_weight_as_it_is(vqx, kind):
    """A graph captured after a warm call, its weight written in place, an
    eager call on the new weight and the freed memory filled with something
    else: every replay is the product with the weight of that moment."""
    print(f"captured linear, {kind}", flush=True)
    M, N, K, bs = (640 if "640" in kind else 40 if "40" in kind else 64), 384, 512, 64
    if kind == "int8 wide":  # decoded inside the product on the first call and in the graph
        N = 12416
    g = torch.Generator(device="cuda").manual_seed(5)
    nf4 = kind.startswith("nf4")
    x = torch.randint(-3, 4, (M, K), generator=g, device="cuda").to(torch.bfloat16)
    sw = torch.ones(N, K // bs, dtype=torch.bfloat16, device="cuda")
    kw = dict(weight_scale=sw, block_size=bs)
    if nf4:
        kw["weight_code"] = torch.arange(-8, 8, device="cuda").to(torch.bfloat16)
    if kind == "outliers":
        # one entry of value 5 per row, at column r
        kw["A_data"] = torch.full((M,), 5.0, dtype=torch.bfloat16, device="cuda")
        kw["A_indices"] = torch.arange(M, dtype=torch.int32, device="cuda")
        kw["A_indptr"] = torch.arange(M + 1, dtype=torch.int32, device="cuda")

    def weight():
        return torch.randint(0 if nf4 else -3, 16 if nf4 else 4, (N, K), generator=g, device="cuda").to(torch.bfloat16)

    def product(w):  # small whole numbers: the product rounds once, the sparse half and its sum once each
        wd = (kw["weight_code"][w.long()] if nf4 else w).double()
        y = (x.double() @ wd.t()).to(torch.bfloat16)
        return y + (5 * wd.t()[:M]).to(torch.bfloat16) if kind == "outliers" else y

    w = weight().t().contiguous().t() if kind == "int8 transposed" else weight()
    for _ in range(3):
        assert torch.equal(Q.linear_mx(x, w, **kw), product(w))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = Q.linear_mx(x, w, **kw)
    for step in range(3):
        w.copy_(weight())
        graph.replay()
        assert torch.equal(y, product(w)), f"step {step}, before an eager call"
        assert torch.equal(Q.linear_mx(x, w, **kw), product(w))
        fill = [torch.full((N, K), 9.0, dtype=torch.bfloat16, device="cuda") for _ in range(8)]
        graph.replay()
        assert torch.equal(y, product(w)), f"step {step}, after an eager call"
        del fill


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


@pytest.mark.gpu
def test_side_stream_waits_for_a_decode_under_way(vqx):
    """The decode is still queued behind other work on the main stream when a
    product on a side stream takes it from the cache."""
    print("side stream behind a decode under way", flush=True)
    M, N, K = 64, 1024, 1024
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randint(-3, 4, (M, K), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randint(-3, 4, (N, K), generator=g, device="cuda").to(torch.bfloat16)
    sw = torch.ones(N, K // 32, dtype=torch.bfloat16, device="cuda")
    want = (x.double() @ w.double().t()).to(torch.bfloat16)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda._sleep(20_000_000)
    first = Q.linear_mx(x, w, weight_scale=sw, block_size=32)
    with torch.cuda.stream(side):
        y = Q.linear_mx(x, w, weight_scale=sw, block_size=32)
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(y, want)
