"""The C++ host path (htr_amd._fast) and the ways around it: without it, with arguments it does not take, with failures behind it."""
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from htr_amd import _native
    _native.lib()
    return torch.device("cuda:0")


@pytest.fixture
def without_fast(monkeypatch):
    from htr_amd import _native
    monkeypatch.setattr(_native, "_fast", None)
    monkeypatch.setitem(sys.modules, "htr_amd._fast", None)          # importing it fails


def _linear(m, n, K, seed, dev):
    from htr_amd import wire
    return tuple(t.to(dev) for t in wire.synth_linear(m, n, K, seed))


def test_missing_extension_is_said_once(without_fast):
    from htr_amd import _native
    with pytest.warns(RuntimeWarning, match="_fast.so"):
        assert _native.fast() is None
    import warnings
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _native.fast() is None


def test_package_ships_every_built_file():
    import fnmatch
    import re
    from htr_amd import build
    patterns = re.findall(r'"([^"]+)"', re.search(r"^htr_amd = \[(.*)\]$", open(os.path.join(ROOT, "pyproject.toml")).read(), re.M).group(1))
    for built in (build.LIB, build.BINDING):
        path = os.path.relpath(built, os.path.join(ROOT, "htr_amd"))
        assert any(fnmatch.fnmatch(path, p) and os.path.dirname(path) == os.path.dirname(p) for p in patterns), path


def test_extension_of_another_build_is_not_used(monkeypatch):
    """Another C ABI or another torch than it was compiled with: launches are prepared in Python."""
    from htr_amd import _native
    module = _native.fast()
    assert module is not None
    abi = _native.lib().htr_abi_version()
    with pytest.raises(ImportError, match="ABI"):
        module.bind(abi + 1, torch.__version__, 0, 0, 0, 0)
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    monkeypatch.setattr(_native, "_fast", None)
    with pytest.warns(RuntimeWarning, match="torch 0.0.1|not 0.0.1"):
        assert _native.fast() is None


def test_a_newer_header_makes_the_extension_stale(monkeypatch, tmp_path):
    from htr_amd import build
    now = os.path.getmtime(build.BINDING)
    for name, age in (("HEADER", 100), ("LIB", 200)):
        f = tmp_path / name
        f.write_text("")
        os.utime(f, (now + age, now + age))
        monkeypatch.setattr(build, name, str(f))
    monkeypatch.setattr(build, "SOURCES", [])
    monkeypatch.setattr(build, "PARTS", [])
    monkeypatch.setattr(build, "BINDING_SOURCE", build.BINDING)
    assert build.is_stale()


@pytest.mark.parametrize("kind", ["tensor", "parameter", "buffer"])
def test_plain_activations_skip_the_dispatcher(monkeypatch, kind):
    """A parameter's rows are a plain tensor: the call does not go through the registered op, whose result would ask for a gradient
    that it cannot give."""
    from htr_amd import ops, wire
    w = wire.synth_linear(256, 384, 4, 51)
    x = torch.randn(2, 3, 384)
    x = {"tensor": lambda: x, "parameter": lambda: torch.nn.Parameter(x), "buffer": lambda: torch.nn.Buffer(x)}[kind]()
    monkeypatch.setattr(ops, "htr_linear_op", lambda *a: pytest.fail("through the dispatcher"))
    monkeypatch.setattr(ops, "_linear_impl", lambda x2, *a: torch.zeros(x2.shape[0], 256))
    assert ops.linear(x, *w).shape == (2, 3, 256)


def _expert_call(monkeypatch, report, waited=None):
    """ops._moe_silu with a stand-in for the device: `report(word address, ticket)` is what its routing kernel does."""
    import htr_amd._fast as real
    from htr_amd import _native, ops

    class Fast:
        wait_word = staticmethod(lambda word, ticket, seconds: real.wait_word(word, ticket, min(seconds, 0.01)))

        @staticmethod
        def moe(x, ids, weights, gate_up, down, word, ticket, stream):
            report(word, ticket)
            return "queued"

    class Stream:
        synchronize = staticmethod(lambda: waited.append(1) if waited is not None else None)

    monkeypatch.setattr(_native, "fast", lambda: Fast)
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 0)
    monkeypatch.setattr(ops, "_ticket_page", lambda: torch.zeros(ops._TICKET_WORDS, dtype=torch.int32))
    monkeypatch.setattr(ops, "_FREE_WORDS", {})
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream)
    return ops._moe_silu(torch.zeros(1, 128), None, None, [1, 2, 3], [1, 2, 3])


def _store(word, value):
    import ctypes
    ctypes.c_uint32.from_address(word).value = value


def test_report_of_the_routing_kernel(monkeypatch):
    assert _expert_call(monkeypatch, lambda word, ticket: _store(word, ticket << 1)) == "queued"
    with pytest.raises(IndexError, match="0 .. 2"):
        _expert_call(monkeypatch, lambda word, ticket: _store(word, ticket << 1 | 1))


def test_report_of_another_call_is_not_taken_for_this_one(monkeypatch):
    """After the wait ran out and the stream was drained, the word has to hold this call's ticket: another one's is an error."""
    waited = []
    for low in (0, 1):
        with pytest.raises(RuntimeError, match="not reported"):
            _expert_call(monkeypatch, lambda word, ticket: _store(word, (ticket + 256) << 1 | low), waited)
    assert len(waited) == 2


def test_capture_is_that_of_the_stream_the_layer_goes_to(monkeypatch):
    """Not the current device's: a layer on another device than the current one is captured, or not, on its own stream."""
    from htr_amd import _native
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    asked, given = [], []

    class Lib:
        htr_stream_capture_id = staticmethod(lambda stream: asked.append(stream) or 7)

    monkeypatch.setattr(_native, "lib", lambda real=_native.lib(): Lib)
    assert _expert_call(monkeypatch, lambda word, ticket: given.append((word, ticket))) == "queued"
    assert asked == [0] and given == [(0, 0)]


def test_words_of_calls_in_flight_differ(monkeypatch):
    from htr_amd import ops
    monkeypatch.setattr(ops, "_ticket_page", lambda: torch.zeros(ops._TICKET_WORDS, dtype=torch.int32))
    monkeypatch.setattr(ops, "_FREE_WORDS", {})
    words = [ops._take_word(0) for _ in range(3 * ops._TICKET_WORDS + 5)]
    assert len(set(words)) == len(words)
    ops._FREE_WORDS[0].append(words[7])
    assert ops._take_word(0) == words[7]          # given back, used again: no new page per call


@pytest.mark.gpu
def test_calls_without_the_extension(dev, without_fast):
    """Every call of a stream, not only the first one, which has no workspace yet."""
    from htr_amd import ops
    print("linear and experts without the extension", flush=True)
    w, x = _linear(256, 384, 4, 51, dev), torch.randn(3, 384, device=dev).bfloat16()
    with pytest.warns(RuntimeWarning):
        first = [ops.linear(x, *w) for _ in range(3)]
    gate_up, down = [_linear(256, 128, 4, 60 + e, dev) for e in range(2)], [_linear(128, 128, 4, 70 + e, dev) for e in range(2)]
    xe, ids, we = torch.randn(5, 128, device=dev).bfloat16(), torch.tensor([[0], [1], [1], [0], [1]], device=dev), torch.rand(5, 1, device=dev)
    layer = ops.moe_experts(xe, ids, we, gate_up, down)
    from htr_amd import _native
    _native._fast = None
    sys.modules.pop("htr_amd._fast")
    assert _native.fast() is not None
    assert all(torch.equal(y, ops.linear(x, *w)) for y in first)
    whole = ops.moe_experts(xe, ids, we, gate_up, down)
    assert float((whole - layer).norm() / layer.norm()) <= 1e-3          # the same products, rounded alike


@pytest.mark.gpu
@pytest.mark.parametrize("M", [20, 200])
def test_two_threads_on_one_stream(dev, M):
    """Calls of two launches each (rotation, product) from two threads on one stream, which share its workspace: each one's
    launches stay together, in the C++ host path (20 rows, float32) and in the Python one (200 rows)."""
    import threading
    from htr_amd import ops
    print(f"two threads on one stream M={M}", flush=True)
    w = _linear(4096, 4096, 4, 52, dev)
    xs = [torch.randn(M, 4096, device=dev, generator=torch.Generator(device=dev).manual_seed(i)) for i in range(2)]
    want = [ops.linear(x, *w) for x in xs]
    torch.cuda.synchronize()
    wrong = [0, 0]

    def work(i):
        ys = [ops.linear(xs[i], *w) for _ in range(100)]
        torch.cuda.synchronize()
        wrong[i] = sum(not torch.equal(y, want[i]) for y in ys)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == [0, 0]


@pytest.mark.gpu
def test_interpreter_lock_is_free_during_launches(dev):
    """In the place of the library's launches, the interpreter's own PyGILState_Check: it returns 0, which is success, only while
    this thread does not hold the lock.  No kernel runs."""
    import ctypes
    from htr_amd import _native, ops
    print("interpreter lock", flush=True)
    module, L = _native.fast(), _native.lib()
    at = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value
    check = at(ctypes.pythonapi.PyGILState_Check)
    w, x = _linear(256, 384, 4, 51, dev), torch.randn(3, 384, device=dev).bfloat16()
    gate_up, down = [_linear(256, 128, 4, 60, dev)], [list(_linear(128, 128, 4, 70, dev))]
    xe, ids, we = torch.randn(5, 128, device=dev).bfloat16(), torch.zeros(5, 1, dtype=torch.int64, device=dev), torch.rand(5, 1, device=dev)
    stream = ops._raw_stream(0)
    module.bind(L.htr_abi_version(), str(torch.__version__), check, at(L.htr_stream_capture_id), at(L.htr_moe_scratch_bytes), check)
    try:
        assert module.linear(x, *w, None, 0, 0, 0, stream) is not None
        assert module.moe(xe, ids, we, gate_up, down, 0, 0, stream) is not None
    finally:
        _native._fast = None
        _native.fast()


@pytest.mark.gpu
def test_a_refused_launch_of_the_layer_is_an_error(dev):
    """A status of the runtime from the library's call (here from a function in its place) is raised, and the layer is not run again."""
    import ctypes
    from htr_amd import _native, ops
    print("refused launch", flush=True)
    module, L = _native.fast(), _native.lib()
    at = lambda fn: ctypes.cast(fn, ctypes.c_void_p).value
    res, args = _native.SIGNATURES["htr_moe_experts"]
    refuse = ctypes.CFUNCTYPE(res, *args)(lambda *a: 8)
    gate_up, down = [_linear(256, 128, 4, 60, dev)], [_linear(128, 128, 4, 70, dev)]
    xe, ids, we = torch.randn(5, 128, device=dev).bfloat16(), torch.zeros(5, 1, dtype=torch.int64, device=dev), torch.rand(5, 1, device=dev)
    module.bind(L.htr_abi_version(), str(torch.__version__), at(L.htr_linear), at(L.htr_stream_capture_id), at(L.htr_moe_scratch_bytes), at(refuse))
    try:
        with pytest.raises(RuntimeError, match="status 8"):
            ops.moe_experts(xe, ids, we, gate_up, down)
    finally:
        _native._fast = None
        _native.fast()


@pytest.mark.gpu
def test_what_the_extension_leaves_to_the_general_path(dev):
    """linear(): None, and nothing launched, for every form that is not the plain decode call; the general path then runs it or says
    what is wrong."""
    from htr_amd import _native, ops
    print("ways out of the extension's linear", flush=True)
    fast = _native.fast()
    m, n = 256, 384
    w, x = _linear(m, n, 4, 51, dev), torch.randn(3, n, device=dev).bfloat16()
    want, bias = ops.linear(x, *w), torch.randn(m, device=dev).bfloat16()
    stream = ops._raw_stream(0)
    ws = ops._WORKSPACES[(0, stream)]
    call = lambda x=x, w=w, bias=None, ptr=ws.ptr, size=ws.size, failed=0: fast.linear(x, *w, bias, ptr, size, failed, stream)
    assert torch.equal(call(), want) and call(bias=bias) is not None
    upto = lambda rows, x=x: fast.linear(x, *w, None, ws.ptr, ws.size, 0, stream, rows)      # as ops calls it
    assert torch.equal(upto(2048), want) and torch.equal(upto(3), want) and upto(2) is None
    assert upto(128, x.repeat(43, 1)) is None and torch.equal(upto(2048, x.repeat(43, 1)), ops.linear(x.repeat(43, 1), *w))      # 129 rows
    assert upto(4096, x.repeat(683, 1)) is None                                   # 2049 rows: more than one launch holds
    flag = torch.ones(1, dtype=torch.int32)
    assert call(failed=flag.data_ptr()) is None                                   # an earlier launch gave up
    assert call(size=256) is None and call(ptr=ws.ptr + 8) is None                # too small, misaligned
    assert call(bias=bias.float()) is None and call(bias=bias[:-1]) is None and call(bias=bias.cpu()) is None
    wide = torch.randn(3, 2 * n, device=dev).bfloat16()
    assert call(x=wide[:, ::2]) is None and call(x=wide) is None and call(x=x.double()) is None and call(x=x.cpu()) is None
    assert call(x=x[:0]) is None and call(x=x.repeat(43, 1)) is None              # no rows, 129 rows
    for k, t in enumerate((w[0][:, :, ::2], w[1].float(), w[2][:-1], w[3].cpu())):
        assert call(w=tuple(t if i == k else o for i, o in enumerate(w))) is None
    assert torch.equal(ops.linear(x[1], *w), want[1]) and torch.equal(call(x=x[1]), want[1])      # one dimension
    assert torch.equal(ops.linear(x.reshape(1, 3, 1, n), *w), want.reshape(1, 3, 1, m))
    strided = torch.stack([x, x], dim=-1)[..., 0]
    assert not strided.is_contiguous() and torch.equal(ops.linear(strided, *w), want)
    for wrong in (bias.float(), bias[:-1]):
        with pytest.raises(RuntimeError, match="bias"):
            ops.linear(x, *w, wrong)


@pytest.mark.gpu
def test_what_the_extension_leaves_to_the_two_grouped_launches(dev):
    """moe(): None for more than 4096 experts, experts of several shapes or bits, other index types; the general path runs what it ran."""
    from htr_amd import _native, ops
    print("ways out of the extension's expert layer", flush=True)
    fast, stream = _native.fast(), ops._raw_stream(0)
    gate_up, down = [_linear(256, 128, 4, 60 + e, dev) for e in range(3)], [_linear(128, 128, 4, 70 + e, dev) for e in range(3)]
    x, w = torch.randn(6, 128, device=dev).bfloat16(), torch.rand(6, 1, device=dev)
    ids = torch.tensor([[0], [1], [1], [0], [1], [0]], device=dev)
    want = ops.moe_experts(x, ids, w, gate_up, down)
    near = lambda y: float((y - want).norm() / want.norm()) <= 1e-3               # the same products, rounded alike
    call = lambda ids=ids, w=w, gate_up=gate_up, down=down: fast.moe(x, ids, w, gate_up, down, 0, 0, stream)
    assert torch.equal(call(), want)
    many = [gate_up + [gate_up[2]] * 4094, down + [down[2]] * 4094]
    assert call(gate_up=many[0], down=many[1]) is None and near(ops.moe_experts(x, ids, w, *many))
    for other in (_linear(512, 128, 4, 80, dev), _linear(256, 128, 3, 80, dev), None):      # an expert that no token chose
        mixed = [gate_up[0], gate_up[1], other]
        assert call(gate_up=mixed) is None and near(ops.moe_experts(x, ids, w, mixed, down))
    with pytest.raises(RuntimeError, match="same m, n and K"):
        ops.moe_experts(x, ids.clamp(max=1) + 1, w, [gate_up[0], gate_up[1], _linear(256, 128, 3, 80, dev)], down)
    assert call(ids=ids.short()) is None and near(ops.moe_experts(x, ids.short(), w, gate_up, down))
    assert call(ids=ids[:5]) is None and call(w=w.long()) is None and call(down=down[:2]) is None


@pytest.mark.gpu
def test_expert_numbers_out_of_range_under_capture(dev):
    """Nothing can be raised from a replay: such a token is not a number, the others are as without it."""
    from htr_amd import ops
    print("bad expert numbers under capture", flush=True)
    gate_up, down = [_linear(256, 128, 4, 60 + e, dev) for e in range(3)], [_linear(128, 128, 4, 70 + e, dev) for e in range(3)]
    x, w = torch.randn(6, 128, device=dev).bfloat16(), torch.rand(6, 2, device=dev)
    good = torch.tensor([[0, 1], [1, 2], [2, 0], [0, 2], [1, 0], [2, 1]], device=dev)
    want = ops.moe_experts(x, good, w, gate_up, down)
    ids = good.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.moe_experts(x, ids, w, gate_up, down)
    for token, bad in ((1, 3), (4, -1), (1, 1 << 40)):
        ids.copy_(good)
        ids[token, 1] = bad
        graph.replay()
        torch.cuda.synchronize()
        others = [t for t in range(6) if t != token]
        assert bool(torch.isnan(y[token]).all()) and torch.equal(y[others], want[others])
        ids.copy_(good)
        graph.replay()
        assert torch.equal(y, want)
