"""k_linear_wide (65 rows and more) against the oracle: edges of its 32- and 256-row tiles, every K, splits, types and alignments; and who
takes a call beyond 128 rows: the rule, what was measured on both of its sides, and the two host paths that follow it."""
import ctypes

import numpy as np
import pytest
import torch

REL_TOL = 1e-3          # float32 results against decode-then-matmul in float64, max norm; activations are rounded to float16 (2e-4)
WIDE = 1 << 27


def _plan(L, m, n, K, M, nsplit):
    out = (ctypes.c_int * 6)()
    return list(out) if L.htr_linear_plan(m, n, K, M, nsplit, out) == 0 else None


@pytest.fixture(scope="module")
def L():
    from htr_amd import _native
    return _native.lib()


@pytest.mark.parametrize("m,n", [(128, 128), (1024, 4096), (6144, 4096), (14336, 4096), (4096, 14336), (152064, 4096)])
def test_wide_plan(L, m, n):
    nblk, rbs = n // 128, m // 128
    for M in (65, 128, 129, 256, 257, 512, 513, 2048):
        cb, wgs, tiles, S, prerot, lds = _plan(L, m, n, 4, M, WIDE)
        assert tiles == -(-M // 256) and prerot == 1 and lds <= 160 * 1024 and 1 <= S <= 8 and cb == -(-nblk // S)
        last = wgs // rbs - S * (tiles - 1)                                       # splits of the last tile
        assert wgs == rbs * (S * (tiles - 1) + last) and 1 <= last <= 8 and (wgs <= 256 or S == last == 1)
        need = L.htr_workspace_bytes(m, n, 4, M, WIDE)
        assert need >= 256 + M * n * 2 and (S == last == 1 or need >= 2 * rbs * last * (M - 256 * (tiles - 1)) * 512)
    assert _plan(L, m, n, 4, 128, 0)[3] == _plan(L, m, n, 4, 128, WIDE)[3]         # the policy from 65 rows to 128
    for want in (1, 2, 3, 8):
        p = _plan(L, m, n, 4, 300, WIDE | want)
        assert (p is None) == (want > nblk or -(-nblk // -(-nblk // want)) != want) and (p is None or p[3] == want)


def test_the_longest_rows_have_a_plan(L):
    """Up to what a launch takes in columns (65535 blocks) 65 to 128 rows have one, as every other row count."""
    for n in (8384512, 8388480):
        for M in (64, 65, 127, 128):
            assert _plan(L, 128, n, 4, M, 0) is not None and L.htr_workspace_bytes(128, n, 4, M, 0) >= 256 + M * n * 2
    assert _plan(L, 128, 8388480, 4, 129, WIDE) is None and L.htr_workspace_bytes(128, 8388480, 4, 129, WIDE) == 0      # 2^31 bytes of activations


def test_route(L):
    wide = lambda m, n, M, x=0, eager=0: L.htr_linear_route(m, n, 4, M, x, eager)
    assert wide(4096, 4096, 128) == 0 and wide(4096, 4096, 129) == WIDE and wide(14336, 4096, 512) == WIDE
    assert wide(14336, 4096, 2048) == -1 and wide(1024, 1024, 1024) == -1          # dequantize and multiply
    assert wide(512, 512, 512) == -1 and wide(512, 512, 512, eager=1) == WIDE      # where the host's time counts
    # float32 activations are rounded to float16 where a launch always took them, and nowhere else
    for eager in (0, 1):
        assert wide(4096, 4096, 384, 2, eager) == wide(4096, 14336, 512, 2, eager) == WIDE
        assert wide(4096, 4096, 385, 2, eager) == wide(4096, 14336, 513, 2, eager) == wide(2048, 2048, 129, 2, eager) == wide(14336, 4096, 2048, 2, eager) == -1
    # refused as htr_linear refuses it, and not to be mistaken for "dequantize"
    assert [wide(4096, 4096, 2049), wide(100, 128, 200), wide(128, 128, 200, 3), L.htr_linear_route(128, 128, 9, 200, 0, 1)] == [-5, -4, -6, -3]


# m, n, K, rows, type: us in a graph, wide kernel / dequantization and product, and eager, each with one of them at least 15 % ahead
_MEASURED = [(256, 4352, 3, 1089, 1, (36.7, 26.0), (36.0, 29.6)),
             (256, 7168, 3, 1112, 0, (40.4, 27.8), (41.0, 29.8)),
             (384, 512, 6, 579, 1, (20.3, 15.3), (19.8, 30.0)),
             (512, 384, 4, 810, 1, (19.0, 14.9), (18.6, 29.7)),
             (512, 768, 4, 753, 0, (21.3, 12.4), (20.9, 24.7)),
             (512, 8192, 2, 761, 0, (38.8, 30.9), (38.5, 32.3)),
             (512, 12672, 5, 208, 1, (37.4, 49.5), (36.4, 49.7)),
             (768, 384, 4, 1137, 0, (20.2, 11.6), (20.0, 25.0)),
             (768, 5248, 2, 1833, 1, (52.9, 42.8), (52.7, 43.6)),
             (768, 7168, 4, 934, 0, (41.5, 33.6), (41.9, 33.9)),
             (1152, 8960, 3, 347, 1, (34.5, 56.7), (34.4, 54.9)),
             (1408, 3456, 5, 746, 1, (34.5, 40.6), (33.9, 41.4)),
             (3200, 384, 8, 194, 0, (17.1, 12.4), (16.5, 25.8)),
             (4736, 2304, 6, 1437, 1, (55.7, 68.9), (55.9, 68.8)),
             (5760, 256, 5, 254, 0, (17.8, 13.2), (17.8, 25.4)),
             (7168, 1408, 2, 174, 0, (20.3, 29.6), (19.8, 30.5)),
             (9344, 256, 4, 269, 0, (18.0, 13.9), (17.6, 25.3)),
             (13568, 1152, 4, 177, 0, (22.6, 36.2), (21.8, 35.6)),
             (19328, 8832, 2, 733, 0, (266.3, 318.5), (264.6, 310.7)),
             (20352, 384, 2, 187, 1, (18.1, 42.3), (17.6, 42.1))]


@pytest.mark.parametrize("m,n,K,M,x,graph,eager", _MEASURED)
def test_route_follows_what_was_measured(L, m, n, K, M, x, graph, eager):
    for mode, (wide, dequantized) in enumerate((graph, eager)):
        route = L.htr_linear_route(m, n, K, M, x, mode)
        assert route == (-1 if dequantized < wide else WIDE), (mode, route)


def test_what_was_fused_is_never_dequantized(L):
    """Rows and matrices that ops.fused_rows_per_launch names are fused for every type, width and mode: a dequantized weight is rounded
    to bfloat16."""
    from htr_amd import ops
    shapes = [(m, n) for m in (1024, 4096, 6144, 10880, 14336, 17024, 17408, 17664, 28672) for n in (1408, 4096, 5120, 8192, 12544, 14336)]
    for m, n in shapes:
        limit = ops.fused_max_rows(m, n)
        for M in {129, 160, 192, 256, 257, 264, 282, 288, 311, 320, 384, 385, 512, 513}:
            fused = M <= limit
            assert (ops.fused_rows_per_launch(m, n, M) > 0) == fused
            routes = {L.htr_linear_route(m, n, K, M, x, eager) for K in (2, 4, 8) for x in (0, 1, 2) for eager in (0, 1)}
            assert not fused or routes == {WIDE}, (m, n, M, routes)
            assert routes <= {WIDE, -1} and (fused or L.htr_linear_route(m, n, 4, M, 2, 1) == -1)


@pytest.mark.parametrize("m,n,M", [(17408, 5120, 264), (16640, 11264, 311), (17024, 13696, 282), (6144, 4096, 333), (4096, 4096, 400), (2048, 2048, 700)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_general_path_asks_the_library(L, monkeypatch, m, n, M, dtype):
    """What the C++ host path does with these calls (htr_linear_route's answer) is what ops._linear_impl does, outside of a capture and in one."""
    from htr_amd import ops
    code = {torch.bfloat16: 0, torch.float32: 2}[dtype]
    x = torch.empty(1, dtype=dtype).expand(M, n)
    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        route = L.htr_linear_route(m, n, 4, M, code, 0 if capturing else 1)
        want = (0, 0) if route == -1 else (M, route)
        assert ops._route(x, None, m, n, 4, M, ops.fused_rows_per_launch(m, n, M)) == want


def test_a_shared_capture_buffer_that_is_too_small(L, monkeypatch):
    """It cannot grow while a capture is in progress: the call then goes where it went before the wide kernel was there."""
    from types import SimpleNamespace
    from htr_amd import ops
    x = lambda M, n: SimpleNamespace(dtype=torch.bfloat16, device=torch.device("cuda", 0), requires_grad=False)
    monkeypatch.setattr(ops, "_followed", lambda *a: False)
    monkeypatch.setattr(ops, "SHARE_CAPTURE_WORKSPACE", True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    for m, n, M in ((4096, 4096, 200), (14336, 4096, 484)):
        assert L.htr_linear_route(m, n, 4, M, 0, 0) == WIDE
        before = ops.fused_rows_per_launch(m, n, M)
        need = L.htr_workspace_bytes(m, n, 4, M, WIDE)
        for held, want in ((None, (before, 0)), (need - 1, (before, 0)), (need, (M, WIDE))):
            table = {} if held is None else {(0, "shared"): SimpleNamespace(buf=SimpleNamespace(numel=lambda: held))}
            monkeypatch.setattr(ops, "_WORKSPACES", table)
            assert ops._route(x(M, n), None, m, n, 4, M, before) == want


def _case(m, n, K, M, seed, dtype=torch.bfloat16):
    from htr_amd import wire
    qw, sc, su, sv = wire.synth_linear(m, n, K, seed)
    return (qw, sc, su, sv), torch.randn(M, n, generator=torch.Generator().manual_seed(seed)).to(dtype)


def _ref(oracle, w, x, bias=None):
    qw, sc, su, sv = w
    y = oracle.c_linear(x.float().numpy(), qw.numpy(), sc.numpy(), su.numpy(), sv.numpy())
    return y if bias is None else y + bias.double().numpy()


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle as o
    return o


# K, rows, m, n, splits of every tile (0: policy), activation type, elements by which x and y are off a 16-byte boundary
_CASES = [(4, 65, 256, 512, 0, "bf16", 0), (4, 96, 256, 128, 1, "bf16", 0), (4, 127, 256, 384, 3, "f16", 0), (4, 129, 256, 512, 2, "bf16", 0),
          (4, 255, 128, 1024, 8, "bf16", 0), (4, 256, 256, 256, 2, "bf16", 0), (4, 257, 256, 512, 4, "bf16", 0), (4, 333, 384, 1408, 0, "f16", 0),
          (4, 513, 128, 640, 5, "bf16", 0), (4, 40, 128, 256, 2, "bf16", 0), (4, 300, 128, 384, 0, "f32", 0), (4, 70, 128, 256, 1, "bf16", 1),
          (2, 97, 128, 384, 1, "bf16", 0), (3, 160, 128, 256, 2, "bf16", 0), (5, 97, 256, 512, 0, "f16", 0), (6, 200, 128, 384, 3, "bf16", 0),
          (7, 66, 128, 256, 1, "bf16", 0), (8, 288, 128, 512, 4, "bf16", 0), (4, 2048, 128, 128, 1, "bf16", 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("K,M,m,n,S,xt,off", _CASES)
def test_wide_kernel(dev, oracle, L, K, M, m, n, S, xt, off):
    from htr_amd import _native
    print(f"wide kernel K={K} M={M} {m}x{n} S={S} {xt} off={off}", flush=True)
    dtype = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[xt]
    w, x = _case(m, n, K, M, 500 + 7 * K + M, dtype)
    d = [t.to(dev) for t in w]
    room = torch.zeros(M * n + off, dtype=dtype, device=dev)
    xd = room[off:].view(M, n).copy_(x)
    bias = torch.randn(m, generator=torch.Generator().manual_seed(M))
    ns = WIDE | S
    need = L.htr_workspace_bytes(m, n, K, M, ns)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    ref = _ref(oracle, w, x, bias)
    code = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}
    # float32 results; then those of the activations' type, from an address that allows no wide stores
    for yt, o, tol in ((torch.float32, 0, REL_TOL), (dtype, off, REL_TOL + (0 if xt == "f32" else 2.0 ** -8 if xt == "bf16" else 2.0 ** -11))):
        outs = []
        b = bias.to(yt).to(dev)
        for _ in range(2):                                                        # again on the same workspace: the slots are clean
            y = torch.full((M * m + o,), float("nan"), dtype=yt, device=dev)
            _native.check(L.htr_linear(*[t.data_ptr() for t in d], xd.data_ptr(), b.data_ptr(), y[o:].data_ptr(), m, n, K, M, code[dtype], code[yt], ns,
                                       ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
            torch.cuda.synchronize()
            outs.append(y[o:].view(M, m))
        assert torch.equal(outs[0], outs[1])
        want = ref if yt == torch.float32 else ref - bias.double().numpy() + b.double().cpu().numpy()
        err = np.abs(outs[0].double().cpu().numpy() - want).max() / np.abs(want).max()
        assert err <= tol, (yt, err)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,M,splits", [(5504, 1408, 257, (4, 1)), (2816, 3712, 260, (8, 3)), (6144, 4096, 333, (3, 2)), (2176, 7040, 280, (8, 4)),
                                          (5504, 1280, 513, (2, 1)), (1920, 3712, 530, (6, 3))])
def test_last_tile_with_a_split_of_its_own(dev, oracle, L, m, n, M, splits):
    """Plans of the policy whose last tile is split otherwise than the full ones: its workgroups and its slots start behind theirs."""
    _, wgs, tiles, S, _, _ = _plan(L, m, n, 4, M, WIDE)
    assert (S, wgs // (m // 128) - S * (tiles - 1)) == splits
    test_wide_kernel(dev, oracle, L, 4, M, m, n, 0, "bf16", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,S", [(97, 4), (128, 8), (300, 2), (513, 5)])
def test_grid_beyond_the_compute_units(dev, oracle, L, M, S):
    """On a device of fewer compute units than the grid has workgroups (the planner's override) the last split finishes every row."""
    m, n = 1024, 2048
    try:
        assert L.htr_plan_device_override(8, 160 * 1024) == 0
        if _plan(L, m, n, 4, M, WIDE | S) is None:                                # 16 column blocks in 5 splits: one would be empty
            n = 1920
        assert _plan(L, m, n, 4, M, WIDE | S)[1] > 8
        test_wide_kernel(dev, oracle, L, 4, M, m, n, S, "bf16", 0)
    finally:
        assert L.htr_plan_device_override(0, 0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M", [97, 200, 333])
def test_captured_and_replayed(dev, L, M):
    """A captured call of the wide kernel, replayed with new inputs and eager work in between, gives what the eager call gives."""
    from htr_amd import ops
    print(f"wide kernel in a graph M={M}", flush=True)
    m = n = 4096
    w, x = _case(m, n, 4, M, 80)
    d, x_in = [t.to(dev) for t in w], x.to(dev)
    other, x_other = [t.to(dev) for t in _case(384, 512, 3, 70, 81)[0]], torch.randn(70, 512, device=dev).bfloat16()
    assert M <= 128 or {L.htr_linear_route(m, n, 4, M, 0, eager) for eager in (0, 1)} == {WIDE}
    ops.linear(x_in, *d)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.linear(x_in, *d)
    for i in range(3):
        x_in.copy_(torch.randn(M, n, generator=torch.Generator().manual_seed(i)))
        ops.linear(x_other, *other)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.linear(x_in, *d)), i


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,M", [(512, 1024, 129), (2048, 2048, 700), (4096, 4096, 400)])
def test_float32_activations_stay_float32(dev, m, n, M, monkeypatch):
    """Beyond the rows that were always fused: the float32 product with the dequantized weight, bit for bit, on both host paths."""
    from htr_amd import _native, ops
    print(f"float32 {m}x{n} M={M}", flush=True)
    w, x = _case(m, n, 4, M, 78, torch.float32)
    d, xd = [t.to(dev) for t in w], x.to(dev)
    want = torch.nn.functional.linear(xd, ops.dequant_w(*d).float())
    for fast in (None, False):
        monkeypatch.setattr(_native, "_fast", fast)
        for _ in range(2):
            assert torch.equal(ops.linear(xd, *d), want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,M", [(4096, 4096, 65), (4096, 4096, 200), (2048, 2048, 700), (17408, 2048, 264)])
def test_rows_beyond_64_through_ops(dev, oracle, m, n, M, monkeypatch):
    """Both host paths take the same route and give the same result; what torch differentiates goes on being differentiated."""
    from htr_amd import _native, ops
    print(f"through ops {m}x{n} M={M}", flush=True)
    w, x = _case(m, n, 4, M, 77)
    d, xd = [t.to(dev) for t in w], x.to(dev)
    ref = _ref(oracle, w, x)
    first = ops.linear(xd, *d)
    again = ops.linear(xd, *d)                                                    # with the workspace of the first: in C++
    monkeypatch.setattr(_native, "_fast", False)
    assert torch.equal(first, again) and torch.equal(first, ops.linear(xd, *d))
    wide = _native.lib().htr_linear_route(m, n, 4, M, 0, 1) >= 0
    # bfloat16 results, and bfloat16 weights where the weight is dequantized
    assert np.abs(first.double().cpu().numpy() - ref).max() / np.abs(ref).max() <= (REL_TOL + 2.0 ** -8 if wide else 2.0 ** -6)
    monkeypatch.setattr(_native, "_fast", None)
    leaf = xd.clone().requires_grad_()
    y = ops.linear(leaf, *d)
    assert y.requires_grad == (M > 128 and ops.fused_rows_per_launch(m, n, M) == 0)


def _followed_by_dequantization(L, m, n, M):
    assert {L.htr_linear_route(m, n, 4, M, x, eager) for x in (0, 1, 2) for eager in (0, 1)} == {-1}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("cast", [None, torch.bfloat16, torch.float16])
def test_dequantization_and_product_on_both_host_paths(dev, oracle, L, dtype, cast, monkeypatch):
    """Bias, more dimensions and autocast where the weight is dequantized: C++ and Python give the same, near the oracle's product."""
    from htr_amd import _native, ops
    m, n, M = 1024, 2048, 1024
    print(f"dequantized {dtype}, autocast {cast}", flush=True)
    _followed_by_dequantization(L, m, n, M)
    w, x = _case(m, n, 4, M, 82, dtype)
    d, xd, bias = [t.to(dev) for t in w], x.to(dev), torch.randn(m, generator=torch.Generator().manual_seed(3)).to(dtype).to(dev)
    got = {}
    for path in (None, False):                                                    # C++, Python
        monkeypatch.setattr(_native, "_fast", path)
        with torch.autocast("cuda", dtype=cast or torch.bfloat16, enabled=cast is not None):
            got[path] = [ops.linear(xd, *d), ops.linear(xd, *d, bias), ops.linear(xd.view(4, M // 4, n), *d, bias)]
        if path is None:
            assert _native._fast not in (None, False)
    assert all(torch.equal(a, b) for a, b in zip(got[None], got[False]))
    plain, biased, three = got[None]
    assert all(y.dtype == dtype for y in got[None]) and three.shape == (4, M // 4, m) and torch.equal(three.view(M, m), biased)
    for y, ref in ((plain, _ref(oracle, w, x)), (biased, _ref(oracle, w, x, bias.cpu()))):
        assert np.abs(y.double().cpu().numpy() - ref).max() / np.abs(ref).max() <= 2.0 ** -6      # bfloat16 weights, bfloat16 or cast results


@pytest.mark.gpu
def test_what_torch_follows_beyond_128_rows(dev, L):
    """Derivatives where the weight is dequantized, of the activations and of the bias, forward and backward, and vmap (in float32, where
    torch's products of batches are safe)."""
    from torch.autograd import forward_ad
    from htr_amd import ops
    m, n, M = 1024, 2048, 1024
    print("followed by torch", flush=True)
    _followed_by_dequantization(L, m, n, M)
    w, x = _case(m, n, 4, M, 83, torch.float32)
    d, xd = [t.to(dev) for t in w], x.to(dev)
    g = torch.Generator(device=dev).manual_seed(4)
    t, bias, bt = (torch.randn(*shape, device=dev, generator=g) for shape in ((M, n), (m,), (m,)))
    W = ops.dequant_w(*d).float()
    near = lambda a, b: float((a - b).norm() / b.norm()) <= 1e-5                  # float32 sums in another order
    want, moved = xd @ W.T + bias, t @ W.T
    with forward_ad.dual_level():
        for call, tangent in ((lambda: ops.linear(forward_ad.make_dual(xd, t), *d, bias), moved),
                              (lambda: ops.linear(xd, *d, forward_ad.make_dual(bias, bt)), bt.expand(M, m))):
            y = forward_ad.unpack_dual(call())
            assert near(y.primal, want) and near(y.tangent, tangent)
    both = torch.func.vmap(lambda a: ops.linear(a, *d, bias))(torch.stack([xd, t]))
    assert near(both[0], want) and near(both[1], moved + bias)
    leaf, lb = xd.clone().requires_grad_(), bias.clone().requires_grad_()
    ops.linear(leaf, *d, lb).backward(moved)
    assert near(leaf.grad, moved @ W) and near(lb.grad, moved.sum(0))
    assert ops.linear(xd, *d, lb).requires_grad and not ops.linear(leaf.detach(), *d, lb.detach()).requires_grad
    with torch.no_grad():
        assert not ops.linear(leaf, *d, lb).requires_grad and near(ops.linear(leaf, *d, lb), want)


@pytest.mark.gpu
@pytest.mark.parametrize("lead", [(1,), (1, 1)])
def test_a_prompt_cut_from_a_longer_buffer(dev, lead):
    """Contiguous rows under outer dimensions of size 1 whose strides are the buffer's: one product of matrices, never a batched one
    (torch's own linear takes one for this layout), with the result of the rows alone."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from htr_amd import _native, ops
    m = n = 2048
    M = 700
    print(f"prompt cut from a longer buffer, {len(lead)} outer dimensions", flush=True)
    assert _native.lib().htr_linear_route(m, n, 4, M, 0, 1) == -1 and _native.fast() is not None
    w, x = _case(m, n, 4, M, 79)
    d, rows = [t.to(dev) for t in w], x.to(dev)
    buffer = torch.zeros(*lead, M + 100, n, dtype=torch.bfloat16, device=dev)
    cut = buffer[..., :M, :]
    cut.copy_(rows)
    assert cut.is_contiguous() and cut.stride(0) != M * n
    called = []

    class Record(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            called.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    with Record():
        y = ops.linear(cut, *d)
    assert "mm" in called and not {"bmm", "baddbmm"} & set(called), called
    assert y.shape == (*lead, M, m) and torch.equal(y.reshape(M, m), ops.linear(rows, *d))
