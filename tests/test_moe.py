"""ops.moe_experts with the default activation: the whole layer in one library call, against the per-expert composition on the
CPU oracle with the same rounding between the two linears."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from htr_amd import _native
    _native.lib()
    return torch.device("cuda:0")


def _layer(E, H, F, K1, K2, seed):
    from htr_amd import wire
    return [wire.synth_linear(2 * F, H, K1, seed + e) for e in range(E)], [wire.synth_linear(H, F, K2, seed + 500 + e) for e in range(E)]


def _composition(oracle, x, ids, w, gate_up, down, F):
    y = np.zeros((x.shape[0], x.shape[1]))
    for e in range(len(gate_up)):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        h = torch.from_numpy(oracle.c_linear(x[tok].float().numpy(), *[t.numpy() for t in gate_up[e]])).float()
        h = (torch.nn.functional.silu(h[:, :F]) * h[:, F:]).to(x.dtype).float().numpy()
        np.add.at(y, tok.numpy(), oracle.c_linear(h, *[t.numpy() for t in down[e]]) * w[tok, slot].double().numpy()[:, None])
    return y


def _to(dev, ws):
    return [tuple(t.to(dev) for t in w) for w in ws]


# tokens per expert on both sides of a 32-row tile and of a 64-row entry, experts without tokens, one token, one expert
@pytest.mark.parametrize("dtype,counts,top,K1,K2,H,F", [(torch.bfloat16, (1, 0, 32, 33), 1, 4, 4, 256, 128), (torch.float16, (64, 65, 0, 3), 1, 3, 5, 128, 384),
                                                        (torch.bfloat16, (130,), 1, 4, 4, 256, 256), (torch.float32, (7, 40, 2), 1, 2, 4, 384, 128),
                                                        (torch.bfloat16, (1,), 1, 4, 4, 128, 128), (torch.float16, None, 3, 4, 4, 2176, 256)])
@pytest.mark.parametrize("id_type", [torch.int64, torch.int32])
def test_whole_layer_matches_the_composition(dev, oracle, dtype, counts, top, K1, K2, H, F, id_type):
    """Bound: two chained linears of 1e-3 each with a rounding to `dtype` between them (bf16: 2^-9 per element of the hidden
    vector, averaged over F products), 4e-3 as for the 64-expert configuration; float16 and float32 stay within 2e-3."""
    from htr_amd import ops
    print(f"moe {dtype} {counts} top {top} K {K1}/{K2} H {H} F {F} {id_type}", flush=True)
    g = torch.Generator().manual_seed(31)
    if counts is None:
        E, T = 5, 37
        ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)])
    else:
        E, T = len(counts), sum(counts)
        ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)][:, None]
    gate_up, down = _layer(E, H, F, K1, K2, 600)
    x = torch.randn(T, H, generator=g).to(dtype)
    w = torch.rand(T, top, generator=g)
    y = ops.moe_experts(x.to(dev), ids.to(id_type).to(dev), w.to(dev), _to(dev, gate_up), _to(dev, down)).cpu().numpy()
    ref = _composition(oracle, x, ids, w, gate_up, down, F)
    rel = float(np.abs(y - ref).max() / np.abs(ref).max())
    assert y.dtype == np.float32 and rel <= (4e-3 if dtype == torch.bfloat16 else 2e-3), rel


@pytest.mark.parametrize("E", [63, 64, 65, 129])
def test_number_of_experts_around_one_launch_of_addresses(dev, E):
    """Up to 64 experts' addresses travel with the routing launch, more of them through a table: a pair's result does not depend on
    how many experts stand beside its own, so every size must give, bit for bit, what the chosen experts alone give."""
    from htr_amd import ops
    print(f"moe: {E} experts", flush=True)
    gate_up, down = (_to(dev, part) for part in _layer(E, 128, 128, 4, 4, 640))
    g = torch.Generator().manual_seed(E)
    few = torch.tensor([0, 1, E // 2, E - 2, E - 1])
    pick = torch.stack([torch.randperm(5, generator=g)[:2] for _ in range(11)])
    x, w = torch.randn(11, 128, generator=g).bfloat16().to(dev), torch.rand(11, 2, generator=g).to(dev)
    chosen = few[pick].to(dev)
    y = ops.moe_experts(x, chosen, w, gate_up, down)
    assert torch.equal(y, ops.moe_experts(x, pick.to(dev), w, [gate_up[e] for e in few], [down[e] for e in few]))
    graph = torch.cuda.CUDAGraph()                                                # the addresses are recorded with the launch
    with torch.cuda.graph(graph):
        z = ops.moe_experts(x, chosen, w, gate_up, down)
    for _ in range(3):
        graph.replay()
        assert torch.equal(z, y)


def test_expert_numbers_out_of_range_and_graph_capture(dev):
    from htr_amd import ops
    print("moe: bad ids, capture", flush=True)
    gate_up, down = (_to(dev, ws) for ws in _layer(3, 128, 128, 4, 4, 700))
    x = torch.randn(6, 128, device=dev).bfloat16()
    ids = torch.tensor([[0], [2], [1], [1], [0], [2]], device=dev)
    w = torch.ones(6, 1, device=dev)
    good = ops.moe_experts(x, ids, w, gate_up, down)
    for bad in (3, -1):
        with pytest.raises(IndexError):
            ops.moe_experts(x, torch.where(ids == 2, bad, ids), w, gate_up, down)
    assert torch.equal(ops.moe_experts(x, ids, w, gate_up, down), good)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.moe_experts(x, ids, w, gate_up, down)
    for _ in range(3):
        x.copy_(torch.randn(6, 128, device=dev))
        ids.copy_(ids.roll(1, 0))
        want = ops.moe_experts(x, ids, w, gate_up, down)
        graph.replay()
        assert torch.equal(y, want)


def test_another_activation_takes_the_two_grouped_launches(dev, oracle):
    from htr_amd import ops
    print("moe: relu", flush=True)
    gate_up, down = _layer(3, 256, 128, 4, 4, 800)
    g = torch.Generator().manual_seed(9)
    x, ids, w = torch.randn(20, 256, generator=g).bfloat16(), torch.randint(0, 3, (20, 1), generator=g), torch.rand(20, 1, generator=g)
    args = (x.to(dev), ids.to(dev), w.to(dev), _to(dev, gate_up), _to(dev, down))
    relu = ops.moe_experts(*args, activation=torch.relu)
    silu_by_hand = ops.moe_experts(*args, activation=lambda t: torch.nn.functional.silu(t))
    whole = ops.moe_experts(*args)
    assert not torch.allclose(relu, whole)
    # the same products, rounded alike; only the order of the float32 sums over the slots could differ
    assert float((silu_by_hand - whole).norm() / whole.norm()) <= 1e-3


def test_gradient_of_the_routing_weights(dev, oracle):
    """The default activation keeps y differentiable in the routing weights, backward and forward, as any other one does."""
    from htr_amd import ops
    print("moe: gradient of the routing weights", flush=True)
    gate_up, down = _layer(4, 256, 128, 4, 4, 820)
    g = torch.Generator().manual_seed(10)
    x, w = torch.randn(9, 256, generator=g).bfloat16(), torch.rand(9, 2, generator=g)
    ids = torch.stack([torch.randperm(4, generator=g)[:2] for _ in range(9)])
    gy = torch.randn(9, 256, generator=g)
    args = [x.to(dev), ids.to(dev), _to(dev, gate_up), _to(dev, down)]
    # d sum(gy y) / d w[t, j] is the product of gy[t] with what slot j alone gives
    want = torch.zeros(9, 2, dtype=torch.float64)
    for j in range(2):
        only = torch.zeros(9, 2)
        only[:, j] = 1.0
        want[:, j] = (torch.from_numpy(_composition(oracle, x, ids, only, gate_up, down, 128)) * gy.double()).sum(1)
    wd = w.to(dev).requires_grad_()
    y = ops.moe_experts(args[0], args[1], wd, *args[2:])
    assert y.requires_grad
    (y * gy.to(dev)).sum().backward()
    assert float((wd.grad.cpu().double() - want).norm() / want.norm()) <= 4e-3      # as for the layer's result in bfloat16
    with torch.no_grad():
        assert not ops.moe_experts(args[0], args[1], wd, *args[2:]).requires_grad
    with torch.autograd.forward_ad.dual_level():
        y, t = torch.autograd.forward_ad.unpack_dual(
            ops.moe_experts(args[0], args[1], torch.autograd.forward_ad.make_dual(w.to(dev), torch.ones(9, 2, device=dev)), *args[2:]))
        alone = ops.moe_experts(args[0], args[1], torch.ones(9, 2, device=dev), *args[2:])
        assert t is not None and float((t - alone).norm() / alone.norm()) <= 1e-3      # the result is linear in the weights


def test_collections_that_load_experts_on_demand(dev):
    """Anything but a plain list or tuple is asked for the experts that some token chose, and for no other."""
    from htr_amd import ops
    print("moe: experts on demand", flush=True)
    gate_up, down = (_to(dev, ws) for ws in _layer(4, 128, 128, 4, 4, 840))

    class OnDemand:
        def __init__(self, experts):
            self.experts, self.asked = experts, set()

        def __len__(self):
            return len(self.experts)

        def __getitem__(self, e):
            if not 0 <= e < len(self.experts):
                raise IndexError(e)
            self.asked.add(e)
            return self.experts[e]

    x = torch.randn(6, 128, device=dev).bfloat16()
    ids, w = torch.tensor([[0], [2], [2], [0], [2], [2]], device=dev), torch.rand(6, 1, device=dev)
    lazy = [OnDemand(gate_up), OnDemand(down)]
    y = ops.moe_experts(x, ids, w, *lazy)
    assert all(c.asked == {0, 2} for c in lazy)
    whole = ops.moe_experts(x, ids, w, gate_up, tuple(down))
    assert float((whole - y).norm() / y.norm()) <= 1e-3          # the same products, rounded alike
    with pytest.raises(TypeError):
        ops.moe_experts(x, ids, w, (t for t in gate_up), (t for t in down))


def test_more_than_65535_tokens(dev):
    """Each token's result is its own: the same bits as in calls of 30000."""
    from htr_amd import ops
    print("moe: 70000 tokens", flush=True)
    gate_up, down = (_to(dev, ws) for ws in _layer(2, 128, 128, 4, 4, 860))
    x, ids, w = torch.randn(70000, 128, device=dev).bfloat16(), torch.randint(0, 2, (70000, 1), device=dev), torch.rand(70000, 1, device=dev)
    parts = [ops.moe_experts(x[i:i + 30000], ids[i:i + 30000], w[i:i + 30000], gate_up, down) for i in range(0, 70000, 30000)]
    assert torch.equal(ops.moe_experts(x, ids, w, gate_up, down), torch.cat(parts))
