"""The work that users of this package have it do, as cases with inputs, one pass, work and tolerance.

Families ("kind"):
  linear   one `ops.linear` call, not captured: any row count, from a single decode row to a long prefill
  layer    the four packed linears of consecutive decoder layers (q/k/v fused, o, gate/up fused, down), captured once in a
           HIP graph and replayed per token step, as serving stacks run decode
  moe      `ops.moe_experts`: routing, the experts' gate/up, the activation, the experts' down projection
  search   `encode.viterbi`: one batch of tiles of the encoder's trellis search
  encode   `encode.encode_group`: whole matrices through the encoder
"""
import math

import torch

from htr_amd import encode, ops, wire

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_TILE_STATES = 1 << 16        # trellis states per step of the search
_TILE_STEPS = 256             # weights per tile


def listed():
    return [
        # decode, one token: the k or v projection of a 9B-class model (GQA 32/8), the smallest linear of a layer
        dict(name="k_proj_1_row", kind="linear", m=1024, n=4096, K=4, rows=1, dtype="bf16", bias=False),
        # decode, one token: the quantized output head, the largest single linear
        dict(name="lm_head_1_row", kind="linear", m=152064, n=4096, K=4, rows=1, dtype="bf16", bias=False),
        # decode, one token, serving: eight 9B-class layers in one graph
        dict(name="layers_1_row_graph", kind="layer", layers=8, hidden=4096, kv=2048, inter=14336, K=4, rows=1, dtype="bf16"),
        # decode, 32 sequences at once, serving
        dict(name="layers_32_rows_graph", kind="layer", layers=8, hidden=4096, kv=2048, inter=14336, K=3, rows=32, dtype="bf16"),
        # decode of a batch that is no power of two, long rows
        dict(name="down_proj_13_rows", kind="linear", m=4096, n=14336, K=3, rows=13, dtype="bf16", bias=False),
        # a short prompt or a speculative batch, float16 with bias, five bits
        dict(name="gate_proj_97_rows", kind="linear", m=14336, n=4096, K=5, rows=97, dtype="f16", bias=True),
        # prefill of one ragged prompt
        dict(name="qkv_proj_333_rows", kind="linear", m=6144, n=4096, K=4, rows=333, dtype="bf16", bias=False),
        # prefill in chunks of 2048 tokens
        dict(name="gate_proj_2048_rows", kind="linear", m=14336, n=4096, K=4, rows=2048, dtype="bf16", bias=False),
        # routed experts in decode: 16 tokens, top 6 of 64
        dict(name="experts_16_tokens", kind="moe", tokens=16, experts=64, top=6, hidden=2048, inter=1408, K=4, dtype="bf16"),
        # routed experts in prefill
        dict(name="experts_500_tokens", kind="moe", tokens=500, experts=64, top=6, hidden=2048, inter=1408, K=4, dtype="bf16"),
        # encoder: the batch of tiles that encode_group hands to the search for tall matrices
        dict(name="search_1024_tiles", kind="search", tiles=1024, K=4),
        # encoder: the gate/up pair of one expert on one Hessian, whole
        dict(name="encode_expert_gate_up", kind="encode", parts=2, m=1408, n=1024, K=3),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, unit=1):
    """A log-uniform multiple of `unit` between lo and hi (both multiples of it)."""
    return min(hi, max(lo, unit * round(_log_uniform(rng, lo, hi) / unit)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "layer", "moe", "moe", "search", "encode"))
    K = rng.choice((2, 3, 4, 4, 4, 5))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16"))
    if kind == "linear":
        rows = rng.choice((1, _size(rng, 2, 32), _size(rng, 1, 2048), _size(rng, 33, 2048)))
        return dict(kind=kind, m=_size(rng, 256, 28672, 128), n=_size(rng, 256, 14336, 128), K=K, rows=rows,
                    dtype=rng.choice((dtype, dtype, dtype, "f32")), bias=rng.random() < 0.3)
    if kind == "layer":
        hidden = _size(rng, 1024, 5120, 128)
        return dict(kind=kind, layers=rng.randint(2, 8), hidden=hidden, kv=128 * rng.choice((4, 8, 16)),
                    inter=128 * round(hidden * rng.uniform(2.5, 3.5) / 128), K=K, rows=rng.choice((1, _size(rng, 2, 64))), dtype=dtype)
    if kind == "moe":
        experts = rng.choice((8, 16, 32, 64))
        return dict(kind=kind, tokens=_size(rng, 1, 512), experts=experts, top=rng.randint(1, min(8, experts // 2)),
                    hidden=_size(rng, 512, 4096, 128), inter=_size(rng, 256, 2048, 128), K=K, dtype=dtype)
    if kind == "search":
        return dict(kind=kind, tiles=_size(rng, 16, 1024), K=K)
    return dict(kind=kind, parts=rng.randint(1, 2), m=_size(rng, 256, 1408, 128), n=_size(rng, 256, 1024, 128), K=K)


# ---- inputs: everything is drawn on the GPU by one generator per state
def _weight(gen, m, n, K, su=None):
    """One packed linear: every bit string is a valid circular trellis stream, row scales are lognormal(0, 0.25)."""
    dev = gen.device
    qw = torch.randint(-(2 ** 31), 2 ** 31, (m // 16, n // 16, 8 * K), dtype=torch.int32, device=dev, generator=gen)
    scales = torch.exp(0.25 * torch.randn(m, device=dev, generator=gen)).half()
    if su is None:
        su = torch.randint(0, 256, (n // 8,), dtype=torch.uint8, device=dev, generator=gen)
    sv = torch.randint(0, 256, (m // 8,), dtype=torch.uint8, device=dev, generator=gen)
    return qw, scales, su, sv


def _activations(gen, rows, n, dtype):
    return torch.randn(rows, n, device=gen.device, generator=gen).to(_DTYPES[dtype])


def _layer_shapes(case):
    h, f = case["hidden"], case["inter"]
    return ((h + case["kv"], h), (h, h), (2 * f, h), (h, f))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        w = _weight(gen, case["m"], case["n"], case["K"])
        x = _activations(gen, case["rows"], case["n"], case["dtype"])
        bias = torch.randn(case["m"], device=dev, generator=gen).to(x.dtype) if case["bias"] else None
        return dict(kind=kind, x=x, w=w, bias=bias)
    if kind == "layer":
        calls = []
        for _ in range(case["layers"]):
            for m, n in _layer_shapes(case):
                calls.append((_activations(gen, case["rows"], n, case["dtype"]), _weight(gen, m, n, case["K"])))
        side = torch.cuda.Stream(dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            for x, w in calls[:4]:
                ops.linear(x, *w)
        torch.cuda.current_stream(dev).wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = [ops.linear(x, *w) for x, w in calls]
        return dict(kind=kind, graph=graph, calls=calls, outs=outs)
    if kind == "moe":
        T, E, H, F, K = case["tokens"], case["experts"], case["hidden"], case["inter"], case["K"]
        gate_up = [_weight(gen, 2 * F, H, K) for _ in range(E)]
        down = [_weight(gen, H, F, K) for _ in range(E)]
        # a router with popular and unpopular experts; tokens prefer different ones
        logits = torch.randn(T, E, device=dev, generator=gen) + 0.5 * torch.randn(E, device=dev, generator=gen)
        probs, ids = torch.topk(torch.softmax(logits, dim=-1), case["top"], dim=-1)
        return dict(kind=kind, x=_activations(gen, T, H, case["dtype"]), ids=ids, probs=probs / probs.sum(-1, keepdim=True),
                    gate_up=gate_up, down=down)
    if kind == "search":
        # what the encoder hands over: rotated weights over their row scale, squared row scales with mean 1 per tile
        x = torch.randn(case["tiles"], _TILE_STEPS, device=dev, generator=gen)
        rs = torch.exp(0.25 * torch.randn(case["tiles"], 16, 1, device=dev, generator=gen)) ** 2
        w = (rs / rs.mean(dim=1, keepdim=True)).expand(-1, -1, 16).reshape(case["tiles"], _TILE_STEPS).contiguous()
        return dict(kind=kind, x=x, w=w, K=case["K"], cb=wire.codebook_f32(dev))
    m, n = case["m"], case["n"]
    # the Hessian of 2 n activations whose channels have different sizes and share a common part
    acts = torch.randn(2 * n, n, device=dev, generator=gen) + 0.3 * torch.randn(2 * n, 1, device=dev, generator=gen)
    acts = acts * torch.exp(0.5 * torch.randn(n, device=dev, generator=gen))
    hess = (acts.double().T @ acts.double() / (2 * n)).float()
    jobs = [dict(W=0.02 * torch.randn(m, n, device=dev, generator=gen), H=hess) for _ in range(case["parts"])]
    return dict(kind=kind, jobs=jobs, K=case["K"], seed=seed)


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return ops.linear(state["x"], *state["w"], state["bias"])
    if kind == "layer":
        state["graph"].replay()
        return state["outs"]
    if kind == "moe":
        return ops.moe_experts(state["x"], state["ids"], state["probs"], state["gate_up"], state["down"])
    if kind == "search":
        return encode.viterbi(state["x"], state["w"], state["cb"], state["K"])
    return encode.encode_group(state["jobs"], state["K"], seed=state["seed"])


# ---- the work a pass cannot do without
def _search_work(tiles):
    """Two passes (free, then tail-biting); per step every state's cost is one addition and one comparison."""
    return 2 * tiles * _TILE_STEPS * _TILE_STATES * 2


def _active_experts(case):
    """Experts that some token chose, in expectation for even routing; every one of them has its weights read."""
    return case["experts"] * (1.0 - (1.0 - case["top"] / case["experts"]) ** case["tokens"])


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, rows = case["m"], case["n"], case["rows"]
        es = _DTYPES[case["dtype"]].itemsize
        return {"bytes": wire.payload_bytes(m, n, case["K"]) + rows * (m + n) * es, "flops": 2 * rows * m * n}
    if kind == "layer":
        shapes, rows = _layer_shapes(case), case["rows"]
        return {"bytes": case["layers"] * sum(wire.payload_bytes(m, n, case["K"]) + 2 * rows * (m + n) for m, n in shapes),
                "flops": case["layers"] * sum(2 * rows * m * n for m, n in shapes)}
    if kind == "moe":
        H, F, T = case["hidden"], case["inter"], case["tokens"]
        packed = wire.payload_bytes(2 * F, H, case["K"]) + wire.payload_bytes(H, F, case["K"])
        return {"bytes": _active_experts(case) * packed + T * H * (2 + 4) + T * case["top"] * (8 + 4),
                "flops": 2 * T * case["top"] * 3 * F * H}
    if kind == "search":
        return {"bytes": case["tiles"] * _TILE_STEPS * (4 + 4 + 8), "flops": _search_work(case["tiles"])}
    m, n, parts = case["m"], case["n"], case["parts"]
    feedback = parts * m * n * n                 # every column block's error into all earlier columns
    factor = n ** 3 / 3 + 4 * 128 * n * n        # one Cholesky factorisation and the Hessian's rotation
    return {"bytes": 4 * n * n + parts * (4 * m * n * 3 + wire.payload_bytes(m, n, case["K"])),
            "flops": parts * _search_work(m * n // 256) + feedback + factor}


def tolerance(case):
    """Relative 2-norm error against the same product in float64, measured and multiplied by about four: the activations
    are rounded to float16 in the rotated basis (2e-4) and bfloat16 results once more (1.7e-3); long prefills form the
    weight in bfloat16 (2.4e-3 with a bfloat16 result).  The encoder's results are whole numbers and what follows from them."""
    kind = case["kind"]
    if kind in ("search", "encode"):
        return "exact"
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 8e-3 if case.get("rows", 0) > 128 else 1.5e-3}
