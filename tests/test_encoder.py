"""The matrix encoder (htr_amd/encode.py; htr/encode.py:45-110 of the reference) and its GPU trellis search.

CPU: the encoder's host logic around the CPU oracle's Viterbi must reproduce, bit for bit, what the reference's
encode_group produced for the same inputs (tests/golden/encode_small.npz, written by tests/golden/make_encoder_golden.py).
GPU: the library's search against the oracle's on identical inputs (states bit-exact), and the whole encoder on the
device against the bars of the reference's own round-trip test (tests/test_release.py:53-73)."""
import os

import numpy as np
import pytest
import torch

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def enc_gold():
    return np.load(os.path.join(HERE, "golden", "encode_small.npz"), allow_pickle=False)


@pytest.fixture(scope="module")
def vit_gold():
    return np.load(os.path.join(HERE, "golden", "viterbi.npz"), allow_pickle=False)


@pytest.fixture()
def oracle_search(oracle):
    from htr_amd import encode
    old = encode.VITERBI
    encode.VITERBI = lambda x, w, cb, K: torch.from_numpy(oracle.c_viterbi(x.numpy(), w.numpy(), K).astype(np.int64))
    yield encode
    encode.VITERBI = old


def _same(result, gold, tag):
    assert np.array_equal(result["qweight"].numpy(), gold[f"{tag}_qweight"])
    assert np.array_equal(result["scales"].numpy().view(np.uint16), gold[f"{tag}_scales_f16bits"])
    assert np.array_equal(result["su"].numpy(), gold[f"{tag}_su"]) and np.array_equal(result["sv"].numpy(), gold[f"{tag}_sv"])
    assert np.array_equal(result["What"].numpy(), gold[f"{tag}_What"])


def test_encoder_reproduces_reference_on_its_round_trip_matrix(oracle_search, enc_gold):
    from htr_amd import wire
    w = torch.from_numpy(enc_gold["a_W"])
    r = oracle_search.encode_group([{"W": w, "H": torch.eye(128)}], 4, max_batch=8)[0]
    _same(r, enc_gold, "a")
    # the bars of the reference's own test (tests/test_release.py:69-73)
    actual = wire.dequant(r["qweight"], r["scales"], r["su"], r["sv"])
    assert torch.equal(actual, r["What"]) and tuple(r["qweight"].shape) == (8, 8, 32)
    assert bool(torch.isfinite(actual).all())
    assert float((actual - w).square().sum() / w.square().sum()) < 0.02


def test_encoder_reproduces_reference_with_hessian_and_shared_signs(oracle_search, enc_gold):
    H = torch.from_numpy(enc_gold["b_H"])
    jobs = [{"W": torch.from_numpy(enc_gold["b0_W"]), "H": H}, {"W": torch.from_numpy(enc_gold["b1_W"]), "H": H}]
    rs = oracle_search.encode_group(jobs, 3, seed=4321, max_batch=64)
    _same(rs[0], enc_gold, "b0")
    _same(rs[1], enc_gold, "b1")
    assert np.array_equal(rs[0]["su"].numpy(), rs[1]["su"].numpy())          # one input sign vector for the group


@pytest.mark.parametrize("K", [2, 3, 4, 5])
def test_cpu_search_matches_reference_vectors(vit_gold, K):
    """CPU tensors take the torch search (the GPU kernel's formulation): bit-identical to the reference's vectors,
    the all-ties row included."""
    from htr_amd import encode
    x, w = torch.from_numpy(vit_gold[f"k{K}_x"]), torch.from_numpy(vit_gold[f"k{K}_w"])
    st = encode.viterbi(x, w, None, K)
    assert st.dtype == torch.int64 and np.array_equal(st.numpy().astype(np.uint16), vit_gold[f"k{K}_states"])


@pytest.mark.parametrize("K,B,T,tailbite", [(6, 2, 256, True), (8, 2, 64, True), (4, 3, 100, False), (4, 2, 1, True), (3, 2, 17, False)])
def test_cpu_search_matches_oracle(oracle, K, B, T, tailbite):
    from htr_amd import encode
    g = torch.Generator().manual_seed(100 * K + T)
    x = torch.randn(B, T, generator=g) * 1.2
    w = torch.rand(B, T, generator=g) + 0.25
    x[0, : T // 2] = 0.0
    st = encode.viterbi_cpu(x, w, K, tailbite).numpy()
    assert np.array_equal(st.astype(np.uint32), oracle.c_viterbi(x.numpy(), w.numpy(), K, tailbite=tailbite))


def test_encoder_on_cpu_tensors_without_a_hook(enc_gold):
    """encode_group on CPU tensors with VITERBI unset (the reference falls back to its portable search there,
    htr/encode.py:10-12, 48): the torch search reproduces the reference's round-trip matrix bit for bit."""
    from htr_amd import encode
    assert encode.VITERBI is None
    r = encode.encode_group([{"W": torch.from_numpy(enc_gold["a_W"]), "H": torch.eye(128)}], 4, max_batch=8)[0]
    _same(r, enc_gold, "a")


def test_matrices_of_one_hessian_share_a_factorisation(oracle_search, enc_gold, monkeypatch):
    """Two matrices that come with the same Hessian object under a shared input sign vector are factored once and fed
    back with one product; the result is the one of separate factorisations (the reference's fixture)."""
    calls = []
    real = oracle_search._feedback_factor
    monkeypatch.setattr(oracle_search, "_feedback_factor", lambda Hd: (calls.append(1), real(Hd))[1])
    H = torch.from_numpy(enc_gold["b_H"])
    jobs = [{"W": torch.from_numpy(enc_gold[f"b{i}_W"]), "H": H} for i in range(2)]
    rs = oracle_search.encode_group(jobs, 3, seed=4321, max_batch=64)
    assert len(calls) == 1
    for i, r in enumerate(rs):
        assert np.array_equal(r["qweight"].numpy(), enc_gold[f"b{i}_qweight"])
    calls.clear()
    oracle_search.encode_group([{"W": jobs[0]["W"], "H": H}, {"W": jobs[1]["W"], "H": H.clone()}], 3, seed=4321, max_batch=64)
    assert len(calls) == 2


def test_sign_draws_and_hessian_preparation():
    from htr_amd import encode
    su, sv = encode.make_signs(256, 128, 99, 2, True)
    su2, sv2 = encode.make_signs(256, 128, 99, 5, True)
    assert torch.equal(su, su2) and not torch.equal(sv, sv2) and set(su.tolist()) == {-1.0, 1.0}
    a, b = encode.make_signs(256, 128, 99, 2, False)
    g = torch.Generator().manual_seed(99 + 7919 * 2)
    assert torch.equal(a, (torch.randint(0, 2, (256,), generator=g) * 2 - 1).float())
    assert torch.equal(b, (torch.randint(0, 2, (128,), generator=g) * 2 - 1).float())
    H = torch.diag(torch.tensor([2.0, 0.0, 4.0]))
    W = torch.ones(2, 3)
    Hp, Wp = encode.prep_H(H, W, damp=0.5)
    mean = (2.0 + 1.0 + 4.0) / 3                                             # dead diagonal entry becomes 1
    assert torch.allclose(torch.diag(Hp), torch.tensor([2.0, 1.0, 4.0], dtype=torch.float64) + 0.5 * mean)
    assert torch.equal(Wp, torch.tensor([[1.0, 0.0, 1.0], [1.0, 0.0, 1.0]]))


# ---------------------------------------------------------------------------------------------------------------- GPU
@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from htr_amd import _native
    _native.lib()
    return torch.device("cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("K", [2, 3, 4, 5])
def test_gpu_search_matches_reference_vectors(dev, vit_gold, K):
    from htr_amd import encode
    print(f"viterbi golden K={K}", flush=True)
    x, w = torch.from_numpy(vit_gold[f"k{K}_x"]), torch.from_numpy(vit_gold[f"k{K}_w"])
    st = encode.viterbi(x.to(dev), w.to(dev), None, K).cpu().numpy()
    assert np.array_equal(st.astype(np.uint16), vit_gold[f"k{K}_states"])


@pytest.mark.gpu
@pytest.mark.parametrize("K,B,T,tailbite", [(2, 5, 256, True), (3, 7, 256, True), (4, 9, 256, True), (5, 6, 256, True),
                                            (6, 3, 256, True), (7, 2, 256, True), (8, 3, 256, True), (8, 2, 256, False), (8, 2, 9, True),
                                            (4, 3, 256, False), (3, 4, 100, True),
                                            (4, 2, 1, True), (2, 2, 17, False)])
def test_gpu_search_matches_oracle(dev, oracle, K, B, T, tailbite):
    from htr_amd import encode
    print(f"viterbi K={K} B={B} T={T} tailbite={tailbite}", flush=True)
    g = torch.Generator().manual_seed(1000 * K + B + T)
    x = torch.randn(B, T, generator=g) * 1.2
    w = torch.rand(B, T, generator=g) + 0.25
    x[0, : T // 2] = 0.0                                                     # long runs of equal costs
    st = encode.viterbi(x.to(dev), w.to(dev), None, K, tailbite=tailbite).cpu().numpy()
    want = oracle.c_viterbi(x.numpy(), w.numpy(), K, tailbite=tailbite)
    assert np.array_equal(st.astype(np.uint32), want)


@pytest.mark.gpu
@pytest.mark.parametrize("K,B,lengths", [(2, 3, (2, 3, 4, 5, 6, 8, 9, 30)), (3, 3, (2, 3, 4, 5, 7, 8, 29)), (4, 3, (2, 3, 4, 5, 6, 31)),
                                         (5, 2, (2, 3, 20)), (6, 2, (2, 21)), (7, 2, (2, 22)), (8, 2, (2, 23)), (4, 600, (11,))])
@pytest.mark.parametrize("tailbite", [True, False])
def test_gpu_search_at_the_edges_of_its_trace_back(dev, oracle, K, B, lengths, tailbite):
    """Lengths around multiples of the steps that the trace back resolves in one turn (4, 3, 2, 1 at K = 2, 3, 4, 5 and
    more), and more tiles than workgroups, so that a workgroup takes several in turn.  Whole numbers: exact."""
    from htr_amd import encode
    for T in lengths:
        print(f"viterbi K={K} B={B} T={T} tailbite={tailbite}", flush=True)
        g = torch.Generator().manual_seed(77 * K + B + T)
        x = torch.randn(B, T, generator=g)
        w = torch.rand(B, T, generator=g) + 0.25
        st = encode.viterbi(x.to(dev), w.to(dev), None, K, tailbite=tailbite).cpu().numpy()
        assert np.array_equal(st.astype(np.uint32), oracle.c_viterbi(x.numpy(), w.numpy(), K, tailbite=tailbite))


@pytest.mark.gpu
@pytest.mark.parametrize("K", range(2, 9))
@pytest.mark.parametrize("tailbite", [True, False])
def test_gpu_search_takes_the_first_of_equal_costs(dev, oracle, K, tailbite):
    """Equal costs in every step (no weight, no target, targets and weights of a few values) and infinite ones, where the trace back's
    masks decide: the first index, as in the oracle.  Exact."""
    from htr_amd import encode
    g = torch.Generator().manual_seed(90 + K)
    for T in (2, 3, 5, 8, 14):
        x, w = torch.randn(8, T, generator=g), torch.rand(8, T, generator=g) + 0.25
        x[0], w[1] = 0.0, 0.0
        w[2] *= torch.arange(T) % 2
        x[3], w[3] = x[3].round(), (4 * w[3]).round()
        x[4], w[4] = 0.0, 1.0
        x[5, T // 2] = float("inf")
        w[6, T // 2] = float("inf")
        x[7] *= 1e20                                                  # every cost overflows
        print(f"viterbi ties K={K} T={T} tailbite={tailbite}", flush=True)
        st = encode.viterbi(x.to(dev), w.to(dev), None, K, tailbite=tailbite).cpu().numpy()
        assert np.array_equal(st.astype(np.uint32), oracle.c_viterbi(x.numpy(), w.numpy(), K, tailbite=tailbite))


@pytest.mark.gpu
def test_gpu_search_within_a_scratch_limit(dev, oracle, monkeypatch):
    """MAX_SCRATCH_BYTES bounds the scratch also where it does not hold one workgroup per compute unit; no tiles at all, and a number
    of bits that is refused whatever the number of tiles."""
    from htr_amd import _native, encode
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(11, 19, generator=g).to(dev), (torch.rand(11, 19, generator=g) + 0.25).to(dev)
    want = encode.viterbi(x, w, None, 4)
    monkeypatch.setattr(encode, "_SCRATCH", {})
    for tiles in (3, 0):                                              # 3: four launches; 0: less than one tile, one at a time
        monkeypatch.setattr(encode, "MAX_SCRATCH_BYTES", max(1, tiles * _native.lib().htr_viterbi_workspace_bytes(1, 19, 4)))
        print(f"viterbi, scratch for {tiles} tiles", flush=True)
        assert torch.equal(encode.viterbi(x, w, None, 4), want)
        if tiles:
            assert max(t.numel() for t in encode._SCRATCH.values()) <= encode.MAX_SCRATCH_BYTES
    assert encode.viterbi(x[:0], w[:0], None, 4).shape == (0, 19)
    with pytest.raises(RuntimeError, match="K 9"):
        encode.viterbi(x[:0], w[:0], None, 9)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [2, 4, 8])
def test_gpu_search_with_scratch_at_any_address(dev, K):
    """The C entry takes the scratch where it is, as it always did; the stored arrays find their own 16-byte boundary in it."""
    from htr_amd import _native, encode
    L = _native.lib()
    g = torch.Generator().manual_seed(6)
    x, w = torch.randn(5, 21, generator=g).to(dev), (torch.rand(5, 21, generator=g) + 0.25).to(dev)
    want = encode.viterbi(x, w, None, K)
    need = L.htr_viterbi_workspace_bytes(5, 21, K)
    for offset in (1, 8, 15):
        print(f"viterbi K={K}, scratch {offset} bytes off", flush=True)
        buf, out = torch.empty(need + offset, dtype=torch.uint8, device=dev), torch.empty(5, 21, dtype=torch.int16, device=dev)
        _native.check(L.htr_viterbi(x.data_ptr(), w.data_ptr(), 5, 21, K, 1, out.data_ptr(), buf.data_ptr() + offset, need,
                                    torch.cuda.current_stream().cuda_stream))
        assert torch.equal(out.long() & 0xFFFF, want)


@pytest.mark.gpu
def test_gpu_search_refuses_another_codebook(dev):
    from htr_amd import encode, wire
    print("viterbi: codebook check", flush=True)
    x, w = torch.zeros(1, 16), torch.ones(1, 16)
    cb = wire.codebook_f32(dev)
    assert encode.viterbi(x.to(dev), w.to(dev), cb, 4).shape == (1, 16)
    with pytest.raises(RuntimeError, match="not the HTR-W1 codebook"):
        encode.viterbi(x.to(dev), w.to(dev), cb * 2.0, 4)
    assert encode.viterbi(x, w, None, 4).shape == (1, 16)           # CPU tensors: the torch search


@pytest.mark.gpu
def test_gpu_encoder_round_trip(dev, enc_gold):
    """The reference's round-trip test on the device: encode the seed-12 matrix with the library's search, reopen, decode.
    torch's device linear algebra need not match the CPU's last bits, so the comparison with the CPU fixture is by
    share of identical tiles; the decode identity and the error bar are exact requirements."""
    from htr_amd import encode, ops, wire
    print("encoder round trip", flush=True)
    w = torch.from_numpy(enc_gold["a_W"]).to(dev)
    r = encode.encode_group([{"W": w, "H": torch.eye(128, device=dev)}], 4, max_batch=8)[0]
    assert tuple(r["qweight"].shape) == (8, 8, 32)
    d = [r[k].to(dev) for k in ("qweight", "scales", "su", "sv")]
    actual = wire.dequant(*d)
    assert torch.equal(actual, r["What"]) and bool(torch.isfinite(actual).all())
    assert float((actual - w).square().sum() / w.square().sum()) < 0.02
    same = float((r["qweight"].numpy() == enc_gold["a_qweight"]).all(axis=2).mean())
    assert same >= 0.9, same
    # the packed linear on the encoded matrix reproduces x @ What^T
    x = torch.randn(3, 128, generator=torch.Generator().manual_seed(1)).to(dev)
    y = ops.linear_f32out(x, *d)
    ref = x @ actual.T
    assert float((y - ref).abs().max() / ref.abs().max()) <= 1e-3


def test_codebook_check_is_not_fooled_by_a_reused_address(monkeypatch):
    """A table that was checked once is known by its memory only while that memory is its own and unchanged."""
    from htr_amd import encode, wire
    monkeypatch.setattr(encode, "_CHECKED_CB", {})
    good = wire.codebook_f32("cpu").clone()
    encode._check_codebook(good)
    encode._check_codebook(good)
    assert len(encode._CHECKED_CB) == 1
    with pytest.raises(RuntimeError, match="codebook"):
        encode._check_codebook(good.flip(0).contiguous())
    good[3] += 1.0                                                    # changed in place
    with pytest.raises(RuntimeError, match="codebook"):
        encode._check_codebook(good)
    address = wire.codebook_f32("cpu").clone()
    encode._check_codebook(address)
    held, at = address.untyped_storage().data_ptr(), address.data_ptr()
    del address
    others = [torch.zeros(wire.S) for _ in range(8)]                  # would take freed memory of the same size
    assert all(t.data_ptr() != at for t in others) and held == at
    for _ in range(40):
        encode._check_codebook(wire.codebook_f32("cpu").clone())
    assert len(encode._CHECKED_CB) <= 16


@pytest.mark.gpu
@pytest.mark.parametrize("K,sizes,n,shared,max_batch", [(2, [(128, 0)], 128, False, 8), (3, [(256, 0), (384, 0)], 256, True, 1024), (4, [(128, 0), (128, 1), (256, 1)], 384, True, 11),
                                                       (5, [(1280, 0)], 128, True, 64)])
def test_gpu_encoder_blocks_match_the_torch_lines(dev, monkeypatch, K, sizes, n, shared, max_batch):
    """_NativeBlocks against _TorchBlocks with the same search (a hook selects them): every output bit for bit.  One and several matrices and Hessians, a dead input column, batches that do not divide the tiles."""
    from htr_amd import encode
    print(f"encoder blocks K={K} {sizes} n={n}", flush=True)
    g = torch.Generator().manual_seed(K)
    hessians = []
    for i in range(2):
        a = torch.randn(2 * n, n, generator=g) * torch.exp(0.5 * torch.randn(n, generator=g))
        a[:, 5 + i] = 0
        hessians.append((a.T @ a / (2 * n)).to(dev))
    jobs = [dict(W=(0.02 * torch.randn(m, n, generator=g)).to(dev), H=hessians[h]) for m, h in sizes]
    got = encode.encode_group(jobs, K, seed=7, shared_su=shared, max_batch=max_batch)
    monkeypatch.setattr(encode, "VITERBI", lambda x, w, cb, k: encode.viterbi(x, w, cb, k))
    want = encode.encode_group(jobs, K, seed=7, shared_su=shared, max_batch=max_batch)
    for a, b in zip(got, want):
        for name in b:
            assert torch.equal(a[name], b[name]), name


def test_encoder_block_launches_refuse_wrong_sizes():
    from htr_amd import _native
    L = _native.lib()
    p = [1 << 12] * 7
    assert L.htr_encode_targets(None, *p[1:3], 16, 16, 0, p[3], None) == 1 and L.htr_encode_targets(p[0] + 4, *p[1:3], 16, 16, 0, p[3], None) == L.htr_encode_targets(*p[:3], 16, 16, 0, p[3] + 8, None) != 0
    for rows, n, col in ((0, 16, 0), (8, 16, 0), (16, 24, 0), (16, 16, 16), (16, 32, 8), (16, 16, -16), (1 << 31, 16, 0)):
        bad = L.htr_encode_targets(*p[:3], rows, n, col, p[3], None)
        assert bad == L.htr_encode_quantized(*p[:4], rows, n, col, *p[4:7], None) == L.htr_encode_targets(*p[:3], 8, 16, 0, p[3], None) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("K,lengths", [(2, (10, 13, 14, 17, 18, 21, 22)), (3, (9, 10, 11, 13, 14, 16, 17, 20)), (4, (7, 8, 9, 10, 11, 12, 13, 14, 256)),
                                       (5, (4, 5, 6, 7, 8, 9, 10, 11)), (6, (5, 6, 9)), (7, (5, 6, 7, 10)), (8, (5, 7, 8, 256))])
@pytest.mark.parametrize("tailbite", [True, False])
def test_gpu_search_with_few_stored_arrays(dev, oracle, K, lengths, tailbite):
    """Lengths with one to ten stored arrays, around the four that the trace back has in flight and its loop takes at a time, and the
    longest.  The states are whole numbers: exact."""
    from htr_amd import encode
    for T in lengths:
        print(f"viterbi K={K} T={T} tailbite={tailbite}", flush=True)
        g = torch.Generator().manual_seed(91 * K + T)
        x = torch.randn(2, T, generator=g)
        w = torch.rand(2, T, generator=g) + 0.25
        st = encode.viterbi(x.to(dev), w.to(dev), None, K, tailbite=tailbite).cpu().numpy()
        assert np.array_equal(st.astype(np.uint32), oracle.c_viterbi(x.numpy(), w.numpy(), K, tailbite=tailbite))


@pytest.mark.parametrize("default", [torch.float64, torch.bfloat16])
def test_buffers_of_the_encoder_blocks_do_not_follow_the_default_type(default):
    """htr_encode_quantized writes float32 errors: a buffer of torch's default type would be read as other numbers, or be too short."""
    from types import SimpleNamespace
    from htr_amd import encode
    G = SimpleNamespace(Wt=torch.zeros(32, 128), wg=torch.zeros(2, 256))
    before = torch.get_default_dtype()
    torch.set_default_dtype(default)
    try:
        blocks = encode._NativeBlocks(G, None, 4, 1024)
    finally:
        torch.set_default_dtype(before)
    assert blocks.err.dtype == torch.float32 and blocks.err.shape == (32, 16)
    assert blocks.x.dtype == torch.float32 and blocks.x.shape == (2, 256) and blocks.states.dtype == torch.int16


@pytest.mark.parametrize("shape", [(6, 1), (6,), (6, 64), (6, 256), (1, 6)])
def test_dead_columns_of_a_matrix_that_does_not_fit_the_hessian_are_refused(shape):
    from htr_amd import encode
    H = torch.diag(torch.arange(128).float())
    with pytest.raises(IndexError):
        encode.prep_H(H, torch.ones(shape))
    with pytest.raises(IndexError):
        encode.prep_H(H[:1], torch.ones(6, 128))


def test_dead_columns_of_a_matrix_with_further_dimensions():
    from htr_amd import encode
    H = torch.diag((torch.arange(128) != 5).float())
    W = torch.ones(6, 128, 3)
    Hd, Wd = encode.prep_H(H, W, damp=0.0)
    assert torch.equal(Wd[:, 5], torch.zeros(6, 3)) and int((Wd == 0).sum()) == 18 and bool((W == 1).all())
    assert torch.equal(Hd, torch.eye(128, dtype=torch.float64))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(0,), (0, 128)])
def test_gpu_encoder_takes_matrices_without_rows(dev, rows):
    """A matrix of 0 rows, alone and beside another one: empty results, as on the CPU, and the other as by itself."""
    from htr_amd import encode
    print(f"encoder, matrices of {rows} rows", flush=True)
    g = torch.Generator().manual_seed(3)
    a = torch.randn(256, 128, generator=g)
    H = (a.T @ a / 256).to(dev)
    jobs = [dict(W=0.02 * torch.randn(m, 128, generator=g).to(dev), H=H) for m in rows]
    got = encode.encode_group(jobs, 4, seed=5)
    assert [tuple(r["qweight"].shape) for r in got] == [(m // 16, 8, 32) for m in rows] and got[0]["What"].shape == (0, 128)
    if len(rows) > 1:
        other = encode.encode_group([dict(W=jobs[0]["W"].new_zeros(128, 128), H=H), jobs[1]], 4, seed=5)[1]
        assert torch.equal(got[1]["qweight"], other["qweight"]) and torch.equal(got[1]["What"], other["What"])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
def test_dead_columns_by_masks_are_those_by_index(dtype):
    """What is not a number, infinite or a negative zero in a dead column as well, and a matrix that is a transposed view."""
    from htr_amd import encode
    g = torch.Generator().manual_seed(11)
    H = torch.randn(128, 128, generator=g)
    W = torch.randn(128, 6, generator=g).to(dtype).T
    for c, v in ((0, float("nan")), (7, -0.0), (127, float("inf"))):
        H[c, c] = 0
        W[2, c] = v
    Hd, Wd = encode.prep_H(H, W, damp=0.0)
    dead = torch.diag(H) == 0
    want_H, want_W = H.double(), W.clone()
    want_H[dead, dead] = 1.0
    want_W[:, dead] = 0
    assert torch.equal(Hd, want_H) and torch.equal(Wd, want_W) and Wd.dtype == dtype and Wd.stride() == want_W.stride()
    assert not torch.signbit(Wd[:, dead]).any() and bool(torch.isnan(W[2, 0]))
