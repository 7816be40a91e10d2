"""GPT-2 124M chunked prefill + greedy generation on the GPU vs the transformers oracle, mirroring the reference's
build_generate tests (tests/models/test_gpt2.py:64-106): one prefill call then one call per token must match HF
generate token for token; every chunk's last-row logits (chunks at pos > 0, longer than a 32-query block, not
aligned, interleaved with decode steps) match HF's full forward within max rel err 1e-4."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(gpu):
    from lokinfer_amd import gpt2 as G
    from oracle import gpt2 as O

    sd = G.random_weights()
    return G, O, sd, O.model(sd)


def rel(got, exp):
    return np.abs(got - exp).max() / np.abs(exp).max()


def test_prefill_logits_and_generate(setup):
    G, O, sd, m = setup
    model = G.Gpt2Generator(sd)
    got = model(O.GEN_PROMPT, 0)
    assert rel(got, O.last_logits(m, O.GEN_PROMPT)) <= 1e-4
    hf = O.greedy(m, O.GEN_PROMPT, 32)
    assert G.generate(G.Gpt2Generator(sd), O.GEN_PROMPT, 32) == hf  # fresh caches
    # the reference op sequence for the decode steps (fused=False) generates the same tokens
    assert G.generate(G.Gpt2Generator(sd, fused=False, sk=(0, 0)), O.GEN_PROMPT, 8) == hf[:8]


def test_two_chunk_prefill(setup):
    G, O, sd, m = setup
    model = G.Gpt2Generator(sd)
    p = O.GEN_PROMPT
    model(p[:6], 0)
    assert rel(model(p[6:], 6), O.last_logits(m, p)) <= 1e-4


def test_multi_chunk_prefill(setup):
    G, O, sd, m = setup
    model = G.Gpt2Generator(sd)
    ids = np.random.default_rng(3).integers(0, G.VOCAB, 300).astype(np.int64)
    pos = 0
    for n in (40, 70, 1, 117, 1, 71):
        got = model(ids[pos:pos + n], pos)
        pos += n
        assert rel(got, O.last_logits(m, ids[:pos])) <= 1e-4, (pos, n)


def test_prefill_512_then_decode(setup):
    """The decode benchmark's configuration reached through one 512-token prefill chunk instead of 512 steps: the
    step at pos 512 matches the oracle's decode step and its argmax."""
    G, O, sd, m = setup
    ids, nxt = O.decode_inputs()
    ref, _ = O.decode_step(m, O.prefill(m, ids), nxt)
    model = G.Gpt2Generator(sd)
    model.prefill(ids)
    got = model([nxt], 512)[0]
    assert rel(got, ref) <= 1e-4
    assert int(np.argmax(got)) == int(np.argmax(ref))


def test_chunk_graph_equals_eager(setup):
    G, O, sd, m = setup
    a, b = G.Gpt2Generator(sd), G.Gpt2Generator(sd, chunk_graph=True)
    ids = np.random.default_rng(5).integers(0, G.VOCAB, 96).astype(np.int64)
    for pos in (0, 32, 64):  # the same T three times: graph capture, then replays
        la, lb = a(ids[pos:pos + 32], pos), b(ids[pos:pos + 32], pos)
        assert np.array_equal(la, lb), pos


def test_generate_to_cache_capacity(setup):
    """A 1000-token prompt in one chunk, then decode steps up to position 1023 (the last cache row; 16 decode chunks
    and 32 key tiles of the cache attention): every step's logits match HF's full forward over the tokens so far."""
    G, O, sd, m = setup
    model = G.Gpt2Generator(sd)
    ids = np.random.default_rng(9).integers(0, G.VOCAB, 1024).astype(np.int64)
    got = model(ids[:1000], 0)
    assert rel(got, O.last_logits(m, ids[:1000])) <= 1e-4
    for pos in (1000, 1001, 1023):
        if pos > 1001:
            for p in range(1002, pos):
                model(ids[p:p + 1], p)
        got = model(ids[pos:pos + 1], pos)
        assert rel(got, O.last_logits(m, ids[:pos + 1])) <= 1e-4, pos
    with pytest.raises(ValueError):
        model(ids[:2], 1023)  # past the cache: refused on the host


def test_capture_with_collectable_models(setup):
    """Regression: models hold their compiled function and it holds them back, so only the cycle collector frees
    them, and a collection during a graph capture destroyed their captured graphs mid-capture. Unreachable models
    are left behind and the collector is made to run on (nearly) every allocation while a new model captures; the
    capture must succeed and give the eager logits."""
    import gc

    G, O, sd, m = setup
    for _ in range(2):
        d = G.Gpt2Generator(sd)
        d([5, 6, 7], 0)
        d([8], 3)  # captures the decode graph
        del d  # now only reachable through its own cycle
    old = gc.get_threshold()
    gc.set_threshold(1)
    try:
        a = G.Gpt2Generator(sd, graph=True)
        a([5, 6, 7], 0)
        la = a([8], 3)
    finally:
        gc.set_threshold(*old)
    assert gc.isenabled()
    b = G.Gpt2Generator(sd, graph=False)
    b([5, 6, 7], 0)
    assert np.array_equal(la, b([8], 3))


@pytest.mark.parametrize("chunk_graph", [False, True])
def test_chunks_follow_written_weights(setup, chunk_graph):
    """The prompt chunk runs on the weights as they are, like the decode step: after an in-place write its logits are a
    fresh model's, and after a second one, and when a weight's tensor was replaced."""
    import torch

    G, O, sd, m = setup
    ids = np.random.default_rng(6).integers(0, G.VOCAB, 90).astype(np.int64)
    model = G.Gpt2Generator(sd, chunk_graph=chunk_graph)
    first = model(ids, 0)
    new, fc, proj = dict(sd), "transformer.h.3.mlp.c_fc.weight", "transformer.h.0.attn.c_attn.weight"
    for step in range(3):
        for k, f in ((fc, 1.5), (proj, -0.5)):
            new[k] = new[k] * np.float32(f)
            if step == 0:
                model.w[k].t.mul_(f)
            elif step == 1:
                with torch.inference_mode():
                    model.w[k].t.copy_(torch.from_numpy(new[k]))
            elif not chunk_graph:
                model.w[k] = type(model.w[k])(torch.from_numpy(new[k]).to(model.w[k].t.device))
            else:
                model.w[k].t.data.copy_(torch.from_numpy(new[k]))
                model.split_weights()
        got = model(ids, 0)
        assert np.array_equal(got, G.Gpt2Generator(new)(ids, 0)) and not np.array_equal(got, first)


def test_chunks_follow_swapped_memory(setup):
    """A weight whose tensor was given other memory (`.data = x`, which torch does not count as a write)."""
    import torch

    G, O, sd, m = setup
    ids = np.random.default_rng(7).integers(0, G.VOCAB, 40).astype(np.int64)
    model, new, k = G.Gpt2Generator(sd), dict(sd), "transformer.h.5.mlp.c_proj.weight"
    first = model(ids, 0)
    new[k] = new[k] * np.float32(1.5)
    model.w[k].t.data = torch.from_numpy(new[k]).to(model.w[k].t.device)
    got = model(ids, 0)
    assert np.array_equal(got, G.Gpt2Generator(new)(ids, 0)) and not np.array_equal(got, first)


def test_split_weights_ready_on_any_stream(setup, monkeypatch):
    """A model built on one stream, where laying a weight out takes long, runs at once on another."""
    import torch

    G, O, sd, m = setup
    ids = np.random.default_rng(8).integers(0, G.VOCAB, 40).astype(np.int64)
    want = G.Gpt2Generator(sd)(ids, 0)
    lay = G.ops.split_weight

    def late(*a, **kw):
        torch.cuda._sleep(20_000_000)  # some 10 ms on the device
        return lay(*a, **kw)

    monkeypatch.setattr(G.ops, "split_weight", late)
    with torch.cuda.stream(torch.cuda.Stream()):
        model = G.Gpt2Generator(sd)
    with torch.cuda.stream(torch.cuda.Stream()):
        assert np.array_equal(model(ids, 0), want)


@pytest.mark.parametrize("sk", [(5, 4), (2, 7), (-1, 4), (2, -4)])
def test_refuses_split_factors(setup, sk):
    """Split-K factors that do not divide K into multiples of 16 are refused at every chunk length."""
    G, O, sd, m = setup
    model = G.Gpt2Generator(sd, sk=sk)
    for t in (2, 40, 700):
        with pytest.raises(G.ops.OpError):
            model(np.zeros(t, np.int64), 0)
