"""The engine on small models built in memory, against the CPU oracle's forward and against
itself: the counterpart of x0ne-core/oracle/tests/gpu_engine.rs.

Bit for bit where the reference's own suite asks it: the same request twice, graph against
eager, the device's greedy tokens against the host's, the synthetic weights drawn on the device
against the oracle's generator. Within the model-level tolerance (logits within 0.05 of the row's
largest magnitude, KL <= 0.02, gpu_engine.rs:29-32) against the oracle, with the greedy tokens
equal to the oracle's up to the first position whose top-2 margin the tolerance could flip."""
import json

import numpy as np
import pytest

from common import (LOGITS_ATOL_OF_MAX, LOGITS_KL, O, reference_tensors, safetensors_bytes, tiny, top_two,
                    wide, worst_ratio)

pytestmark = pytest.mark.gpu


class Fixture:
    def __init__(self, cfg, seed):
        self.cfg = cfg
        self.tensors = reference_tensors(cfg, seed)
        self.file = safetensors_bytes(self.tensors)
        self.model = O.Model(cfg, weights_bf16=True)
        for name, (_, bits) in self.tensors.items():
            self.model.set(name, bits)

    def engine(self, max_ctx, page_seed=7, f64_sums=False):
        """The f32 path unless asked (these tests hold its kernels to the oracle's tolerances);
        f64_sums None gives the engine's default."""
        from x0ne_core import Engine, EngineOptions
        return Engine.load_from(self.cfg.to_json(), {"model.safetensors": self.file},
                                EngineOptions(max_ctx=max_ctx, page_seed=page_seed, f64_sums=f64_sums))

    def tokens(self, seed, n):
        return O.Rng(seed).tokens(n, self.cfg.vocab)


def assert_logits(what, got, want):
    scale = float(np.abs(want).max())
    atol = LOGITS_ATOL_OF_MAX * scale
    r, at = worst_ratio(got, want, atol, 0.0)
    kl = O.kl(want, got)
    exact = bool((np.asarray(got, np.float32).view(np.uint32) == np.asarray(want, np.float32).view(np.uint32)).all())
    print(f"MEASURE {what}: worst logit ratio {r:.5f} of {atol:.4f}, KL {kl:.3e}, bit-equal {exact}")
    assert r <= 1.0, f"{what}: logit {at}: got {got[at]} want {want[at]}"
    assert kl <= LOGITS_KL, f"{what}: KL {kl}"
    first, second = top_two(want)
    if first - second > 2 * atol:
        assert O.argmax(got) == O.argmax(want), f"{what}: argmax"


FIXTURES = [("1 layer 2/1", lambda: Fixture(tiny(1, 2, 1, False), 1)),
            ("2 layers 4/2", lambda: Fixture(tiny(2, 4, 2, False), 2)),
            ("3 layers 16/8 tied", lambda: Fixture(wide(), 3))]


@pytest.mark.parametrize("name,make", FIXTURES, ids=[f[0] for f in FIXTURES])
def test_every_route_gives_the_oracle_logits_at_every_position(name, make):
    from x0ne_core import DecodeMode, Route
    f = make()
    e = f.engine(256)
    ids = f.tokens(11, 40)
    want = f.model.logits(ids)
    positions = list(range(len(ids)))
    rows = {}
    for mode in [DecodeMode.GRAPH, DecodeMode.EAGER]:
        e.set_decode_mode(mode)
        for route in [Route.PREFILL, Route.DECODE]:
            got = e.logits_at(ids, positions, route)
            rows[(mode, route)] = got
            for p in positions:
                assert_logits(f"{name} {mode.name} {route.name} pos {p}", got[p], want[p])
            assert e.client_data_is_zero() and e.host_buffers_are_zero()
    # Graph and eager replay the same decode launches: the same bits (gpu_engine.rs:155-158). The
    # prefill passes (GEMMs over many rows) agree with them within the model tolerance.
    base = rows[(DecodeMode.GRAPH, Route.DECODE)]
    for p in positions:
        eager = rows[(DecodeMode.EAGER, Route.DECODE)][p]
        assert (eager.view(np.uint32) == base[p].view(np.uint32)).all(), f"{name} pos {p}: graph = eager"
        for mode in [DecodeMode.GRAPH, DecodeMode.EAGER]:
            assert_logits(f"{name} prefill against decode pos {p}", rows[(mode, Route.PREFILL)][p], base[p])
        assert (rows[(DecodeMode.GRAPH, Route.PREFILL)][p].view(np.uint32) ==
                rows[(DecodeMode.EAGER, Route.PREFILL)][p].view(np.uint32)).all(), f"{name} pos {p}: prefill twice"
    print(f"MEASURE {name}: {e.describe()}")


@pytest.mark.parametrize("chunk", [1 << 30, 16, 7])
@pytest.mark.parametrize("name,make", FIXTURES, ids=[f[0] for f in FIXTURES])
def test_the_exact_mode_prefill_passes_give_the_decode_steps_bits(name, make, chunk):
    """The exact mode's prefill passes (the f64-sum GEMM on the f64 matrix cores, the f64 causal
    attention) round where its decode step rounds and sum every product in f64, so a prompt's
    logits through passes of `chunk` rows are the decode route's bit for bit at every position,
    and both are the oracle's within the model tolerance; the greedy tokens agree."""
    from x0ne_core import Engine, EngineOptions, Route
    f = make()
    e = Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=96, page_seed=5, prefill_chunk=min(chunk, 96), f64_sums=True))
    assert e.exact() and f"prefill passes of {min(chunk, 96)} rows" in e.describe(), e.describe()
    ids = f.tokens(15, 50)
    want = f.model.logits(ids)
    every = list(range(len(ids)))
    passes = e.logits_at(ids, every, Route.PREFILL)
    steps = e.logits_at(ids, every, Route.DECODE)
    for p in every:
        assert_logits(f"{name} exact chunk {chunk} pos {p}", passes[p], want[p])
        assert (passes[p].view(np.uint32) == steps[p].view(np.uint32)).all(), \
            f"{name} exact chunk {chunk} pos {p}: the passes' logits differ from the decode steps'"
    g = e.greedy(ids[:45], 6)
    assert g.size == 6 and e.client_data_is_zero()
    want_g = [int(np.argmax(r)) for r in e.logits_at(np.concatenate([ids[:45], g[:-1]]), list(range(44, 50)),
                                                       Route.DECODE)]
    assert g.tolist() == want_g, f"{name} exact chunk {chunk}: greedy {g.tolist()} against {want_g}"
    e.close()


@pytest.mark.parametrize("chunk", [1 << 30, 16, 7])
def test_prefill_passes_across_chunk_boundaries_give_the_oracle_logits(chunk):
    """A prompt cut in passes of `chunk` rows (gpu_engine.rs:229-302): the logits at and around
    every boundary are the oracle's, and the first pass's rows equal those of that pass alone."""
    from x0ne_core import Engine, EngineOptions, Route
    f = Fixture(wide(), 6)
    e = Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=96, page_seed=5, prefill_chunk=min(chunk, 96), f64_sums=False))
    c = min(chunk, 96)
    assert f"prefill passes of {c} rows" in e.describe(), e.describe()
    ids = f.tokens(14, 50)
    want = f.model.logits(ids)
    keep = sorted(set(p for b in range(0, 50, c) for p in (b - 1, b, b + 1) if 0 <= p < 50) | {0, 49})
    got = e.logits_at(ids, keep, Route.PREFILL)
    for row, p in zip(got, keep):
        assert_logits(f"chunk {c} position {p}", row, want[p])
    first = [p for p in keep if p < min(c, 50)]
    alone = e.logits_at(ids[:min(c, 50)], first, Route.PREFILL)
    for row, one, p in zip(got, alone, first):
        assert (row.view(np.uint32) == one.view(np.uint32)).all(), f"chunk {c} position {p}: the first pass alone"
    g = e.greedy(ids[:45], 6)
    assert g.size == 6 and e.client_data_is_zero()


def test_the_same_request_twice_gives_the_same_bits():
    f = Fixture(wide(), 4)
    e = f.engine(128)
    ids = f.tokens(12, 30)
    a = e.logits_at(ids, [0, 15, 29])
    g1 = e.greedy(ids[:10], 20)
    b = e.logits_at(ids, [0, 15, 29])
    g2 = e.greedy(ids[:10], 20)
    for x, y in zip(a, b):
        assert (x.view(np.uint32) == y.view(np.uint32)).all()
    assert (g1 == g2).all()
    assert e.client_data_is_zero() and e.host_buffers_are_zero()


@pytest.mark.parametrize("which", [0, 1])
def test_greedy_on_the_device_is_greedy_on_the_host(which):
    from x0ne_core import FormatError, GREEDY_AHEAD_MAX
    f = [Fixture(tiny(2, 4, 2, False), 8), Fixture(wide(), 9)][which]
    e = f.engine(256)
    for prompt_len, n in [(1, 1), (1, 40), (17, 2), (30, 100), (150, 57)]:
        prompt = f.tokens(16 + prompt_len, prompt_len)
        engine = e.greedy(prompt, n)
        assert engine.size == n
        host = []
        s = e.session(prompt)
        for i in range(n):
            t = O.argmax(s.logits())
            host.append(t)
            if i + 1 < n:
                s.step(t)
        s.finish()
        assert host == engine.tolist(), f"prompt {prompt_len}, {n} tokens: host greedy against the engine's"
        for ahead in [1, 2, 3, GREEDY_AHEAD_MAX]:
            g = e.session(prompt).into_greedy_ahead(n, ahead)
            device = []
            for i in range(n):
                device.append(g.next_token())
                assert g.taken() == i + 1
                assert g.position() < prompt_len + n
                assert g.position() <= prompt_len + i + ahead
            with pytest.raises(FormatError):
                g.next_token()
            g.finish()
            assert device == engine.tolist(), f"{ahead} ahead"
            assert e.client_data_is_zero() and e.host_buffers_are_zero()
        # The oracle, until its choice is within the tolerance of another.
        f.model.reset()
        logits = f.model.extend(prompt)
        compared = 0
        for i, t in enumerate(engine):
            scale = float(np.abs(logits).max())
            first, second = top_two(logits)
            if first - second <= 2 * LOGITS_ATOL_OF_MAX * scale:
                break
            assert t == O.argmax(logits), f"prompt {prompt_len}: token {i} against the oracle"
            compared += 1
            if i + 1 < n:
                logits = f.model.step(int(t))
        print(f"MEASURE greedy prompt {prompt_len}: compared {compared} of {n} tokens with the oracle")


@pytest.mark.parametrize("q_heads,kv_heads", [(2, 2), (4, 2), (8, 2), (8, 1)])
@pytest.mark.parametrize("np_,batch,chunk", [(65, 5, 0), (77, 5, 176), (95, 2, 0), (96, 3, 192), (113, 4, 2048)])
def test_prompts_of_any_length_share_a_pass_and_keep_their_bits(q_heads, kv_heads, np_, batch, chunk):
    """Prompts of more than 64 ids go through a pass together, each sequence's rows at the next multiple
    of 16 (77 ids in passes of 176 rows: two at a time, the fifth alone), QK-norm + RoPE and the attention
    of all of them in one launch each: tokens and last logits are the bits each sequence gets alone."""
    from x0ne_core import Engine, EngineOptions
    f = Fixture(tiny(2, q_heads, kv_heads, False), 23)
    e = Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=128, page_seed=4, prefill_chunk=chunk, max_batch=5))
    prompts = np.stack([f.tokens(500 + b, np_) for b in range(batch)])
    toks, _, logits = e.greedy_batch(prompts, 4, logits=True)
    assert e.client_data_is_zero()
    for b in range(batch):
        t1, _, l1 = e.greedy_batch(prompts[b:b + 1], 4, logits=True)
        assert (t1[0] == toks[b]).all() and (l1[0].view(np.uint32) == logits[b].view(np.uint32)).all(), f"sequence {b}"


@pytest.mark.parametrize("which,np_,chunk", [(0, 21, 16), (1, 21, 16), (0, 80, 0), (1, 80, 0)])
def test_batched_greedy_is_each_sequence_alone_and_the_oracle(which, np_, chunk):
    """B independent prompts decoded together (the batched step: few-row GEMMs, one attention
    launch over every sequence's own pages): each sequence's tokens and last logits are the bits
    it gets alone or in another batch order, graph and eager alike; they are the oracle's greedy
    tokens until the oracle's top-2 margin is within the tolerance, and its logits within the
    model tolerance; and the client bytes are zeroed after. Prompts of 21 ids go in passes of 16
    rows, one sequence at a time; prompts of 80 ids (more than 64, a multiple of 16) share one
    prefill pass of 320 rows (the default pass size, min(2048, max_ctx x max_batch)), and alone
    take a pass of 80: the same bits either way."""
    from x0ne_core import DecodeMode, Engine, EngineOptions
    f = [Fixture(tiny(2, 4, 2, False), 21), Fixture(wide(), 22)][which]
    e = Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=128, page_seed=9, prefill_chunk=chunk, max_batch=4))
    B, n = 4, 30
    prompts = np.stack([f.tokens(300 + b, np_) for b in range(B)])
    toks, times, logits = e.greedy_batch(prompts, n, logits=True)
    assert toks.shape == (B, n) and (np.diff(times) >= 0).all()
    assert e.client_data_is_zero() and e.host_buffers_are_zero()
    order = [2, 0, 3, 1]
    t2, _, l2 = e.greedy_batch(prompts[order], n, logits=True)
    for i, b in enumerate(order):
        assert (t2[i] == toks[b]).all(), f"sequence {b} in another order"
        assert (l2[i].view(np.uint32) == logits[b].view(np.uint32)).all(), f"sequence {b} logits in another order"
    for b in [0, 3]:
        t1, _, l1 = e.greedy_batch(prompts[b:b + 1], n, logits=True)
        assert (t1[0] == toks[b]).all() and (l1[0].view(np.uint32) == logits[b].view(np.uint32)).all(), \
            f"sequence {b} alone"
    e.set_decode_mode(DecodeMode.EAGER)
    te, _, le = e.greedy_batch(prompts, n, logits=True)
    e.set_decode_mode(DecodeMode.GRAPH)
    assert (te == toks).all() and (le.view(np.uint32) == logits.view(np.uint32)).all(), "eager = graph"
    for b in range(B):
        f.model.reset()
        ol = f.model.extend(prompts[b])
        compared = 0
        for i in range(n):
            scale = float(np.abs(ol).max())
            first, second = top_two(ol)
            if first - second <= 2 * LOGITS_ATOL_OF_MAX * scale:
                break
            assert toks[b, i] == O.argmax(ol), f"sequence {b} token {i} against the oracle"
            compared += 1
            if i + 1 < n:
                ol = f.model.step(int(toks[b, i]))
        print(f"MEASURE batched greedy sequence {b}: compared {compared} of {n} tokens with the oracle")
        f.model.reset()
        want = f.model.logits(np.concatenate([prompts[b], toks[b, :-1]]))[-1]
        assert_logits(f"batched sequence {b} last logits", logits[b], want)
    assert e.client_data_is_zero() and e.host_buffers_are_zero()


def test_batched_greedy_refusals():
    from x0ne_core import Engine, EngineOptions, FormatError, NotImplementedFeature
    f = Fixture(tiny(1, 2, 1, False), 23)
    single = f.engine(64)
    with pytest.raises(NotImplementedFeature):
        single.greedy_batch(np.zeros((1, 3), np.uint32), 2)
    e = Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=64, page_seed=2, max_batch=2))
    with pytest.raises(FormatError):
        e.greedy_batch(np.zeros((3, 3), np.uint32), 2)  # above max_batch
    with pytest.raises(FormatError):
        e.greedy_batch(np.full((2, 3), f.cfg.vocab, np.uint32), 2)  # outside the vocabulary
    with pytest.raises(FormatError):
        e.greedy_batch(np.zeros((2, 60), np.uint32), 6)  # 60 + 6 - 1 > 64
    assert e.greedy_batch(np.zeros((2, 60), np.uint32), 5)[0].shape == (2, 5)
    with pytest.raises(NotImplementedFeature):
        Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                         EngineOptions(max_ctx=64, f64_sums=True, max_batch=2))
    assert e.client_data_is_zero() and e.host_buffers_are_zero()
    # The single-sequence paths still run on a batched engine (sequence 0's pages).
    g = e.greedy(f.tokens(5, 9), 7)
    assert (g == single.greedy(f.tokens(5, 9), 7)).all()


def test_session_refusals_and_scrub():
    from x0ne_core import FormatError
    f = Fixture(tiny(1, 2, 1, False), 5)
    e = f.engine(64)
    with pytest.raises(FormatError):
        e.session([])
    with pytest.raises(FormatError):
        e.session([f.cfg.vocab])
    with pytest.raises(FormatError):
        e.session(list(range(65)))
    s = e.session([1, 2, 3])
    with pytest.raises(FormatError):
        e.session([1])  # one session at a time
    with pytest.raises(FormatError):
        s.step(f.cfg.vocab)
    assert s.position() == 3
    s.step(4)
    assert s.position() == 4
    assert not e.client_data_is_zero()
    s.finish()
    assert e.client_data_is_zero() and e.host_buffers_are_zero()
    s = e.session(list(range(60)))
    for t in range(4):
        s.step(t)
    with pytest.raises(FormatError):
        s.step(1)  # max_ctx
    s.finish()
    with pytest.raises(FormatError):
        e.greedy(list(range(60)), 6)  # 60 + 6 - 1 > 64
    assert e.greedy(list(range(60)), 5).size == 5


def synthetic_config(layers=2, hidden=256, inter=512, q=4, kv=2, vocab=1000, tied=False):
    return tiny(layers, q, kv, tied, hidden=hidden, inter=inter, vocab=vocab, max_pos=4096)


def test_synthetic_weights_are_the_oracles_draws_bit_for_bit():
    """The device initialiser (init.hip) and the oracle's generator draw the same bf16 bits."""
    from x0ne_core import Engine, EngineOptions
    cfg = synthetic_config()
    e = Engine.load_synthetic(cfg.to_json(), 0, 0.02, EngineOptions(max_ctx=64))
    a = e.arena()
    slices = {}
    for label, _, sl in a.slices():
        slices.setdefault(label, []).append(sl)
    names = [n for n, _ in cfg.tensors()]
    sizes = dict(cfg.tensors())

    def draws(name):
        i = names.index(name)
        if name.endswith("norm.weight") or "layernorm" in name:
            return np.full(sizes[name], 0x3F80, np.uint16)
        return O.normal_bf16(O.tensor_key(0, i), 0, sizes[name], 0.02)

    def read(label, k):
        sl = slices[label][k]
        return a.read_array(sl, 0, sl.len // 2, np.uint16)

    got = read("embed", 0)
    assert (got == draws("model.embed_tokens.weight")).all(), "embedding"
    for l in range(cfg.layers):
        p = f"model.layers.{l}."
        qkv = np.concatenate([draws(p + "self_attn.q_proj.weight"), draws(p + "self_attn.k_proj.weight"),
                              draws(p + "self_attn.v_proj.weight")])
        assert (read("qkv", l) == qkv).all(), f"layer {l} qkv"
        assert (read("o", l) == draws(p + "self_attn.o_proj.weight")).all(), f"layer {l} o"
        gu = np.concatenate([draws(p + "mlp.gate_proj.weight"), draws(p + "mlp.up_proj.weight")])
        assert (read("gate_up", l) == gu).all(), f"layer {l} gate_up"
        assert (read("down", l) == draws(p + "mlp.down_proj.weight")).all(), f"layer {l} down"
        assert (read("input_norm", l) == 0x3F80).all() and (read("post_norm", l) == 0x3F80).all()
    assert (read("lm_head", 0) == draws("lm_head.weight")).all(), "lm_head"


def test_synthetic_greedy_against_the_oracle():
    """N(0, 0.02) weights drawn on both sides from seed 0: the device's greedy tokens against the
    oracle's, with the oracle's top-2 margins printed."""
    from x0ne_core import Engine, EngineOptions
    cfg = synthetic_config(layers=3, hidden=512, inter=1536, q=8, kv=4, vocab=4096)
    e = Engine.load_synthetic(cfg.to_json(), 0, 0.02, EngineOptions(max_ctx=256, page_seed=3))
    m = O.Model(cfg, weights_bf16=True)
    m.init_normal(0, 0.02)
    prompt = O.Rng(0).tokens(20, cfg.vocab)
    n = 64
    dev = e.greedy(prompt, n)
    want, margins = m.greedy(prompt, n)
    agree = 0
    for a, b in zip(dev, want):
        if a != b:
            break
        agree += 1
    print(f"MEASURE synthetic greedy: {agree} of {n} tokens equal to the oracle's; smallest margin "
          f"{margins[:max(agree, 1)].min():.3e}; first mismatch margin {margins[agree] if agree < n else None}")
    logits_dev = e.logits_at(np.concatenate([prompt, dev[:-1]]), [19, 40, 82])
    m.reset()
    full = m.logits(np.concatenate([prompt, dev[:-1]]))
    for p, row in zip([19, 40, 82], logits_dev):
        assert_logits(f"synthetic pos {p}", row, full[p])
    assert agree == n or margins[agree] < 2 * LOGITS_ATOL_OF_MAX * float(np.abs(full[19 + agree]).max())


def oracle_fixture(name):
    import os
    with open(os.path.join(os.path.dirname(__file__), "golden", f"oracle_greedy_{name}.json")) as fh:
        return json.load(fh)


def check_against_fixture(fx, f64, min_agree, max_ctx_extra=16):
    """Greedy tokens and teacher-forced logits of the synthetic engine against the oracle's
    fixture (tests/golden/make_oracle_greedy.py: per step the oracle's token, top-2 margin, row
    scale max|logit|, log-sum-exp and its 16 largest logits). Returns the agreement count."""
    from x0ne_core import Engine, EngineOptions, Route
    prompt = np.array(fx["prompt"], np.uint32)
    want = np.array(fx["tokens"], np.uint32)
    margins, scales = np.array(fx["margins"]), np.array(fx["scales"])
    n = want.size
    e = Engine.load_synthetic(fx["config"], fx["seed"], fx["std"],
                              EngineOptions(max_ctx=prompt.size + n + max_ctx_extra, page_seed=1, f64_sums=f64))
    if f64 is None:  # the default options: a dense engine of one sequence runs the exact mode
        assert e.exact(), e.describe()
        f64 = True
    assert e.exact() == f64
    got = e.greedy(prompt, n)
    agree = next((i for i in range(n) if got[i] != want[i]), n)
    mode = "f64" if f64 else "f32"
    # Teacher-forced on the oracle's tokens: the logits at every generated position.
    ids = np.concatenate([prompt, want[:-1]])
    at = list(range(prompt.size - 1, ids.size))
    rows = e.logits_at(ids, at, Route.DECODE)
    worst = worst_lse = 0.0
    flips = []
    for i, row in enumerate(rows):
        tol = LOGITS_ATOL_OF_MAX * scales[i]
        top = np.array(fx["top_ids"][i])
        err = float(np.abs(row[top].astype(np.float64) - np.array(fx["top_logits"][i])).max())
        lse = abs(O.logsumexp(row) - fx["logsumexp"][i])
        worst, worst_lse = max(worst, err / tol), max(worst_lse, lse / tol)
        if O.argmax(row) != int(want[i]):
            flips.append(i)
            # The reference's rule with this row's scale: only a choice within twice the
            # tolerance of the runner-up may go the other way (gpu_engine.rs:421-439).
            assert margins[i] < 2 * tol, f"{mode}: step {i} argmax differs at margin {margins[i]:.3e}"
        if f64:
            assert err <= 1e-5 * scales[i], f"f64 sums: step {i}: top logits {err:.3e} from the oracle's"
    if f64:  # the exact mode's prefill passes: the decode steps' bits
        passes = e.logits_at(ids, at, Route.PREFILL)
        for i, (row, row_p) in enumerate(zip(rows, passes)):
            assert (row.view(np.uint32) == row_p.view(np.uint32)).all(), f"f64 sums: step {i}: passes against steps"
    print(f"MEASURE {fx['what']}, {mode} sums: {agree} of {n} greedy tokens equal to the oracle's "
          f"(first mismatch margin {margins[agree] if agree < n else None}); teacher-forced: top-16 logits within "
          f"{worst:.3f} and log-sum-exp within {worst_lse:.3f} of the 0.05 x row-scale tolerance, argmax differs at "
          f"{flips}; {e.describe()}")
    assert worst <= 1.0 and worst_lse <= 1.0, mode
    assert agree >= min_agree, f"{mode}: {agree} tokens equal, fewer than {min_agree}"
    e.close()
    return agree


def test_qwen3_8b_greedy_is_the_oracle_fixture():
    """The bench workload itself (Qwen3-8B shape, N(0, 0.02) bf16 weights from seed 0, the
    20-token splitmix64 prompt) against the CPU oracle's 64 greedy steps
    (tests/golden/oracle_greedy_8b.json). The exact mode (f64 sums in the projections and
    attention) gives all 64 tokens and the oracle's top logits to 1e-5 of the row scale. The
    fp32 path: teacher-forced on the oracle's tokens its top-16 logits and log-sum-exp stay within
    the model tolerance (0.05 of each row's own scale) at all 64 positions, an argmax that differs
    does so only where the oracle's margin is within twice that tolerance, and its own greedy
    run agrees up to the first step whose oracle margin is within twice the tolerance (the
    reference's rule, gpu_engine.rs:421-437). 55 of the 64 margins are, the first at step 0, so
    the free run is held to no count: 19 equal on this build, 37 with the few-row GEMM's former
    summation order over the 20 prompt rows. The engine's default options (EngineOptions
    { max_ctx }, what the bench times) are the exact mode: all 64."""
    fx = oracle_fixture("8b")
    assert check_against_fixture(fx, None, 64) == 64
    tol2 = 2 * LOGITS_ATOL_OF_MAX * np.array(fx["scales"])
    first_tie = next((i for i, m in enumerate(fx["margins"]) if m < tol2[i]), len(fx["margins"]))
    check_against_fixture(fx, False, first_tie)


def test_qwen3_0_6b_greedy_is_the_oracle_fixture():
    """BASELINE config 1's shape (Qwen3-0.6B: 28 layers, hidden 1024, 16 q / 8 kv heads, tied
    embeddings) with the same synthetic weights and prompt: the exact mode gives the oracle's 64
    greedy tokens, the fp32 path its logits within the model tolerance (oracle_greedy_0_6b.json)."""
    fx = oracle_fixture("0_6b")
    assert check_against_fixture(fx, None, 64) == 64
    check_against_fixture(fx, False, 1)


def test_a_model_directory_loads_as_its_files_in_memory(tmp_path):
    """Engine::load (engine.rs:292-297) from a directory, single file and sharded over an index,
    gives the in-memory load's tokens and logits bit for bit."""
    from x0ne_core import Engine, EngineOptions, Route
    f = Fixture(wide(), 9)
    ids = f.tokens(21, 12)
    opts = EngineOptions(max_ctx=64, page_seed=3, f64_sums=False)
    e = f.engine(64, page_seed=3)
    want_tokens = e.greedy(ids, 8)
    want_logits = e.logits_at(ids, [11], Route.PREFILL)[0]
    e.close()
    single = tmp_path / "single"
    single.mkdir()
    (single / "config.json").write_text(json.dumps(f.cfg.to_json()))
    (single / "model.safetensors").write_bytes(f.file)
    names = list(f.tensors)
    half = len(names) // 2
    shards = tmp_path / "shards"
    shards.mkdir()
    (shards / "config.json").write_text(json.dumps(f.cfg.to_json()))
    (shards / "model-00001-of-00002.safetensors").write_bytes(
        safetensors_bytes({k: f.tensors[k] for k in names[:half]}))
    (shards / "model-00002-of-00002.safetensors").write_bytes(
        safetensors_bytes({k: f.tensors[k] for k in names[half:]}))
    wm = {k: ("model-00001-of-00002.safetensors" if i < half else "model-00002-of-00002.safetensors")
          for i, k in enumerate(names)}
    (shards / "model.safetensors.index.json").write_text(json.dumps({"metadata": {}, "weight_map": wm}))
    for d in (single, shards):
        e = Engine.load(str(d), opts)
        assert e.config["hidden_size"] == f.cfg.hidden
        got_tokens = e.greedy(ids, 8)
        got_logits = e.logits_at(ids, [11], Route.PREFILL)[0]
        e.close()
        assert list(got_tokens) == list(want_tokens), d.name
        assert (got_logits.view(np.uint32) == want_logits.view(np.uint32)).all(), d.name


def test_a_batched_engine_holds_its_weights_in_panels_too():
    """An engine for batches (max_batch > 1) keeps a second copy of every projection and of the
    LM head in 16-row panels, filled at load from the row-major copy: each is the host's panel
    layout of the row-major bits (gemm.hip, FEW_W_PANEL); an engine of one sequence has none."""
    from x0ne_core import Engine, EngineOptions
    from x0ne_core.ops import to_panels
    cfg = synthetic_config(vocab=1024, tied=True)
    e = Engine.load_synthetic(cfg.to_json(), 5, 0.02, EngineOptions(max_ctx=64, max_batch=2))
    assert "in 16-row panels" in e.describe(), e.describe()
    a = e.arena()
    slices = {}
    for label, _, sl in a.slices():
        slices.setdefault(label, []).append(sl)

    def read(label, k):
        sl = slices[label][k]
        return a.read_array(sl, 0, sl.len // 2, np.uint16)

    h, qkv_rows = cfg.hidden, (cfg.q_heads + 2 * cfg.kv_heads) * cfg.head_dim
    shapes = {"qkv": (qkv_rows, h), "o": (h, cfg.q_heads * cfg.head_dim), "gate_up": (2 * cfg.inter, h),
              "down": (h, cfg.inter)}
    for l in range(cfg.layers):
        for name, (rows, cols) in shapes.items():
            want = to_panels(read(name, l).reshape(rows, cols))
            assert (read(name + "_panel", l) == want).all(), f"layer {l} {name}"
    assert (read("lm_head_panel", 0) == to_panels(read("embed", 0).reshape(cfg.vocab, h))).all(), "tied head"
    e.close()
    one = Engine.load_synthetic(cfg.to_json(), 5, 0.02, EngineOptions(max_ctx=64))
    assert not any(label.endswith("_panel") for label, _, _ in one.arena().slices())



@pytest.mark.parametrize("route_name", ["PREFILL", "DECODE"])
def test_the_statistics_of_a_pass_are_those_of_its_logits_rows(route_name):
    """Engine::run / stats (engine.rs:928-1006, gpu_engine.rs:159-182): per position the argmax of
    the row (metrics::argmax), its log-sum-exp within 1e-4 relative and the next id's
    log-probability within 1e-3 (NaN at the last position); the rows run keeps are the bits
    logits_at gives; the client bytes are zero after; a kept position outside the ids is refused."""
    from x0ne_core import FormatError, Route
    f = Fixture(wide(), 31)
    e = f.engine(64, page_seed=4)
    route = getattr(Route, route_name)
    ids = f.tokens(41, 24)
    every = list(range(len(ids)))
    rows = e.logits_at(ids, every, route)
    stats, kept = e.run(ids, route, keep=[0, 7, 23])
    for k, p in enumerate([0, 7, 23]):
        assert (kept[k].view(np.uint32) == rows[p].view(np.uint32)).all(), f"run row {p}"
    assert np.array_equal(e.stats(ids, route).view(np.uint32), stats.view(np.uint32)), "stats is run without rows"
    for p, s in enumerate(stats):
        row = rows[p].astype(np.float64)
        assert int(s["argmax"]) == O.argmax(rows[p]), f"argmax at {p}"
        lse = O.logsumexp(rows[p])
        assert abs(float(s["logsumexp"]) - lse) <= 1e-4 * max(abs(lse), 1.0), f"log-sum-exp at {p}"
        if p + 1 < len(ids):
            assert abs(float(s["next_logprob"]) - (row[ids[p + 1]] - lse)) <= 1e-3, f"log-probability at {p}"
        else:
            assert np.isnan(s["next_logprob"])
    assert e.client_data_is_zero()
    with pytest.raises(FormatError):
        e.run(ids, route, keep=[len(ids)])


def moe_of_dense(f, experts: int, top_k: int, router_bits=None):
    """The Qwen3-MoE checkpoint and config whose every expert is the dense fixture's MLP: the same
    attention, norms and vocabulary, mlp.experts.e.* = mlp.*, the router `router_bits` (zeros:
    every logit equal, so the routing takes experts 0 .. top_k - 1 at equal weights)."""
    cfg = f.cfg.to_json()
    cfg.update({"model_type": "qwen3_moe", "decoder_sparse_step": 1, "norm_topk_prob": True,
                "num_experts": experts, "num_experts_per_tok": top_k, "moe_intermediate_size": f.cfg.inter,
                "mlp_only_layers": []})
    out = {k: v for k, v in f.tensors.items() if ".mlp." not in k}
    h = f.cfg.hidden
    for l in range(f.cfg.layers):
        p = f"model.layers.{l}.mlp."
        out[p + "gate.weight"] = ((experts, h), np.zeros(experts * h, np.uint16) if router_bits is None
                                  else router_bits[l])
        for e in range(experts):
            for leaf in ("gate_proj", "up_proj", "down_proj"):
                out[f"{p}experts.{e}.{leaf}.weight"] = f.tensors[p + leaf + ".weight"]
    return json.dumps(cfg), safetensors_bytes(out)


@pytest.mark.parametrize("experts,top_k", [(1, 1), (2, 2)])
def test_a_moe_of_identical_experts_is_the_dense_model(experts, top_k):
    """A Qwen3-MoE engine (router GEMV, routing, expert GEMVs through the device-held ids, SwiGLU,
    f32 down rows, weighted combination) whose experts all equal the dense MLP: top-1 weighs its
    expert exactly 1, and two experts with equal router logits route to [0, 1] at 0.5 each, so
    the combination is exact; the logits are the dense oracle's within the model tolerance
    (gpu_engine.rs:29-32) at every position, and its very bits in the exact mode (a MoE engine's
    default, f64 sums as the oracle's), graph and eager give the same bits, the routing
    diagnostic reads [0 .. top_k) at every layer and position, and the client bytes are zeroed."""
    from x0ne_core import DecodeMode, Engine, EngineOptions, Route
    f = Fixture(wide(), 41)
    text, file = moe_of_dense(f, experts, top_k)
    e = Engine.load_from(text, {"model.safetensors": file}, EngineOptions(max_ctx=64, page_seed=6))
    assert "MoE, %d experts" % experts in e.describe(), e.describe()
    ids = f.tokens(42, 20)
    want = f.model.logits(ids)
    at = [0, 5, 11, 19]
    graph = e.logits_at(ids, at, Route.DECODE)
    assert e.exact(), e.describe()
    for row, p in zip(graph, at):
        assert_logits(f"moe {experts}/{top_k} position {p}", row, want[p])
        assert (row.view(np.uint32) == want[p].view(np.uint32)).all(), f"moe position {p}: the oracle's bits"
    e.set_decode_mode(DecodeMode.EAGER)
    eager = e.logits_at(ids, at, Route.DECODE)
    for a, b, p in zip(graph, eager, at):
        assert (a.view(np.uint32) == b.view(np.uint32)).all(), f"graph and eager at {p}"
    e.set_decode_mode(DecodeMode.GRAPH)
    route = e.moe_routing(ids[:6]).reshape(6, f.cfg.layers, top_k)
    assert (route == np.arange(top_k, dtype=np.uint32)).all(), route
    dev = e.greedy(ids[:12], 8)
    f.model.reset()
    oracle, margins = f.model.greedy(ids[:12], 8)
    agree = int(np.argmin(np.append(dev == oracle, False)))
    if agree < 8:
        full = f.model.logits(np.concatenate([ids[:12], oracle[:-1]]))
        assert margins[agree] < 2 * LOGITS_ATOL_OF_MAX * float(np.abs(full[11 + agree]).max())
    assert e.client_data_is_zero()


class HostMoe:
    """The MoE decode step composed on the host from the oracle's kernels (oracle/src/lib.rs): the
    dense step of model.rs:196-262 with each layer's MLP replaced as engine.rs:795-815 does it:
    router GEMV (f32 logits) -> moe_route -> expert [gate; up] GEMVs (bf16) -> SwiGLU (bf16) ->
    expert down GEMVs (f32) -> the weighted combination (bf16)."""

    def __init__(self, cfg, experts, top_k, mi, tensors):
        self.c, self.E, self.K, self.mi = cfg, experts, top_k, mi
        self.W = {k: O.bf16_values(b).astype(np.float32) for k, (_, b) in tensors.items()}
        self.inv = O.inv_freq_f32(cfg.head_dim, cfg.theta)

    def layer(self, l, leaf):
        return self.W[f"model.layers.{l}.{leaf}.weight"]

    def run(self, ids):
        c, hd = self.c, self.c.head_dim
        qd, kvd, h = c.q_heads * hd, c.kv_heads * hd, c.hidden
        K = [[] for _ in range(c.layers)]
        V = [[] for _ in range(c.layers)]
        rows, routes, router_logits = [], [], []
        for pos, tok in enumerate(ids):
            residual = np.zeros(h, np.float32)
            delta = O.embedding(self.W["model.embed_tokens.weight"], h, int(tok))
            route_p, logit_p = [], []
            for l in range(c.layers):
                residual, x = O.add_rmsnorm(residual, delta, self.layer(l, "input_layernorm"), c.eps)
                x = O.bf16_round(x)
                wqkv = np.concatenate([self.layer(l, "self_attn.q_proj"), self.layer(l, "self_attn.k_proj"),
                                       self.layer(l, "self_attn.v_proj")])
                qkv = O.bf16_round(O.gemv(wqkv, qd + 2 * kvd, h, x))
                q, k, v = O.qk_norm_rope(qkv, self.layer(l, "self_attn.q_norm"), self.layer(l, "self_attn.k_norm"),
                                         self.inv, c.q_heads, c.kv_heads, hd, pos, c.eps)
                K[l].append(O.bf16_round(k))
                V[l].append(v)
                attn = O.bf16_round(O.attention_decode(O.bf16_round(q), np.concatenate(K[l]), np.concatenate(V[l]),
                                                       pos + 1, c.q_heads, c.kv_heads))
                delta = O.bf16_round(O.gemv(self.layer(l, "self_attn.o_proj"), h, qd, attn))
                residual, x = O.add_rmsnorm(residual, delta, self.layer(l, "post_attention_layernorm"), c.eps)
                x = O.bf16_round(x)
                lg = O.gemv(self.W[f"model.layers.{l}.mlp.gate.weight"], self.E, h, x)
                eids, wts = O.moe_route(lg, self.E, self.K)
                gu_all = np.concatenate([np.concatenate([self.W[f"model.layers.{l}.mlp.experts.{e}.gate_proj.weight"],
                                                         self.W[f"model.layers.{l}.mlp.experts.{e}.up_proj.weight"]])
                                         for e in range(self.E)])
                gu = O.bf16_round(O.moe_gemv(gu_all, self.E, 2 * self.mi, h, eids, x, self.K))
                act = O.bf16_round(np.concatenate([O.swiglu(gu[s * 2 * self.mi:(s + 1) * 2 * self.mi])
                                                   for s in range(self.K)]))
                d_all = np.concatenate([self.W[f"model.layers.{l}.mlp.experts.{e}.down_proj.weight"]
                                        for e in range(self.E)])
                y = O.moe_gemv(d_all, self.E, h, self.mi, eids, act, 1)
                delta = O.bf16_round(O.moe_combine(y, wts, h, self.K))
                route_p.append(eids)
                logit_p.append(lg)
            residual, x = O.add_rmsnorm(residual, delta, self.W["model.norm.weight"], c.eps)
            head = self.W["model.embed_tokens.weight"] if c.tied else self.W["lm_head.weight"]
            rows.append(O.gemv(head, c.vocab, h, O.bf16_round(x)))
            routes.append(np.stack(route_p))
            router_logits.append(np.stack(logit_p))
        return rows, np.stack(routes), router_logits


def test_a_random_moe_routes_each_token_to_distinct_experts():
    """Eight experts of their own, two per token, a random router, against the MoE step composed
    from the oracle's kernels (HostMoe): the engine's routing at every layer and position is the
    host's (a differing pick only where the host's two router logits are within the GEMV
    tolerance of each other, the comparison ending there), its logits within the model tolerance
    at every position; the step is the same bits graph and eager and over repeated requests;
    greedy decoding runs through the captured graph; a dense engine has no routing to report."""
    from x0ne_core import DecodeMode, Engine, EngineOptions, Route
    f = Fixture(tiny(2, 4, 2, False), 43)
    g = np.random.default_rng(44)
    text, _ = moe_of_dense(f, 8, 2)
    cfg = json.loads(text)
    cfg["moe_intermediate_size"] = 64
    out = {k: v for k, v in f.tensors.items() if ".mlp." not in k}
    h = f.cfg.hidden

    def bits(*shape):
        vals = g.normal(0, 0.1, size=int(np.prod(shape))).astype(np.float32)
        return shape, (vals.view(np.uint32) >> 16).astype(np.uint16)

    for l in range(f.cfg.layers):
        p = f"model.layers.{l}.mlp."
        out[p + "gate.weight"] = bits(8, h)
        for x in range(8):
            out[f"{p}experts.{x}.gate_proj.weight"] = bits(64, h)
            out[f"{p}experts.{x}.up_proj.weight"] = bits(64, h)
            out[f"{p}experts.{x}.down_proj.weight"] = bits(h, 64)
    e = Engine.load_from(json.dumps(cfg), {"model.safetensors": safetensors_bytes(out)},
                         EngineOptions(max_ctx=64, page_seed=2))
    ids = f.tokens(45, 16)
    route = e.moe_routing(ids).reshape(16, f.cfg.layers, 2)
    assert (route < 8).all() and (route[..., 0] != route[..., 1]).all()
    assert len(set(route.reshape(-1).tolist())) > 2, "the router spreads the tokens"
    want_rows, want_route, router_logits = HostMoe(f.cfg, 8, 2, 64, out).run(ids)
    upto = len(ids)
    for p in range(len(ids)):
        for l in range(f.cfg.layers):
            if (route[p, l] != want_route[p, l]).any():
                lg = router_logits[p][l]
                picked = sorted(set(route[p, l].tolist()) ^ set(want_route[p, l].tolist()))
                gap = abs(float(lg[picked[0]]) - float(lg[picked[-1]]))
                assert gap <= 1e-3 * float(np.abs(lg).max()), f"position {p} layer {l}: routing differs at gap {gap}"
                upto = min(upto, p)
    rows = e.logits_at(ids, list(range(upto)), Route.DECODE)
    for p in range(upto):
        assert_logits(f"random moe position {p}", rows[p], want_rows[p])
    same = sum(int((rows[p].view(np.uint32) == want_rows[p].view(np.uint32)).all()) for p in range(upto))
    print(f"MEASURE random MoE: routing equal to the host's at {upto} of {len(ids)} positions, logits compared "
          f"there, {same} of them bit-equal")
    assert upto >= 8
    # A MoE engine sums in f64 by default, as the oracle's kernels do: the same routing and bits.
    assert e.exact() and upto == len(ids) and same == upto
    a = e.logits_at(ids, [3, 15], Route.DECODE)
    b = e.logits_at(ids, [3, 15], Route.DECODE)
    e.set_decode_mode(DecodeMode.EAGER)
    c = e.logits_at(ids, [3, 15], Route.DECODE)
    e.set_decode_mode(DecodeMode.GRAPH)
    for x, y, z in zip(a, b, c):
        assert (x.view(np.uint32) == y.view(np.uint32)).all() and (x.view(np.uint32) == z.view(np.uint32)).all()
        assert np.isfinite(x).all()
    assert e.greedy(ids[:10], 6).size == 6 and e.client_data_is_zero()
    dense = f.engine(64)
    assert dense.moe_routing(ids).size == 0


@pytest.mark.parametrize("which", [0, 1])
def test_the_decode_attention_kernels_agree_inside_the_engine(which):
    """gpu_engine.rs:722-769: the per-head kernel and split-K agree within the model tolerance
    against the oracle and each other at positions around the 64- and 256-key tile edges; the
    merge kernel and the last-block merge give the same bits; switching back gives the first
    bits again. A switch re-captures the graph and leaves the client bytes zeroed; it is refused
    while a session is open, and the last-block merge is refused without a grouped kernel."""
    from x0ne_core import DecodeAttention, FormatError, GpuError, SplitMerge
    f = [Fixture(tiny(2, 4, 2, False), 14), Fixture(wide(), 15)][which]
    e = f.engine(700)
    ids = f.tokens(25, 520)
    keep = [0, 63, 64, 127, 128, 129, 255, 256, 300, 519]
    want = f.model.logits(ids)
    assert e.decode_attention() == DecodeAttention.SPLIT_K
    assert e.split_merge() == SplitMerge.LAST_BLOCK
    split = e.logits_at(ids, keep)
    e.set_decode_attention(DecodeAttention.PER_HEAD)
    assert e.client_data_is_zero() and "per head" in e.describe()
    per_head = e.logits_at(ids, keep)
    e.set_decode_attention(DecodeAttention.SPLIT_K)
    for a, b, p in zip(split, per_head, keep):
        assert_logits(f"split-K at {p}", a, want[p])
        assert_logits(f"per-head at {p}", b, want[p])
        assert_logits(f"split-K against per-head at {p}", a, b)
    e.set_split_merge(SplitMerge.KERNEL)
    assert "merge Kernel" in e.describe()
    kernel_merge = e.logits_at(ids, keep)
    for a, b, p in zip(split, kernel_merge, keep):
        assert (a.view(np.uint32) == b.view(np.uint32)).all(), f"the two merges differ at {p}"
    e.set_split_merge(SplitMerge.LAST_BLOCK)
    again = e.logits_at(ids, keep)
    for a, b, p in zip(split, again, keep):
        assert (a.view(np.uint32) == b.view(np.uint32)).all(), f"split-K again at {p}"
    print(f"MEASURE P = {e.splits()}, {e.describe()}")
    s = e.session(ids[:5])
    with pytest.raises(FormatError):
        e.set_decode_attention(DecodeAttention.PER_HEAD)
    with pytest.raises(FormatError):
        e.set_split_merge(SplitMerge.KERNEL)
    # A refused change leaves every piece of state as it was: the getters, the description and
    # the graph (the session still decodes with the split-K kernel's bits).
    assert e.decode_attention() == DecodeAttention.SPLIT_K
    assert e.split_merge() == SplitMerge.LAST_BLOCK
    assert "merge LastBlock" in e.describe()
    s.finish()
    # Between requests the same change is taken and captured again.
    e.set_decode_attention(DecodeAttention.PER_HEAD)
    assert e.decode_attention() == DecodeAttention.PER_HEAD
    again_per_head = e.logits_at(ids, keep)
    for a, b, p in zip(per_head, again_per_head, keep):
        assert (a.view(np.uint32) == b.view(np.uint32)).all(), f"per-head after a refused change at {p}"
    e.set_decode_attention(DecodeAttention.SPLIT_K)
    ex = Engine_exact(f)
    from x0ne_core import NotImplementedFeature
    with pytest.raises(NotImplementedFeature):
        ex.set_decode_attention(DecodeAttention.PER_HEAD)
    with pytest.raises(NotImplementedFeature):
        ex.set_split_merge(SplitMerge.KERNEL)
    ungrouped = Fixture(tiny(1, 3, 1, False), 16)
    u = ungrouped.engine(64)
    with pytest.raises(GpuError):
        u.set_split_merge(SplitMerge.LAST_BLOCK)
    assert u.split_merge() == SplitMerge.KERNEL


def Engine_exact(f):
    from x0ne_core import Engine, EngineOptions
    return Engine.load_from(f.cfg.to_json(), {"model.safetensors": f.file},
                            EngineOptions(max_ctx=64, page_seed=3, f64_sums=True))
