"""Two portions inside prompts as one iteration (MK_CFG_PAIR_PORTIONS): the same logits, tokens, caches, states and scheduler tensors, bit by
bit, as portions one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _any_pair(monkeypatch):
    """Offline launches begin with pairs where there is one, however little these small models gain by it."""
    monkeypatch.setenv("FLEET_MK_PAIRS_WORTH", "1")


# linears that run for both portions at once: split in slices and left to the stage behind or summed by the last to arrive, whole, in ranges of
# four to six tiles; and such that do not (reductions that are no multiple of 512 slices)
SHAPES = {
    "wide": dict(hidden_size=4096, num_q_heads=32, num_kv_heads=8, intermediate_size=1536),
    "mixed": dict(hidden_size=2048, num_q_heads=24, num_kv_heads=6, intermediate_size=6144),
    "long": dict(hidden_size=2048, num_q_heads=16, num_kv_heads=2, intermediate_size=12288),
    "narrow": dict(hidden_size=1024, num_q_heads=32, num_kv_heads=4, intermediate_size=6144),
    "experts": dict(hidden_size=2048, num_q_heads=32, num_kv_heads=4, intermediate_size=0, num_experts=16, num_experts_per_tok=4, moe_intermediate_size=768),
}


@pytest.mark.parametrize("name,lengths,B,portion,steps", [
    ("wide", (64 * 4 + 7,), 64, 64, 100), ("wide", (64 * 5,), 64, 64, 3), ("wide", (129, 200, 65), 64, 64, 100), ("wide", (150, 90, 33), 64, 20, 7), ("mixed", (64 * 3 + 1,), 64, 64, 100),
    ("mixed", (180, 75), 40, 40, 100), ("long", (64 * 4 + 63,), 64, 64, 2), ("experts", (64 * 4 + 30,), 64, 64, 100), ("wide", (64, 65), 33, 33, 100)])
def test_offline(name, lengths, B, portion, steps):
    _offline(name, lengths, B, portion, steps, len(lengths))


@pytest.mark.parametrize("R,steps", [(1, 100), (1, 3), (1, 5), (2, 100)])
def test_requests_that_wait(R, steps):
    """Prompts that begin when others have been answered: behind the first iteration that is not of two portions, and where a launch begins."""
    _offline("wide", (200, 150, 300), 64, 64, steps, R)


@pytest.mark.parametrize("workgroups,name,B", [(32, "wide", 64), (48, "wide", 64), (32, "mixed", 40), (48, "narrow", 64)])
def test_grids_smaller_than_a_portion(workgroups, name, B):
    """Rows of the second portion start again at the first workgroup; "narrow": where a linear left its sum to them."""
    _offline(name, (B * 4 + 7, 70), B, B, 100, 2, num_workers=workgroups)


def _offline(name, lengths, B, portion, steps, R, **kw):
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    shape = Qwen3Shape(head_dim=128, num_layers=2, vocab_size=512, **SHAPES[name])
    g = torch.Generator().manual_seed(5)
    prompts = [torch.randint(0, 512, (n,), generator=g) for n in lengths]
    w, max_seq, outs = random_weights(shape, seed=2), max(lengths) + 6, []
    for pairs in (True, False):
        dec = Qwen3Decoder(shape, w, max_num_batched_tokens=B, max_num_batched_requests=R, max_seq_length=max_seq, page_size=16, eos_token_id=0x7FFFFFFF, max_tokens_per_request=portion,
                           pair_portions=pairs, total_requests=len(lengths), **kw)
        assert dec.mpk.stats()["paired_portions"] == pairs
        dec.load_prompts(prompts)
        out, fin = [], False
        while not fin:
            fin = dec.mpk.run_steps(steps)
            # (rows behind the last iteration's tokens are of older ones)
            out += [dec.logits().clone(), torch.tensor(dec.mpk.stats()["iterations"])] + [v.clone() for k, v in dec.meta.items() if k != "input_tokens"]
        out += [dec.k_cache.clone(), dec.v_cache.clone()]
        outs.append([t.cpu() for t in out])
        dec.mpk.finalize()
    assert len(outs[0]) == len(outs[1]) and all(torch.equal(a, b) for a, b in zip(*outs))


def _model(family):
    import generate
    make, sizes = generate.SHAPES[family + "-2k"]
    torch.manual_seed(7)
    return generate.random_model(make(**sizes, layers={"suborax": 2, "dodonex": 4, "bukatar": 4, "vizonex": 4}[family], vocab=1000, **({"positions": 512} if family == "vizonex" else {})))[0]


def _kept(builder):
    """What the iterations of a layer-list model leave for later ones: caches, states and rings, and the batch slots' state slots."""
    for name in ("k_cache", "v_cache", "latent_cache", "state", "tail", "canon", "state_slots"):
        held = getattr(builder, name, None)
        for t in held.values() if isinstance(held, dict) else held if isinstance(held, list) else [] if held is None else [held]:
            yield t


@pytest.mark.parametrize("family", ["suborax", "dodonex", "bukatar", "vizonex"])
@pytest.mark.parametrize("lengths,R,portion,steps", [((64 * 4 + 7, 64 * 3), 1, 64, 100), ((200, 150, 33), 3, 30, 5), ((90,) * 40, 34, 64, 100)])
def test_offline_families(family, lengths, R, portion, steps):
    """The scheduler's pairs in the other kernels, and what goes on behind them: states that move between slots, scans, rings, experts; a batch
    of more requests than a portion has rows for."""
    import generate
    model = _model(family)
    g = torch.Generator().manual_seed(6)
    prompts = [torch.randint(0, 1000, (n,), generator=g) for n in lengths]
    max_seq, outs = max(lengths) + 6, []
    for pairs in (True, False):
        gen = generate.Generator(max_seq, model_config=model, batch=R, max_num_batched_tokens=64, max_tokens_per_request=portion, page_size=64, total_requests=len(lengths), eos_token_id=-1,
                                 pair_portions=pairs)
        assert gen.mpk.stats()["paired_portions"] == pairs
        gen.load_prompts(prompts)
        out, fin = [], False
        while not fin:
            fin = gen.mpk.run_steps(steps)
            out += [gen.logits().clone(), torch.tensor(gen.mpk.stats()["iterations"])] + [v.clone() for k, v in gen.meta.items() if k != "input_tokens"]
        kept = [t.clone() for t in _kept(gen.model.model_builder)]
        out += kept
        outs.append([t.cpu() for t in out])
        gen.finalize()
    assert kept and len(outs[0]) == len(outs[1]) and all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("entry", ["mk_enqueue_steps", "mk_enqueue_steps_static"])
def test_in_a_callers_graph(entry):
    """A captured launch that begins with pairs, replayed over prompts of other lengths (without any pair as well), the program's own work in between."""
    import ctypes
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    from mirage import _capi
    lib = _capi.load()
    shape = Qwen3Shape(head_dim=128, num_layers=2, vocab_size=512, **SHAPES["wide"])
    w, gen = random_weights(shape, seed=2), torch.Generator().manual_seed(8)
    decs = [Qwen3Decoder(shape, w, max_num_batched_tokens=64, max_num_batched_requests=2, max_seq_length=400, page_size=16, eos_token_id=0x7FFFFFFF, max_tokens_per_request=64, pair_portions=p)
            for p in (True, False)]
    draw = lambda lengths: [torch.randint(0, 512, (n,), generator=gen) for n in lengths]
    decs[0].load_prompts(draw((300, 200)))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _capi.check(getattr(lib, entry)(decs[0].mpk._handle, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), 9))
    _capi.check(lib.mk_wait(decs[0].mpk._handle, ctypes.c_void_p(0), None))
    for lengths in ((300, 200), (20, 7), (390, 64), (129, 100)):
        prompts, outs = draw(lengths), []
        for dec in decs:
            dec.k_cache.zero_()
            dec.v_cache.zero_()
            dec.load_prompts(prompts)
            graph.replay() if dec is decs[0] else dec.mpk.run_steps(9)
            torch.cuda.synchronize()
            outs.append([t.clone() for t in (dec.logits()[:2], dec.meta["step"], dec.meta["tokens"], dec.k_cache, dec.v_cache)])
            assert dec.mpk.stats()["aborted"] == 0 and dec.mpk.stats()["iterations"] == 9
        assert all(torch.equal(a, b) for a, b in zip(*outs)), lengths
    for dec in decs:
        dec.mpk.finalize()


@pytest.mark.parametrize("family", ["suborax", "dodonex", "bukatar", "vizonex"])
def test_session(family):
    """Prompts of several requests, some of which begin or end inside a pair, then steps of one token each."""
    from mirage.mpk import ServingSession
    model = _model(family)
    g = torch.Generator().manual_seed(9)
    prompts = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in (300, 215, 170)]
    outs = []
    for pairs in (True, False):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=1536, max_requests=3, max_seq_length=512)
        assert s._second > 0
        s._second, calls = s._second if pairs else 0, []
        run = s.mpk.persistent_kernel.enqueue_batches
        s.mpk.persistent_kernel.enqueue_batches = lambda *a, **k: (calls.append(1), run(*a, **k))
        out = [s.step(list(enumerate(prompts)), [[len(p) - 1] for p in prompts])]
        out += [s.step([(r, [3 + i]) for r in range(3)], [[0]] * 3) for i in range(2)]
        out.append(s.step([(0, prompts[1][:190])], [[189]]))
        assert len(calls) >= 3 if pairs else not calls
        outs.append([(lg.cpu(), greedy) for lg, greedy in out])
        s.finalize()
    for (a, ga), (b, gb) in zip(*outs):
        assert torch.isfinite(a).all() and torch.equal(a, b) and ga == gb


@pytest.mark.parametrize("family", ["suborax", "bukatar"])
def test_wanted_rows_and_rounding(family):
    """Which rows are wanted decides which rows share a pass, and with that the order of sums: 16-bit logits differ by rounding at most.  (Sessions of these
    families are 0.003 to 0.013 from 64-bit results, in 2-norms; two of them differ by no more than both together, 0.026.)"""
    from mirage.mpk import ServingSession
    model = _model(family)
    g = torch.Generator().manual_seed(9)
    prompts = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in (300, 215, 170)]
    last = []
    for want in ([[len(p) - 1] for p in prompts], [list(range(len(p))) for p in prompts], [[0, len(p) - 1] for p in prompts]):
        outs = []
        for _ in range(2):
            s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=1536, max_requests=3, max_seq_length=512)
            out, _ = s.step(list(enumerate(prompts)), want)
            ends = torch.tensor([len(w) for w in want]).cumsum(0) - 1
            outs.append(out[ends.cuda()].double().cpu())
            s.finalize()
        assert torch.equal(*outs)
        last.append(outs[0])
    for other in last[1:]:
        assert (other - last[0]).norm() / last[0].norm() < 0.026


def test_descriptions_that_are_copied():
    """Both descriptions in front of the launch, where they are long (mk_set_host_batch's words by a copy), against fetched ones."""
    from mirage.mpk import ServingSession
    model, outs = _model("suborax"), []
    toks = torch.randint(0, 1000, (300,), generator=torch.Generator().manual_seed(9)).tolist()
    for whole in (False, True):
        s = ServingSession.open(model_config=model, max_tokens=64 * 4000, max_requests=2, max_seq_length=512)
        put, calls = s._put, []
        if whole:
            s._put = lambda at, ids, desc: put(at, ids, desc + [0] * (s._second - 2 * s.max_rows - len(desc)))
        run = s.mpk.persistent_kernel.enqueue_batches
        s.mpk.persistent_kernel.enqueue_batches = lambda *a, **k: (calls.append(a), run(*a, **k))
        outs.append(s.step([("a", toks)], [[299]]))
        assert len(calls) == 2 and all((a[0] + a[2] > 8000) == whole for a in calls)
        s.finalize()
    assert torch.equal(outs[0][0], outs[1][0]) and outs[0][1] == outs[1][1]


def test_descriptions_that_do_not_fit():
    from mirage import _capi
    from mirage.mpk import ServingSession
    s = ServingSession.open(model_config=_model("suborax"), max_tokens=512, max_requests=2, max_seq_length=256)
    pk, at, n = s.mpk.persistent_kernel, s._second, len(s._dev)
    for bad in ((0, at, 4), (at + 1, at, 4), (4, at, 0), (4, at, n - at + 1), (4, at + 1, 4)):
        with pytest.raises(_capi.MkError, match="mk_set_host_batch named"):
            pk.enqueue_batches(*bad)
    cache = [c.clone() for c in s.mpk.model_builder.k_cache]
    for rows in ((64, 2), (2, 64)):  # too few rows beside another portion: nothing runs
        words = s._put(0, *s._describe([("a", list(range(rows[0])))])[:2])
        words2 = s._put(at, *s._describe([("b", list(range(rows[1])))])[:2])
        pk.enqueue_batches(words, at, words2)
        with pytest.raises(_capi.MkError, match="fewer than three rows"):
            pk.wait()
        s.end("a")
        s.end("b")
    assert all(torch.equal(a, b) for a, b in zip(cache, s.mpk.model_builder.k_cache))
    s.finalize()


def test_words_that_do_not_hold_both_descriptions():
    """The second description is read behind the graph's own tensors: launches where that lies outside the named words are refused."""
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    from mirage import _capi
    from mirage.mpk import ServingSession
    shape = Qwen3Shape(head_dim=128, num_layers=2, vocab_size=512, **SHAPES["wide"])
    dec = Qwen3Decoder(shape, random_weights(shape, seed=2), max_num_batched_tokens=64, max_num_batched_requests=2, max_seq_length=200, page_size=16, max_tokens_per_request=64,
                       kernel_mode="online_notoken")
    assert dec.mpk.stats()["paired_portions"]
    dec.mpk.attach_host_batch(torch.zeros(4096, dtype=torch.int32, pin_memory=True), torch.zeros(4096, dtype=torch.int32, device="cuda"))  # (its tensors lie elsewhere)
    with pytest.raises(_capi.MkError, match="the ids and all index tensors"):
        dec.mpk.enqueue_batches(4, 2048, 4)
    dec.mpk.finalize()
    s = ServingSession.open(model_config=_model("suborax"), max_tokens=512, max_requests=2, max_seq_length=256)
    pk, at, n = s.mpk.persistent_kernel, s._second, len(s._dev)
    pk._g.set_host_batch(s._host.data_ptr(), s._dev.data_ptr(), n - 1, s._sampled.data_ptr())
    with pytest.raises(_capi.MkError, match="the ids and all index tensors"):
        pk.enqueue_batches(4, at, 4)
    s.finalize()


def test_graphs_that_run_portions_one_by_one():
    from mirage import _capi
    from suborax_helpers import CONFIGS, weights
    from mirage.mpk import MirageModelConfig, ServingSession
    cfg = CONFIGS[sorted(CONFIGS)[0]]
    s = ServingSession.open(model_config=MirageModelConfig(architecture=cfg, state_dict={k: v.cuda() for k, v in weights(cfg).items()}), max_tokens=512, max_requests=2, max_seq_length=256)
    assert s._second == 0 and s.mpk.persistent_kernel.stats()["paired_portions"] == 0  # (linears of this size do not stream through the matrix cores)
    with pytest.raises(_capi.MkError, match="one by one"):
        s.mpk.persistent_kernel.enqueue_batches(4, 8, 4)
    s.finalize()
