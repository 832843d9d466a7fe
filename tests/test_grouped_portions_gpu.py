"""More than two portions inside prompts as one iteration: the same results, bit by bit, as portions one by one, where tasks of the linears and of the attention
end within a portion, a pair or a tile."""
import pytest
import torch

from test_paired_portions_gpu import SHAPES, _any_pair, _kept, _model, _offline  # noqa: F401  (_any_pair: a fixture)

pytestmark = pytest.mark.gpu

# queries per kv head of four and eight; chunks of two, four and eight; rows of an output that are no multiple of a task's
SHAPES.update({
    "eight": dict(hidden_size=2048, num_q_heads=64, num_kv_heads=8, intermediate_size=6144),
    "odd": dict(hidden_size=4096, num_q_heads=24, num_kv_heads=6, intermediate_size=5120),
})


@pytest.mark.parametrize("name,lengths,B,portion,R", [
    ("wide", (64 * 9 + 5,), 64, 64, 1), ("wide", (64 * 16 + 1,), 64, 64, 1), ("eight", (64 * 7 + 40,), 64, 64, 1), ("long", (64 * 6 + 9,), 64, 64, 1), ("narrow", (64 * 5 + 33,), 64, 64, 1),
    ("odd", (64 * 8 + 17,), 64, 64, 1), ("wide", (300, 290, 280, 270), 64, 20, 4), ("wide", (90,) * 12, 64, 9, 12), ("mixed", (50 * 7 + 3, 50 * 5), 50, 50, 2), ("experts", (64 * 8 + 30,), 64, 64, 1),
    ("wide", (33 * 7 + 2,), 33, 33, 1)])
def test_offline(name, lengths, B, portion, R):
    _offline(name, lengths, B, portion, 1000, R)


@pytest.mark.parametrize("steps", [4, 6, 9])
def test_launches_that_end_inside(steps):
    """The last iteration of a launch runs alone, whatever could run beside it."""
    _offline("wide", (64 * 12 + 3,), 64, 64, steps, 1)


def test_pages_that_hold_no_whole_tile():
    """Pages of four and of twenty-four positions: tiles of sixteen reach into others, and no page is a power of two."""
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    shape = Qwen3Shape(head_dim=128, num_layers=2, vocab_size=512, **SHAPES["wide"])
    w, prompt = random_weights(shape, seed=2), torch.randint(0, 512, (64 * 6 + 11,), generator=torch.Generator().manual_seed(5))
    for page in (4, 24):
        outs = []
        for pairs in (True, False):
            dec = Qwen3Decoder(shape, w, max_num_batched_tokens=64, max_num_batched_requests=1, max_seq_length=400, page_size=page, eos_token_id=0x7FFFFFFF, max_tokens_per_request=64, pair_portions=pairs)
            dec.load_prompts([prompt])
            dec.mpk.run_steps(7)
            outs.append([t.clone().cpu() for t in (dec.logits()[:11], dec.k_cache, dec.v_cache)])
            dec.mpk.finalize()
        assert all(torch.equal(a, b) for a, b in zip(*outs)), page


def test_values_that_are_not_finite():
    """An infinity in a row of values reaches the positions that see it and no others, in whichever portion they are."""
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    shape = Qwen3Shape(head_dim=128, num_layers=1, vocab_size=512, **SHAPES["wide"])
    w, prompt = random_weights(shape, seed=2), torch.randint(0, 511, (64 * 4 + 9,), generator=torch.Generator().manual_seed(5))
    w["embed"][511] = float("inf")
    prompt[150] = 511
    outs = []
    for pairs in (True, False):
        dec = Qwen3Decoder(shape, w, max_num_batched_tokens=64, max_num_batched_requests=1, max_seq_length=280, page_size=16, eos_token_id=0x7FFFFFFF, max_tokens_per_request=64, pair_portions=pairs)
        dec.load_prompts([prompt])
        dec.mpk.run_steps(5)
        outs.append([t.clone().cpu().view(torch.int16) for t in (dec.k_cache, dec.v_cache)])
        dec.mpk.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("family", ["suborax", "dodonex", "bukatar", "vizonex"])
def test_session(family):
    """As many passes in a launch as run together, prompts of one token among them, and portions in which every request brings one row."""
    from mirage.mpk import ServingSession
    model, g = _model(family), torch.Generator().manual_seed(9)
    lengths = (70, 1, 2, 3) + (2,) * 40 + (500, 330)
    prompts = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in lengths]
    outs = []
    for together in (8, 4, 0):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 64, max_requests=48, max_seq_length=512)
        s._second, s._together, held = s._second if together else 0, together, []
        run = s.mpk.persistent_kernel.enqueue_batches
        s.mpk.persistent_kernel.enqueue_batches = lambda *a, **k: (held.append(k["hold"]), run(*a, **k))
        out = [s.step(list(enumerate(prompts)), [[n - 1] for n in lengths])]
        out += [s.step([(r, [3 + i]) for r in range(len(lengths))], [[0]] * len(lengths)) for i in range(2)]
        assert any(held) if together == 8 else True
        outs.append([(lg.cpu(), greedy) for lg, greedy in out])
        s.finalize()
    for other in outs[:2]:
        for (a, ga), (b, gb) in zip(other, outs[2]):
            assert torch.isfinite(a).all() and torch.equal(a, b) and ga == gb


# flex attention: more chunks than LDS holds, units in pairs; five queries a kv head and two slices of value dims; units one by one; a window and kept positions
# whose tiles lie apart; positions in chunks.  Requests that begin inside a portion: units whose tiles are not the same ones
@pytest.mark.parametrize("family,sizes", [
    ("suborax", dict(heads=16, kv_heads=4)), ("suborax", dict(heads=20, kv_heads=4, dim=96, vdim=160)), ("suborax", dict(heads=8, kv_heads=2, dim=64, vdim=64)),
    ("suborax", dict(heads=16, kv_heads=8, dim=160)), ("bukatar", dict(window=100, keep_first=40)), ("vizonex", dict(chunk=128))])
def test_flex_attention(family, sizes):
    import generate
    from mirage.mpk import ServingSession
    make, base = generate.SHAPES[family + "-2k"]
    torch.manual_seed(7)
    model = generate.random_model(make(**{**base, **sizes}, layers={"suborax": 2}.get(family, 4), vocab=1000, **({"positions": 1024} if family == "vizonex" else {})))[0]
    g = torch.Generator().manual_seed(9)
    lengths = (64 * 9 + 5, 333, 70)
    prompts, outs = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in lengths], []
    for together in (8, 0):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 64, max_requests=3, max_seq_length=640)
        assert s.mpk.persistent_kernel.stats()["paired_portions"]
        s._second, s._together = s._second if together else 0, together
        outs.append([s.step(list(enumerate(prompts)), [[n - 1] for n in lengths])[0].cpu(), s.step([(r, [3]) for r in range(3)], [[0]] * 3)[0].cpu()])
        s.finalize()
    assert all(torch.isfinite(a).all() and torch.equal(a, b) for a, b in zip(*outs))


def test_portions_of_single_rows():
    """Portions in which every request brings one row append keys and values in the attention itself, beside portions whose rows are prepared ahead of it."""
    from mirage.mpk import ServingSession
    model, outs = _model("suborax"), []
    for grouped in (True, False):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 64, max_requests=40, max_seq_length=512)
        passes = [[(r, [r + 1]) for r in range(40)], [(0, list(range(50)))], [(r, [r + 7]) for r in range(40)], [(1, list(range(30))), (2, list(range(30)))]]
        if grouped:
            s._passes(passes)
        else:
            for p in passes:
                s._unread = True
                s._pass(p)
        outs.append([c.clone().cpu() for c in s.mpk.model_builder.k_cache + s.mpk.model_builder.v_cache] + [s.step([(0, [5]), (1, [6]), (3, [7])], [[0]] * 3)[0].cpu()])
        s.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def test_batches_that_do_not_fit():
    from mirage import _capi
    from mirage.mpk import ServingSession
    s = ServingSession.open(model_config=_model("suborax"), max_tokens=1024, max_requests=2, max_seq_length=512)
    pk, at, apart = s.mpk.persistent_kernel, s._second, s._apart
    assert s._together == pk.stats()["portions_together"] == 8
    with pytest.raises(_capi.MkError, match="from word 0 on"):
        pk.enqueue_batches(4, at, 4, at=apart, hold=True)
    with pytest.raises(_capi.MkError, match="no batches are held"):
        pk._g.enqueue_held(pk._stream_ptr(None))
    words = [s._put(i // 2 * apart + i % 2 * at, *s._describe([("a", list(range(64)))])[:2]) for i in range(8)]
    for p in range(4):
        pk.enqueue_batches(words[2 * p], at, words[2 * p + 1], at=p * apart, hold=True)
    with pytest.raises(_capi.MkError, match="8 batches together"):
        pk.enqueue_batches(4, at, 4, at=apart, hold=True)
    with pytest.raises(_capi.MkError, match="mk_set_host_batch named"):
        pk.enqueue_batches(4, at, 4, at=4 * apart, hold=True)
    pk._g.enqueue_held(pk._stream_ptr(None))
    pk.wait()
    assert pk.stats()["iterations"] == 8
    cache = [c.clone() for c in s.mpk.model_builder.k_cache]
    for rows in ((64, 64, 64, 2), (2, 64, 64, 64), (64, 64, 2, 64)):  # (one too small: nothing runs)
        s.end("b")
        words = [s._put(i // 2 * apart + i % 2 * at, *s._describe([("b", list(range(n)))])[:2]) for i, n in enumerate(rows)]
        pk.enqueue_batches(words[0], at, words[1], hold=True)
        pk.enqueue_batches(words[2], at, words[3], at=apart)
        with pytest.raises(_capi.MkError, match="fewer than three rows"):
            pk.wait()
    assert all(torch.equal(a, b) for a, b in zip(cache, s.mpk.model_builder.k_cache))
    s.finalize()


def test_out_of_pages_behind_some_passes():
    """What has been described runs, then the error comes; what the requests have in the cache is what ran."""
    from mirage.mpk import ServingSession
    model, outs = _model("suborax"), []
    for grouped in (True, False):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 7, max_requests=2, max_seq_length=448)
        if not grouped:
            s._second = 0
        with pytest.raises(RuntimeError, match="out of cache pages"):
            s.step([(r, [i % 900 for i in range(300)]) for r in "ab"])
        outs.append([c.clone().cpu() for c in s.mpk.model_builder.k_cache] + [torch.tensor([r.length for r in s.requests.values()])])
        s.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def test_single_rows_whose_sums_lie_apart():
    """As above where the projection runs portion by portion, since the output one streams no weights (2560 values, 128 tiles): its slices are the next portion's a moment later."""
    import generate
    from mirage.mpk import ServingSession
    make, base = generate.SHAPES["suborax-2k"]
    torch.manual_seed(7)
    model, outs = generate.random_model(make(**{**base, "heads": 16, "kv_heads": 8, "dim": 160}, layers=2, vocab=1000))[0], []
    for grouped in (True, False):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 64, max_requests=40, max_seq_length=512)
        assert s.mpk.persistent_kernel.stats()["paired_portions"]
        passes = [[(r, [r + 1]) for r in range(40)], [(0, list(range(50)))], [(r, [r + 7]) for r in range(40)], [(r, [r + 9]) for r in range(36)]]
        if grouped:
            s._passes(passes)
        else:
            for p in passes:
                s._unread = True
                s._pass(p)
        outs.append([c.clone().cpu() for c in s.mpk.model_builder.k_cache + s.mpk.model_builder.v_cache] + [s.step([(0, [5]), (1, [6]), (3, [7])], [[0]] * 3)[0].cpu()])
        s.finalize()
    assert all(torch.isfinite(a).all() and torch.equal(a, b) for a, b in zip(*outs))


def test_attention_layers_of_unequal_shape():
    """Heads of 128, attended for all portions at once with more chunks than LDS holds, and of 160, portion by portion, by turns: both leave partial results in the same words, and little is
    streamed between them (two layers have a feed-forward)."""
    import generate
    from mirage.mpk import ServingSession
    make, base = generate.SHAPES["suborax-2k"]
    torch.manual_seed(7)
    cfg = make(**{**base, "heads": 16, "kv_heads": 4}, layers=1, vocab=1000)
    narrow = {**cfg["layers"][0], "mlp": None}
    wide = {**narrow, "mixer": {**narrow["mixer"], "dim": 160}}
    cfg["layers"] = [{**narrow, "mlp": cfg["layers"][0]["mlp"]}, wide, narrow, wide, narrow, {**wide, "mlp": cfg["layers"][0]["mlp"]}, narrow]
    model, g = generate.random_model(cfg)[0], torch.Generator().manual_seed(9)
    lengths, outs = (64 * 16 + 5, 64 * 9), []
    prompts = [torch.randint(0, 1000, (n,), generator=g).tolist() for n in lengths]
    for together in (8, 0):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=64 * 64, max_requests=2, max_seq_length=1088)
        assert s.mpk.persistent_kernel.stats()["paired_portions"]
        s._second, s._together = s._second if together else 0, together
        outs.append([s.step([(i, p)], [[len(p) - 1]])[0].cpu() for i, p in enumerate(prompts)] + [s.step([(r, [3]) for r in range(2)], [[0]] * 2)[0].cpu()])
        outs[-1] += [c.clone().cpu() for c in s.mpk.model_builder.k_cache + s.mpk.model_builder.v_cache]
        s.finalize()
    assert all(torch.isfinite(a).all() and torch.equal(a, b) for a, b in zip(*outs))


def test_batches_that_a_failed_caller_has_left():
    """Held batches of a caller that failed before it could launch them: the next one's first batches, from word 0 on, begin anew, and so do requests; descriptions that overlap are refused."""
    from mirage import _capi
    from mirage.mpk import ServingSession
    model, outs = _model("suborax"), []
    toks = torch.randint(0, 1000, (64 * 6 + 9,), generator=torch.Generator().manual_seed(9)).tolist()
    for left in (False, True):
        s = ServingSession.open(model_config=model, dtype=torch.bfloat16, max_tokens=2048, max_requests=2, max_seq_length=512)
        pk, at, apart = s.mpk.persistent_kernel, s._second, s._apart
        if left:
            words = [s._put(i // 2 * apart + i % 2 * at, *s._describe([("gone", list(range(64)))])[:2]) for i in range(4)]
            s.end("gone")
            pk.enqueue_batches(words[0], at, words[1], hold=True)
            with pytest.raises(_capi.MkError, match="behind those that end at word"):
                pk.enqueue_batches(words[2], at, words[3], at=at, hold=True)
            pk.enqueue_batches(words[2], at, words[3], at=apart, hold=True)
        outs.append([s.step([("a", toks)], [[len(toks) - 1]])[0].cpu()] + [c.clone().cpu() for c in s.mpk.model_builder.k_cache])
        assert pk.stats()["iterations"] == 7
        if left:
            pk.enqueue_batches(words[0], at, words[1], hold=True)
            pk._g.init_requests()
            with pytest.raises(_capi.MkError, match="no batches are held"):
                pk._g.enqueue_held(pk._stream_ptr(None))
        s.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def test_numbers_of_words_whose_sums_wrap():
    from mirage import _capi
    from mirage.mpk import ServingSession
    s = ServingSession.open(model_config=_model("suborax"), max_tokens=1024, max_requests=2, max_seq_length=512)
    pk, at, apart, most = s.mpk.persistent_kernel, s._second, s._apart, 2 ** 63 - 2
    for words, second, words2 in ((4, at, most), (4, most, 4), (most, most, 4), (4, most, most)):
        with pytest.raises(_capi.MkError, match="mk_set_host_batch named"):
            pk.enqueue_batches(words, second, words2)
        for far in (0, apart, most):
            with pytest.raises(_capi.MkError, match="mk_set_host_batch named"):
                pk._g.hold_batches(far, words, second, words2)
    with pytest.raises(_capi.MkError, match="mk_set_host_batch named"):
        pk._g.hold_batches(most, 4, at, 4)
    with pytest.raises(_capi.MkError, match="words behind those"):
        pk.attach_more_batches(most)
    s.finalize()


@pytest.mark.parametrize("workgroups", [2, 8, 16])
def test_convolutions_that_read_what_scans_leave(workgroups):
    """Where few workgroups have the small linear between a convolution and its scan run for all portions: not before the portion in front has left its last inputs."""
    _offline_grid("bukatar", workgroups, 8)


@pytest.mark.parametrize("family", ["suborax", "bukatar"])
def test_fewer_wavefronts_than_portions(family):
    """One workgroup has four wavefronts, each of which prepares rows of one portion: no more portions run together."""
    _offline_grid(family, 1, 4)


def _offline_grid(family, workgroups, together):
    import generate
    model, outs = _model(family), []
    prompt = torch.randint(0, 1000, (64 * 9 + 5,), generator=torch.Generator().manual_seed(6))
    for pairs in (True, False):
        gen = generate.Generator(600, model_config=model, batch=1, max_num_batched_tokens=64, max_tokens_per_request=64, page_size=64, eos_token_id=-1, pair_portions=pairs, num_workers=workgroups)
        assert gen.mpk.stats()["portions_together"] == (together if pairs else 1)
        gen.load_prompts([prompt])
        gen.mpk.run_steps(10)
        outs.append([t.clone().cpu() for t in [gen.logits()[:5], *_kept(gen.model.model_builder)]])
        gen.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))
