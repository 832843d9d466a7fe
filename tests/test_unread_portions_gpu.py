"""Iterations whose logits and sampled tokens nobody reads end with the last stage that writes caches or recurrent states: what later
iterations compute is, bit for bit, what it is behind iterations that were run whole."""
import importlib

import pytest
import torch

from helpers import make_meta, make_mpk
from test_online_modes import _cfg, _decoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("family,dtype", [("suborax", torch.bfloat16), ("suborax", torch.float32), ("dodonex", torch.bfloat16), ("bukatar", torch.bfloat16), ("vizonex", torch.bfloat16)])
@pytest.mark.parametrize("lengths", [(150,), (65, 130, 3)])
def test_session(family, dtype, lengths):
    """Prompts in portions of which only the last rows are wanted, against the same passes with every row wanted."""
    _session(family, "even", dtype, lengths)


# (the last layer of these routes tokens to experts)
@pytest.mark.parametrize("family,dtype", [("bukatar", torch.bfloat16), ("bukatar", torch.float32), ("vizonex", torch.bfloat16), ("vizonex", torch.float32)])
def test_session_of_a_model_that_ends_with_experts(family, dtype):
    _session(family, "odd", dtype, (65, 130, 3))


def _session(family, kind, dtype, lengths):
    from mirage.mpk import MirageModelConfig, ServingSession
    h = importlib.import_module(family + "_helpers")
    cfg = h.CONFIGS[kind]
    w = {k: v.cuda() for k, v in h.weights(cfg).items()}
    outs = []
    for every in (False, True):
        s = ServingSession.open(model_config=MirageModelConfig(architecture=cfg, state_dict=w), dtype=dtype, max_tokens=512, max_requests=3, max_seq_length=192)
        calls, pk = [], s.mpk.persistent_kernel
        ingest = pk.enqueue_ingest
        pk.enqueue_ingest = lambda **kw: (calls.append(1), ingest(**kw))
        ps = [h.prompt(cfg, n, seed=r) for r, n in enumerate(lengths)]
        lg, greedy = s.step(list(enumerate(ps)), [list(range(n)) if every else [n - 1] for n in lengths])
        ends = torch.tensor(lengths).cumsum(0) - 1
        out = [lg[ends.cuda()] if every else lg, torch.tensor(greedy)]
        for i in range(2):
            lg, greedy = s.step([(r, [7 + i]) for r in range(len(ps))], [[0]] * len(ps))
            out += [lg, torch.tensor(greedy)]
        assert (len(calls) > 0) != every
        outs.append([t.cpu() for t in out])
        s.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("requests,portion", [(1, 8), (1, 64), (2, 8), (5, 16)])
def test_offline(requests, portion):
    """One launch (the portions inside prompts end early) against launches of one iteration (each of which is run whole); prompts that end
    with a portion, inside one and at the end of the sequence, and a batch in which one request decodes while another ingests."""
    from oracle.qwen3_ref import make_model_weights, make_prompt
    cfg = _cfg()
    w = make_model_weights(cfg, seed=47)
    max_seq = 96
    prompts = [make_prompt(cfg, n, 600 + i) for i, n in enumerate((64, 75, 17, 95, 40)[:requests])]
    outs = []
    for whole in (False, True):
        dec = _decoder(cfg, w, max_num_batched_tokens=64, max_num_batched_requests=requests, max_seq_length=max_seq, page_size=16, max_tokens_per_request=portion)
        dec.load_prompts(prompts)
        n, done = 40, False
        if whole:
            for _ in range(n):
                done = done or dec.mpk.run_steps(1)
        else:
            dec.mpk.run_steps(n)
        outs.append([t.cpu().clone() for t in (dec.meta["tokens"], dec.meta["step"], dec.k_cache, dec.v_cache, dec.logits()[:requests])])
        dec.mpk.finalize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))


def _described(mpk_meta, rows):
    one = lambda *v: torch.tensor(v, dtype=torch.int32)
    mpk_meta["qo_indptr_buffer"].copy_(one(0, rows))
    mpk_meta["paged_kv_indptr_buffer"].copy_(one(0, 1))
    mpk_meta["paged_kv_last_page_len_buffer"].copy_(one(rows))
    torch.cuda.synchronize()


def test_what_an_unread_batch_leaves():
    """Caches as the whole pass writes them, logits as they were; the offline mode has no such launch."""
    from mirage import _capi
    from oracle.qwen3_ref import make_model_weights
    cfg = _cfg()
    w = make_model_weights(cfg, seed=48)
    on = _decoder(cfg, w, max_num_batched_tokens=8, max_num_batched_requests=1, max_seq_length=16, page_size=16, kernel_mode="online_notoken")
    on.meta["input_tokens"].copy_(torch.arange(8).view(-1, 1))
    _described(on.meta, 8)
    on.mpk()
    lg, k = on.logits().clone(), on.k_cache.clone()
    on.k_cache.zero_()
    on.meta["input_tokens"][0] = 99
    on.mpk.enqueue_ingest()
    on.mpk.wait()
    assert torch.equal(on.logits(), lg)
    other = on.k_cache.clone()
    assert not torch.equal(other, k)
    on.mpk()
    assert torch.equal(on.k_cache, other) and not torch.equal(on.logits(), lg)
    on.mpk.finalize()
    off = _decoder(cfg, w, max_num_batched_tokens=8, max_num_batched_requests=1, max_seq_length=16, page_size=16)
    with pytest.raises(_capi.MkError, match="host describes"):
        off.mpk.enqueue_ingest()
    off.mpk.finalize()


def test_stage_times_of_an_unread_batch():
    """Stages that were left out show no times, those that ran show this batch's."""
    from oracle.qwen3_ref import make_model_weights
    cfg = _cfg()
    on = _decoder(cfg, make_model_weights(cfg, seed=48), max_num_batched_tokens=8, max_num_batched_requests=1, max_seq_length=16, page_size=16, kernel_mode="online_notoken")
    _described(on.meta, 8)
    on.mpk()
    before = on.mpk.stage_profile(raw=True)
    ran = [line[3] > 0 for line in before]
    on.mpk.enqueue_ingest()
    on.mpk.wait()
    for old, new, r in zip(before, on.mpk.stage_profile(raw=True), ran):
        if old[0].endswith("unread=skip"):
            assert tuple(new[1:]) == (0, 0, 0, 0)
        elif r:
            assert new[3] > old[3]
    assert any(line[0].endswith("unread=skip") for line in before)
    on.mpk()
    assert [line[3] > 0 for line in on.mpk.stage_profile(raw=True)] == ran
    on.mpk.finalize()


@pytest.mark.parametrize("carried", [False, True])
def test_rows_carried_from_one_iteration_to_the_next(carried):
    """A stage at the end whose output an iteration reads before it is written again runs in every iteration."""
    import mirage as mi
    g = torch.Generator().manual_seed(3)
    x, W, acc = (torch.randn(8, 64, generator=g).to(torch.bfloat16).cuda(), torch.randn(64, 64, generator=g).to(torch.bfloat16).cuda(), torch.zeros(8, 64, dtype=torch.bfloat16, device="cuda"))
    meta = make_meta(1, 64, 8, 1, 8)
    pk = make_mpk(meta, 64, 8, 1, 8, 64, mode="onepass")
    tx, tW, ta = pk.attach_input(x, "x"), pk.attach_input(W, "W"), pk.attach_input(acc, "acc")
    if carried:
        pk.linear_with_residual_layer(input=tx, weight=tW, residual=ta, output=ta, grid_dim=(1, 1, 1), block_dim=(256, 1, 1))
    else:
        pk.linear_layer(input=tx, weight=tW, output=ta, grid_dim=(1, 1, 1), block_dim=(128, 1, 1))
    pk.compile()
    _described(meta, 8)
    pk.enqueue_ingest()
    pk.wait()
    assert bool((acc != 0).any()) == carried
    pk.finalize()


@pytest.mark.parametrize("B,R,total,portion,page_size,max_seq", [(64, 1, 2, 64, 16, 150), (64, 2, 3, 16, 4, 90), (64, 5, 9, 64, 16, 120), (40, 3, 6, 30, 8, 100), (64, 40, 50, 2, 8, 30)])
def test_scheduler_of_portions(B, R, total, portion, page_size, max_seq):
    """Long portions of one, two and many requests: the same batches, entry for entry, as the scheduler oracle's."""
    import numpy as np
    from demo_qwen3 import Qwen3Decoder, Qwen3Shape, random_weights
    from oracle.sched_ref import SchedulerOracle
    shape = Qwen3Shape(hidden_size=1024, num_q_heads=8, num_kv_heads=2, head_dim=128, intermediate_size=512, num_layers=1, vocab_size=512)
    rng = np.random.default_rng(B + R + total)
    prompts = [torch.from_numpy(rng.integers(0, shape.vocab_size, size=int(rng.integers(1, max_seq - 3)))) for _ in range(total)]
    pages = R * ((max_seq + page_size - 1) // page_size)
    dec = Qwen3Decoder(shape, random_weights(shape, seed=1), max_num_batched_tokens=B, max_num_batched_requests=R, max_seq_length=max_seq, page_size=page_size, max_num_pages=pages,
                       total_requests=total, eos_token_id=0x7FFFFFFF, max_tokens_per_request=portion)
    dec.load_prompts(prompts)
    orc = SchedulerOracle([p.tolist() for p in prompts], R, B, pages, page_size, max_seq, max_new_per_req=portion)
    out = None
    while True:
        n = orc.step(out)
        fin = dec.mpk.run_steps(1)
        if n == 0:
            assert fin
            break
        assert not fin
        nreq = int((orc["request_ids"] >= 0).sum())
        for ours, theirs, m in (("step", "step", total), ("input_tokens", "input_tokens", n), ("qo_indptr_buffer", "qo_indptr", R + 1), ("paged_kv_indptr_buffer", "kv_indptr", R + 1),
                                ("paged_kv_last_page_len_buffer", "kv_last_page_len", nreq), ("paged_kv_indices_buffer", "kv_indices", int(orc["kv_indptr"][R]))):
            assert np.array_equal(dec.meta[ours].cpu().numpy().reshape(-1)[:m], orc[theirs].reshape(-1)[:m]), ours
        out = dec.meta["output_tokens"].cpu().numpy().reshape(-1)
    assert np.array_equal(dec.meta["tokens"].cpu().numpy(), orc["tokens"])
    dec.mpk.finalize()
