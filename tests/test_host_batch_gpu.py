"""Batches that a launch fetches from pinned memory by itself (mk_set_host_batch / mk_enqueue_batch)."""
import pytest
import torch

from suborax_helpers import CONFIGS, prompt, weights

pytestmark = pytest.mark.gpu


def _session(**kw):
    from mirage.mpk import MirageModelConfig, ServingSession
    cfg = CONFIGS[sorted(CONFIGS)[0]]
    return cfg, ServingSession.open(model_config=MirageModelConfig(architecture=cfg, state_dict={k: v.cuda() for k, v in weights(cfg).items()}), **kw)


@pytest.mark.parametrize("max_requests", [1, 3, 64])
def test_as_copied(max_requests):
    """The same steps with the batch fetched by the launch and with copies on the stream: logits and tokens equal bit by bit."""
    outs = []
    for fetched in (True, False):
        cfg, s = _session(max_tokens=64 * max_requests * 2, max_requests=max_requests, max_seq_length=128)
        s._fetched = fetched
        ps = [prompt(cfg, 1 + (7 * r) % 70, seed=r) for r in range(max_requests)]
        out = [s.step(list(enumerate(ps)), [[len(p) - 1] for p in ps])]
        out += [s.step([(r, [7 + i]) for r in range(max_requests)], [[0]] * max_requests) for i in range(3)]
        outs.append([(lg.cpu(), greedy) for lg, greedy in out])
        s.finalize()
    for (a, ga), (b, gb) in zip(*outs):
        assert torch.equal(a, b) and ga == gb


def test_every_word_arrives_and_none_behind():
    """A workgroup moves 2048 words a turn: sizes around one and two turns, and the least a batch has."""
    cfg, s = _session(max_tokens=32 * 4500, max_requests=2, page_size=32, max_seq_length=64)
    pk, n0 = s.mpk.persistent_kernel, 2 * s.max_rows + 4 * 2 + 2 + 1
    s.step([("a", [5])], [[0]])
    least = s._host[:n0].clone()
    g = torch.Generator().manual_seed(3)
    for words in (n0, 255, 256, 257, 2047, 2048, 2049, 4096, 4097, len(s._dev) - 1, len(s._dev)):
        s._host.copy_(torch.randint(0, 1 << 30, s._host.shape, generator=g, dtype=torch.int32))
        s._host[:n0] = least
        s._dev.fill_(-7)
        s._sampled.fill_(-1)
        want = torch.full_like(s._host, -7, pin_memory=False)
        want[:words] = s._host[:words]
        pk.enqueue_batch(words)
        pk.wait()
        assert torch.equal(s._dev.cpu(), want)
        assert s._sampled[0] == s.mpk.output_tokens.view(-1)[0].item()
        s._dev.fill_(-7)
        s._sampled.fill_(-1)
        pk.enqueue_ingest(host_words=words)
        pk.wait()
        assert torch.equal(s._dev.cpu(), want) and (s._sampled == -1).all()
    s.finalize()


@pytest.mark.parametrize("ingest", [False, True])
def test_descriptions_that_are_copied(ingest):
    """Long descriptions reach the device by a copy in front of the launch: the same words, on both sides of that line."""
    cfg, s = _session(max_tokens=32 * 7000, max_requests=2, page_size=32, max_seq_length=64)
    pk, n0 = s.mpk.persistent_kernel, 2 * s.max_rows + 4 * 2 + 2 + 1
    want, _ = s.step([("a", [5])], [[0]])
    g = torch.Generator().manual_seed(4)
    for words in (7167, 7168, 7169, 14000):
        s._host[n0:] = torch.randint(0, 1 << 30, s._host[n0:].shape, generator=g, dtype=torch.int32)
        s._dev.fill_(-7)
        s.logits().zero_()
        (pk.enqueue_ingest(host_words=words) if ingest else pk.enqueue_batch(words))
        pk.wait()
        assert torch.equal(s._dev[:words].cpu(), s._host[:words]) and (s._dev[words:] == -7).all()
        assert torch.equal(s.logits()[:1].float(), want) != ingest
    s.finalize()


def test_views_of_the_logits():
    """A view per call, whatever mode the first one was asked for in and whatever became of an earlier one; none behind finalize()."""
    cfg, s = _session(max_tokens=256, max_requests=2, max_seq_length=64)
    with torch.inference_mode():
        s.step([("a", [5])], [[0]])
        s.logits()
    view = s.logits()
    assert not view.is_inference() and view.data_ptr() == s.logits().data_ptr()
    shape = view.shape
    view.unsqueeze_(0).requires_grad_()
    assert s.logits().shape == shape and not s.logits().requires_grad
    lg, _ = s.step([("a", [6])], [[0]])
    assert torch.equal(lg, s.logits()[:1].float())
    s.finalize()
    with pytest.raises(RuntimeError):
        s.logits()


def test_memory_of_another_kind_is_refused():
    cfg, s = _session(max_tokens=256, max_requests=2, max_seq_length=64)
    pk, host, dev, tokens = s.mpk.persistent_kernel, s._host, s._dev, s._sampled
    named = pk._g.set_host_batch
    n = len(dev)
    with pytest.raises(Exception, match="mk_set_host_batch named"):
        pk.enqueue_batch(n + 1)
    for bad in ((torch.zeros(n, dtype=torch.int32).data_ptr(), dev.data_ptr(), n, None), (dev.data_ptr(), dev.data_ptr(), n, None), (host.data_ptr(), host.data_ptr(), n, None),
                (host.data_ptr(), 0, n, None), (host.data_ptr() + 2, dev.data_ptr(), n - 1, None), (host.data_ptr(), dev.data_ptr(), n, dev.data_ptr()), (host.data_ptr(), dev.data_ptr(), 0, None)):
        with pytest.raises(Exception):
            named(*bad)
        with pytest.raises(Exception, match="mk_set_host_batch named"):  # (nothing is named any more)
            pk.enqueue_batch(1)
    pk.attach_host_batch(host, dev, tokens)
    assert s.step([("a", [5])], [[0]])[1][0] is not None
    s.finalize()
