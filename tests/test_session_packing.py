"""How ServingSession packs the tokens of a step: passes of rows that nobody reads first, as long as such rows fill them."""
import pytest
import torch


@pytest.mark.parametrize("lengths,want", [
    ((11, 1), None), ((40, 33, 9), None), ((8,), None), ((9,), None), ((17, 16, 15, 1), None), ((30, 30), ((0, 29), (29,))), ((30, 25), ((12, 29), (3, 24))), ((3, 2, 2), None), ((64,), ((),))])
def test_order_of_rows(lengths, want):
    from mirage.mpk.serving import PagePool, ServingSession
    s = ServingSession.__new__(ServingSession)
    s.page_size, s.max_rows, s.max_requests, s.rows_per_request, s.max_seq = 4, 8, 4, 8, 64
    s.pool, s.requests, s.mpk = PagePool(64), {}, type("M", (), {})()
    want = [[n - 1] for n in lengths] if want is None else [list(w) for w in want]
    passes, unread, state = [], [], {}

    def run(batch):
        assert 0 < sum(len(t) for _, t in batch) <= 8 and len(batch) <= 4
        for rid, toks in batch:
            assert list(toks) == [100 * rid + state.get(rid, 0) + j for j in range(len(toks))]  # in order, none twice
            state[rid] = state.get(rid, 0) + len(toks)
        passes.append([x for _, t in batch for x in t])
        unread.append(s._unread)
        return [x + 1000 for x in passes[-1]]  # the token after a row

    s._pass = run
    s.logits = lambda: torch.tensor([float(x) for x in passes[-1]])[:, None]
    lg, greedy = s.step([(r, [100 * r + j for j in range(n)]) for r, n in enumerate(lengths)], want)
    assert state == dict(enumerate(lengths)) and greedy == [1000 + 100 * r + n - 1 for r, n in enumerate(lengths)]
    assert (lg is None and not any(want)) or lg.flatten().tolist() == [100.0 * r + p for r, w in enumerate(want) for p in w]
    read = {100 * r + p for r, (w, n) in enumerate(zip(want, lengths)) for p in (*w, n - 1)}
    assert [not read & set(p) for p in passes] == unread
    free = sum(min([n - 1, *w]) for w, n in zip(want, lengths))  # rows in front of the first one read
    assert sum(unread) >= free // 8 and len(passes) <= -(-sum(lengths) // 8) + 1


@pytest.mark.parametrize("seed", range(4))
def test_no_more_passes_than_in_order(seed):
    """Rows that nobody reads go first only where that costs no pass: entries beyond the batch's slots, portions that cannot fill one.  (Where portions are
    shorter than a pass it can be one more for a long prompt that has waited.)"""
    import random
    from mirage.mpk.serving import PagePool, ServingSession

    def passes(lengths, want, rows, slots, portion, first):
        s = ServingSession.__new__(ServingSession)
        s.page_size, s.max_rows, s.max_requests, s.rows_per_request, s.max_seq, s._unread_first = 4, rows, slots, portion, 1000, first
        s.pool, s.requests, s.mpk = PagePool(64), {}, type("M", (), {})()
        sizes = []
        s._pass = lambda batch: (sizes.append(sum(len(t) for _, t in batch)), [0] * rows)[1]
        s.logits = lambda: torch.zeros(rows, 1)
        s.step([(r, [0] * n) for r, n in enumerate(lengths)], want)
        assert sum(sizes) == sum(lengths)
        return len(sizes)

    rng = random.Random(seed)
    assert passes([3] * 64, None, 64, 16, 64, True) == 4 and passes([16, 5], None, 8, 1, 8, True) == 3
    for _ in range(400):
        rows, slots = rng.choice([4, 8, 16]), rng.randint(1, 6)
        portion = rng.choice([rows, rows, rng.randint(1, rows)])
        lengths = [rng.choice([1, rng.randint(1, 6), rng.randint(1, 40)]) for _ in range(rng.randint(1, 9))]
        want = [sorted(rng.sample(range(n), min(n, rng.choice([0, 1, 1, 2])))) if rng.random() < 0.4 else [n - 1] for n in lengths]
        assert passes(lengths, want, rows, slots, portion, True) <= passes(lengths, want, rows, slots, portion, False) + (portion < rows)
