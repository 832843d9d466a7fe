"""ServingSession: the host loop of the serving mode (MPK in "online_notoken" mode).

The caller says, step by step, which requests bring which tokens; the session keeps every live request's pages, packs the
tokens of a step into passes of at most `max_num_batched_tokens` rows (single decoded tokens beside portions of prompts,
at most `max_tokens_per_request` rows of one request per pass), describes each pass in the meta tensors and launches the
megakernel once for it.  What a request has in the cache is its pages, its length and, where the model has recurrent layers,
its state slot, so a request may pause for any number of steps, and a portion may end anywhere.

`generate` is the greedy loop on top: continuous batching over a list of prompts with as many live requests as there are
batch slots and pages.
"""
from dataclasses import dataclass, field
from typing import Dict, List, Sequence, Tuple

import torch

from .mpk import MPK, MPKMetadata


MAX_TOGETHER = 8  # passes of which no row is wanted that may be one launch (as many as the kernels run together)


class PagePool:
    """Free list of cache pages (or state slots).  What is given back is handed out again first."""

    def __init__(self, num_pages: int, what: str = "cache pages"):
        self.num_pages, self.what = num_pages, what
        self._free = list(range(num_pages - 1, -1, -1))

    def __len__(self):
        return len(self._free)

    def take(self, n: int) -> List[int]:
        if n > len(self._free):
            raise RuntimeError(f"out of {self.what}: {n} asked for, {len(self._free)} of {self.num_pages} free")
        return [self._free.pop() for _ in range(n)]

    def give(self, pages: List[int]):
        self._free.extend(reversed(pages))


@dataclass
class _Request:
    pages: List[int] = field(default_factory=list)
    length: int = 0  # positions whose keys and values are in the cache
    slot: int = -1   # recurrent-state slot (models with recurrent layers)


class ServingSession:
    # models with recurrent layers: the tensor that names every batch slot's state slot, and the pool of state slots
    state_slots = slots = None
    # sessions opened here: a pass's ids and description in pinned memory, the device tensor they go to, and a pinned place for the sampled
    # tokens.  The launch fetches and leaves them itself (_fetched), so that nothing but the launch is on the stream and a pass waits for the
    # device once
    _host = _dev = _sampled = None
    _fetched = False
    # two passes of which no row is wanted may be one launch (enqueue_batches): word the second one's description begins at, 0: not in this graph.  Or
    # more of them, _together at most, each two with descriptions _apart words behind those of the two in front (in _words: _host is where those begin)
    _second = 0
    _together = 2
    _apart = 0
    _words = _every = None
    _view = None  # of the logits
    # rows that nobody reads go into passes of their own, in front (see step).  Which rows share a pass decides in which order attention, experts and linears
    # of few rows add, so that 16-bit results depend, in rounding, on the rows that are wanted; 32-bit sessions keep the rows in order, and their results
    # are the same bit by bit whichever are wanted (16.2 ms for three prompts and their steps of a 2048-wide model, 15.7 with those rows in front)
    _unread_first = True
    _unread = False  # nobody reads the logits or the sampled tokens of the pass that runs

    def __init__(self, mpk: MPK):
        if mpk.metadata.mode != "online_notoken":
            raise ValueError("a serving session drives an MPK in online_notoken mode")
        self.mpk = mpk
        pk = mpk.persistent_kernel
        self.page_size, self.max_rows, self.max_requests = pk.page_size, pk.max_num_batched_tokens, pk.max_num_batched_requests
        self.rows_per_request, self.max_seq = pk.max_tokens_per_request, min(pk.max_seq_length, mpk.model_builder.max_positions or pk.max_seq_length)
        self.pool = PagePool(pk.max_num_pages)
        # one state slot per batch slot: the kernel starts a request's state from zero where its position is zero
        self.state_slots = getattr(mpk.model_builder, "state_slots", None)
        if self.state_slots is not None:
            self.slots = PagePool(self.max_requests, "state slots")
        self._unread_first = mpk.metadata.dtype != torch.float32
        self.requests: Dict[object, _Request] = {}
        mpk._ensure_compiled()

    @staticmethod
    def open(model_path: str = None, model_config=None, model_name: str = None, dtype=torch.bfloat16, max_tokens: int = 4096, max_requests: int = 4,
             page_size: int = 64, max_rows: int = 64, max_seq_length: int = None, device: str = "cuda") -> "ServingSession":
        """Build and compile the model found at `model_path` (class chosen by its config.json) or given as `model_config`,
        with a cache of `max_tokens` positions."""
        pages = max(1, max_tokens // page_size)
        max_seq = max_seq_length or pages * page_size
        # the batch description of a pass travels in one piece: the five index tensors are slices of one buffer, behind which there is room for a
        # second description
        R = max_requests
        words = 2 * max_rows + 4 * R + 2 + pages
        second = (words + 1) // 2 * 2
        apart = second + second
        every = torch.zeros(MAX_TOGETHER // 2 * apart, dtype=torch.int32, device=device)
        dev = every[:second + words]
        ids, block = dev[:2 * max_rows].view(torch.int64).view(max_rows, 1), dev[2 * max_rows:words]
        qo, kv, last, slots, idx = block.split([R + 1, R + 1, R, R, pages])
        meta = MPKMetadata(mode="online_notoken", max_seq_length=max(2, max_seq), max_num_batched_requests=R, max_num_batched_tokens=max_rows, max_num_pages=pages,
                           page_size=page_size, device=device, weight_from_model=model_path is not None, model_path=model_path, model_name=model_name,
                           model_config=model_config, max_tokens_per_request=min(max_rows, 64), dtype=dtype, qo_indptr_buffer=qo, paged_kv_indptr_buffer=kv,
                           paged_kv_last_page_len_buffer=last, paged_kv_indices_buffer=idx, state_slots_buffer=slots, input_tokens=ids)
        mpk = MPK(meta)
        mpk.build()
        session = ServingSession(mpk)
        host = torch.empty(2 * max_rows + len(every), dtype=torch.int32, pin_memory=True)
        session._sampled, session._words = host[:2 * max_rows].view(torch.int64), host[2 * max_rows:]
        session._host, session._dev = session._words[:len(dev)], dev
        mpk.persistent_kernel.attach_host_batch(session._host, dev, session._sampled)
        session._fetched = True
        stats = mpk.persistent_kernel.stats()
        if stats["paired_portions"]:
            session._second, session._apart, session._together, session._every = second, apart, min(MAX_TOGETHER, stats["portions_together"]), every
            mpk.persistent_kernel.attach_more_batches(len(every) - len(dev))
        return session

    # ------------------------------------------------------------------ steps
    def logits(self) -> torch.Tensor:
        """Logits of the rows of the last pass (a view of the library's tensor)."""
        if self._view is None or self.mpk.persistent_kernel.__finalized__:  # (making one takes 5 us; of a finalized kernel's memory there is none to be had)
            with torch.inference_mode(False):
                self._view = self.mpk.model_builder.logits.to_torch()
        return self._view.detach()  # (the caller's own: what it does to its shape stays with it)

    def step(self, entries: Sequence[Tuple[object, Sequence[int]]], want: Sequence[Sequence[int]] = None):
        """Run `entries` = (request, its next tokens) as one batch.  Returns (logits, next tokens): float32 rows for the
        wanted places (want[i] indexes entries[i]'s tokens) in order, or None, and the greedy token after each entry.

        Tokens that do not fit one pass are spread over several, and how depends on `want`: in a 16-bit session the same tokens with other places
        wanted give logits, caches and so perhaps greedy tokens that differ as two orders of the same sums do (relative 5e-3 measured, each as far from
        64-bit results as the other); the same call gives the same bits.  A 32-bit session's results do not depend on `want`."""
        if len({rid for rid, _ in entries}) != len(entries):
            raise ValueError("a request may appear once in a step")
        want = want if want is not None else [[] for _ in entries]
        for rid, toks in entries:
            r = self.requests.get(rid)
            if (r.length if r else 0) + len(toks) > self.max_seq:
                raise ValueError(f"request {rid!r} would grow beyond max_seq_length={self.max_seq}")
        found = [dict.fromkeys(w) for w in want]  # place -> (logits of a run of rows, row of the run)
        greedy = [None] * len(entries)
        done = [0] * len(entries)
        # shorter portions first, so that single tokens share their pass with the head of the longer ones
        order = sorted(range(len(entries)), key=lambda i: len(entries[i][1]))

        # places in front of the first one whose logits are wanted (the last one's greedy token always is): as long as they fill passes, passes
        # are made of them alone, which are run without what only logits need, two at a time where the graph can.  A pass holds at most
        # max_requests requests: where more have tokens left, or those there are cannot fill it, such passes would come on top of the others
        # (64 entries of 3 tokens at 16 requests and 64 rows: seven passes instead of four)
        whole = [len(e[1]) for e in entries]
        ahead = self._unread_first and sum(whole) > self.max_rows
        inner = [min([n - 1, *f]) for n, f in zip(whole, found)] if ahead else whole

        def fill(ends, done):
            batch, room = [], self.max_rows
            for i in order:
                n = min(ends[i] - done[i], self.rows_per_request, room)
                if n > 0 and len(batch) < self.max_requests:
                    batch.append((i, n))
                    room -= n
            return batch, room

        def next_batch(done):
            batch, room = [], 1
            if ahead and sum(max(0, h - d) for h, d in zip(inner, done)) >= self.max_rows and sum(d < n for n, d in zip(whole, done)) <= self.max_requests:
                batch, room = fill(inner, done)
            if room:
                batch, _ = fill(whole, done)
            # (portions in the middle of their prompts, of which no row is wanted)
            return batch, all(done[i] + n < whole[i] and not any(done[i] <= p < done[i] + n for p in found[i]) for i, n in batch)

        def tokens(batch, done):
            return [(entries[i][0], entries[i][1][done[i]:done[i] + n]) for i, n in batch]

        while True:
            batch, unread = next_batch(done)
            if not batch:
                break
            if unread and self._second and self._fetched and self.mpk.persistent_kernel.profiler_tensor is None:
                # (as many neighbours as run together, two by two)
                ahead_of, then, passes = [], list(done), []
                while batch and unread and 2 * sum(n for _, n in batch) > self.max_rows and len(passes) < self._together:
                    passes.append(tokens(batch, then))
                    then = list(then)
                    for i, n in batch:
                        then[i] += n
                    ahead_of.append(then)
                    batch, unread = next_batch(then)
                pairs = len(passes) // 2
                if pairs:
                    self._passes(passes[:2 * pairs])
                    done = ahead_of[2 * pairs - 1]
                    continue
                batch, unread = next_batch(done)
            self._unread = unread
            sampled = self._pass(tokens(batch, done))
            row, wanted = 0, []
            for i, n in batch:
                lo, hi = done[i], done[i] + n
                wanted += [(row + p - lo, i, p) for p in found[i] if lo <= p < hi]
                if hi == len(entries[i][1]):
                    sampled = self.mpk.output_tokens.view(-1).tolist() if sampled is None else sampled
                    greedy[i] = sampled[row + n - 1]
                row, done[i] = row + n, hi
            wanted.sort()
            a = 0
            while a < len(wanted):  # neighbouring rows are copied together
                b = a + 1
                while b < len(wanted) and wanted[b][0] == wanted[b - 1][0] + 1:
                    b += 1
                run = self.logits()[wanted[a][0]:wanted[a][0] + b - a].to(torch.float32, copy=True)
                for k in range(a, b):
                    found[wanted[k][1]][wanted[k][2]] = (run, k - a)
                a = b
        rows = [found[i][p] for i in range(len(entries)) for p in want[i]]
        if not rows:
            return None, greedy
        run = rows[0][0]
        if len(rows) == len(run) and all(r is run and k == j for j, (r, k) in enumerate(rows)):
            return run, greedy
        return torch.stack([r[k] for r, k in rows]), greedy

    def _describe(self, batch):
        """The requests of a pass have its rows from now on: their ids, and the five index tensors one behind the other."""
        ps = self.page_size
        ids, qo, kv, last, slots, pages = [], [0], [0], [], [], []
        for rid, toks in batch:
            r = self.requests.get(rid)
            if r is None:
                r = _Request(slot=-1 if self.slots is None else self.slots.take(1)[0])
                self.requests[rid] = r
            r.length += len(toks)
            need = -(-r.length // ps) - len(r.pages)
            if need > 0:
                try:
                    r.pages += self.pool.take(need)
                except RuntimeError:
                    r.length -= len(toks)
                    raise
            ids += list(toks)
            pages += r.pages
            qo.append(len(ids))
            kv.append(len(pages))
            last.append(r.length - (len(r.pages) - 1) * ps)
            slots.append(max(r.slot, 0))
        pad = self.max_requests - len(batch)
        return ids, qo + [qo[-1]] * pad + kv + [kv[-1]] * pad + last + [0] * pad + slots + [0] * pad + pages, len(pages)

    def _put(self, at, ids, desc):
        """A description in pinned memory, from word `at` on; its length."""
        n, host = 2 * self.max_rows, (self._host if self._words is None else self._words).numpy()[at:]
        # plain numbers as they are; what else torch takes for ids (tensors of one value among it) by way of torch, which costs 6.5 us
        host[:2 * len(ids)].view("int64")[:] = ids if set(map(type, ids)) == {int} else torch.tensor(ids, dtype=torch.int64).numpy()
        host[n:n + len(desc)] = desc
        return n + len(desc)

    def _passes(self, batches):
        """Passes of which nobody reads logits or sampled tokens, an even number of them, as one launch."""
        pk, stream, words = self.mpk.persistent_kernel, torch.cuda.current_stream(self._dev.device), []
        try:
            for i, batch in enumerate(batches):
                words.append(self._put(i // 2 * self._apart + i % 2 * self._second, *self._describe(batch)[:2]))
        finally:  # (out of pages, or not ids: the passes in front have happened all the same)
            pairs = len(words) // 2
            for p in range(pairs):
                pk.enqueue_batches(words[2 * p], self._second, words[2 * p + 1], default_stream=stream, at=p * self._apart, hold=p + 1 < pairs)
            if pairs:
                pk.wait(default_stream=stream)
            if len(words) % 2:
                if pairs:  # (described behind the others: once more, where a pass by itself is)
                    self._words[:words[-1]].copy_(self._words[pairs * self._apart:pairs * self._apart + words[-1]])
                pk.enqueue_ingest(default_stream=stream, host_words=words[-1])
                pk.wait(default_stream=stream)

    def _pass(self, batch):
        unread, self._unread = self._unread, False
        ids, desc, num_pages = self._describe(batch)
        R, m = self.max_requests, self.mpk
        if self._host is not None:
            words = self._put(0, ids, desc)
            pk = m.persistent_kernel
            if self._fetched and pk.profiler_tensor is None:
                stream = torch.cuda.current_stream(self._dev.device)  # (the logits' copies', whichever device is current)
                if unread:
                    pk.enqueue_ingest(default_stream=stream, host_words=words)
                else:
                    pk.enqueue_batch(words, default_stream=stream)
                pk.wait(default_stream=stream)
                return None if unread else self._sampled.tolist()
            self._dev[:words].copy_(self._host[:words], non_blocking=True)
            if pk.profiler_tensor is not None:  # (the whole call also writes the trace)
                m()
                return None
            stream = torch.cuda.current_stream(self._dev.device) if self._dev.is_cuda else None
            if unread:
                pk.enqueue_ingest(default_stream=stream)
                pk.wait(default_stream=stream)
                return None
            pk.enqueue_steps(1, default_stream=stream)
            self._sampled.copy_(m.output_tokens.view(-1), non_blocking=True)
            pk.wait(default_stream=stream)
            return self._sampled.tolist()
        t = torch.tensor(desc, dtype=torch.int32)
        for dst, lo, n in ((m.qo_indptr_buffer, 0, R + 1), (m.paged_kv_indptr_buffer, R + 1, R + 1), (m.paged_kv_last_page_len_buffer, 2 * R + 2, R),
                           (self.state_slots, 3 * R + 2, R), (m.paged_kv_indices_buffer, 4 * R + 2, num_pages)):
            if dst is not None:
                dst[:n].copy_(t[lo:lo + n])
        m.input_tokens.view(-1)[:len(ids)].copy_(torch.tensor(ids, dtype=torch.int64))
        m()

    def end(self, rid):
        """The request is finished: its pages and its state slot go back to their pools."""
        r = self.requests.pop(rid, None)
        if r is not None:
            self.pool.give(r.pages)
            if self.slots is not None:
                self.slots.give([r.slot])

    # ------------------------------------------------------------------ greedy generation
    def generate(self, prompts: Sequence[Sequence[int]], max_new_tokens: int, eos_token_id: int = -1) -> List[List[int]]:
        """Greedy continuation of every prompt, continuously batched: a request is admitted when a batch slot and the pages
        for its whole length are free; prompts enter in portions beside the running requests' tokens, a pass a step (no two run
        together, as they do in one step over a whole prompt)."""
        out = [list(p) for p in prompts]
        need = [-(-(len(p) + max_new_tokens) // self.page_size) for p in prompts]
        for i, p in enumerate(prompts):
            if not p or need[i] > self.pool.num_pages or len(p) + max_new_tokens - 1 > self.max_seq:
                raise ValueError(f"prompt {i} is empty or its {len(p) + max_new_tokens} positions exceed the cache or max_seq_length={self.max_seq}")
        waiting, live, reserved = list(range(len(prompts))), {}, 0
        while waiting or live:
            while waiting and len(live) < self.max_requests and reserved + need[waiting[0]] <= self.pool.num_pages:
                i = waiting.pop(0)
                live[i] = 0  # tokens of out[i] already in the cache
                reserved += need[i]
            entries, room = [], self.max_rows
            for i in sorted(live, key=lambda i: len(out[i]) - live[i]):
                n = min(len(out[i]) - live[i], self.rows_per_request, room)
                if n > 0:
                    entries.append((i, n))
                    room -= n
            _, greedy = self.step([(("generate", i), out[i][live[i]:live[i] + n]) for i, n in entries])
            for (i, n), tok in zip(entries, greedy):
                live[i] += n
                if live[i] < len(out[i]):
                    continue
                out[i].append(tok)
                if len(out[i]) - len(prompts[i]) == max_new_tokens or tok == eos_token_id:
                    self.end(("generate", i))
                    reserved -= need[i]
                    del live[i]
        return out

    def finalize(self):
        self.mpk.finalize()
