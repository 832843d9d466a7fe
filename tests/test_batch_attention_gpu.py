"""Attention of many requests (a workgroup takes two units at a time where contexts are about equally long, four wavefronts take one
otherwise) and sampling, at the sizes where their splits change, against plain torch in 32 bits."""
import pytest
import torch

from helpers import make_meta, make_mpk

pytestmark = pytest.mark.gpu
D = 128


def _lens(kind, R):
    g = torch.Generator().manual_seed(R)
    if kind == "near":  # up to 256 positions above the average
        return torch.randint(1, 300, (R,), generator=g).tolist()
    if kind == "one long":
        return [40] * (R - 1) + [900]
    return [int(kind)] * R


# (33 requests of 8 kv heads: 264 units on 256 workgroups; the second of a pair is missing nearly everywhere)
@pytest.mark.parametrize("R,kind,new,ps,nkv,qpk", [(33, "near", 1, 16, 8, 4), (64, "near", 1, 64, 8, 4), (64, "1", 1, 16, 8, 4), (64, "17", 1, 4, 8, 4), (64, "300", 1, 1, 8, 4), (50, "near", 1, 16, 8, 8),
                                                   (64, "one long", 1, 64, 8, 4), (40, "near", 2, 16, 8, 4), (64, "520", 1, 2048, 5, 8)])
def test_attention_of_many_requests(R, kind, new, ps, nkv, qpk):
    """`new`: rows of the first requests, as many as 64 rows allow."""
    _check(_lens(kind, R), new, ps, nkv, qpk, 7 * R + len(kind))


# (requests of 1024 pages fill a unit's page list when two are taken at a time, of 1025 are taken one at a time; two, three and five turns of a
# workgroup, of which the longest contexts just allow two units at a time or just do not, on either side of the line that the rule draws)
@pytest.mark.parametrize("lens,ps,nkv,qpk,max_seq", [([1024] * 64, 1, 5, 8, 1024), ([1024] * 64, 1, 5, 8, 1025), ([1024] + [1000] * 63, 1, 8, 4, 1024),
                                                     ([20] * 63 + [430], 16, 8, 4, 1024), ([20] * 63 + [500], 16, 8, 4, 1024), ([455] * 64, 16, 12, 4, 1024), ([480] * 64, 16, 12, 4, 1024),
                                                     ([345] * 64, 16, 12, 8, 1024), ([370] * 64, 16, 12, 8, 1024), ([980] * 64, 16, 20, 4, 1024), ([1000] * 64, 16, 20, 4, 1024)])
def test_attention_at_the_limits_of_two_units_at_a_time(lens, ps, nkv, qpk, max_seq):
    _check(lens, 1, ps, nkv, qpk, sum(lens), max_seq)


def _check(lens, new, ps, nkv, qpk, seed, max_seq=None):
    import mirage as mi
    R, cached = len(lens), [n - 1 for n in lens]
    rows = [new if i < (64 - R) // max(1, new - 1) and new > 1 else 1 for i in range(R)]
    total, longest = sum(rows), max(c + n for c, n in zip(cached, rows))
    need = [-(-(c + n) // ps) for c, n in zip(cached, rows)]
    pages, max_seq = sum(need), max_seq or -(-(longest + 1) // ps) * ps
    meta = make_meta(R, max_seq, 64, R, pages)
    pk = make_mpk(meta, max_seq, 64, R, pages, ps, mode="onepass")
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()
    qkv, kc, vc, out = rnd(64, nkv * (qpk + 2) * D), rnd(pages, ps, nkv, D), rnd(pages, ps, nkv, D), torch.zeros(64, nkv * qpk * D, dtype=torch.bfloat16, device="cuda")
    k0, v0 = kc.clone(), vc.clone()
    pk.paged_attention_layer(input=pk.attach_input(qkv, "qkv"), k_cache=pk.attach_input(kc, "kc"), v_cache=pk.attach_input(vc, "vc"), q_norm=None, k_norm=None, cos_pos_embed=None,
                             sin_pos_embed=None, output=pk.attach_input(out, "out"), grid_dim=(R, nkv, 1), block_dim=(128, 1, 1))
    pk.compile()
    order = torch.randperm(pages, generator=g)
    first = torch.tensor([0] + need).cumsum(0)
    qo = torch.tensor([0] + rows).cumsum(0)
    i32 = lambda t: torch.as_tensor(t).to(torch.int32)
    meta["qo_indptr_buffer"].copy_(i32(qo))
    meta["paged_kv_indptr_buffer"].copy_(i32(first))
    meta["paged_kv_indices_buffer"].copy_(i32(order))
    meta["paged_kv_last_page_len_buffer"].copy_(i32([c + n - (p - 1) * ps for c, n, p in zip(cached, rows, need)]))
    torch.cuda.synchronize()
    pk()
    x = qkv.float().view(64, nkv, qpk + 2, D)
    for r in range(R):
        own = order[first[r]:first[r + 1]].cuda()
        a, n, L = int(qo[r]), rows[r], cached[r]
        K, V = (torch.cat([c[own].float().view(-1, nkv, D)[:L], x[a:a + n, :, qpk + i]]) for i, c in enumerate((k0, v0)))
        assert torch.equal(kc[own].view(-1, nkv, D)[L:L + n], qkv.view(64, nkv, qpk + 2, D)[a:a + n, :, qpk]), f"appended keys of request {r}"
        assert torch.equal(vc[own].view(-1, nkv, D)[L:L + n], qkv.view(64, nkv, qpk + 2, D)[a:a + n, :, qpk + 1]), f"appended values of request {r}"
        for t in range(n):
            end = L + t + 1
            s = (x[a + t, :, :qpk, None] * K[:end].transpose(0, 1)[:, None]).sum(-1) / D ** 0.5
            want = (s.softmax(-1)[..., None] * V[:end].transpose(0, 1)[:, None]).sum(2)
            got = out[a + t].view(nkv, qpk, D).float()
            # one rounding to bf16; weights of cached positions keep 16 bits, scores come from 32-bit sums
            bound = want.abs() * 2.0 ** -8 + float(V.abs().max()) * 2.0 ** -13
            assert bool(((got - want).abs() <= bound).all()), f"request {r} token {t}: off by {float((got - want).abs().max())}"
    assert bool((out[total:] == 0).all()) and pk.stats()["aborted"] == 0
    pk.finalize()


# (pieces of sixteen bytes, five of them a lane and turn: 163840 logits; rows that do not begin on sixteen bytes)
@pytest.mark.parametrize("V", [1, 8, 1000, 1001, 4104, 163848, 200001])
@pytest.mark.parametrize("B", [1, 17, 64])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_sampling(B, V, dtype):
    """The first of the largest values, wherever it lies; rows of the lowest values there are."""
    meta = make_meta(B, 64, B, B, B)
    pk = make_mpk(meta, 64, B, B, B, 64, mode="onepass")
    logits = torch.randn(B, V, generator=torch.Generator().manual_seed(V + B)).to(dtype).cuda()
    top = torch.finfo(dtype).max
    at = [(i * V) // 7 + i for i in range(7)] + [0, V - 1]
    want = []
    for r in range(B):
        if r == 1:
            logits[r] = -top
        elif V > 1:
            a, b = min(at[r % 9], V - 1), min(at[(r + 4) % 9], V - 1)
            logits[r, a] = logits[r, b] = top
    if dtype == torch.float32:  # (32-bit sampling runs beside other 32-bit stages)
        f32 = lambda name, *shape: pk.attach_input(torch.zeros(*shape, device="cuda"), name)
        pk.embed_scaled_layer(pk.attach_input(meta["input_tokens"], "ids"), f32("table", 4, 64), f32("rows32", B, 64), f32("rows", B, 64), 1.0)
    pk.argmax_layer(input=pk.attach_input(logits, "logits"), output=pk.attach_input(meta["output_tokens"], "out"), grid_dim=(1, 1, 1), block_dim=(128, 1, 1))
    pk.compile()
    for M in sorted({1, B // 2 + 1, B}):
        meta["output_tokens"].fill_(-5)
        torch.cuda.synchronize()
        pk.run_once(list(range(M)), [0] * M)
        want = [int((logits[r] == logits[r].max()).nonzero()[0]) for r in range(M)]
        assert meta["output_tokens"].view(-1).tolist() == want + [-5] * (B - M)
    pk.finalize()
