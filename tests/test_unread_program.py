"""Which stages at a program's end an iteration whose logits and sampled tokens nobody reads leaves out (marked in the listing), on
host-only graphs: none of what a later iteration reads before it is written again."""
import pytest
import torch

import mirage as mi
from helpers import make_meta

B, R, PS, PAGES, SEQ = 8, 2, 64, 4, 128


def _pk(mode="onepass"):
    return mi.PersistentKernel(mode=mode, world_size=1, mpi_rank=0, num_workers=256, num_local_schedulers=0, num_remote_schedulers=0, max_seq_length=SEQ, max_num_batched_requests=R,
                               max_num_batched_tokens=B, max_num_pages=PAGES, page_size=PS, meta_tensors=make_meta(R, SEQ, B, R, PAGES, device="cpu"), profiler_tensor=None, trace_name=None,
                               spec_decode_config=None, use_cutlass_kernel=False, eos_token_id=2)


def _attach(pk, name, *shape, dtype=torch.bfloat16):
    """(the caller's tensor: rows and columns of it can be attached beside it)"""
    t = torch.zeros(*shape, dtype=dtype)
    return pk.attach_input(t, name), t


def _skipped(pk):
    """One entry per stage: does an unread iteration leave it out?"""
    return [line.endswith(" unread=skip") for line in pk.describe_program().splitlines()]


def _linear(pk, x, n, out, name="w", res=None):
    w, _ = _attach(pk, name, n, x.dim(1))
    if res is None:
        pk.linear_layer(input=x, weight=w, output=out, grid_dim=(1, 1, 1), block_dim=(128, 1, 1))
    else:
        pk.linear_with_residual_layer(input=x, weight=w, residual=res, output=out, grid_dim=(1, 1, 1), block_dim=(256, 1, 1))


@pytest.mark.parametrize("carried", [False, True])
def test_query_latents_written_for_the_next_iteration(carried):
    pk, H, rank, rot = _pk(), 2, 32, 32
    q, _ = _attach(pk, "q", B, H * 64)
    ql, _ = _attach(pk, "ql", B, H * rank)
    other, _ = _attach(pk, "other", B, H * rank)
    cache, _ = _attach(pk, "cache", PAGES, PS, rank + rot)
    cos, sin = (_attach(pk, n, SEQ, rot // 2, dtype=torch.float32)[0] for n in ("cos", "sin"))
    out, _ = _attach(pk, "out", B, H * rank)
    pk.latent_attention_layer(q, ql, cache, cos, sin, out, H, rank, rot, 64, 0, 1.0)
    _linear(pk, out, H * rank, ql if carried else other)
    assert _skipped(pk) == [False, False, not carried]


def test_norm_that_finishes_the_sum_of_the_stage_in_front():
    """The linear behind a convolution over time keeps the request's ring and runs in every iteration; the sum over its slices of K is
    left to the norm behind it, which therefore runs as well."""
    pk, n = _pk(), 64
    x, xo, xp, g = (_attach(pk, k, *s, dtype=torch.float32)[0] for k, s in (("x", (B, n)), ("xo", (B, n)), ("xp", (B, n)), ("g", (n,))))
    y, rows, conv, z, out, last = (_attach(pk, k, B, n)[0] for k in ("y", "rows", "conv", "z", "out", "last"))
    taps, ring = _attach(pk, "taps", 4, n)[0], _attach(pk, "ring", R, 4, n)[0]
    slots, _ = _attach(pk, "slots", R, dtype=torch.int32)
    pk.residual_prenorm_layer(y, x, xo, rows, weight=g)
    pk.ring_conv_layer(rows, taps, ring, slots, conv, identity=True)
    _linear(pk, conv, n, z)
    pk.residual_prenorm_layer(z, xo, xp, out, weight=g)
    _linear(pk, out, n, last, "w2")
    kinds = [line.split()[1] for line in pk.describe_program().splitlines()]
    assert kinds == ["MX_PRENORM[multi-token", "DU_CONV[portions]", "LINEAR", "MX_PRENORM[multi-token", "LINEAR"]
    assert "sum=next" in pk.describe_program().splitlines()[2]
    assert _skipped(pk) == [False] * 4 + [True]


def _rows(pk, t, name):
    """Some rows of a tensor attached already."""
    return pk.attach_input(t, name)


def _chain(build):
    """A small program in bf16: `build(pk, x, y, S)` records it over row tensors x, y [B, 64] and S [4 B, 64], whose rows can be attached by themselves."""
    pk = _pk()
    x, y = _attach(pk, "x", B, 64)[0], _attach(pk, "y", B, 64)[0]
    build(pk, x, y, torch.zeros(4 * B, 64, dtype=torch.bfloat16))
    return _skipped(pk)


@pytest.mark.parametrize("parent", [False, True])
def test_halves_of_a_tensor_attached_beside_it(parent):
    """The first half is written anew in every iteration, the second one is a running sum."""
    def build(pk, x, y, S):
        if parent:
            _rows(pk, S, "S")
        first, second = _rows(pk, S[:B], "first"), _rows(pk, S[B:2 * B], "second")
        _linear(pk, x, 64, first)
        _linear(pk, first, 64, second, "w2", res=second)
    assert _chain(build) == [False, False]


@pytest.mark.parametrize("shift", [0, 1, B - 1, B])
def test_rows_of_neighbouring_tokens(shift):
    """A stage reads rows that overlap, `shift` tokens further on, those that the program's first stage writes; the last one writes all of them."""
    def build(pk, x, y, S):
        _rows(pk, S[2:], "other part")
        _linear(pk, x, 64, _rows(pk, S[:B], "a"))
        _linear(pk, _rows(pk, S[shift:shift + B], "b"), 64, y, "w2")
        _linear(pk, y, 64, _rows(pk, S[:B], "c"), "w3")
    # (with shift B the stage reads nothing that another one writes)
    assert _chain(build) == [shift in (0, B)] * 3


@pytest.mark.parametrize("n", [64, 128])
def test_columns_carried_beside_rewritten_ones(n):
    """The first stage writes n columns of rows of 128, all of which are read; the last one writes all."""
    pk = _pk()
    x, y, wide = _attach(pk, "x", B, 64)[0], _attach(pk, "y", B, 64)[0], _attach(pk, "wide", B, 128)[0]
    _linear(pk, x, n, wide)
    _linear(pk, wide, 64, y, "w2")
    _linear(pk, y, 128, wide, "w3")
    assert _skipped(pk) == [n == 128] * 3


def test_columns_that_nobody_writes():
    """Rows of 128 of which all stages write the same 64: the others are the caller's."""
    pk = _pk()
    x, y, wide = _attach(pk, "x", B, 64)[0], _attach(pk, "y", B, 64)[0], _attach(pk, "wide", B, 128)[0]
    _linear(pk, x, 64, wide)
    _linear(pk, wide, 64, y, "w2")
    _linear(pk, y, 64, wide, "w3")
    assert _skipped(pk) == [True] * 3


def test_token_ids_sampled_for_the_next_iteration():
    pk = _pk()
    ids, _ = _attach(pk, "ids", B, 1, dtype=torch.int64)
    table, x, logits = _attach(pk, "table", 32, 64)[0], _attach(pk, "x", B, 64)[0], _attach(pk, "logits", B, 32)[0]
    pk.embed_layer(ids, table, x, grid_dim=(1, 1, 1), block_dim=(128, 1, 1), input_source=1)
    _linear(pk, x, 32, logits)
    pk.argmax_layer(input=logits, output=ids, grid_dim=(1, 1, 1), block_dim=(128, 1, 1))
    assert _skipped(pk) == [False] * 4


@pytest.mark.parametrize("used", [False, True])
def test_padding(used):
    """Rows of 64 values of which 60 are real: padding is zero before and after a norm, unless another stage uses those columns."""
    pk = _pk()
    x, xo, g = (_attach(pk, k, *s, dtype=torch.float32)[0] for k, s in (("x", (B, 64)), ("xo", (B, 64)), ("g", (64,))))
    ids, _ = _attach(pk, "ids", B, 1, dtype=torch.int64)
    table, rows, z = _attach(pk, "table", 32, 60)[0], _attach(pk, "rows", B, 64)[0], _attach(pk, "z", B, 64)[0]
    pk.embed_scaled_layer(ids, table, x, rows)
    _linear(pk, rows, 64, z)
    if used:
        _linear(pk, z, 64, rows, "w2")
    pk.residual_rmsnorm_layer(None, x, g, xo, rows, width=60)
    assert _skipped(pk) == ([False] * 4 if used else [False, True, True])


@pytest.mark.parametrize("family,kind", [("suborax", "even"), ("suborax", "odd"), ("suborax", "one_layer"), ("dodonex", "even"), ("dodonex", "odd"), ("bukatar", "even"), ("bukatar", "odd"), ("bukatar", "wide"),
                                         ("vizonex", "even"), ("vizonex", "odd"), ("vizonex", "taps")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_models_end_behind_their_last_cache_or_state(family, kind, dtype):
    import importlib
    from mirage.mpk import MPK, MirageModelConfig, MPKMetadata
    h = importlib.import_module(family + "_helpers")
    m = MPK(MPKMetadata(mode="online_notoken", max_seq_length=256, max_num_batched_requests=4, max_num_batched_tokens=64, max_num_pages=8, page_size=64, device="cpu", num_workers=256, dtype=dtype,
                        model_config=MirageModelConfig(architecture=h.CONFIGS[kind], state_dict=h.weights(h.CONFIGS[kind]))))
    m.build()
    pk = m.persistent_kernel
    kinds, skipped = [line.split()[1] for line in pk.describe_program().splitlines()], _skipped(pk)
    first = skipped.index(True)
    assert all(skipped[first:]) and kinds[first - 1].split("[")[0] in ("FX_ATTN", "MX_LATENT_MERGE", "MX_DELTA_OUT", "HY_SCAN", "DU_SCAN")
    assert not any(k.startswith(("FX_", "MX_LATENT", "MX_DELTA", "HY_SCAN", "HY_CONV", "DU_")) and not k.startswith("FX_ADDNORM") for k in kinds[first:])


@pytest.mark.parametrize("carried", [False, True])
def test_shares_written_for_the_next_iteration(carried):
    """The router writes the shares of the chosen experts, which a norm at the program's beginning weights its summands with."""
    pk, E, top, n = _pk(), 4, 2, 32
    shares, _ = _attach(pk, "shares", B, 4, dtype=torch.float32)
    other, _ = _attach(pk, "other", B, 4, dtype=torch.float32)
    y, _ = _attach(pk, "y", B, top * n)
    x, xo = (_attach(pk, k, B, n, dtype=torch.float32)[0] for k in ("x", "xo"))
    rows, _ = _attach(pk, "rows", B, n)
    pk.residual_prenorm_layer(y, x, xo, rows, slot_weights=shares, slots=top, slot_columns=n)
    logits, _ = _attach(pk, "logits", B, E, dtype=torch.float32)
    ids, _ = _attach(pk, "ids", B, top, dtype=torch.int32)
    pk.expert_route_layer(logits, ids, shares if carried else other, E, top)
    w, _ = _attach(pk, "w", E * n, n)
    out, _ = _attach(pk, "out", B, top * n)
    pk.expert_linear_layer(rows, w, ids, out, E, top, n, n, n)
    assert _skipped(pk) == [not carried] * 3
