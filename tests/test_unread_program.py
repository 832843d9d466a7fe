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
