"""Prefill launches that may split their tiles, over block tables wider than the lengths need.

Whether a small batch splits is decided from the lengths, on the device; the table's width only
allows it. Short prompts on a wide table therefore run whole tiles, and must give the bits of the
same call on a table that allows no split. With single-token requests, past 2,048 positions the
decode items' merge and the tiles' run in one launch.
"""
import numpy as np
import pytest
import torch

import oracle
from ccinfer_amd import prefill_attention, prefill_attention_fp8
from ccinfer_amd import workloads as W
from tests._util import assert_attn_close, f32, say, u16
from tests.test_gpu_fp8 import quantised_cache

pytestmark = pytest.mark.gpu


def _work(gpu, prefix, news, hq, hkv, d):
    return W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                            share_pairs=(), hq=hq, hkv=hkv, d=d)


def _widen(w, width):
    table = np.full((w.batch, width), -1, np.int32)
    table[:, :w.block_table.shape[1]] = w.block_table
    return torch.from_numpy(table)


@pytest.mark.parametrize("width", [128, 129, 2048])  # decode items inside the tile launch, or not
@pytest.mark.parametrize("prefix,news,hq,hkv,d", [
    (0, (200,), 16, 8, 128),
    (0, (2,), 32, 8, 128),
    (48, (64, 30, 129), 16, 8, 128),
    (32, (20, 400, 77), 32, 8, 64),
    (16, (33, 300), 8, 2, 96),
])
def test_short_prompts_on_wide_tables(gpu, prefix, news, hq, hkv, d, width):
    say(f"wide table {width} prefix={prefix} new={news} {hq}/{hkv} d={d}")
    w = _work(gpu, prefix, news, hq, hkv, d)
    m = w.device_meta(gpu)
    wide = _widen(w, width).to(gpu)
    lens = (m["query_start_loc"], m["context_lens"])
    tight = prefill_attention(w.q, w.k_cache, w.v_cache, m["block_table"], *lens)
    got = prefill_attention(w.q, w.k_cache, w.v_cache, wide, *lens)
    assert torch.equal(got.view(torch.int16), tight.view(torch.int16))
    if d in (64, 128):
        kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
        tight = prefill_attention_fp8(w.q, kc, vc, ks, vs, m["block_table"], *lens)
        got = prefill_attention_fp8(w.q, kc, vc, ks, vs, wide, *lens)
        assert torch.equal(got.view(torch.int16), tight.view(torch.int16))


@pytest.mark.parametrize("width", [None, 2048])
@pytest.mark.parametrize("prefix,news,hq,hkv,d", [
    (1904, (1, 100, 1), 16, 8, 128),                 # up to 2,048 positions
    (2608, (1, 100, 1, 1, 1, 300), 16, 8, 128),      # flat plan of the decode items
    (2608, (1, 40), 32, 8, 64),                      # fixed splits
    (4000, (1, 60, 1), 8, 2, 96),
    (5008, (1, 7) + (1,) * 5, 8, 4, 32),
    (1504, (2, 1) * 32, 1, 1, 128),                  # the most requests of a launch that splits
    (1504, (2, 1) * 32 + (2,), 1, 1, 128),           # one more
    (1504, (1,) * 9, 1, 1, 128),                     # single-token requests only
])
def test_mixed_batches(gpu, prefix, news, hq, hkv, d, width):
    say(f"mixed, wide table {width} prefix={prefix} new={news} {hq}/{hkv} d={d}")
    w = _work(gpu, prefix, news, hq, hkv, d)
    m = w.device_meta(gpu)
    table = m["block_table"] if width is None else _widen(w, width).to(gpu)
    lens = (m["query_start_loc"], m["context_lens"])
    out = torch.empty_like(w.q)
    call = lambda: prefill_attention(w.q, w.k_cache, w.v_cache, table, *lens, output=out)
    call()
    first = out.clone()
    want = oracle.prefill(u16(w.q), u16(w.k_cache), u16(w.v_cache), w.block_table,
                          w.query_start_loc, w.context_lens)
    assert_attn_close(f32(first), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), first.view(torch.int16))


def test_lengths_change_between_replays(gpu):
    """A captured call splits or not by the lengths it finds at each replay; a request whose
    context is shorter than its query, and rows of no request, stay as they are."""
    say("prefill split decided at replay")
    w = _work(gpu, 3008, (40, 200), 16, 8, 128)
    m = w.device_meta(gpu)
    ctx, out = m["context_lens"].clone(), torch.empty_like(w.q)
    call = lambda: prefill_attention(w.q, w.k_cache, w.v_cache, m["block_table"],
                                     m["query_start_loc"], ctx, output=out)
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for lens in ((3048, 3208), (100, 260), (3048, 199), (39, 199), (41, 3208)):
        ctx.copy_(torch.tensor(lens, dtype=torch.int32))
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        want = oracle.prefill(u16(w.q), u16(w.k_cache), u16(w.v_cache), w.block_table,
                              w.query_start_loc, np.asarray(lens, np.int32))
        for b, (lo, hi) in enumerate(((0, 40), (40, 240))):
            if lens[b] < hi - lo:
                assert (out[lo:hi] == 7.0).all()
            else:
                assert_attn_close(f32(out[lo:hi]), want[lo:hi], str(lens))
