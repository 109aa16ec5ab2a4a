"""Edges of the pipelined prefill kernel (head dims 64 / 128, bf16 and fp8) against the oracle.

The kernel walks 64-key tiles in 32-key halves, three stages deep, with rings of three tiles:
the cases put the last key, the causal diagonal and the wavefronts' last rows on and beside
the edges of halves, tiles and rings, for each split of a workgroup into heads and rows, and
let the scores of a row grow or fall along the keys so that the reference of its softmax
moves often, or never. Reference behaviour: src/kernel/attention/prefill_attn.cu:80-241.
Bar: max-abs <= 2e-2, mean-abs <= 2e-3 on every row; slots no request may read are poisoned.
"""
import numpy as np
import pytest
import torch

import oracle
from ccinfer_amd import _lib, prefill_attention, prefill_attention_fp8, prefill_workspace_size
from ccinfer_amd import workloads as W
from tests._util import assert_attn_close, f32, say, u16
from tests.test_gpu_fp8 import quantised_cache

pytestmark = pytest.mark.gpu

# new tokens per request; the prefix goes in front of each
SHAPES = [
    (0, (2, 31, 32, 33, 63, 64, 65)),
    (16, (47, 48, 49, 95, 112, 113)),
    (64, (64, 127, 128, 129, 192, 193)),
    (176, (15, 16, 17, 80, 257)),
    (1024, (2, 63, 320)),
]


def _ramp(w, kind):
    """Scales the K rows along each request's positions: a row's scores grow or fall."""
    if kind == "flat":
        return
    for b in range(w.batch):
        n = int(w.context_lens[b])
        pos = np.arange(n)
        slot = w.block_table[b, pos // 16].astype(np.int64) * 16 + pos % 16
        f = 0.2 + 6.0 * pos / n if kind == "grow" else 6.2 - 6.0 * pos / n
        idx = torch.from_numpy(slot).to(w.k_cache.device)
        f = torch.from_numpy(f.astype(np.float32)).to(w.k_cache.device)
        w.k_cache[idx] = (w.k_cache[idx].float() * f[:, None, None]).to(torch.bfloat16)


def _poison(w, k, v, kbad, vbad):
    used = np.zeros(w.num_blocks * 16, bool)
    for b in range(w.batch):
        pos = np.arange(int(w.context_lens[b]))
        used[w.block_table[b, pos // 16] * 16 + pos % 16] = True
    rows = torch.from_numpy(np.nonzero(~used)[0]).to(k.device)
    k[rows] = kbad
    v[rows] = vbad


@pytest.mark.parametrize("kind", ["flat", "grow", "fall"])
@pytest.mark.parametrize("d,hq,hkv", [(128, 3, 3), (128, 4, 2), (128, 8, 2), (64, 4, 4), (64, 8, 2),
                                      (96, 4, 2)])
def test_bf16_edges(gpu, d, hq, hkv, kind):
    for prefix, news in SHAPES:
        say(f"pipelined prefill d={d} {hq}/{hkv} {kind} prefix={prefix} new={news}")
        w = W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                             share_pairs=(), hq=hq, hkv=hkv, d=d)
        _ramp(w, kind)
        _poison(w, w.k_cache, w.v_cache, float("nan"), float("inf"))
        m = w.device_meta(gpu)
        out = prefill_attention(w.q, w.k_cache, w.v_cache, m["block_table"], m["query_start_loc"],
                                m["context_lens"])
        torch.cuda.synchronize()
        want = oracle.prefill(u16(w.q), u16(w.k_cache), u16(w.v_cache), w.block_table,
                              w.query_start_loc, w.context_lens)
        assert_attn_close(f32(out), want, f"prefix {prefix}")


@pytest.mark.parametrize("kind", ["flat", "grow"])
@pytest.mark.parametrize("d,hq,hkv", [(128, 4, 2), (64, 3, 3), (64, 8, 2)])
def test_fp8_edges(gpu, d, hq, hkv, kind):
    for prefix, news in SHAPES:
        say(f"pipelined fp8 prefill d={d} {hq}/{hkv} {kind} prefix={prefix} new={news}")
        w = W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                             share_pairs=(), hq=hq, hkv=hkv, d=d)
        _ramp(w, kind)
        kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
        _poison(w, kc, vc, 0x7F, 0x7F)  # E4M3 NaN
        m = w.device_meta(gpu)
        out = prefill_attention_fp8(w.q, kc, vc, ks, vs, m["block_table"], m["query_start_loc"],
                                    m["context_lens"])
        torch.cuda.synchronize()
        want = oracle.prefill_fp8(u16(w.q), kc.cpu().numpy(), vc.cpu().numpy(), ks.cpu().numpy(),
                                  vs.cpu().numpy(), w.block_table, w.query_start_loc,
                                  w.context_lens)
        assert_attn_close(f32(out), want, f"prefix {prefix}")


# Launches that fill at most half the CUs split their tiles' key ranges (prefill_attn.hip, "Split
# tiles"): prefix, new tokens of each request, query heads, kv heads, head dim.
SPLIT = [
    (1136, (17,), 16, 8, 128),
    (1984, (512,), 16, 8, 128),
    (3008, (64, 1, 200), 32, 8, 128),
    (9008, (40, 1), 4, 4, 64),
    (4000, (257, 100), 8, 2, 64),
    (2992, (129,), 8, 2, 96),
    (1200, (2, 3, 1, 5, 6), 1, 1, 128),
    (0, (1600,), 4, 2, 128),
]


@pytest.mark.parametrize("holes", [False, True])
@pytest.mark.parametrize("prefix,news,hq,hkv,d", SPLIT)
def test_split_tiles(gpu, prefix, news, hq, hkv, d, holes):
    say(f"split prefill prefix={prefix} new={news} {hq}/{hkv} d={d} holes={holes}")
    w = W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                         share_pairs=(), hq=hq, hkv=hkv, d=d)
    _ramp(w, "grow")
    if holes:
        w.block_table[0, 3:9] = -1
        w.block_table[-1, w.block_table.shape[1] // 2 + 1] = -1
    m = w.device_meta(gpu)
    size = prefill_workspace_size(w.batch, int(w.query_start_loc[-1]), w.mbpr, hq, hkv, d)
    outs = []
    for fill in (0xFF, 0x3C):  # the workspace needs no initialisation
        ws = torch.full((size,), fill, dtype=torch.uint8, device=gpu)
        outs.append(prefill_attention(w.q, w.k_cache, w.v_cache, m["block_table"],
                                      m["query_start_loc"], m["context_lens"], workspace=ws))
    # a workspace without room for the partials (the size also holds two copies of the q rows)
    rows = 2 * (-(-w.q.numel() * 2 // 256) * 256)
    ws = torch.empty(size - rows - (1 << 20), dtype=torch.uint8, device=gpu)
    whole = torch.empty_like(w.q)
    code = _lib.load().ccinfer_prefill_attention(
        *(x.data_ptr() for x in (w.q, w.k_cache, w.v_cache, m["block_table"], m["query_start_loc"],
                                 m["context_lens"], whole)),
        w.batch, w.q.shape[0], w.mbpr, hq, hkv, d, 16, ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream().cuda_stream)
    assert code == 0
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    want = oracle.prefill(u16(w.q), u16(w.k_cache), u16(w.v_cache), w.block_table,
                          w.query_start_loc, w.context_lens)
    assert_attn_close(f32(outs[0]), want, "split")
    assert_attn_close(f32(whole), want, "whole")
    assert not torch.equal(outs[0], whole)  # the batch did split
    if not holes and d in (64, 128):
        kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
        o8 = prefill_attention_fp8(w.q, kc, vc, ks, vs, m["block_table"], m["query_start_loc"],
                                   m["context_lens"])
        torch.cuda.synchronize()
        want = oracle.prefill_fp8(u16(w.q), kc.cpu().numpy(), vc.cpu().numpy(), ks.cpu().numpy(),
                                  vs.cpu().numpy(), w.block_table, w.query_start_loc,
                                  w.context_lens)
        assert_attn_close(f32(o8), want, "split fp8")
