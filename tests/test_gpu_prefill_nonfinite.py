"""Prefill with non-finite values: what a NaN or Inf may reach in the pipelined kernel.

Every query row attends by itself (src/kernel/attention/prefill_attn.cu:80-241: one row's
running max, sum and accumulator), so a NaN or Inf in one query row leaves every other row as
it is without it. The comparison is with the same call without the bad row, at the suite's bar:
wavefronts move the references of their rows together, which changes roundings only.

A key past a row's causal limit has probability 0 there, and 0 * NaN is NaN, so a non-finite
cache row reaches earlier rows where the kernel multiplies it at all: in the 32-key half that
holds the last key of the row's wavefront (32 query rows), never past it.
"""
import pytest
import torch

from ccinfer_amd import prefill_attention, prefill_attention_fp8
from ccinfer_amd import workloads as W
from tests._util import assert_attn_close, f32, say
from tests.test_gpu_fp8 import quantised_cache

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")

# prefix, new tokens of each request, query heads, kv heads, head dim
WHOLE = [
    (0, (10, 16, 17), 16, 8, 128),       # partial tiles: rows past the end repeat the first row
    (48, (40, 200), 3, 3, 128),
    (0, (130, 33), 32, 8, 64),
    (16, (70, 100), 4, 2, 96),           # padded head dim
]
SPLIT = [
    (1984, (512,), 16, 8, 128),
    (3008, (20, 200), 32, 8, 128),
    (4000, (257,), 8, 2, 64),
]


def _inputs(gpu, prefix, news, hq, hkv, d):
    return W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                            share_pairs=(), hq=hq, hkv=hkv, d=d)


def _calls(gpu, w, hkv, d):
    """The bf16 call and, where it exists, the fp8 call, as functions of q."""
    m = w.device_meta(gpu)
    meta = (m["block_table"], m["query_start_loc"], m["context_lens"])
    yield "bf16", lambda q: prefill_attention(q, w.k_cache, w.v_cache, *meta)
    if d in (64, 128):
        kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
        yield "fp8", lambda q: prefill_attention_fp8(q, kc, vc, ks, vs, *meta)


# prefix, new tokens, position of the bad cache row, query heads, kv heads, head dim: the rows of
# wavefronts whose last key lies in an earlier 32-key half must not change a bit.
LATER_KEYS = [
    (0, 128, 40, 4, 2, 128),
    (0, 128, 100, 4, 2, 128),
    (16, 200, 150, 3, 3, 64),
    (0, 64, 63, 4, 2, 96),
    (1136, 256, 1391, 4, 4, 128),    # split: the last piece lies above the first wavefronts
    (1136, 256, 1300, 4, 4, 128),
    (4000, 256, 4255, 3, 3, 64),
    (2992, 129, 3100, 8, 2, 96),
]


@pytest.mark.parametrize("prefix,new,pos,hq,hkv,d", LATER_KEYS)
def test_rows_before_a_bad_cache_row(gpu, prefix, new, pos, hq, hkv, d):
    w = _inputs(gpu, prefix, (new,), hq, hkv, d)
    clean = [r for r in range(new) if (prefix + r // 32 * 32 + 31) // 32 < pos // 32]
    assert 0 < len(clean) <= pos - prefix
    slot = int(w.block_table[0, pos // 16]) * 16 + pos % 16
    m = w.device_meta(gpu)
    meta = (m["block_table"], m["query_start_loc"], m["context_lens"])
    want = prefill_attention(w.q, w.k_cache, w.v_cache, *meta)
    say(f"bad cache row prefix={prefix} new={new} pos={pos} {hq}/{hkv} d={d}")
    for k, v in ((NAN, NAN), (1.0, INF), (INF, 1.0)):
        kc, vc = w.k_cache.clone(), w.v_cache.clone()
        kc[slot], vc[slot] = k, v
        got = prefill_attention(w.q, kc, vc, *meta)
        assert torch.equal(got[clean].view(torch.int16), want[clean].view(torch.int16)), (k, v)
    if d in (64, 128):
        kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
        want = prefill_attention_fp8(w.q, kc, vc, ks, vs, *meta)
        kc[slot], vc[slot] = 0x7F, 0x7F  # E4M3 NaN
        got = prefill_attention_fp8(w.q, kc, vc, ks, vs, *meta)
        assert torch.equal(got[clean].view(torch.int16), want[clean].view(torch.int16)), "fp8"


@pytest.mark.parametrize("bad", [NAN, INF])
@pytest.mark.parametrize("prefix,news,hq,hkv,d", WHOLE + SPLIT)
def test_query_rows_are_independent(gpu, prefix, news, hq, hkv, d, bad):
    w = _inputs(gpu, prefix, news, hq, hkv, d)
    starts = [int(x) for x in w.query_start_loc]
    for kind, call in _calls(gpu, w, hkv, d):
        want = f32(call(w.q))
        for b, n in enumerate(news):
            for r in sorted({0, 5, n // 2, n - 1}):
                row, head = starts[b] + r, (r + b) % hq
                say(f"bad query row {kind} {bad} {hq}/{hkv} d={d} prefix={prefix} new={n} row={r}")
                q = w.q.clone()
                q[row, head] = bad
                got = f32(call(q))
                if bad != bad:
                    assert (got[row, head] != got[row, head]).all()
                got[row, head] = want[row, head]
                assert_attn_close(got, want, f"{kind}, bad row {r} of {n}")


@pytest.mark.parametrize("prefix,news,hq,hkv,d", WHOLE[1:2] + SPLIT + [
    (1136, (64, 256), 4, 4, 128),
    (2992, (129,), 8, 2, 96),
])
def test_infinite_value_row(gpu, prefix, news, hq, hkv, d):
    """A cached V row of +Inf under finite scores makes every output +Inf (its probability is
    positive, the other values finite), never NaN: no partial sum is multiplied by 0."""
    w = _inputs(gpu, prefix, news, hq, hkv, d)
    m = w.device_meta(gpu)
    meta = (m["block_table"], m["query_start_loc"], m["context_lens"])
    for pos in (0, prefix - 1):
        say(f"infinite value row prefix={prefix} new={news} {hq}/{hkv} d={d} pos={pos}")
        v = w.v_cache.clone()
        for b in range(len(news)):
            v[int(w.block_table[b, pos // 16]) * 16 + pos % 16] = INF
        assert (f32(prefill_attention(w.q, w.k_cache, v, *meta)) == INF).all()
