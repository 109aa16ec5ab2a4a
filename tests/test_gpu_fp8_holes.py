"""fp8 prefill over block tables with holes in many key tiles, whole and split.

The fp8 staging keeps the validity of a tile's rows in a ring of four tiles and the block ids of a
piece from the piece's first tile on: the holes here lie past the fourth tile, several in a ring's
turn, in whole tiles and in pieces. Slots no request may read hold E4M3 NaN. Reference:
src/kernel/attention/prefill_attn.cu:120-150 (negative block ids are skipped).
"""
import numpy as np
import pytest
import torch

import oracle
from ccinfer_amd import prefill_attention_fp8
from ccinfer_amd import workloads as W
from tests._util import assert_attn_close, f32, say, u16
from tests.test_gpu_fp8 import quantised_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prefix,news,hq,hkv,d", [
    (1008, (70, 33, 300, 64, 5, 2, 128, 90) * 3, 16, 8, 128),   # whole: more tiles than CUs / 2
    (1008, (70, 33, 300, 64, 5, 2, 128, 90) * 3, 32, 8, 64),
    (1984, (512,), 16, 8, 128),                             # split
    (3008, (64, 1, 200), 32, 8, 128),
    (4000, (257, 100), 8, 2, 64),
])
def test_fp8_holes(gpu, prefix, news, hq, hkv, d):
    say(f"fp8 prefill with holes prefix={prefix} new={news} {hq}/{hkv} d={d}")
    w = W.prefill_prefix(device=gpu, seed=prefix + d, n_seqs=len(news), prefix=prefix, new=news,
                         share_pairs=(), hq=hq, hkv=hkv, d=d)
    for b in range(w.batch):
        w.block_table[b, 3 + b::9] = -1       # one block in 144 positions
        w.block_table[b, 40:46] = -1          # a tile and a half
    kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
    used = np.zeros(w.num_blocks * 16, bool)
    for b in range(w.batch):
        pos = np.arange(int(w.context_lens[b]))
        blk = w.block_table[b, pos // 16]
        used[(blk * 16 + pos % 16)[blk >= 0]] = True
    bad = torch.from_numpy(np.nonzero(~used)[0]).to(gpu)
    kc[bad], vc[bad] = 0x7F, 0x7F
    m = w.device_meta(gpu)
    got = prefill_attention_fp8(w.q, kc, vc, ks, vs, m["block_table"], m["query_start_loc"],
                                m["context_lens"])
    torch.cuda.synchronize()
    want = oracle.prefill_fp8(u16(w.q), kc.cpu().numpy(), vc.cpu().numpy(), ks.cpu().numpy(),
                              vs.cpu().numpy(), w.block_table, w.query_start_loc, w.context_lens)
    assert_attn_close(f32(got), want)
