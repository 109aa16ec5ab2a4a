"""Workspaces of the Python prefill calls: with and without the memory for split tiles."""
import pytest
import torch

from ccinfer_amd import (CcinferError, prefill_attention, prefill_attention_fp8,
                         prefill_workspace_size)
from ccinfer_amd import workloads as W
from tests._util import assert_attn_close, f32, say
from tests.test_gpu_fp8 import quantised_cache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(16, 8, 128), (8, 2, 64)])
def test_workspace_without_split_memory(gpu, hq, hkv, d):
    """A workspace smaller than the size query by the memory for split tiles is taken and runs
    the tiles whole; one too small for those is refused as an invalid argument."""
    say(f"prefill workspace {hq}/{hkv} d={d}")
    w = W.prefill_prefix(device=gpu, seed=d, n_seqs=1, prefix=4000, new=(200,), share_pairs=(),
                         hq=hq, hkv=hkv, d=d)
    m = w.device_meta(gpu)
    meta = (m["block_table"], m["query_start_loc"], m["context_lens"])
    kc, vc, ks, vs = quantised_cache(gpu, w, hkv, d)
    size = prefill_workspace_size(1, 200, w.mbpr, hq, hkv, d)
    rows = 2 * (-(-w.q.numel() * 2 // 256) * 256)  # the query's copies, not needed here
    small = torch.empty(size - rows - (1 << 20), dtype=torch.uint8, device=gpu)
    for call in (lambda ws: prefill_attention(w.q, w.k_cache, w.v_cache, *meta, workspace=ws),
                 lambda ws: prefill_attention_fp8(w.q, kc, vc, ks, vs, *meta, workspace=ws)):
        split, whole = call(None), call(small)
        assert_attn_close(f32(whole), f32(split))
        assert not torch.equal(split, whole)
        with pytest.raises(CcinferError) as e:
            call(small[:64])
        assert e.value.code == 6
