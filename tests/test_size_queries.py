"""The workspace size queries of the Python interface: what they take and what they remember."""
import numpy as np
import pytest
import torch

import ccinfer_amd as cc
from ccinfer_amd import ops

QUERIES = [
    (cc.decode_workspace_size, (4, 256, 16, 8, 128)),
    (cc.decode_shared_workspace_size, (4, 256, 16, 8, 128)),
    (cc.prefill_workspace_size, (4, 600, 256, 16, 8, 128)),
]


@pytest.mark.parametrize("query,args", QUERIES)
def test_whole_numbers_of_any_kind(query, args):
    """Anything with __index__ counts by its value, also a 0-d array, which cannot be hashed."""
    want = query(*args)
    for kind in (np.int64, np.array, torch.tensor):
        assert query(*(kind(a) for a in args)) == want
    assert query(*args, cache_block_size=np.array(16)) == want
    with pytest.raises(Exception):
        query(float(args[0]), *args[1:])


@pytest.mark.parametrize("query,args", QUERIES)
def test_a_changed_tensor_is_read_again(query, args):
    batch = torch.tensor(args[0])
    assert query(batch, *args[1:]) == query(*args)
    batch.fill_(64)
    assert query(batch, *args[1:]) == query(64, *args[1:]) != query(*args)


@pytest.mark.parametrize("query,args", QUERIES)
def test_remembered_size(query, args):
    """The calls' own look-up: plain ints are remembered, other block sizes are asked for."""
    assert ops._size(query, *args, 16) == query(*args, 16)
    block = torch.tensor(16)
    assert ops._size(query, *args, block) == query(*args, 16)
    block.fill_(48)
    assert ops._size(query, *args, block) == query(*args, 48)
    assert ops._size(query, *args, np.array(32)) == query(*args, 32)
