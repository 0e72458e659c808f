"""Radix select at the edges of its chunks (256 scores) and of the scores it keeps in registers (2048), with many ties,
against the oracle, exactly."""
import pytest
import torch

from acache_amd import ops
from oracle import acache_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("largest", [True, False])
@pytest.mark.parametrize("distinct", [3, 40, 100000])
def test_chunk_and_register_edges(device, distinct, largest):
    g = torch.Generator().manual_seed(distinct)
    lens = [1, 2, 255, 256, 257, 511, 513, 1791, 2047, 2048, 2049, 2304, 2305, 5000]
    picks = [1, 1, 254, 1, 129, 300, 512, 7, 2046, 410, 2000, 2303, 1, 1777]
    scores = [torch.randint(0, distinct, (n,), generator=g).float() - distinct // 2 for n in lens]
    cu = lambda v: torch.tensor([0] + torch.tensor(v).cumsum(0).tolist(), dtype=torch.int32)
    cu_a, cu_k = cu(lens), cu(picks)
    out = ops.topk_anchors(torch.cat(scores).to(device), cu_a.to(device), cu_k.to(device), int(cu_k[-1]), largest=largest).cpu()
    for b, (s, k) in enumerate(zip(scores, picks)):
        assert out[cu_k[b]:cu_k[b + 1]].tolist() == O.topk_anchors(s, k, largest=largest), (lens[b], k)
