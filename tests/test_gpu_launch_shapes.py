"""Launch shapes that depend on the sizes of a call: each rule of a dispatch at the sizes where it can go wrong."""

import pytest
import torch

from turboquant_amd.paged import PagedKVPool
from turboquant_amd.quantizer import TurboQuantProd

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def _i32(x, dev):
    return torch.tensor(x, dtype=torch.int32, device=dev)


@pytest.mark.parametrize("d,B,H", [(128, 2, 3), (128, 65, 2), (256, 130, 1), (128, 1024, 2), (256, 1024, 1), (128, 1025, 1)])
def test_ragged_append_numbers_only_the_pages_that_exist(gpu, d, B, H):
    """Most runs of the batch are empty; the others start and end anywhere in a page, the first and the last sequence and
    the ones beside a multiple of 64 among them.  Up to 1024 sequences the tiles are numbered through an index of the
    existing pages, beyond that over all of them: the pages must equal one append per sequence, byte for byte."""
    g = torch.Generator().manual_seed(d + B)
    per_seq = 9
    runs, starts = [0] * B, [int(x) for x in torch.randint(0, 17, (B,), generator=g)]
    live = sorted({0, 1, B - 1} | {b for c in range(64, B, 64) for b in (c - 1, c)})
    for i, b in enumerate(live):
        runs[b] = (1, 16, 17, 31, 100, 3, 127)[i % 7]
    if B == 65:
        runs[0] = 0                                                    # an empty sequence in front
    rows = sum(runs) + 2
    row0 = [1 + sum(runs[:b]) for b in range(B)]
    k = torch.randn(rows, H, d, generator=g).bfloat16().to(gpu)
    v = torch.randn(rows, H, d, generator=g).bfloat16().to(gpu)
    table = torch.randperm(B * per_seq, generator=g).view(B, per_seq).to(torch.int32).to(gpu)
    tq = TurboQuantProd(d, bits=3, device=gpu)
    pa, pb = (PagedKVPool(tq, H, B * per_seq, value_bits=2, dtype=torch.bfloat16, device=gpu) for _ in range(2))
    _say(f"ragged append d={d} B={B} H={H} rows={rows}")
    pa.append_ragged(k, v, _i32(row0, gpu), _i32(runs, gpu), _i32(starts, gpu), table, max_run=max(runs))
    for b in range(B):
        if runs[b]:
            pb.append(k[None, row0[b]:row0[b] + runs[b]], v[None, row0[b]:row0[b] + runs[b]], table[b:b + 1],
                      start_pos=_i32([starts[b]], gpu))
    torch.cuda.synchronize()
    assert torch.equal(pa.data, pb.data)
    assert int((pa.data != 0).sum()) > 0
