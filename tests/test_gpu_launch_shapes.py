"""Launch shapes that depend on the sizes of a call: each rule of a dispatch at the sizes where it can go wrong."""

import copy

import pytest
import torch

from turboquant_amd.paged import PagedKVPool
from turboquant_amd.quantizer import TurboQuantProd
from tests.test_gpu_parity import _decode_case, _make_pool
from tests.test_gpu_parity_scores import _set_option

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


# 256 compute units: up to 1024 tiles at head_dim 128 and 512 at 256 every group of tiles has one to itself, and no index is built
@pytest.mark.parametrize("d,H,B,max_run", [(128, 8, 2, 1009), (128, 8, 2, 1010), (256, 4, 2, 1009), (256, 4, 2, 1010), (128, 3, 7, 770)])
def test_ragged_append_of_few_sequences_with_and_without_the_index(gpu, d, H, B, max_run):
    """The longest run first, last or in the middle, an empty one and one of a single token: against one append per sequence, byte for
    byte (the kernels and their arithmetic are the same, only the numbering of the tiles differs)."""
    g = torch.Generator().manual_seed(d + max_run)
    width = max_run // 16 + 3
    k, v = (torch.randn(max_run + 64, H, d, generator=g).bfloat16().to(gpu) for _ in range(2))
    tq = TurboQuantProd(d, bits=3, device=gpu)
    for long_at in sorted({0, B // 2, B - 1}):
        runs = [(1, 0, 15, 16, 17, 0, 2)[b % 7] for b in range(B)]
        runs[long_at] = max_run - 1 if long_at else max_run
        row0 = [sum(runs[:b]) for b in range(B)]
        starts = [int(x) for x in torch.randint(0, 17, (B,), generator=g)]
        table = torch.randperm(B * width, generator=g).view(B, width).to(torch.int32).to(gpu)
        pa, pb = (PagedKVPool(tq, H, B * width, value_bits=2, dtype=torch.bfloat16, device=gpu) for _ in range(2))
        _say(f"few ragged runs d={d} H={H} runs={runs}")
        pa.append_ragged(k, v, _i32(row0, gpu), _i32(runs, gpu), _i32(starts, gpu), table, max_run=max_run)
        for b in range(B):
            if runs[b]:
                rows = slice(row0[b], row0[b] + runs[b])
                pb.append(k[None, rows], v[None, rows], table[b:b + 1], start_pos=_i32([starts[b]], gpu))
        torch.cuda.synchronize()
        assert torch.equal(pa.data, pb.data)
        assert int((pa.data != 0).sum()) > 0


def _ragged_pool(gpu, d, key_bits, vb, H, lens, dtype, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    tq = TurboQuantProd(d, bits=key_bits, device=gpu)
    B, width = len(lens), max(1, max(-(-n // 16) for n in lens))
    table = torch.rand(B * width, generator=g, device=gpu).argsort().to(torch.int32).view(B, width).contiguous()
    pool = PagedKVPool(tq, H, B * width, value_bits=vb, dtype=dtype, device=gpu)
    rows = sum(lens)
    k = torch.randn(rows, H, d, generator=g, device=gpu).to(dtype)
    v = torch.randn(rows, H, d, generator=g, device=gpu).to(dtype)
    run = _i32(lens, gpu)
    row0 = (torch.cumsum(run, 0) - run).to(torch.int32)
    pool.append_ragged(k, v, row0, run, torch.zeros_like(run), table, max_run=max(lens))
    return pool, table, run, g


# (head_dim, key bits, heads per KV head, KV heads, sequences): workgroups of 4 and of 8 wavefronts, a share per wavefront (more
# pairs than workgroups fit), the merge in the launch, more shares than one pass of it takes
@pytest.mark.parametrize("d,kb,G,H,B", [(128, 3, 4, 2, 3), (128, 3, 5, 8, 16), (128, 4, 5, 8, 97), (128, 3, 12, 8, 97),
                                        (64, 3, 4, 4, 200), (256, 3, 8, 2, 5), (256, 2, 4, 4, 90), (128, 2, 1, 1, 1024)])
@pytest.mark.parametrize("ring", [0, 40])
def test_shares_by_length_give_what_equal_shares_give(gpu, d, kb, G, H, B, ring):
    """A step whose workgroups may be dealt out by length against the same step with two equal shares per sequence: the same
    sums in another order, the weights rounded to bf16 relative to another reference.  Either is within 2^-7 of the largest |value|
    of a row of the oracle's result (the bound of the decode tests), so they are within twice that of each other."""
    g = torch.Generator().manual_seed(B + d)
    longest = 9000 if B < 300 else 1500
    lens = [int(longest * 2.0 ** (-11.0 * float(x))) for x in torch.rand(B, generator=g)]
    lens[0] = longest
    if B > 4:
        lens[1], lens[2], lens[B // 2], lens[-1] = 0, 1, 64, 63
    dtype = torch.float16 if kb == 4 else torch.bfloat16
    pool, table, seq, dg = _ragged_pool(gpu, d, kb, 4, H, lens, dtype, 31 * B + d)
    q = torch.randn(B, H * G, d, generator=dg, device=gpu).to(dtype)
    _say(f"by length d={d} kb={kb} G={G} H={H} B={B} ring={ring}")
    if ring:
        exact = torch.randn(2, pool.num_pages, 16, H, d, generator=dg, device=gpu).to(dtype)
        outs = [pool.decode_attention_ring(q, table, seq, exact[0], exact[1], ring, max_len=longest, n_split=n).float()
                for n in (None, 2, None)]
    else:
        outs = [pool.decode_attention(q, table, seq, max_len=longest, n_split=n).float() for n in (None, 2, None)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[2])
    a, b = outs[0], outs[1]
    scale = b.abs().amax(-1, keepdim=True).clamp_min(1e-6)
    assert float(((a - b).abs() / scale).max()) <= 2.0 ** -6 and float((a - b).norm() / b.norm()) <= 6e-3
    if B > 4:
        assert not a[1].any()                            # an empty sequence


# (head_dim, key bits, heads per KV head, KV heads, lengths of the few sequences): more than eight shares each, merged by a kernel of
# its own from parts that lie where the most shares would end
@pytest.mark.parametrize("d,kb,G,H,lens", [(128, 3, 4, 1, [30000, 900, 0]), (128, 3, 4, 2, [24001, 3000, 11, 24000, 7000]), (256, 3, 8, 1, [30011, 64, 2000]),
                                           (256, 2, 4, 2, [20000, 100, 1, 0, 5000]), (64, 3, 4, 2, [30000, 2000]), (128, 5, 4, 2, [26000, 500, 1700])])
@pytest.mark.parametrize("recent", [None, 128])
def test_dozens_of_shares_by_length_against_the_oracle(gpu, d, kb, G, H, lens, recent):
    from tests.test_gpu_parity import _decode_case
    B, tail = len(lens), None
    if recent:                                           # (with few groups of heads the exact tail is several parts)
        tail = [recent, 3, 0, 77, recent][:B]
    for seed in (1, 2):
        _say(f"oracle, by length d={d} kb={kb} G={G} H={H} lens={lens} recent={tail}")
        _decode_case(gpu, d, kb, 4, B, H * G, H, lens, tail, seed=seed)


# one share per sequence, walked by four, two and one wavefronts, and 5-bit keys, whose operands are in LDS
@pytest.mark.parametrize("d,kb,G,H,B", [(128, 3, 4, 8, 60), (128, 3, 4, 8, 97), (64, 3, 4, 8, 200), (256, 3, 8, 4, 60), (128, 5, 4, 8, 60)])
@pytest.mark.parametrize("ring", [0, 40])
@pytest.mark.parametrize("in_launch", [1, 0])
def test_very_uneven_lengths_split_sequences_and_merge_them_either_way(gpu, d, kb, G, H, B, ring, in_launch):
    """One long sequence among short ones: the schedule deals the long one out (the result is not that of equal shares bit for
    bit), merged by the workgroup or wavefront that finishes last, or by a kernel of its own."""
    from turboquant_amd import _ffi
    lens = [6000] + [40 + 7 * b % 200 for b in range(B - 1)]
    lens[5], lens[B // 2] = 0, 1
    pool, table, seq, dg = _ragged_pool(gpu, d, kb, 4, H, lens, torch.bfloat16, B + d)
    q = torch.randn(B, H * G, d, generator=dg, device=gpu).bfloat16()
    exact = torch.randn(2, pool.num_pages, 16, H, d, generator=dg, device=gpu).bfloat16() if ring else None
    _say(f"one long sequence d={d} kb={kb} G={G} H={H} B={B} ring={ring} in_launch={in_launch}")
    n = pool.default_splits(B, 6000, H * G)
    try:
        _ffi.check(_ffi.lib().tq_set_option(b"merge_in_kernel", in_launch), "tq_set_option")
        a, again, b = (_step(pool, q, table, seq, 6000, k, exact, ring).float() for k in (None, None, n))
        torch.cuda.synchronize()
    finally:
        _ffi.check(_ffi.lib().tq_set_option(b"merge_in_kernel", 1), "tq_set_option")
    assert torch.equal(a, again) and not torch.equal(a[0], b[0])
    scale = b.abs().amax(-1, keepdim=True).clamp_min(1e-6)
    assert float(((a - b).abs() / scale).max()) <= 2.0 ** -6            # (twice the bound against the oracle)
    assert not a[5].any() and torch.equal(a[B // 2], b[B // 2])


@pytest.mark.parametrize("d,H,G,B", [(128, 8, 4, 16), (128, 8, 4, 97), (256, 2, 8, 4)])
def test_a_captured_step_reads_the_lengths_of_every_replay(gpu, d, H, G, B):
    """Captured with one set of lengths and replayed with others - equal, uneven, empty sequences, shorter -, eager steps in between."""
    N = 8000 if B < 50 else 1500
    pool, table, seq, dg = _ragged_pool(gpu, d, 3, 4, H, [N] * B, torch.bfloat16, B)
    q = torch.randn(B, H * G, d, generator=dg, device=gpu).bfloat16()
    sets = [[N] * B, [max(1, int(N * 0.6 ** b)) for b in range(B)], [N if b == 1 else 0 for b in range(B)], [N // 3] * B,
            [1 + (97 * b) % N for b in range(B)]]
    lens, out = seq.clone(), torch.empty_like(q)
    step = lambda o: pool.decode_attention(q, table, lens, max_len=N, out=o)
    _say(f"captured step d={d} H={H} B={B}")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(out)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(out)
    for new in sets + sets[::-1]:
        lens.copy_(_i32(new, gpu))
        want = step(torch.empty_like(q))
        torch.cuda.synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), new


def _step(pool, q, table, seq, longest, n_split, exact, ring):
    if ring:
        return pool.decode_attention_ring(q, table, seq, exact[0], exact[1], ring, max_len=longest, n_split=n_split)
    return pool.decode_attention(q, table, seq, max_len=longest, n_split=n_split)


# (head_dim, key bits, heads per KV head, KV heads, sequences, tokens): one share per sequence walked by four, two and one wavefronts
# and by a workgroup of eight; a few shares, merged in the launch; dozens, merged by a kernel of their own; 5-bit keys
_EQUAL = [(128, 3, 4, 8, 64, 2048), (128, 3, 4, 8, 96, 700), (128, 4, 5, 8, 128, 512), (64, 3, 4, 8, 100, 700), (128, 3, 4, 8, 192, 333),
          (128, 3, 4, 8, 300, 200), (128, 3, 4, 8, 32, 8192), (128, 2, 4, 2, 16, 4000), (256, 3, 8, 2, 128, 2048), (256, 3, 8, 2, 4, 33000),
          (128, 3, 4, 8, 2, 33000), (128, 5, 4, 8, 64, 700)]


@pytest.mark.parametrize("d,kb,G,H,B,N", _EQUAL)
@pytest.mark.parametrize("ring", [0, 40])
def test_steps_of_equal_length_are_those_of_equal_shares(gpu, d, kb, G, H, B, N, ring):
    """A step whose sequences are as long as one another, or nearly, gains nothing from shares by length and has to be the step with
    that many equal shares, bit for bit: it once split sequences between wavefronts and took half as long again."""
    pool, table, seq, dg = _ragged_pool(gpu, d, kb, 4, H, [N] * B, torch.bfloat16, B + d)
    q = torch.randn(B, H * G, d, generator=dg, device=gpu).bfloat16()
    exact = torch.randn(2, pool.num_pages, 16, H, d, generator=dg, device=gpu).bfloat16() if ring else None
    n = pool.default_splits(B, N, H * G)
    nearly = seq - torch.randint(0, max(2, N // 25), (B,), generator=dg, device=gpu).to(torch.int32)
    nearly[0] = N
    for name, lens in (("equal", seq), ("nearly equal", nearly)):
        _say(f"{name} lengths d={d} kb={kb} G={G} H={H} B={B} N={N} ring={ring} splits={n}")
        outs = [_step(pool, q, table, lens, N, k, exact, ring) for k in (None, n)]
        torch.cuda.synchronize()
        assert torch.equal(*outs) and bool(outs[0].any())


@pytest.mark.parametrize("d,B,H,T,dtype", [(128, 32, 8, 1, torch.bfloat16), (128, 300, 2, 1, torch.float16), (128, 3, 2, 70, torch.bfloat16),
                                           (256, 5, 1, 17, torch.float16), (64, 7, 3, 1, torch.bfloat16), (128, 4, 1, 3, torch.float32),
                                           (576, 9, 1, 1, torch.bfloat16), (128, 2, 4, 1500, torch.bfloat16)])
def test_append_of_the_newest_tokens_takes_the_lengths(gpu, d, B, H, T, dtype):
    """Lengths with the new tokens, or the positions they begin at: every kernel of an append, the rows that begin or end on a page
    boundary and a sequence whose length leaves no room for its tokens among them.  Byte for byte."""
    g = torch.Generator(device=gpu).manual_seed(d + B + T)
    tq = TurboQuantProd(d, bits=3, device=gpu)
    per_seq = -(-(T + 40) // 16)
    table = torch.randperm(B * per_seq, generator=g, device=gpu).view(B, per_seq).to(torch.int32)
    lens = _i32([T + (0, 15, 16, 17, 33, -1)[b % 6] for b in range(B)], gpu)
    k, v = torch.randn(2, B, T, H, d, generator=g, device=gpu).to(dtype)
    _say(f"newest d={d} B={B} H={H} T={T} {dtype}")
    pools = [PagedKVPool(tq, H, B * per_seq, value_bits=4, value_group_size=32, dtype=dtype, device=gpu) for _ in range(2)]
    pools[0].append(k, v, table, start_pos=lens - T)
    assert pools[1]._append_newest(k, v, table, lens)
    torch.cuda.synchronize()
    assert torch.equal(pools[0].data, pools[1].data) and bool(pools[0].data.any())


# every count of column tiles per wavefront, 1 .. 4 bits, groups of one tile (up to a tile per compute unit) and of several, and
# one tile more and less than that
@pytest.mark.parametrize("d,key_bits,vb,dtype", [(64, 3, 2, torch.bfloat16), (192, 2, 4, torch.float16), (320, 5, 2, torch.bfloat16),
                                                 (448, 3, 4, torch.float32), (576, 4, 4, torch.bfloat16), (640, 4, 2, torch.float16),
                                                 (704, 5, 4, torch.bfloat16), (768, 3, 4, torch.bfloat16)])
@pytest.mark.parametrize("tokens", [1, 33, 4096, 4111])
def test_appends_at_other_head_sizes_on_both_quantisers(gpu, d, key_bits, vb, dtype, tokens):
    """Rows on a 16-byte boundary go to the matrix-core key quantiser and the chunked value kernel, the same rows one element
    further into a buffer to the vector-ALU kernels: values and scales byte for byte; an index or a sign may flip where an
    fp32 sum meets a threshold (and a flipped index changes a tenth of its vector's signs): 1e-4 of the codes; norms are
    equal."""
    g = torch.Generator(device=gpu).manual_seed(d + tokens)
    tq = TurboQuantProd(d, bits=key_bits, device=gpu)
    pages = -(-tokens // 16) + 1
    table = torch.arange(pages, dtype=torch.int32, device=gpu)[None]
    start = _i32([5], gpu)
    _say(f"append d={d} bits={key_bits}/{vb} {dtype} tokens={tokens}")
    x = torch.randn(2, 1, tokens, 1, d, generator=g, device=gpu).to(dtype)
    x[0, 0, tokens // 2] = 0
    got = []
    for pad in (0, 1):
        buf = torch.zeros(2 * tokens * d + 16, dtype=dtype, device=gpu)
        rows = buf[pad:pad + 2 * tokens * d].view(2, 1, tokens, 1, d)
        rows.copy_(x)
        pool = PagedKVPool(tq, 1, pages, value_bits=vb, value_group_size=32, dtype=dtype, device=gpu)
        pool.append(rows[0], rows[1], table, start_pos=start)
        got.append((pool, pool.export_flat(table[0], tokens + 5)))
    torch.cuda.synchronize()
    (pa, a), (pb, b) = got
    L = pa.layout
    assert torch.equal(pa.data[..., L.off_vdata:], pb.data[..., L.off_vdata:])
    codes = tokens * d
    assert int((a[0] != b[0]).sum()) <= max(1, 1e-4 * codes)
    assert int(sum(((a[1] ^ b[1]) >> s & 1).sum() for s in range(8))) <= max(d // 4, 2e-4 * codes)
    assert torch.equal(a[2], b[2])                       # both add the squares in one order
    flipped = (a[0] != b[0]).any(-1)
    assert int(flipped.sum()) <= max(1, 3e-3 * tokens)
    assert torch.allclose(a[3][~flipped], b[3][~flipped], rtol=1e-5, atol=1e-6)
    assert int((a[0] != 0).sum()) > 0


def _both_quantisers(gpu, quantizer, x):
    """Codes of the same rows on a 16-byte boundary (matrix-core kernel) and one element further on (vector-ALU kernel)."""
    codes = []
    for pad in (0, 1):
        buf = torch.empty(x.numel() + 16, dtype=x.dtype, device=gpu)
        rows = buf[pad:pad + x.numel()].view(x.shape)
        rows.copy_(x)
        codes.append(quantizer.quantize(rows))
    return codes


# sizes with one to four column tiles per wavefront, one to four index bits, every input type; vectors as models make them, with a
# few channels ten times as large, with nearly all of their length in one channel, and far from the origin
@pytest.mark.parametrize("d,key_bits,dtype", [(64, 3, torch.bfloat16), (192, 4, torch.float16), (320, 3, torch.float32), (384, 2, torch.bfloat16),
                                              (448, 3, torch.float16), (576, 4, torch.bfloat16), (576, 5, torch.float16), (704, 4, torch.float32),
                                              (768, 4, torch.bfloat16), (768, 5, torch.bfloat16)])
@pytest.mark.parametrize("values", ["plain", "outliers", "spike", "offset"])
def test_codes_do_not_depend_on_the_quantiser_that_a_row_reaches(gpu, d, key_bits, dtype, values):
    """The two key quantisers add their products in different orders; an index whose coordinate lies on a threshold within
    rounding, and a sign whose projection is zero within it, must come out alike all the same: indices, signs and norms are
    equal.  (65536 vectors of 576, 4-bit keys: two dozen indices and some thirty signs lie that near.)  The residual norm is a sum
    of d squares in two orders, each relative error below d 2^-24."""
    n = 65536 if d != 64 else 262144
    g = torch.Generator(device=gpu).manual_seed(d * 7 + key_bits)
    x = torch.randn(n, d, generator=g, device=gpu)
    if values == "outliers":
        x[:, torch.randperm(d, generator=g, device=gpu)[:4]] *= 10
    elif values == "spike":
        x *= 0.01
        x[torch.arange(n, device=gpu), torch.randint(0, d, (n,), generator=g, device=gpu)] = 50.0
    elif values == "offset":
        x = torch.rand(n, d, generator=g, device=gpu) + 1
    x = x.to(dtype)
    x[7], x[8] = 0, x[9]
    _say(f"codes of both quantisers d={d} bits={key_bits} {dtype} {values}")
    a, b = _both_quantisers(gpu, TurboQuantProd(d, bits=key_bits, device=gpu), x)
    torch.cuda.synchronize()
    for name in ("mse_indices", "qjl_signs", "norms"):
        assert int((getattr(a, name) != getattr(b, name)).sum()) == 0, name
    assert torch.allclose(a.residual_norms, b.residual_norms, rtol=d * 2.0 ** -24, atol=0)


def test_a_vector_without_a_residual_keeps_its_signs(gpu):
    """Keys that are de-quantised and quantised again have a residual of rounding errors, so every projection is zero within
    rounding and all signs are decided by the sums in order."""
    d = 576
    g = torch.Generator(device=gpu).manual_seed(5)
    tq = TurboQuantProd(d, bits=4, device=gpu)
    mse = tq.mse_quantizer
    x = mse.dequantize(mse.quantize(torch.randn(96, d, generator=g, device=gpu)))
    _say("vectors without a residual")
    a, b = _both_quantisers(gpu, tq, x)
    torch.cuda.synchronize()
    for name in ("mse_indices", "qjl_signs", "norms"):
        assert int((getattr(a, name) != getattr(b, name)).sum()) == 0, name


# the matrix-core quantiser with a run-time size numbers ragged tiles with 256 of its 256 .. 768 threads; at head_dim 768 the index
# of many runs leaves room for one tile per workgroup only
@pytest.mark.parametrize("d,key_bits,B,H", [(64, 3, 65, 2), (192, 3, 130, 1), (320, 4, 257, 1), (576, 4, 65, 3), (576, 4, 1024, 1),
                                            (704, 4, 130, 1), (768, 4, 40, 8), (768, 4, 300, 1), (768, 3, 1024, 1)])
def test_ragged_append_of_other_head_sizes(gpu, d, key_bits, B, H):
    """Against one append per sequence, byte for byte, and against the vector-ALU kernel (rows one element off the boundary) but for
    the residual norms - whose last bits also tell that two kernels ran."""
    g = torch.Generator().manual_seed(d + B)
    runs = [int(x) for x in torch.randint(0, 40, (B,), generator=g)]
    runs[B // 2] = 200
    runs[0], runs[-1] = 0, 17
    starts = [int(x) for x in torch.randint(0, 17, (B,), generator=g)]
    rows, width = sum(runs), 15
    row0 = [sum(runs[:b]) for b in range(B)]
    buf = torch.randn(2 * rows * H * d + 16, generator=g).bfloat16().to(gpu)
    k, v = buf[:2 * rows * H * d].view(2, rows, H, d)
    off = torch.empty_like(buf)
    ko, vo = off[1:1 + 2 * rows * H * d].view(2, rows, H, d)
    ko.copy_(k), vo.copy_(v)
    table = torch.randperm(B * width, generator=g).view(B, width).to(torch.int32).to(gpu)
    tq = TurboQuantProd(d, bits=key_bits, device=gpu)
    pa, pb, pc = (PagedKVPool(tq, H, B * width, value_bits=4, dtype=torch.bfloat16, device=gpu) for _ in range(3))
    _say(f"ragged append d={d} bits={key_bits} B={B} H={H} rows={rows}")
    args = _i32(row0, gpu), _i32(runs, gpu), _i32(starts, gpu), table
    pa.append_ragged(k, v, *args, max_run=max(runs))
    pc.append_ragged(ko, vo, *args, max_run=max(runs))
    for b in range(B):
        if runs[b]:
            s = slice(row0[b], row0[b] + runs[b])
            pb.append(k[None, s], v[None, s], table[b:b + 1], start_pos=_i32([starts[b]], gpu))
    torch.cuda.synchronize()
    assert torch.equal(pa.data, pb.data)
    meta = slice(pa.layout.off_meta, pa.layout.off_meta + 8 * 16)
    ma, mc = (p.data[..., meta].contiguous().view(torch.float32) for p in (pa, pc))
    assert torch.equal(ma[..., 0::2], mc[..., 0::2]) and not torch.equal(ma, mc)
    assert torch.allclose(ma, mc, rtol=d * 2.0 ** -24, atol=0)
    pa.data[..., meta] = pc.data[..., meta]
    assert torch.equal(pa.data, pc.data)


@pytest.mark.parametrize("d,key_bits,vb,dtype", [(64, 3, 2, torch.bfloat16), (320, 3, 4, torch.float16), (576, 4, 4, torch.bfloat16), (576, 4, 2, torch.float16),
                                                 (384, 2, 4, torch.bfloat16), (704, 5, 2, torch.float16)])
@pytest.mark.parametrize("layout", ["tokens first", "heads first", "every other token"])
def test_odd_values_and_strides_at_other_head_sizes(gpu, d, key_bits, vb, dtype, layout):
    """Infinities, NaN, zeros, the type's largest and smallest numbers, in rows that lie apart: the matrix-core quantiser and the chunked
    value kernel (rows on a 16-byte boundary) against the vector-ALU kernels (one element further on), all bytes but those of
    the residual norms, which agree but for the order of the sum."""
    B, T, H = 2, 37, 3
    g = torch.Generator(device=gpu).manual_seed(d + vb)
    x = torch.randn(2, B, T, H, d, generator=g, device=gpu).to(dtype)
    big, small = torch.finfo(dtype).max, torch.finfo(dtype).tiny
    for t, odd in enumerate((float("inf"), -float("inf"), float("nan"), 0.0, big, -big, small)):
        x[:, :, 2 * t, :, (5 * t + 3) % d] = odd
    x[:, 0, 20], x[:, 0, 21], x[:, 1, 22], x[:, 1, 23], x[:, 1, 24] = 0, float("nan"), float("inf"), small, 7.0
    x[:, 0, 25] = torch.finfo(dtype).smallest_normal * x[:, 0, 26].float().sign().to(dtype)
    tq = TurboQuantProd(d, bits=key_bits, device=gpu)
    table = torch.randperm(B * 4, generator=torch.Generator().manual_seed(3)).view(B, 4).to(torch.int32).to(gpu)
    start = _i32([5, 0], gpu)
    _say(f"odd values d={d} bits={key_bits}/{vb} {dtype} {layout}")
    pools = []
    for pad in (0, 1):
        shape = {"tokens first": (2, B, T, H, d), "heads first": (2, B, H, T, d), "every other token": (2, B, 2 * T, H, d)}[layout]
        n = 1
        for k in shape:
            n *= k
        buf = torch.zeros(n + 16, dtype=dtype, device=gpu)
        rows = buf[pad:pad + n].view(shape)
        if layout == "heads first":
            rows = rows.transpose(2, 3)
        elif layout == "every other token":
            rows = rows[:, :, ::2]
        rows.copy_(x)
        pool = PagedKVPool(tq, H, 8, value_bits=vb, dtype=dtype, device=gpu)
        pool.append(rows[0], rows[1], table, start_pos=start)
        pools.append(pool)
    torch.cuda.synchronize()
    L = pools[0].layout
    a, b = (p.data.clone() for p in pools)
    meta = slice(L.off_meta, L.off_meta + 8 * 16)
    ma, mb = (p[..., meta].contiguous().view(torch.float32) for p in (a, b))
    assert torch.equal(torch.nan_to_num(ma[..., 0::2], nan=-1.0), torch.nan_to_num(mb[..., 0::2], nan=-1.0))
    assert torch.allclose(ma, mb, rtol=d * 2.0 ** -24, atol=0, equal_nan=True)
    a[..., meta] = b[..., meta] = 0
    assert torch.equal(a[..., L.off_vdata:], b[..., L.off_vdata:]), "values"
    assert torch.equal(a, b), "keys"


# ------------------------------------------------------------------ sixteen query heads per wavefront (head_dim 512 / 576)
@pytest.mark.parametrize("d,key_bits,vb,Hq,Hkv,dtype,lens,recent,n_split", [
    (576, 4, 4, 9, 1, torch.bfloat16, [1, 33, 200], None, 1),                  # one tile, 7 columns without a head; a sequence of one token
    (576, 4, 4, 16, 1, torch.bfloat16, [700, 96, 97], None, None),             # one full tile: three blocks side by side, a last turn with one
    (576, 3, 2, 17, 1, torch.float16, [300, 31], [0, 9], 2),                   # two tiles, the second with one head; fp16 pages; exact tail
    (576, 4, 2, 64, 2, torch.bfloat16, [513, 64], None, 4),                    # two KV heads of two tiles; splits without tokens
    (576, 3, 4, 40, 1, torch.bfloat16, [2100, 5], None, 1),                    # three tiles: a pair of wavefronts without heads; the table registers move on
    (576, 4, 4, 65, 1, torch.float16, [130, 32], None, 3),                     # five tiles: two workgroups, the second with three idle pairs
    (576, 4, 4, 128, 1, torch.bfloat16, [400, 16, 15], [3, 0, 7], 2),          # eight tiles, exact tail
    (512, 4, 4, 128, 1, torch.float16, [300, 77], None, None),                 # lane-major key words
    (512, 3, 2, 24, 1, torch.bfloat16, [257, 480], None, 2),
    (512, 3, 4, 12, 1, torch.bfloat16, [64, 1000], None, 5),
    (512, 4, 2, 80, 2, torch.bfloat16, [129, 31], [7, 0], None)])
def test_more_than_eight_heads_per_wide_kv_head(gpu, d, key_bits, vb, Hq, Hkv, dtype, lens, recent, n_split):
    """Decode at head_dim 512 / 576 with 9 .. 128 query heads per KV head: every sequence against the oracle on the same
    store, and against the kernel that takes 8 heads per workgroup (operands not packed ahead).  Both round the weighted scales
    to bf16 (2^-9 each) and agree in everything else to fp32: 2^-7 of the largest output bounds two such sums."""
    out = {}
    try:
        for pre in (1, 0):
            _set_option("wide_prepack", pre)
            out[pre] = _decode_case(gpu, d, key_bits, vb, len(lens), Hq, Hkv, lens, recent, seed=40 + Hq + d, n_split=n_split,
                                    dtype=dtype, return_out=True).float()
    finally:
        _set_option("wide_prepack", 1)
    assert float((out[1] - out[0]).abs().max()) <= 2.0 ** -7 * float(out[0].abs().max())


@pytest.mark.parametrize("case", ["page", "all", "scale"])
def test_sixteen_heads_per_wavefront_and_slots_without_tokens(gpu, case):
    """Table entries outside the pool give their tokens no weight, and page slots behind a sequence's last token may hold
    anything (infinite scales and zero points, NaN norms): the results are those of the tokens that exist."""
    d, Hq, N = 576, 32, 200
    pool, tq = _make_pool(gpu, d, 4, 4, 1, 16, torch.bfloat16)
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn(1, N, 1, d, generator=g).bfloat16().to(gpu) for _ in range(2))
    q = torch.randn(1, Hq, d, generator=g).bfloat16().to(gpu)
    table = torch.arange(13, dtype=torch.int32, device=gpu)[None]
    pool.append(k, v, table)
    seq = torch.tensor([N], dtype=torch.int32, device=gpu)
    want = pool.decode_attention(q, table, seq, n_split=2, max_len=N)
    if case == "scale":
        L = pool.layout
        page = pool.data[12, 0]                                   # tokens 192 .. 207, eight of them written
        page[L.off_meta + 64:L.off_meta + 128] = 0xff             # (NaN)
        for off in (L.off_vscale, L.off_vzero):
            sect = page[off:off + 2 * 18 * 16].view(torch.int16).view(18, 16)
            sect[:, 8:] = 0x7f80                                  # (infinity)
        assert torch.equal(pool.decode_attention(q, table, seq, n_split=2, max_len=N), want)
        return
    bad = table.clone()
    if case == "all":
        bad[:] = 99
        assert torch.count_nonzero(pool.decode_attention(q, bad, seq, n_split=2, max_len=N)) == 0
        return
    bad[0, 12] = -1                                               # the last page: what is left is the sequence of 192 tokens
    short = torch.tensor([192], dtype=torch.int32, device=gpu)
    assert torch.equal(pool.decode_attention(q, bad, seq, n_split=1, max_len=N), pool.decode_attention(q, table, short, n_split=1, max_len=N))


@pytest.mark.parametrize("d", [512, 576])
def test_sixteen_heads_per_wavefront_of_two_sequences_and_slots_without_tokens(gpu, d):
    """The same with a second sequence beside it: one alone in few splits takes the kernel of 8 heads per workgroup, whose results it has to
    within the rounding of the weighted scales (2^-9 each)."""
    Hq, N = 32, 200
    pool, tq = _make_pool(gpu, d, 4, 4, 1, 16, torch.bfloat16)
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn(1, N, 1, d, generator=g).bfloat16().to(gpu) for _ in range(2))
    q = torch.randn(1, Hq, d, generator=g).bfloat16().to(gpu).expand(2, Hq, d).contiguous()
    table = torch.arange(13, dtype=torch.int32, device=gpu)[None].repeat(2, 1)
    pool.append(k, v, table[:1])
    both = lambda t, lens, n=2: pool.decode_attention(q, t, _i32(lens, gpu), n_split=n, max_len=N)
    want = both(table, [N, 31])
    one = pool.decode_attention(q[:1], table[:1], _i32([N], gpu), n_split=2, max_len=N)
    assert float((one[0].float() - want[0].float()).abs().max()) <= 2.0 ** -7 * float(one.float().abs().max())
    L = pool.layout
    page = pool.data[12, 0]                                       # tokens 192 .. 207, eight of them written
    page[L.off_meta + 64:L.off_meta + 128] = 0xff
    for off in (L.off_vscale, L.off_vzero):
        page[off:off + 2 * (d // 32) * 16].view(torch.int16).view(d // 32, 16)[:, 8:] = 0x7f80
    assert torch.equal(both(table, [N, 31]), want)
    bad = table.clone()
    bad[0, 12], bad[1] = -1, 99
    assert torch.equal(both(bad, [N, 31], 1)[0], both(table, [192, 31], 1)[0])
    assert torch.count_nonzero(both(bad, [N, 31])[1]) == 0


@pytest.mark.parametrize("d,Hq,B,dtype", [(576, 8, 40, torch.bfloat16), (576, 5, 53, torch.float16), (704, 8, 33, torch.bfloat16),
                                          (320, 7, 80, torch.bfloat16), (576, 128, 3, torch.bfloat16), (576, 128, 17, torch.float16),
                                          (512, 100, 21, torch.bfloat16), (640, 3, 200, torch.float16)])
def test_rotation_of_hundreds_of_rows(gpu, d, Hq, B, dtype):
    """Steps whose rotation passes over the row tiles with the matrix terms in LDS (265 .. 2176 rows, shares of one to three
    tiles per wavefront, a last tile that is not full): the operands are those of the vector-ALU rotation to rounding (sums in another order),
    so the outputs agree within a rounding step of the output type."""
    pool, tq = _make_pool(gpu, d, 4, 4, 1, 6, dtype)
    g = torch.Generator().manual_seed(d + Hq)
    k, v = (torch.randn(1, 90, 1, d, generator=g).to(dtype).to(gpu) for _ in range(2))
    table = torch.arange(6, dtype=torch.int32, device=gpu)
    pool.append(k, v, table[None])
    q = torch.randn(B, Hq, d, generator=g).to(dtype).to(gpu)
    seq = torch.randint(1, 91, (B,), generator=g).to(torch.int32).to(gpu)
    outs = []
    try:
        for opt in (1, 0):
            _set_option("prep_mfma", opt)
            outs.append(pool.decode_attention(q, table, seq, n_split=1, max_len=90).float())
    finally:
        _set_option("prep_mfma", 1)
    assert float((outs[0] - outs[1]).abs().max()) <= 2.0 ** -7 * float(outs[1].abs().max())


@pytest.mark.parametrize("dtype,unit,scale", [(torch.float16, 2.0 ** -15, 2.0 ** 11), (torch.bfloat16, 2.0 ** -69, 2.0 ** 65)])
def test_rotation_of_rows_of_tiny_numbers(gpu, dtype, unit, scale):
    """Rows of fp16 subnormals, of bf16 numbers whose squares are fp32 subnormals, and some of zeros and of single such numbers, with a scale
    that makes their scores count: as the vector-ALU rotation."""
    d, Hq, B = 576, 8, 40
    pool, tq = _make_pool(gpu, d, 4, 4, 1, 6, dtype)
    g = torch.Generator().manual_seed(9)
    k, v = (torch.randn(1, 90, 1, d, generator=g).to(dtype).to(gpu) for _ in range(2))
    table = torch.arange(6, dtype=torch.int32, device=gpu)
    pool.append(k, v, table[None])
    q = torch.rand(B, Hq, d, generator=g) * 2 - 1
    q[::3, 1] = 0
    q[1::3, 2, 5:] = 0
    q[::4, 3] *= 1e3                                                 # (ordinary rows among them)
    q = (q * unit).to(dtype).to(gpu)
    assert int((q != 0).sum()) > q.numel() // 2
    seq = torch.full((B,), 90, dtype=torch.int32, device=gpu)
    outs = []
    try:
        for opt in (1, 0):
            _set_option("prep_mfma", opt)
            outs.append(pool.decode_attention(q, table, seq, n_split=1, max_len=90, scale=scale).float())
    finally:
        _set_option("prep_mfma", 1)
    mean = pool.decode_attention(torch.zeros_like(q), table, seq, n_split=1, max_len=90).float()
    assert float((outs[1] - mean).abs().max()) > 0.1 * float(mean.abs().max())                  # (the scores count)
    assert float((outs[0] - outs[1]).abs().max()) <= 2.0 ** -7 * float(outs[1].abs().max())


# ------------------------------------------------------------------ the exact tail on the matrix cores
@pytest.mark.parametrize("d,Hq,Hkv,B,dtype,rows,n_split", [
    (128, 5, 1, 2, torch.bfloat16, [1, 16], 1), (128, 16, 1, 3, torch.float16, [15, 17, 0], 3), (128, 17, 1, 1, torch.bfloat16, [129], 2),
    (128, 40, 8, 65, torch.float16, [128, 127, 33], 1),               # 520 units: two wavefronts each; matrix-core preparation of fp16 queries
    (128, 24, 8, 67, torch.bfloat16, [200, 64, 3], 2),                # 536 units of three heads, more tiles than a wavefront's four
    (256, 16, 2, 4, torch.bfloat16, [128, 100, 1, 31], 16),           # shares of a unit's tokens (a merge kernel behind)
    (256, 6, 1, 300, torch.float16, [130, 5], 1), (64, 8, 2, 3, torch.bfloat16, [300, 16, 1024], 1), (64, 4, 4, 130, torch.float16, [40, 128], 1),
    (576, 8, 1, 3, torch.bfloat16, [128, 17, 90], 2), (576, 40, 1, 2, torch.float16, [128, 33], 2), (512, 16, 1, 2, torch.bfloat16, [300, 1], 9),
    (576, 16, 2, 2, torch.bfloat16, [1024, 500], 1)])
def test_exact_tail_on_the_matrix_cores(gpu, d, Hq, Hkv, B, dtype, rows, n_split):
    """Exact tokens that start on 16-byte boundaries run on the matrix cores, others on the vector ALU; both take products and
    weights in fp32 and sum in different orders, so the outputs agree within a rounding step of the output type.  The slots
    behind a sequence's last exact token hold NaN and infinity."""
    pool, tq = _make_pool(gpu, d, 3, 4, Hkv, 8, dtype)
    g = torch.Generator().manual_seed(d + B + Hq)
    k, v = (torch.randn(1, 100, Hkv, d, generator=g).to(dtype).to(gpu) for _ in range(2))
    table = torch.arange(7, dtype=torch.int32, device=gpu)
    pool.append(k, v, table[None])
    R = max(rows)
    n_rows = torch.tensor([rows[b % len(rows)] for b in range(B)], dtype=torch.int32)
    rk, rv = (torch.randn(B, R, Hkv, d, generator=g).to(dtype) for _ in range(2))
    for b in range(B):
        rk[b, n_rows[b]:] = float("nan")
        rv[b, n_rows[b]:] = float("inf")
    q = torch.randn(B, Hq, d, generator=g).to(dtype).to(gpu)
    seq = torch.randint(0, 101, (B,), generator=g).to(torch.int32).to(gpu)
    outs = []
    for pad in (0, 1):                                                # (one element in: rows that are not even word-aligned)
        wide = [torch.zeros(B, R, Hkv, d + 2, dtype=dtype, device=gpu) for _ in range(2)]
        for w, x in zip(wide, (rk, rv)):
            w[..., 1:1 + d] = x.to(gpu)
        ks, vs = (wide[0][..., 1:1 + d], wide[1][..., 1:1 + d]) if pad else (rk.to(gpu), rv.to(gpu))
        outs.append(pool.decode_attention(q, table, seq, recent_k=ks, recent_v=vs, recent_len=n_rows.to(gpu), n_split=n_split,
                                          max_len=100).float())
    assert torch.isfinite(outs[0]).all()
    assert float((outs[0] - outs[1]).abs().max()) <= 2.0 ** -7 * float(outs[1].abs().max())


@pytest.mark.parametrize("Hq,Hkv,B,dtype,rows", [
    (16, 2, 16, torch.float16, [16, 3, 0, 64]), (2, 2, 16, torch.bfloat16, [16, 1]),        # tail and preparation on the vector ALU in one launch
    (16, 2, 16, torch.float16, [65, 128]), (32, 2, 16, torch.bfloat16, [16, 5]),            # the tail on the matrix cores, two rounds of workgroups
    (32, 2, 1, torch.float16, [128]), (32, 2, 2, torch.bfloat16, [100, 128]),               # sixteen heads of few sequences
    (8, 2, 128, torch.float16, [16, 9]), (8, 2, 128, torch.bfloat16, [128, 77])])           # three rounds: a launch each
def test_exact_tail_at_head_dim_256_in_each_launch(gpu, Hq, Hkv, B, dtype, rows):
    """The forms of the launch before the page kernel, as above."""
    test_exact_tail_on_the_matrix_cores(gpu, 256, Hq, Hkv, B, dtype, rows, 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_exact_tail_in_place_with_two_wavefronts_per_unit(gpu, dtype):
    """The newest tokens read in place from a paged cache by 528 units, against the same rows gathered (same kernel, same bits up
    to the shared launch's preparation): blocks anywhere, sequences shorter than the ring, a block outside the cache behind the end."""
    d, Hkv, Hq, B, ring = 128, 8, 16, 66, 128
    pool, tq = _make_pool(gpu, d, 3, 4, Hkv, B * 16, dtype)
    g = torch.Generator().manual_seed(3)
    lens = [int(x) for x in torch.randint(1, 250, (B,), generator=g)]
    table = torch.randperm(B * 16, generator=g).view(B, 16).to(torch.int32).to(gpu)
    x = torch.randn(B, 250, Hkv, d, generator=g).to(dtype).to(gpu)
    pool.append(x, x.flip(-1), table)
    cache = torch.randn(2, B * 16, 16, Hkv, d, generator=g).to(dtype).to(gpu)
    q = torch.randn(B, Hq, d, generator=g).to(dtype).to(gpu)
    seq = _i32(lens, gpu)
    got = pool.decode_attention_ring(q, table, seq, cache[0], cache[1], ring, n_split=1, max_len=250).float()
    rk, rv = (torch.zeros(B, ring, Hkv, d, dtype=dtype, device=gpu) for _ in range(2))
    for b, n in enumerate(lens):
        r = min(n, ring)
        pos = torch.arange(n - r, n, device=gpu)
        rk[b, :r], rv[b, :r] = (c[table[b].long()[pos // 16], pos % 16] for c in cache)
    old = _i32([n - min(n, ring) for n in lens], gpu)
    want = pool.decode_attention(q, table, old, recent_k=rk, recent_v=rv, recent_len=_i32([min(n, ring) for n in lens], gpu),
                                 n_split=1, max_len=250).float()
    assert torch.equal(got, want)


# ------------------------------------------------------------------ a token of the cache object in fp32
class _Counted:
    """The library, counting the calls of each entry that it answered."""
    def __init__(self, lib):
        self._lib, self.answered = lib, {}

    def __getattr__(self, name):
        entry = getattr(self._lib, name)

        def call(*args):
            rc = entry(*args)
            if rc == 0:
                self.answered[name] = self.answered.get(name, 0) + 1
            return rc
        return call

    def take(self, *names):
        return sum(self.answered.pop(name, 0) for name in names)


@pytest.fixture
def counted(monkeypatch):
    """The library as the Python methods and the native host side in front of them call it."""
    import ctypes
    from turboquant_amd import _ffi
    real = _ffi.lib()
    assert _ffi.native() is not None, "the native host side is not built"
    host, lib = _ffi._host, _Counted(real)
    seen = {name: ctypes.CFUNCTYPE(*[t for ts in _ffi._SIGNATURES[name] for t in (ts if isinstance(ts, list) else [ts])])(getattr(lib, name))
            for name in _ffi._HOST_CALLS}
    monkeypatch.setattr(_ffi, "lib", lambda: lib)
    host.bind({name: _ffi.address(f) for name, f in seen.items()})
    yield lib
    host.bind({name: _ffi.address(getattr(real, name)) for name in _ffi._HOST_CALLS})


@pytest.mark.parametrize("d,B,H,prompt,buffer,key_bits,vb,gs,n_q", [
    (128, 1, 8, 400, 128, 3, 2, 32, 1), (64, 2, 3, 150, 128, 4, 4, 32, 1), (256, 1, 2, 300, 1, 2, 8, 64, 3), (128, 2, 1, 129, 128, 3, 4, 16, 9),
    (64, 1, 5, 65, 64, 5, 2, 64, 2), (128, 3, 4, 384, 33, 3, 2, 128, 1)])
def test_cache_token_in_few_launches(gpu, counted, d, B, H, prompt, buffer, key_bits, vb, gs, n_q):
    """Tokens, scores and values of the cache object through the entries of their own, against the general paths: codes,
    norms and buffers bit for bit, inner products with the compressed keys bit for bit, everything else within fp32 sums in another
    order.  Prompts as views of a (batch, tokens, heads, d) tensor, the buffer's rows then not behind one another: the
    first token takes the general path, the ones after it do not (all of them do where several batches' tokens lie apart as well)."""
    from turboquant_amd import _ffi, kv_cache as KC
    g = torch.Generator().manual_seed(d + prompt)
    for view in (False, True):
        shape = (B, prompt + 4, H, d) if view else (B, H, prompt + 4, d)
        k, v = (torch.randn(*shape, generator=g).to(gpu) for _ in range(2))
        if view:
            k, v = k.transpose(1, 2), v.transpose(1, 2)
        qs = torch.randn(4, B, H, n_q, d, generator=g).to(gpu)
        results = []
        for how in ("native", "python", "general"):
            fast = how != "general"
            patch = pytest.MonkeyPatch()
            if not fast:
                patch.setattr(KC, "_plain", lambda *t: False)
            if how != "native":
                patch.setattr(_ffi, "_host", None)
            cache = KC.TurboQuantKVCache(d, key_bits=key_bits, value_bits=vb, value_group_size=gs, buffer_size=buffer, device=gpu,
                                         dtype=torch.float32)
            cache.prefill(k[..., :prompt, :], v[..., :prompt, :])
            outs = []
            for i in range(4):
                t = prompt + i
                before = cache.key_quantized
                cache.append(k[..., t:t + 1, :], v[..., t:t + 1, :])
                assert before.norms.shape[-1] == t - buffer                # (what a caller kept is as it was)
                scores = cache.attention_scores(qs[i])
                outs.append((scores, cache.attend(torch.softmax(scores, dim=-1))))
            results.append((cache, outs))
            patch.undo()
            assert counted.take("tq_cache_append") == (0 if not fast else 4 if not view else 3 if B == 1 else 0)
            assert counted.take("tq_cache_scores", "tq_cache_scores_rows") == counted.take("tq_cache_attend") == (4 if fast else 0)
        assert all(torch.equal(x, y) for s, t in zip(results[0][1], results[1][1]) for x, y in zip(s, t))
        (a, oa), _, (b, ob) = results
        assert a.get_seq_length() == b.get_seq_length() and a.memory_bytes() == b.memory_bytes()
        for x, y in zip((*a.key_quantized[:4], *a.value_quantized[:3], a.key_buffer, a.value_buffer),
                        (*b.key_quantized[:4], *b.value_quantized[:3], b.key_buffer, b.value_buffer)):
            assert x.dtype == y.dtype and torch.equal(x, y)
        for (s1, r1), (s2, r2) in zip(oa, ob):
            n_c = s1.shape[-1] - buffer
            assert s1.shape == s2.shape and torch.equal(s1[..., :n_c], s2[..., :n_c])
            assert float((s1 - s2).abs().max()) <= 1e-6 * (d ** 0.5) * float(s2.abs().max())
            assert r1.shape == r2.shape and float((r1 - r2).norm()) <= 2e-6 * float(r2.norm())


def test_cache_codes_at_any_byte(gpu):
    """Code sections that begin one byte into a buffer take the general paths: same codes, and scores and values as from aligned ones
    (inner products of codes bit for bit, the rest within fp32 sums in another order)."""
    from turboquant_amd.kv_cache import TurboQuantKVCache
    g = torch.Generator().manual_seed(2)
    k, v = (torch.randn(1, 3, 302, 128, generator=g).to(gpu) for _ in range(2))
    q = torch.randn(1, 3, 2, 128, generator=g).to(gpu)

    def moved(t):
        return torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)

    results = []
    for odd in (False, True):
        cache = TurboQuantKVCache(128, buffer_size=128, device=gpu, dtype=torch.float32)
        cache.prefill(k[..., :300, :], v[..., :300, :])
        out = []
        for t in (300, 301):
            if odd:
                kq, vq = cache.key_quantized, cache.value_quantized
                cache.key_quantized = kq._replace(mse_indices=moved(kq.mse_indices), qjl_signs=moved(kq.qjl_signs))
                cache.value_quantized = vq._replace(data=moved(vq.data))
                assert cache.value_quantized.data.data_ptr() % 2 == 1
            scores = cache.attention_scores(q)
            out += [scores, cache.attend(torch.softmax(scores, dim=-1))]
            cache.append(k[..., t:t + 1, :], v[..., t:t + 1, :])
            assert cache.seq_len == t + 1
        results.append((cache, out))
    (a, oa), (b, ob) = results
    for x, y in zip((*a.key_quantized[:4], *a.value_quantized[:3]), (*b.key_quantized[:4], *b.value_quantized[:3])):
        assert torch.equal(x, y)
    for x, y in zip(oa, ob):
        assert x.shape == y.shape and float((x - y).norm()) <= 2e-6 * float(y.norm())


def test_cache_token_that_has_to_be_differentiated(gpu):
    """Weights and queries with a gradient take the general paths, through which torch differentiates."""
    from turboquant_amd.kv_cache import TurboQuantKVCache
    g = torch.Generator().manual_seed(1)
    k = torch.randn(1, 2, 300, 128, generator=g).to(gpu)
    cache = TurboQuantKVCache(128, buffer_size=128, device=gpu, dtype=torch.float32)
    cache.prefill(k, k)
    q = torch.randn(1, 2, 1, 128, generator=g).to(gpu).requires_grad_()
    scores = cache.attention_scores(q)
    out = cache.attend(torch.softmax(scores, dim=-1))
    out.sum().backward()
    assert q.grad is not None and torch.isfinite(q.grad).all() and float(q.grad.abs().max()) > 0
    assert torch.allclose(out, cache.attend(torch.softmax(scores, dim=-1).detach()), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("d,B,H,n_c,n_buf,key_bits,vb,gs", [
    (128, 1, 8, 300, 64, 3, 2, 32), (128, 1, 1, 1, 1, 2, 8, 16), (128, 2, 8, 77, 5, 4, 4, 128), (128, 1, 17, 40, 3, 5, 2, 64),
    (256, 3, 11, 129, 2, 3, 4, 32), (256, 1, 2, 1000, 130, 4, 2, 256), (64, 1, 5, 33, 7, 3, 2, 32), (128, 1, 4, 9001, 128, 3, 4, 32)])
def test_cache_token_in_one_launch(gpu, d, B, H, n_c, n_buf, key_bits, vb, gs):
    """A token into the cache object by the launch that quantises and copies at once, by the two behind one another, and by the quantisers
    and concatenations: the same bytes in every section and buffer.  Rows around a tile of sixteen, a section of one token, pieces of 16
    and of 4 bytes, copies of several rounds; channels that are one group, equal, infinite or no numbers."""
    from turboquant_amd import _ffi
    from turboquant_amd.kv_cache import TurboQuantKVCache
    g = torch.Generator().manual_seed(n_c + d)
    k, v = (torch.randn(B, H, n_c + n_buf + 1, d, generator=g).to(gpu) for _ in range(2))
    v[0, 0, n_c, : d // 2] = 2.5
    v[-1, -1, n_c, 3] = float("inf")
    v[0, -1, n_c, 5] = float("nan")
    states = []
    try:
        for how in (-1, 0, None):                              # one launch, two, the general path
            cache = TurboQuantKVCache(d, key_bits=key_bits, value_bits=vb, value_group_size=gs, buffer_size=n_buf, device=gpu, dtype=torch.float32)
            cache.prefill(k[..., :n_c + n_buf, :].contiguous(), v[..., :n_c + n_buf, :].contiguous())
            assert _ffi.lib().tq_set_option(b"append_small", how if how is not None else -1) == 0
            cache.key_buffer, cache.value_buffer = cache.key_buffer.contiguous(), cache.value_buffer.contiguous()
            new = [t[..., n_c + n_buf:, :].contiguous() for t in (k, v)]
            if how is None:
                cache._append(*new)
            else:
                spare = copy.copy(cache)
                launches = _nodes(lambda: spare._append_spill(*new))
                assert launches == (1 if how == -1 and d != 64 else 2)
                assert cache._append_spill(*new)
            states.append([*cache.key_quantized[:4], *cache.value_quantized[:3], cache.key_buffer, cache.value_buffer])
    finally:
        _ffi.lib().tq_set_option(b"append_small", -1)
    for other in states[1:]:
        for a, b in zip(states[0], other):
            assert a.shape == b.shape and torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.parametrize("d,rows,n_buf,how", [(128, 3, 4, -1), (128, 17, 1, 0), (256, 2, 2, -1), (64, 5, 3, -1)])
def test_cache_token_into_an_empty_part(gpu, d, rows, n_buf, how):
    """The library's entry with no compressed tokens yet, whose old sections are not there: the first ones are the quantisers' codes of the row that
    leaves, byte for byte."""
    import ctypes as C
    from turboquant_amd import _ffi
    from turboquant_amd.kv_cache import quantize_values
    lib, tq = _ffi.lib(), TurboQuantProd(d, bits=3, device=gpu)
    g = torch.Generator().manual_seed(d)
    kb, vb = (torch.randn(rows, n_buf, d, generator=g).to(gpu) for _ in range(2))
    key, value = (torch.randn(rows, d, generator=g).to(gpu) for _ in range(2))
    byte = dict(dtype=torch.uint8, device=gpu)
    idx, signs, data = torch.empty(rows, d // 4, **byte), torch.empty(rows, d // 8, **byte), torch.empty(rows, d // 2, **byte)
    norms, rnorms, scales, zeros = (torch.empty(rows, n, device=gpu) for n in (1, 1, d // 32, d // 32))
    nk, nv = torch.empty_like(kb), torch.empty_like(vb)
    work = torch.empty(lib.tq_cache_append_bytes(rows, d, 2, 4, 32), **byte)
    ly = tq._layer()
    _set_option("append_small", how)
    try:
        _ffi.check(lib.tq_cache_append(
            key.data_ptr(), value.data_ptr(), d, d, kb.data_ptr(), vb.data_ptr(), rows * n_buf * d, n_buf * d, d, rows * n_buf * d, n_buf * d, d, rows, rows,
            n_buf, C.byref(ly), 4, 32, 0, *[None] * 7, idx.data_ptr(), signs.data_ptr(), norms.data_ptr(), rnorms.data_ptr(), data.data_ptr(),
            scales.data_ptr(), zeros.data_ptr(), nk.data_ptr(), nv.data_ptr(), work.data_ptr(), _ffi.stream_ptr(gpu)), "tq_cache_append")
        torch.cuda.synchronize()
    finally:
        _set_option("append_small", -1)
    kq, vq = tq.quantize(kb[:, 0]), quantize_values(vb[:, :1], bits=4, group_size=32)
    for got, want in zip((idx, signs, rnorms, norms, data, scales, zeros), (*kq[:4], *vq[:3])):
        assert torch.equal(got.flatten(), want.flatten())
    assert torch.equal(nk, torch.cat([kb[:, 1:], key[:, None]], dim=1)) and torch.equal(nv, torch.cat([vb[:, 1:], value[:, None]], dim=1))


@pytest.mark.parametrize("d,B,H,n_c,n_q,step", [(128, 1, 8, 300, 1, 3), (64, 2, 3, 65, 1, 2), (256, 1, 2, 40, 5, 2), (128, 2, 2, 17, 3, 1)])
def test_cache_scores_of_queries_that_lie_apart(gpu, d, B, H, n_c, n_q, step):
    """A token's slice of a tensor of all queries gives the scores of its copy, bit for bit."""
    from turboquant_amd.kv_cache import TurboQuantKVCache
    g = torch.Generator().manual_seed(d + n_c)
    k, v = (torch.randn(B, H, n_c + 9, d, generator=g).to(gpu) for _ in range(2))
    q = torch.randn(B, H, n_q * step, d, generator=g).to(gpu)
    cache = TurboQuantKVCache(d, key_bits=3, value_bits=2, buffer_size=9, device=gpu, dtype=torch.float32)
    cache.prefill(k, v)
    part = q[..., 1 % step::step, :] if n_q > 1 else q[..., step - 1:, :]
    assert torch.equal(cache.attention_scores(part), cache.attention_scores(part.clone(memory_format=torch.contiguous_format)))
    for pad in (0, 1):                                  # rows on 16-byte boundaries, and a word off them
        wide = torch.randn(B, H, n_q, 2 * d + pad, generator=g).to(gpu)[..., d + pad:]
        assert torch.equal(cache.attention_scores(wide), cache.attention_scores(wide.contiguous()))


@pytest.mark.parametrize("d,H,n_c,n_buf,vb", [(64, 8, 1000, 128, 2), (128, 8, 300, 128, 4), (256, 3, 2000, 33, 2)])
def test_cache_blocks_of_queries_on_either_side_of_the_limit(gpu, counted, d, H, n_c, n_buf, vb):
    """The largest block of queries that takes the entry, and the next one, which takes the general path: results as from products in fp64
    of what the cache holds (fp32 sums, 2e-6 of the norm), and scratch that stays small."""
    from turboquant_amd import kv_cache as KC
    g = torch.Generator().manual_seed(d)
    k, v = (torch.randn(1, H, n_c + n_buf, d, generator=g).to(gpu) for _ in range(2))
    cache = KC.TurboQuantKVCache(d, value_bits=vb, buffer_size=n_buf, device=gpu, dtype=torch.float32)
    cache.prefill(k, v)
    keys = torch.cat([cache.key_quantizer.dequantize(cache.key_quantized), cache.key_buffer], dim=2).double()
    values = torch.cat([KC.dequantize_values(cache.value_quantized), cache.value_buffer], dim=2).double()

    def last(few):
        lo, hi = 1, 1 << 16
        while hi - lo > 1:
            mid = (lo + hi) // 2
            lo, hi = (mid, hi) if few(H * mid, n_c, n_buf, d) else (lo, mid)
        return lo

    most = last(KC.TurboQuantKVCache._few_score_queries)
    for n_q in (most, most + 1):
        q = torch.randn(1, H, n_q, d, generator=g).to(gpu)
        got, want = cache.attention_scores(q), torch.matmul(q.double(), keys.transpose(-2, -1).contiguous()) / d ** 0.5
        assert counted.take("tq_cache_scores", "tq_cache_scores_rows") == (n_q == most)
        assert float((got - want).norm()) <= 2e-6 * float(want.norm())
    most = last(KC.TurboQuantKVCache._few_value_queries)
    assert counted._lib.tq_cache_attend_bytes(H, most, d, n_c, n_buf) <= 32 << 20
    for n_q in (most, most + 1):
        w = torch.softmax(torch.randn(1, H, n_q, n_c + n_buf, generator=g), dim=-1).to(gpu)
        got, want = cache.attend(w), torch.matmul(w.double(), values)
        assert counted.take("tq_cache_attend") == (n_q == most)
        assert float((got - want).norm()) <= 2e-6 * float(want.norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_cache_products_under_autocast(gpu, dtype):
    """Scores and values have the type, and the rounding, that autocast gives the products of the general paths."""
    from turboquant_amd import kv_cache as KC
    g = torch.Generator().manual_seed(4)
    k, v = (torch.randn(1, 2, 300, 128, generator=g).to(gpu) for _ in range(2))
    cache = KC.TurboQuantKVCache(128, buffer_size=128, device=gpu, dtype=torch.float32)
    cache.prefill(k, v)
    q = torch.randn(1, 2, 1, 128, generator=g).to(gpu)
    w = torch.softmax(torch.randn(1, 2, 1, 300, generator=g), dim=-1).to(gpu)
    with torch.autocast("cuda", dtype=dtype):
        scores, out = cache.attention_scores(q), cache.attend(w)
        tail = torch.matmul(q, cache.key_buffer.transpose(-2, -1).contiguous()) * (1 / 128 ** 0.5)
        want = torch.matmul(w[..., :172], KC.dequantize_values(cache.value_quantized)) + torch.matmul(w[..., 172:], cache.value_buffer)
    assert out.dtype == want.dtype == dtype and torch.equal(out, want)
    assert torch.equal(scores[..., 172:], tail.to(scores.dtype))


def test_cache_and_ring_of_tensors_that_are_negated_lazily(gpu):
    """A tensor whose sign torch keeps beside its memory (the imaginary part of a conjugate) is read with that sign."""
    from turboquant_amd.capture import RingBuffer
    from turboquant_amd.kv_cache import TurboQuantKVCache
    g = torch.Generator().manual_seed(6)
    k, v = (torch.randn(1, 2, 302, 128, generator=g).to(gpu) for _ in range(2))
    q = torch.randn(1, 2, 1, 128, generator=g).to(gpu)
    results = []
    for lazy in (False, True):
        neg = torch._neg_view if lazy else torch.neg
        cache = TurboQuantKVCache(128, buffer_size=128, device=gpu, dtype=torch.float32)
        cache.prefill(k[..., :300, :], v[..., :300, :])
        for t in (300, 301):
            cache.append(neg(k[..., t:t + 1, :]), neg(v[..., t:t + 1, :]))
        w = torch.softmax(cache.attention_scores(q), dim=-1)
        ring = RingBuffer(4, 2, 128, device=gpu, dtype=torch.float32)
        ring.write(neg(k[0, :, 0]).view(1, 2, 128), neg(v[0, :, 0]).view(1, 2, 128), 1)
        results.append((cache.key_buffer, cache.value_buffer, cache.attention_scores(q), cache.attend(neg(w)), *ring.peek()))
    for a, b in zip(*results):
        assert a.shape == b.shape and float((a - b).norm()) <= 2e-6 * float(a.norm())


# ------------------------------------------------------------------ inner products and flat codes of small calls
@pytest.mark.parametrize("d,bits,lead,n_k,n_q,dtype", [
    (64, 2, (), 1, 1, torch.float32), (128, 3, (2,), 63, 16, torch.bfloat16), (128, 5, (1, 3), 65, 17, torch.float32),
    (256, 4, (), 64, 33, torch.float16), (320, 3, (2,), 130, 5, torch.float32), (576, 4, (), 100, 40, torch.float32),
    (192, 2, (), 17, 15, torch.float32), (128, 3, (8,), 4097, 31, torch.float32)])
def test_inner_products_on_the_matrix_cores(gpu, d, bits, lead, n_k, n_q, dtype):
    """tq_score against the same codes in float64.  Bound: two fp32 sums of d products each, of numbers that are themselves fp32
    sums of d products of the query with a row of Pi (norm 1) or S (at most `big`): d 2^-24 of the magnitudes, twice."""
    from turboquant_amd.quantizer import TurboQuantProd
    tq = TurboQuantProd(d, bits=bits, device=gpu)
    g = torch.Generator().manual_seed(d + n_k)
    k = torch.randn(*lead, n_k, d, generator=g).to(gpu, dtype)
    q = torch.randn(*lead, n_q, d, generator=g).to(gpu, dtype)
    code = tq.quantize(k)
    got = tq.attention_score(q, code).double().cpu()
    per = 8 // {1: 1, 2: 2, 3: 4, 4: 4}[bits - 1]
    packed = code.mse_indices.cpu().long()
    index = torch.stack([packed >> (8 // per * s) & (1 << 8 // per) - 1 for s in range(per)], -1).flatten(-2)[..., :d]
    sign = torch.stack([code.qjl_signs.cpu().long() >> s & 1 for s in range(8)], -1).flatten(-2)[..., :d].double() * 2 - 1
    cent = tq.mse_quantizer.centroids.double().cpu()[index] * code.norms.double().cpu()[..., None]
    sign = sign * (tq.qjl_scale * code.residual_norms.double().cpu()[..., None])
    Pi, S, q64 = tq.mse_quantizer.Pi.double().cpu(), tq.S.double().cpu(), q.double().cpu()
    rot, sk = q64 @ Pi.T, q64 @ S.T
    want = rot @ cent.transpose(-1, -2) + sk @ sign.transpose(-1, -2)
    big = max(1.0, float(S.norm(dim=1).max()))
    length = q64.norm(dim=-1, keepdim=True) * torch.ones(d, dtype=torch.float64)
    bound = 2 * d * 2 ** -24 * ((rot.abs() + length) @ cent.abs().transpose(-1, -2) + (sk.abs() + big * length) @ sign.abs().transpose(-1, -2))
    assert got.shape == want.shape and bool(((got - want).abs() <= bound + 4e-7 * want.abs()).all())


def test_inner_products_with_more_keys_than_a_grid_counts(gpu):
    """2^30 + 77 keys of 64 (29 GB): more threads along the keys than a launch may have.  The estimates at both ends and around the places where
    a launch ends are those of the same codes alone, bit for bit."""
    from turboquant_amd.quantizer import ProdQuantized, TurboQuantProd
    n = (1 << 30) + 77
    g = torch.Generator(device=gpu).manual_seed(3)
    tq = TurboQuantProd(64, bits=2, device=gpu)
    codes = torch.empty(2, n, 8, dtype=torch.uint8, device=gpu).random_(generator=g)
    norms = torch.empty(2, n, device=gpu).uniform_(0.5, 2.0, generator=g)
    q = torch.randn(1, 64, generator=g, device=gpu)
    got = tq.attention_score(q, ProdQuantized(codes[0], codes[1], norms[0], norms[1], 1))
    for at in (0, (1 << 28) - 40, (1 << 29) - 40, 3 * (1 << 28) - 40, (1 << 30) - 40, n - 100):
        part = slice(at, at + 100)
        want = tq.attention_score(q, ProdQuantized(codes[0, part].clone(), codes[1, part].clone(), norms[0, part].clone(), norms[1, part].clone(), 1))
        assert torch.equal(got[:, part], want)


@pytest.mark.parametrize("d,bits,dtype", [(128, 3, torch.float32), (128, 4, torch.bfloat16), (256, 3, torch.float16)])
def test_flat_codes_of_few_vectors_are_those_of_many(gpu, d, bits, dtype):
    """A tile of 16 vectors per workgroup in small calls, groups of tiles in large ones: codes, norms and de-quantised rows bit for bit."""
    from turboquant_amd.quantizer import ProdQuantized, TurboQuantProd
    tq = TurboQuantProd(d, bits=bits, device=gpu)
    g = torch.Generator().manual_seed(d)
    k = (torch.randn(20000, d, generator=g) * 2).to(gpu, dtype)
    many = tq.quantize(k)
    rows = tq.dequantize(many)
    for n in (1, 15, 16, 17, 33, 8191, 8192, 8193):
        few = tq.quantize(k[5:5 + n])
        for x, y in zip(few[:4], many[:4]):
            assert torch.equal(x, y[5:5 + n])
        assert torch.equal(tq.dequantize(few), rows[5:5 + n])


# ------------------------------------------------------------------ keys and values of a small append in one launch
def _nodes(call):
    """Nodes of a graph that `call` is captured into."""
    import ctypes
    from turboquant_amd import _ffi
    graph, n = torch.cuda.CUDAGraph(keep_graph=True), ctypes.c_size_t()
    with torch.cuda.graph(graph):
        call()
    assert _ffi.lib().hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("d,B,H,T,kb,vb,gs,dtype,ragged", [
    (128, 1, 1, 1, 3, 2, 32, torch.bfloat16, False), (128, 33, 3, 1, 4, 4, 16, torch.float16, False),
    (256, 5, 2, 17, 3, 4, 128, torch.bfloat16, False), (256, 16, 8, 1, 2, 2, 64, torch.float16, False),
    (128, 128, 4, 1, 2, 4, 32, torch.bfloat16, False), (128, 3, 2, 40, 5, 2, 64, torch.bfloat16, True), (256, 7, 1, 33, 4, 4, 32, torch.float16, True)])
def test_small_append_in_one_launch(gpu, d, B, H, T, kb, vb, gs, dtype, ragged):
    """The same pages as two launches write, byte for byte, over pages that hold other tokens already; a sequence whose run
    leaves the block table and one whose page lies outside the pool write nothing there."""
    g = torch.Generator().manual_seed(d + B)
    per_seq = 5
    tq = TurboQuantProd(d, bits=kb, device=gpu)
    table = torch.randperm(B * per_seq, generator=g).view(B, per_seq).to(torch.int32)
    starts = torch.randint(0, 30, (B,), generator=g).to(torch.int32)
    if B > 4:
        starts[2] = per_seq * 16 - 1 if T > 1 else per_seq * 16
        table[3] = B * per_seq + 7
    lens = [T - (b % 3 if ragged else 0) for b in range(B)]
    rows = (sum(lens), H, d) if ragged else (B, T, H, d)
    k, v = (torch.randn(*rows, generator=g).to(gpu, dtype) for _ in range(2))
    fill = torch.randint(0, 256, (B * per_seq,), generator=g, dtype=torch.uint8).to(gpu)
    table_gpu, starts_gpu = table.to(gpu), starts.to(gpu)
    got, nodes = [], []
    for one in (True, False):
        pool = PagedKVPool(tq, H, B * per_seq, value_bits=vb, value_group_size=gs, dtype=dtype, device=gpu)
        pool.data += fill[:, None, None]
        try:
            _set_option("append_small", -1 if one else 0)
            if ragged:
                row0 = _i32([sum(lens[:b]) for b in range(B)], gpu)
                pool.append_ragged(k, v, row0, _i32(lens, gpu), starts.to(gpu), table.to(gpu), max_run=T)
            else:
                pool.append(k, v, table_gpu, start_pos=starts_gpu)
                nodes.append(_nodes(lambda: pool.append(k, v, table_gpu, start_pos=starts_gpu)))
        finally:
            _set_option("append_small", -1)
        got.append(pool.data.clone())
    assert ragged or nodes[0] == nodes[1] - 1
    assert torch.equal(*got) and not torch.equal(got[0], torch.zeros_like(got[0]) + fill[:, None, None])


# ------------------------------------------------------------------ a ring's rows in one launch
@pytest.mark.parametrize("H,d,dtype,n,capacity", [(8, 128, torch.bfloat16, 1, 4), (1, 64, torch.float16, 5, 3), (3, 64, torch.float32, 257, 300),
                                                  (5, 66, torch.bfloat16, 2, 4)])
def test_ring_rows_from_any_layout(gpu, counted, H, d, dtype, n, capacity):
    """Rows of every layout a caller may hand over - side by side, in a wider tensor, heads transposed, one row repeated, misaligned, of
    another type, needing a gradient, the ring's own - end in the ring as torch's copies leave them, whoever copies them."""
    from turboquant_amd.capture import RingBuffer
    g = torch.Generator().manual_seed(n)
    wide = torch.randn(n, 3, H, d, generator=g).to(gpu, dtype)
    flat = torch.randn(n * H * d + 1, generator=g).to(gpu, dtype)
    forms = [wide[:, 1].contiguous(), wide[:, 1], wide[:, 0].transpose(0, 1).contiguous().transpose(0, 1), wide[:1, 2].expand(n, H, d),
             flat[1:].view(n, H, d), wide[:, 2].double(), wide[:, 2].clone().requires_grad_()]
    taken = set()
    for ix, x in enumerate(forms):
        for iy, y in enumerate(forms):
            ring, want = RingBuffer(capacity, H, d, gpu, dtype), RingBuffer(capacity, H, d, gpu, dtype)
            want._write_rows = lambda *a: False
            outs = []
            for r in (ring, want):
                out = [r.write(x, y, n), r.write(x[:1], y[:1], 1)]
                outs.append([t.detach() for o in out if o is not None for t in o] + [t.detach() for t in r.peek()])
            assert len(outs[0]) == len(outs[1]) and all(torch.equal(a, b) for a, b in zip(*outs))
            assert ring._rows.requires_grad == want._rows.requires_grad
            if counted.take("tq_ring_write"):
                taken.add((ix, iy))
    plain = {(i, j) for i in (0, 1, 3) for j in (0, 1, 3)} if H * d * forms[0].element_size() % 16 == 0 else set()
    assert plain <= taken and not any(i in (4, 5, 6) for pair in taken for i in pair)
    ring = RingBuffer(capacity, H, d, gpu, dtype)
    ring.write(forms[0], forms[0], 1)
    before = ring._rows._version
    ring.write(*ring.peek(), 1)
    assert torch.equal(ring._rows[0, 0], ring._rows[0, 1]) and ring._rows._version > before
    with torch.inference_mode():
        r2 = RingBuffer(capacity, H, d, gpu, dtype)
        r2.write(forms[0], forms[1], 1)
        assert torch.equal(r2.peek()[0], forms[0][:1]) and torch.equal(r2.peek()[1], forms[1][:1])
    with pytest.raises(RuntimeError):
        r2.write(forms[0], forms[1], 1)


# ------------------------------------------------------------------ groups of tiles that are heads of one page, and others
@pytest.mark.parametrize("d,H,kb,dtype", [(128, 8, 3, torch.bfloat16), (128, 6, 2, torch.float16), (128, 7, 4, torch.bfloat16), (256, 3, 3, torch.bfloat16),
                                          (256, 4, 4, torch.float16)])
@pytest.mark.parametrize("form", ["runs", "ragged", "blocks"])
def test_append_of_many_heads_is_that_of_each(gpu, d, H, kb, dtype, form):
    """More tiles than a launch of single tiles takes: groups whose tiles are heads of one page share an address, groups that
    begin in one page and end in the next do not.  Every head's pages are those of a pool that holds it alone."""
    g = torch.Generator().manual_seed(10 * d + H)
    B, T = 3, 1500
    tq = TurboQuantProd(d, bits=kb, device=gpu)
    per_seq = T // 16 + 4
    table = torch.randperm(B * per_seq, generator=g).view(B, per_seq).to(torch.int32).to(gpu)
    lens, starts = [T, T - 33, 700], [0, 5, 31]
    if form == "blocks":
        starts = [16, 0, 32]
    k, v = (torch.randn(B, T, H + 1, d, generator=g).to(gpu, dtype) for _ in range(2))
    blocks = torch.randn(2, B * per_seq, 16, H + 1, d, generator=g).to(gpu, dtype)
    src = torch.randperm(B * per_seq, generator=g).view(B, per_seq).to(torch.int32).to(gpu)

    def pages(lo, n):
        pool = PagedKVPool(tq, n, B * per_seq, value_bits=2, dtype=dtype, device=gpu)
        kk, vv = k[:, :, lo:lo + n], v[:, :, lo:lo + n]
        if form == "runs":
            pool.append(kk, vv, table, start_pos=_i32(starts, gpu))
        elif form == "ragged":
            pool.append_ragged(kk.reshape(B * T, n, d), vv.reshape(B * T, n, d), _i32([0, T, 2 * T], gpu), _i32(lens, gpu), _i32(starts, gpu), table,
                               max_run=T)
        else:
            pool.append_from_blocks(blocks[0][:, :, lo:lo + n], blocks[1][:, :, lo:lo + n], src, table, _i32(lens, gpu), start_pos=_i32(starts, gpu),
                                    max_tokens=T)
        return pool.data

    whole = pages(0, H)
    for h in range(H):
        assert torch.equal(whole[:, h], pages(h, 1)[:, 0])


# ------------------------------------------------------------------ the last round of a large append
@pytest.mark.parametrize("d,H,rest", [(128, 8, 8), (128, 8, 512), (128, 8, 520), (128, 3, 301), (256, 2, 2), (256, 2, 256), (256, 2, 258), (256, 1, 511)])
@pytest.mark.parametrize("ragged", [False, True])
def test_last_round_of_single_tiles(gpu, d, H, rest, ragged):
    """`rest` tiles more than whole rounds of 512 workgroups: up to the limit of the rule, one behind it.  The pages are those of
    appends of a few tokens each."""
    g = torch.Generator().manual_seed(d + rest)
    tiles = 512 * (8192 // d // 16)
    pages = -(-(tiles + rest) // H)
    N = 16 * pages - 3
    tq = TurboQuantProd(d, bits=3, device=gpu)
    k, v = (torch.randn(1, N, H, d, generator=g).bfloat16().to(gpu) for _ in range(2))
    table = torch.randperm(2 * pages, generator=g).view(2, pages).to(torch.int32).to(gpu)
    got, want = (PagedKVPool(tq, H, 2 * pages, value_bits=2, device=gpu) for _ in range(2))
    if ragged:
        got.append_ragged(k[0], v[0], _i32([N, 0], gpu), _i32([0, N], gpu), _i32([0, 0], gpu), table, max_run=N)
    else:
        got.append(k, v, table[1:])
    step = 4096
    for t in range(0, N, step):
        want.append(k[:, t:t + step], v[:, t:t + step], table[1:], start_pos=_i32([t], gpu))
    assert torch.equal(got.data, want.data)
