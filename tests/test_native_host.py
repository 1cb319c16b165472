"""The native host side of small calls (csrc/tq_host.cpp) against the Python methods it stands in front of: the same results bit for
bit where it takes a call, and nothing done where it does not."""

import threading

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from turboquant_amd import _ffi
from turboquant_amd.capture import RingBuffer
from turboquant_amd.kv_cache import TurboQuantKVCache
from turboquant_amd.paged import PagedKVPool
from turboquant_amd.quantizer import TurboQuantProd

pytestmark = pytest.mark.gpu


class _Watched:
    """The native side, with the answers it gave; `off` leaves the Python methods alone."""

    def __init__(self, host, off):
        self.host, self.off, self.taken, self.left = host, off, 0, 0

    def __getattr__(self, name):
        def call(*args):
            r = None if self.off else getattr(self.host, name)(*args)
            if r is None or r is False:
                self.left += 1
            else:
                self.taken += 1
            return r
        return call


@pytest.fixture
def both(gpu, monkeypatch):
    """both(run) -> (result with the native side, result without, calls it took, calls it left)"""
    _ffi.lib()
    assert _ffi.native() is not None, "the native host side is not built"
    host = _ffi._host

    def run_both(run):
        out = []
        for off in (False, True):
            watched = _Watched(host, off)
            monkeypatch.setattr(_ffi, "_host", watched)
            out.append(run())
            if not off:
                taken, left = watched.taken, watched.left
        monkeypatch.setattr(_ffi, "_host", host)
        return out[0], out[1], taken, left
    return run_both


def _same(a, b):
    if torch.is_tensor(a):
        return a.dtype == b.dtype and a.is_inference() == b.is_inference() and a.shape == b.shape and torch.equal(a.flatten().view(torch.uint8), b.flatten().view(torch.uint8))
    if isinstance(a, (tuple, list)):
        return len(a) == len(b) and all(_same(x, y) for x, y in zip(a, b))
    return a == b


@pytest.mark.parametrize("d,bits,dtype", [(128, 3, torch.float32), (64, 2, torch.bfloat16), (256, 4, torch.float16), (576, 4, torch.bfloat16)])
@pytest.mark.parametrize("form", ["plain", "one", "rows of a wider tensor", "transposed", "negated", "gradient", "inference", "none"])
def test_codes_scores_and_keys(gpu, both, d, bits, dtype, form):
    q = TurboQuantProd(d, bits=bits, device=gpu)
    g = torch.Generator().manual_seed(d + bits)
    x = torch.randn(3, 40, d, generator=g).to(gpu, dtype)
    y = torch.randn(3, 5, d, generator=g).to(gpu, dtype)
    if form == "one":
        x, y = x[:1, :1].contiguous(), y[:1, :1].contiguous()
    elif form == "rows of a wider tensor":
        x = torch.cat([x, x], dim=-1)[..., :d]
    elif form == "transposed":
        x = x.transpose(0, 1).contiguous().transpose(0, 1)
    elif form == "negated":
        x = torch._neg_view(x)
    elif form == "none":
        x = x[:, :0]

    def run():
        with torch.inference_mode(form == "inference"):
            z = x.clone().requires_grad_() if form == "gradient" else x
            if form == "none":                                 # (its codes have no last dimension to infer)
                with pytest.raises(RuntimeError):
                    q.quantize(z)
                return []
            code = q.quantize(z)
            if form == "negated":                              # (keys are read as their memory holds them)
                return list(code[:4])
            return [*code[:4], q.attention_score(y, code), q.dequantize(code)]
    a, b, taken, left = both(run)
    assert _same(a, b)
    assert taken == {"plain": 3, "one": 3, "inference": 3, "none": 0, "negated": 0}.get(form, 2) and left == (1 if taken < 3 else 0)


@pytest.mark.parametrize("d,Hq,Hkv,bits,vb,dtype", [(128, 8, 2, 3, 4, torch.bfloat16), (64, 6, 2, 4, 2, torch.float16), (256, 4, 1, 3, 2, torch.bfloat16),
                                                     (576, 24, 1, 4, 4, torch.bfloat16), (128, 3, 3, 3, 2, torch.float32)])
def test_pages_and_decode_steps(gpu, both, d, Hq, Hkv, bits, vb, dtype):
    quant = TurboQuantProd(d, bits=bits, device=gpu)
    g = torch.Generator().manual_seed(d + Hq)
    B, T = 3, 70
    k, v = (torch.randn(B, T, Hkv, d, generator=g).to(gpu, dtype) for _ in range(2))
    query = torch.randn(B, Hq, d, generator=g).to(gpu, dtype)
    exact = torch.randn(2, 5 * B, 16, Hkv, d, generator=g).to(gpu, dtype)
    table = torch.randperm(5 * B, generator=g).to(gpu, torch.int32).reshape(B, 5)
    lens = torch.tensor([70, 33, 64], dtype=torch.int32, device=gpu)
    start = torch.tensor([0, 3, 10], dtype=torch.int32, device=gpu)
    longest = 80

    def steps(query, table, lens, k, v):
        def run():
            pool = PagedKVPool(quant, Hkv, 5 * B, value_bits=vb, dtype=dtype, device=gpu)
            pool.append(k, v, table)
            first = pool.data.clone()
            pool.append(k[:, :1], v[:, :1], table, start_pos=start)
            outs = [first, pool.data.clone(), pool.decode_attention(query, table, lens, max_len=longest),
                    pool.decode_attention(query, table, lens, recent_k=k[:, :7], recent_v=v[:, :7], n_split=2),
                    pool.decode_attention(query[:1], table[0], lens[:1], scale=0.3)]
            return outs + [pool.decode_attention_ring(query, table, lens, exact[0], exact[1], 16, max_len=longest)]
        return run
    a, b, taken, left = both(steps(query, table, lens, k, v))
    assert _same(a, b) and (taken, left) == (6, 0)
    # lengths of 64 bits, a query of other strides, and keys and values of different strides are the Python methods' (the one-sequence
    # step's query is one row either way)
    odd = query.transpose(0, 1).contiguous().transpose(0, 1)
    c, e, taken, left = both(steps(odd, table, lens.long(), k, v.transpose(1, 2).contiguous().transpose(1, 2)))
    assert _same(c, e) and _same(a, c) and (taken, left) == ((0, 6) if Hkv > 1 else (2, 4))      # (one KV head: the same strides)
    # what is refused stays refused
    pool = PagedKVPool(quant, Hkv, 5 * B, value_bits=vb, dtype=dtype, device=gpu)
    with pytest.raises(ValueError):
        pool.append(k, v, table[:, :1])                        # 70 tokens do not fit a page
    with pytest.raises(TypeError):
        pool.append(k.double(), v.double(), table)
    with pytest.raises(TypeError):
        pool.decode_attention(query, table, lens, recent_k=k.double(), recent_v=v.double())


@pytest.mark.parametrize("form", ["plain", "step", "narrow", "own rows", "inference", "autocast", "no grad"])
def test_ring_rows(gpu, both, form):
    g = torch.Generator().manual_seed(5)
    k, v = (torch.randn(9, 2, 64, generator=g).to(gpu, torch.bfloat16) for _ in range(2))
    if form == "step":
        k, v = k[::2], v[::2]
    elif form == "narrow":
        k, v = (torch.cat([t, t], dim=-1)[..., 32:96] for t in (k, v))

    def run():
        ring = RingBuffer(8, 2, 64, gpu)
        with torch.inference_mode(form == "inference"), torch.autocast("cuda", torch.bfloat16, enabled=form == "autocast"):
            inner = RingBuffer(8, 2, 64, gpu) if form == "inference" else ring
            was = None if form == "inference" else inner._rows._version
            left = [inner.write(k, v, k.shape[0])]
            if form == "own rows":
                left.append(inner.write(inner._rows[0, 4:6], inner._rows[1, 4:6], 2))
            bumped = form == "inference" or inner._rows._version > was
        return [inner._rows.clone(), inner.size, bumped] + [t if t is None else list(t) for t in left]
    a, b, taken, left = both(run)
    assert _same(a, b) and a[2]
    assert (taken > 0) == (form not in ("narrow", "autocast")) and (left > 0) == (form in ("narrow", "autocast", "own rows"))


def _move_codes(cache):
    """The codes of a cache, one byte into buffers of their own."""
    def moved(t):
        return torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)
    kq, vq = cache.key_quantized, cache.value_quantized
    cache.key_quantized = kq._replace(mse_indices=moved(kq.mse_indices), qjl_signs=moved(kq.qjl_signs))
    cache.value_quantized = vq._replace(data=moved(vq.data))


@pytest.mark.parametrize("form", ["plain", "batches apart", "no value groups", "autocast", "bits put in", "gradient", "codes at odd bytes"])
def test_cache_tokens(gpu, both, form):
    g = torch.Generator().manual_seed(9)
    B, H, n, d = 2, 3, 150, 128
    k, v = (torch.randn(B, H, n + 3, d, generator=g).to(gpu) for _ in range(2))
    w = torch.randn(3, B, H, 2, d, generator=g).to(gpu)
    if form == "batches apart":
        k, v = (torch.cat([t, t], dim=1)[:, :H] for t in (k, v))

    def run():
        cache = TurboQuantKVCache(d, key_bits=3, value_bits=2, value_group_size=128 if form == "no value groups" else 32, buffer_size=64,
                                  device=gpu, dtype=torch.float32)
        cache.prefill(k[..., :n, :], v[..., :n, :])
        if form == "bits put in":
            cache.value_quantized = cache.value_quantized._replace(scales=cache.value_quantized.scales.half())
        outs = []
        with torch.autocast("cuda", torch.bfloat16, enabled=form == "autocast"):
            for i in range(3):
                if form == "codes at odd bytes":                   # (the library refuses what the checks before it let pass)
                    _move_codes(cache)
                if form != "bits put in":
                    cache.append(k[..., n + i:n + i + 1, :], v[..., n + i:n + i + 1, :])
                    if form == "codes at odd bytes":
                        _move_codes(cache)
                x = w[i].clone().requires_grad_() if form == "gradient" else w[i]
                scores = cache.attention_scores(x)
                outs += [scores.detach(), cache.attend(torch.softmax(scores.float(), dim=-1)).detach()]
        return outs + [*cache.key_quantized[:4], *cache.value_quantized[:3], cache.key_buffer, cache.value_buffer, cache.seq_len]
    a, b, taken, left = both(run)
    assert _same(a, b)
    # (a prompt's keys are a slice of the tensor: one call left to Python; where batches lie apart their tokens are too)
    assert (taken, left) == {"plain": (9, 1), "no value groups": (9, 1), "batches apart": (6, 7), "autocast": (0, 13), "bits put in": (3, 7),
                             "gradient": (3, 10), "codes at odd bytes": (3, 13)}[form]


@pytest.mark.parametrize("watch", ["vmap", "forward mode", "dispatch mode", "function mode", "trace", "deterministic"])
def test_what_has_to_see_an_operation_sees_it(gpu, both, watch):
    """Transforms, modes and traces, and fills of new memory: the calls are the Python methods', with their results, derivatives and errors."""
    g = torch.Generator().manual_seed(2)
    quant = TurboQuantProd(128, bits=3, device=gpu)
    k, v = (torch.randn(1, 2, 150, 128, generator=g).to(gpu) for _ in range(2))
    cache = TurboQuantKVCache(128, value_bits=2, buffer_size=64, device=gpu, dtype=torch.float32)
    cache.prefill(k, v)
    code = quant.quantize(k)
    query = torch.randn(1, 2, 3, 128, generator=g).to(gpu)
    weights = torch.softmax(torch.randn(1, 2, 3, 150, generator=g), dim=-1).to(gpu)
    calls = {"codes": (lambda x: list(quant.quantize(x)[:4]), k), "products": (lambda x: quant.attention_score(x, code), query),
             "scores": (cache.attention_scores, query), "values": (cache.attend, weights)}
    if watch == "trace":                                           # (a trace of torch's own operations)
        calls = {"values": calls["values"]}

    class Dispatch(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Dispatch.seen += 1
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        seen = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Function.seen += 1
            return func(*args, **(kwargs or {}))

    def watched(call, x):
        if watch == "vmap":
            return torch.vmap(call)(torch.stack([x, x]))
        if watch == "forward mode":
            with torch.autograd.forward_ad.dual_level():
                out = call(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
                return [y for t in (out if isinstance(out, list) else [out]) for y in torch.autograd.forward_ad.unpack_dual(t) if y is not None]
        if watch == "trace":
            return torch.jit.trace(call, (x,), check_trace=False)(x)
        with {"dispatch mode": Dispatch, "function mode": Function}[watch]():
            return call(x)

    def run():
        outs = []
        Dispatch.seen = Function.seen = 0
        for call, x in calls.values():
            if watch == "deterministic":
                torch.use_deterministic_algorithms(True, warn_only=True)
                try:
                    outs.append(call(x))
                finally:
                    torch.use_deterministic_algorithms(False)
                continue
            try:
                outs.append(watched(call, x))
            except RuntimeError as e:                              # (what the Python methods cannot do they refuse)
                outs.append(type(e).__name__)
        return outs + [Dispatch.seen, Function.seen]
    a, b, taken, left = both(run)
    assert _same(a, b) and taken == 0 and left >= 1
    if watch == "forward mode":
        assert len(a[3]) == 2 and float(a[3][1].abs().max()) > 0           # (the values' sum has a derivative)
    if watch in ("dispatch mode", "function mode"):
        assert a[-2] + a[-1] > 0


def test_threads_share_a_quantiser(gpu, both):
    """Calls of several threads, one of which has the quantiser's descriptors built again and again: the results of one thread alone."""
    quant = TurboQuantProd(128, bits=3, device=gpu)
    g = torch.Generator().manual_seed(8)
    xs = [torch.randn(40 + i, 128, generator=g).to(gpu) for i in range(3)]
    want = [list(quant.quantize(x)[:4]) + [quant.attention_score(x[:5], quant.quantize(x))] for x in xs]
    first = quant.mse_quantizer.quantize(xs[0]).indices

    def run():
        torch.cuda.synchronize()
        wrong = []

        def use(x, result):
            try:
                for _ in range(20):
                    code = quant.quantize(x)
                    if not _same(list(code[:4]) + [quant.attention_score(x[:5], code)], result):
                        wrong.append(x.shape)
            except Exception as e:
                wrong.append(repr(e))

        def rebuild():
            try:
                for _ in range(10):
                    quant.S.add_(0)
                    if not torch.equal(quant.mse_quantizer.quantize(xs[0]).indices, first):
                        wrong.append("first stage")
            except Exception as e:
                wrong.append(repr(e))
        threads = [threading.Thread(target=use, args=a) for a in zip(xs, want)] + [threading.Thread(target=rebuild)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        return wrong
    a, b, taken, left = both(run)
    assert a == b == [] and taken > 0 and left == 0


def test_a_captured_step_and_a_side_stream(gpu, both):
    """Outputs and workspaces come from the pool of the stream that the call runs on, and a captured step replays with new lengths."""
    quant = TurboQuantProd(128, bits=3, device=gpu)
    g = torch.Generator().manual_seed(3)
    k, v = (torch.randn(2, 96, 2, 128, generator=g).to(gpu, torch.bfloat16) for _ in range(2))
    query = torch.randn(2, 8, 128, generator=g).to(gpu, torch.bfloat16)
    table = torch.arange(12, dtype=torch.int32, device=gpu).reshape(2, 6)
    pool = PagedKVPool(quant, 2, 12, value_bits=4, dtype=torch.bfloat16, device=gpu)
    pool.append(k, v, table)
    lens = torch.tensor([96, 50], dtype=torch.int32, device=gpu)

    def run():
        n, outs = lens.clone(), []
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            outs.append(pool.decode_attention(query, table, n, max_len=96))
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = pool.decode_attention(query, table, n, max_len=96)
        for step in range(3):
            n.sub_(step)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, pool.decode_attention(query, table, n, max_len=96))
            outs.append(out.clone())
        return outs
    a, b, taken, left = both(run)
    assert _same(a, b) and left == 0 and taken == 5
