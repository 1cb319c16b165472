"""CPU: host-side logic of the package (no kernel launches): the C-ABI library
loads and exports what include/tq_hip.h declares, argument checking, page
geometry, codebook files, ring / capture policy against the reference's trace,
and the loud failure on CPU tensors."""

import copy
import ctypes as C
import gc
import json
import os
import pickle
import re
import sys
import types
import weakref

import numpy as np
import pytest
import torch

import turboquant_amd
from turboquant_amd import _ffi
from turboquant_amd.capture import KVCaptureEngine, RingBuffer
from turboquant_amd.codebook import compute_lloyd_max_codebook, get_codebook, get_codebook_tensors
from turboquant_amd.quantizer import TurboQuantMSE, TurboQuantProd, _pack_indices, _unpack_indices
from turboquant_amd.kv_cache import ValueQuantized, quantize_values, unpack_values

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "tq_hip.h")).read()
    declared = set(re.findall(r"\b(tq_[a-z_0-9]+)\s*\(", header))
    assert declared, "no declarations found"
    lib = _ffi.lib()
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} declared in tq_hip.h but not exported"
    assert declared == set(_ffi.EXPORTED_SYMBOLS)
    assert lib.tq_version() == _ffi.ABI_VERSION


@pytest.mark.parametrize("d", [128, 256])
def test_split_matrices_sum_exactly_and_follow_the_documented_operand_order(d):
    """The three bf16 terms of a split matrix add up to the fp32 matrix bit for bit, and element
    (row, col) of term t sits where include/tq_hip.h says the matrix-core kernels read it."""
    g = torch.Generator().manual_seed(d)
    m = torch.randn(d, d, generator=g) * torch.logspace(-6, 2, d)[None, :]
    raw = _ffi.split_bf16x3(m)
    assert raw.dtype == torch.int16 and raw.numel() == 3 * d * d
    flat = raw.reshape(-1).view(torch.bfloat16).float()
    t, r, c = torch.meshgrid(torch.arange(3), torch.arange(d), torch.arange(d), indexing="ij")
    pos = ((((t * (d // 16) + r // 16) * (d // 32) + c // 32) * 4 + (c % 32) // 8) * 16 + r % 16) * 8 + c % 8
    assert torch.equal(torch.sort(pos.reshape(-1)).values, torch.arange(3 * d * d))       # a permutation
    terms = flat[pos]                                                                       # (3, d, d) row-major
    want = m.clone()
    for k in range(3):                       # each term is the bf16 rounding of what the terms before it left
        assert torch.equal(terms[k], want.to(torch.bfloat16).float())
        want = want - terms[k]
    assert torch.equal(terms[0] + terms[1] + terms[2], m)
    with pytest.raises(ValueError):
        _ffi.split_bf16x3(torch.zeros(48, 48))


@pytest.mark.parametrize("d", [64, 192, 576])
def test_several_matrices_are_split_as_each_by_itself(d):
    m = torch.randn(3, d, d, generator=torch.Generator().manual_seed(d))
    raw = _ffi.split_bf16x3(m)
    for i in range(3):
        assert raw[i].is_contiguous() and torch.equal(raw[i], _ffi.split_bf16x3(m[i]))


@pytest.mark.parametrize("B", [1, 2, 3, 64, 1024, 1025])
@pytest.mark.parametrize("n_split", [1, 2, 31, 256, 257, 512, 2048])
def test_workspace_of_a_step_by_length_holds_the_equal_shares_it_may_fall_back_to(B, n_split):
    lib = _ffi.lib()
    for Hq, d in ((1, 64), (8, 128), (128, 576)):
        assert lib.tq_decode_workspace_bytes(B, Hq, d, -n_split) >= lib.tq_decode_workspace_bytes(B, Hq, d, n_split)


def _decode_args(n_split, rows=(None, None, 0, 0, 0, 0, None), stages=()):
    """Arguments of a decode entry that end in a refusal before anything is read or launched (a layer of head_dim 100)."""
    ly, layout = _ffi.TqLayer(), _ffi.TqPageLayout()
    ly.d = layout.d = 100
    return (1, 2, 4, 8, 2, 1, 16, 1, 4, 1, 1.0, C.byref(ly), C.byref(layout), *rows, 1, 1, n_split, *stages, None)


@pytest.mark.parametrize("n_split", [0, -1, -64, -(1 << 20), -(1 << 31)])
def test_a_split_count_that_is_not_positive_is_refused(n_split):
    """By every decode entry, with the code of an invalid argument; positive counts get as far as the head size."""
    lib, ring = _ffi.lib(), (1, 1, 64, 4, 4, 16)
    for n, want in ((n_split, -1), (1, -2), (1 << 20, -2)):
        assert lib.tq_decode_attn_paged(*_decode_args(n)) == want
        assert lib.tq_decode_attn_paged_stages(*_decode_args(n, stages=(7,))) == want
        assert lib.tq_decode_attn_paged_ring(*_decode_args(n, rows=ring)) == want
    for n, want in ((n_split, -1), (1 << 20, -1), (1, -2)):
        assert lib.tq_decode_attn_paged_by_length(*_decode_args(n)) == want
        assert lib.tq_decode_attn_paged_ring_by_length(*_decode_args(n, rows=ring)) == want


def test_argument_errors_are_reported_before_any_launch():
    lib = _ffi.lib()
    assert lib.tq_bucketize_pack(None, 4, 128, None, 2, None, None) == -3
    assert lib.tq_sign_pack(None, 4, 128, None, None) == -3
    ly = _ffi.TqLayer()
    ly.d, ly.mse_bits = 100, 2                       # not a multiple of 64
    assert lib.tq_quantize_keys(1, 0, 4, 128, C.byref(ly), 1, 1, 1, 1, None, None, 0, None) == -2
    assert lib.tq_quantize_values(1, 0, 4, 128, 128, 48, 2, 1, 1, 1, None) == -1     # 128 % 48 != 0
    assert lib.tq_quantize_values(1, 0, 4, 128, 128, 32, 3, 1, 1, 1, None) == -2     # 3-bit values
    assert lib.tq_decode_workspace_bytes(0, 8, 128, 4) == 0
    with pytest.raises(ValueError):
        _ffi.check(-1, "x")
    with pytest.raises(RuntimeError):
        _ffi.check(700, "x")
    with pytest.raises(TypeError):
        _ffi.dtype_tag(torch.float64)


@pytest.mark.parametrize("d,mb,vb,gs,dt,per_token", [
    (128, 2, 4, 32, torch.bfloat16, 32 + 16 + 4 + 4 + 64 + 16),      # 136 B: fp32 norm and residual norm
    (256, 2, 2, 32, torch.bfloat16, 64 + 32 + 4 + 4 + 64 + 32),      # 200 B
    (128, 2, 2, 32, torch.float16, 32 + 16 + 4 + 4 + 32 + 16),
    (128, 3, 4, 64, torch.float32, 48 + 16 + 4 + 4 + 64 + 16),
    (64, 2, 2, 32, torch.bfloat16, 16 + 8 + 4 + 4 + 16 + 8),
])
def test_page_layout_geometry(d, mb, vb, gs, dt, per_token):
    L = _ffi.make_page_layout(d, mb, vb, gs, dt)
    assert L.off_keys == 0 and L.key_lane_major == (1 if d % 128 == 0 or d == 64 else 0)
    offs = [L.off_keys, L.off_meta, L.off_vdata, L.off_vscale, L.off_vzero]
    assert offs == sorted(offs) and all(o % 16 == 0 for o in offs)
    used = L.off_vzero + (d // gs) * 16 * (4 if dt == torch.float32 else 2)
    assert used == 16 * per_token
    assert L.page_bytes % 128 == 0 and used <= L.page_bytes < used + 128
    with pytest.raises(ValueError):
        _ffi.make_page_layout(100, 2, 2, 32, torch.bfloat16)
    with pytest.raises(ValueError):
        _ffi.make_page_layout(128, 2, 3, 32, torch.bfloat16)


@pytest.mark.parametrize("d,mb", [(128, 1), (128, 2), (128, 3), (128, 4), (64, 2), (256, 2), (576, 3)])
def test_walsh_terms_reconstruct_the_codebook(d, mb):
    cb = get_codebook(d, mb)
    cent = torch.tensor(cb["centroids"], dtype=torch.float32)
    ly = _ffi.TqLayer()
    _ffi.walsh_terms(cent, mb, ly)
    assert 1 <= ly.n_terms <= 2 ** mb - 1
    # a symmetric codebook is an odd function of the +-1 index bits: only odd-size subsets survive
    assert ly.n_terms == 2 ** (mb - 1)
    for idx in range(2 ** mb):
        val = ly.term_const + sum(ly.term_coef[t] * (bin(idx & ly.term_mask[t]).count("1") & 1)
                                  for t in range(ly.n_terms))
        assert val == pytest.approx(float(cent[idx]), abs=2e-7)
    # an asymmetric codebook keeps every subset
    skew = torch.arange(2 ** mb, dtype=torch.float32) ** 2
    _ffi.walsh_terms(skew, mb, ly)
    for idx in range(2 ** mb):
        val = ly.term_const + sum(ly.term_coef[t] * (bin(idx & ly.term_mask[t]).count("1") & 1)
                                  for t in range(ly.n_terms))
        assert val == pytest.approx(float(skew[idx]), abs=1e-4)


def test_shipped_codebooks_equal_reference_files(golden):
    for d, b in [(64, 1), (64, 2), (64, 3), (64, 4), (128, 1), (128, 2), (128, 3), (128, 4), (576, 3),
                 (256, 1), (256, 2), (256, 3)]:
        ref, got = golden.codebook(d, b), get_codebook(d, b)
        assert got["d"] == d and got["bits"] == b
        assert set(got) == {"centroids", "boundaries", "mse_per_coord", "mse_total", "d", "bits"}
        assert np.allclose(got["centroids"], ref["centroids"], rtol=0, atol=1e-15)
        # the fp32 tensors handed to the kernels are identical
        c, e = get_codebook_tensors(d, b, "cpu")
        assert torch.equal(c, torch.tensor(ref["centroids"], dtype=torch.float32))
        # ... and so are the thresholds, the middle one included: two of the reference's tables hold
        # -4e-17 / -3e-18 there instead of 0, which decides the bucket of a coordinate that is exactly 0
        # (every coordinate of an all-zero vector), so the shipped tables carry the published values
        assert torch.equal(e, torch.tensor(ref["boundaries"], dtype=torch.float32)), (d, b)


def test_rotation_and_sketch_matrices_equal_the_reference_ones(golden):
    """generate_rotation_matrix / generate_qjl_matrix (rotation.py:17-56) against the matrices the
    reference produced for config 1 (seed 42, sketch seed 42 + 1000) and for the other golden cases.
    torch.randn from a seeded CPU generator is bit-stable, so S must match bit for bit; Pi goes
    through LAPACK's QR, whose summation order depends on the BLAS thread count (differences of 1e-6
    between 1 and 8 threads were observed), hence 2e-6."""
    from turboquant_amd.rotation import generate_qjl_matrix, generate_rotation_matrix
    z = golden.npz("config1_full")
    S = generate_qjl_matrix(128, "cpu", seed=42 + 1000)
    assert S.dtype == torch.float32 and torch.equal(S, torch.from_numpy(z["S"]))
    Pi = generate_rotation_matrix(128, "cpu", seed=42)
    ref = torch.from_numpy(z["Pi"])
    assert Pi.shape == ref.shape and (Pi - ref).abs().max() <= 2e-6
    assert (Pi @ Pi.T - torch.eye(128)).abs().max() < 1e-5
    # a wrong sign convention, a transposed factor or a different seed rule would be off by O(1)
    assert (Pi.T - ref).abs().max() > 0.1
    for file, case in golden.key_case_list():
        kc = golden.npz(file)
        d, bits, seed = [int(v) for v in kc[case + ".meta"]]
        if golden.has(file, case + ".S"):
            assert torch.equal(generate_qjl_matrix(d, "cpu", seed=seed + 1000), torch.from_numpy(kc[case + ".S"])), case
        assert (generate_rotation_matrix(d, "cpu", seed=seed) - torch.from_numpy(kc[case + ".Pi"])).abs().max() <= 2e-6, case
    # the quantiser objects draw their matrices through the same two functions, seeds as quantizer.py:107,208
    tq = TurboQuantProd(128, bits=3, device="cpu", seed=42)
    assert torch.equal(tq.S, torch.from_numpy(z["S"]))
    assert (tq.mse_quantizer.Pi - ref).abs().max() <= 2e-6


def test_codebook_solver_known_answer(golden):
    got = compute_lloyd_max_codebook(128, 2)
    ref = golden.codebook(128, 2)
    assert got["centroids"] == pytest.approx(ref["centroids"], abs=1e-15)
    assert got["mse_total"] == pytest.approx(0.11600007032012699, abs=1e-13)
    with pytest.raises(ValueError):
        compute_lloyd_max_codebook(2, 1)


def test_pack_helpers_match_reference_vectors(golden):
    z = golden.npz("packing")
    for bits in (1, 2, 3, 4, 5):
        for d in (128, 13):
            idx = torch.from_numpy(z[f"idx_b{bits}_d{d}"])
            pk = _pack_indices(idx, bits)
            assert pk.dtype == torch.uint8 and np.array_equal(pk.numpy(), z[f"packed_b{bits}_d{d}"])
            assert np.array_equal(_unpack_indices(pk, bits, d).numpy(), z[f"unpacked_b{bits}_d{d}"])
    vq = ValueQuantized(torch.tensor([[0b11100100, 0b00011011]], dtype=torch.uint8), None, None, 2)
    assert unpack_values(vq).tolist() == [[0, 1, 2, 3, 3, 2, 1, 0]]
    vq = ValueQuantized(torch.tensor([[0xA5]], dtype=torch.uint8), None, None, 4)
    assert unpack_values(vq).tolist() == [[5, 10]]


def test_public_surface():
    assert turboquant_amd.__version__ == "0.2.0"
    for name in ("compute_lloyd_max_codebook", "get_codebook", "TurboQuantMSE", "TurboQuantProd", "TurboQuantKVCache",
                 "RingBuffer", "KVCaptureEngine", "CompressedKVStore", "compute_hybrid_attention"):
        assert hasattr(turboquant_amd, name)
    tq = TurboQuantProd(128, bits=3, device=torch.device("cpu"))
    assert set(dict(tq.named_buffers())) >= {"S", "mse_quantizer.Pi", "mse_quantizer.centroids",
                                             "mse_quantizer.boundaries", "mse_quantizer.decision_boundaries"}
    assert set(tq.state_dict()) == {"S", "mse_quantizer.Pi", "mse_quantizer.centroids", "mse_quantizer.boundaries",
                                    "mse_quantizer.decision_boundaries"}
    assert tq.mse_quantizer.bits == 2 and tq.mse_quantizer.n_clusters == 4
    with pytest.raises(AssertionError):
        TurboQuantProd(128, bits=1, device=torch.device("cpu"))


def test_no_cpu_fallback():
    tq = TurboQuantProd(128, bits=3, device=torch.device("cpu"))
    x = torch.randn(4, 128)
    with pytest.raises(RuntimeError, match="GPU only"):
        tq.quantize(x)
    with pytest.raises(RuntimeError, match="GPU only"):
        tq.mse_quantizer.quantize(x)
    with pytest.raises(RuntimeError, match="GPU only"):
        quantize_values(x, 2, 32)


class _TagStore:
    def __init__(self, heads, dim):
        self.num_kv_heads, self.head_dim, self.device = heads, dim, torch.device("cpu")
        self.chunks = []

    @property
    def num_tokens(self):
        return sum(len(c) for c in self.chunks)

    def append_chunk(self, key, value):
        assert torch.equal(key, value)
        self.chunks.append([int(t) for t in key[:, 0, 0].float().tolist()])

    def reset(self):
        self.chunks = []


def test_capture_engine_routes_tokens_like_the_reference(golden):
    for tr in golden.json("capture_trace.json"):
        if tr.get("double_prefill"):
            st = _TagStore(1, 4)
            eng = KVCaptureEngine(st, ring_capacity=4, device="cpu", dtype=torch.float32)
            a = torch.arange(3.0).view(-1, 1, 1).expand(3, 1, 4)
            eng.ingest_prefill(a, a, 3)
            eng.ingest_prefill(a + 10, a + 10, 3)
        else:
            st = _TagStore(2, 8)
            eng = KVCaptureEngine(st, ring_capacity=tr["capacity"], device="cpu", dtype=torch.float32)
            tok = 0
            if tr["prefill"]:
                k = torch.arange(float(tr["prefill"])).view(-1, 1, 1).expand(tr["prefill"], 2, 8)
                eng.ingest_prefill(k, k, tr["prefill"])
                tok = tr["prefill"]
            for _ in range(tr["decodes"]):
                k = torch.full((1, 2, 8), float(tok))
                eng.ingest_decode(k, k, 1)
                tok += 1
            if tr["flush"]:
                eng.flush()
            assert eng.total_compressed_tokens == tr["total_compressed"]
            assert eng.total_buffered_tokens == tr["total_buffered"]
            assert eng.total_tokens == tr["total_compressed"] + tr["total_buffered"]
            assert eng.ring.total_written == tr["ring_total_written"]
        peek = eng.ring.peek()
        ring = [] if peek is None else [int(t) for t in peek[0][:, 0, 0].tolist()]
        assert st.chunks == tr["chunks"]
        assert ring == tr["ring"]


def test_ring_buffer_contract():
    rb = RingBuffer(4, 2, 8, "cpu", torch.float32)
    assert rb.size == 0 and not rb.is_full and rb.peek() is None and rb.drain() is None
    k = torch.arange(6.0).view(-1, 1, 1).expand(6, 2, 8)
    spill = rb.write(k, k, 6)
    assert spill is not None and spill[0][:, 0, 0].tolist() == [0, 1, 2, 3]
    assert rb.size == 2 and rb.total_written == 6
    assert rb.peek()[0][:, 0, 0].tolist() == [4, 5]
    got = rb.drain()
    assert got[0][:, 0, 0].tolist() == [4, 5] and rb.size == 0
    rb.reset()
    assert rb.total_written == 0


def test_paged_cache_ingest_gathers_blocks_in_table_order():
    st = _TagStore(1, 4)
    eng = KVCaptureEngine(st, ring_capacity=4, device="cpu", dtype=torch.float32)
    cache = torch.zeros(2, 5, 4, 1, 4)
    table = torch.tensor([3, 0, 4])
    for logical, phys in enumerate(table.tolist()):
        for s in range(4):
            cache[:, phys, s] = logical * 4 + s
    eng.ingest_prefill_from_paged_cache(cache, 10, table, 4)
    assert st.chunks == [[0, 1, 2, 3, 4, 5]]
    assert eng.ring.peek()[0][:, 0, 0].tolist() == [6, 7, 8, 9]


def test_fp6_digits_of_the_rotation_decode_back_to_it():
    """_ffi.split_fp6x5: the five fp6 (e2m3) digits and block scales of Pi^T, in the lane order of the block-scaled
    MFMA, decode back to the matrix within 2^-22 of each (row, 32-coordinate block)'s largest value (the permuted
    contraction index and the 0.5 / 1 / 2 / 0.5 position factors of the fp4 bit operand included)."""
    from turboquant_amd import _ffi
    from turboquant_amd.rotation import generate_rotation_matrix
    d = 128
    m = generate_rotation_matrix(d, "cpu", seed=42).T.contiguous()
    codes, scales = _ffi.split_fp6x5(m)
    assert tuple(codes.shape) == (d // 16, 1, 5, 64, 6) and tuple(scales.shape) == (d // 16, 1, 64, 2)
    c = codes.numpy().view(np.uint32).astype(np.uint64)
    sc = scales.numpy().view(np.uint32)
    s_idx = np.arange(32)
    coord = 4 * (s_idx % 8) + s_idx // 8
    factor = np.array([0.5, 1.0, 2.0, 0.5])[coord % 4]
    rec = np.zeros((d, d))
    for t in range(5):
        word = sc[:, 0, :, 0] if t < 4 else sc[:, 0, :, 1]                   # [tile][lane]
        e8 = ((word >> (8 * (t % 4))) & 0xFF).astype(np.int64) - 127
        for s_ in range(32):
            lo = 6 * s_
            w, sh = lo // 32, lo % 32
            code = (c[:, 0, t, :, w] >> np.uint64(sh)) & np.uint64(63)
            if sh > 26:
                code |= (c[:, 0, t, :, w + 1] << np.uint64(32 - sh)) & np.uint64(63)
            code = code.astype(np.int64)
            ex, man = (code >> 3) & 3, code & 7
            mag = np.where(ex == 0, man / 8.0, (1 + man / 8.0) * 2.0 ** (ex - 1))
            val = np.where(code & 32, -mag, mag) * 2.0 ** e8 * factor[s_]    # [tile][lane]
            for lane in range(64):
                rec[16 * np.arange(d // 16) + (lane & 15), 32 * (lane >> 4) + coord[s_]] += val[:, lane]
    ref = m.double().numpy()
    blockmax = np.abs(ref).reshape(d, d // 32, 32).max(-1).repeat(32, axis=1)
    assert np.all(np.abs(rec - ref) <= 2.0 ** -22 * 2.0 * blockmax)


def test_quotient_of_bf16_numbers_rounds_like_its_product_with_a_reciprocal():
    """The value quantiser (kv_cache.py:53-99 divides bf16 numbers and rounds to bf16) replaces a / s by
    a * r, r an fp32 reciprocal of s good to one ulp.  Both operands have at most 8 significant bits, so the
    quotient is never a rounding tie of bf16 and never closer than 2^-17 (relative) to one, far more than the
    product's error: the two round to the same bf16 number.  Exhaustive over all pairs of significands, the
    exponent offsets the quantiser can meet, and the three reciprocals nearest to 1 / s."""
    def bf16_bits(f):
        u = f.view(np.uint32).astype(np.uint64)
        return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint32)
    ms = np.arange(128, 256, dtype=np.float32)[:, None, None]
    ma = np.arange(128, 256, dtype=np.float32)[None, :, None]
    a = ma * np.exp2(np.arange(-30, 9, dtype=np.float32))[None, None, :]
    ref = bf16_bits((a / ms).astype(np.float32))
    r0 = (np.float32(1.0) / ms).astype(np.float32)
    for step in (-1, 0, 1):
        r = (r0.view(np.int32) + step).view(np.float32)
        got = bf16_bits((a * r).astype(np.float32))
        assert np.array_equal(got, np.broadcast_to(ref, got.shape)), step


def test_quotient_of_fp16_numbers_is_its_product_with_a_reciprocal_and_one_correction():
    """The value quantiser replaces a / s of fp16 numbers by q + (a - q s) r with q = a r, r an fp32 reciprocal of s good to one ulp:
    the same fp32 number, for all pairs of significands and the three reciprocals nearest to 1 / s (powers of two change nothing
    within the range that the kernel takes it for).  Both multiply-adds round once: their products have 35 and 48 bits."""
    def fma(a, b, c):
        return (np.float64(a) * np.float64(b) + np.float64(c)).astype(np.float32)
    s = np.arange(1024, 2048, dtype=np.float32)[:, None]
    a = np.arange(1024, 2048, dtype=np.float32)[None, :]
    ref = (a / s).astype(np.float32)
    r0 = (np.float32(1.0) / s).astype(np.float32)
    for step in (-1, 0, 1):
        r = (r0.view(np.int32) + step).view(np.float32)
        q = (a * r).astype(np.float32)
        assert np.array_equal(fma(fma(-q, s, a), r, q), ref), step


def test_bench_refuses_more_than_one_gpu_and_its_shape_table_is_well_formed():
    """bench.py measures one GPU: --gpus 2 exits with a message instead of running; the shapes of its table mode
    are ones the entry points accept (query heads a multiple of KV heads, head sizes a multiple of 64 up to 768,
    key bits 2 - 5, value bits 2 / 4 / 8) and the byte count per token and head follows the page layout."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert res.returncode == 2 and "one GPU" in res.stderr and res.stdout.strip() == ""
    sys.path.insert(0, root)
    import bench
    assert len(set(bench.SHAPE_TABLE)) == len(bench.SHAPE_TABLE)
    for (B, N, Hq, Hkv, d, kb, vb) in bench.SHAPE_TABLE:
        assert B > 0 and N > 0 and Hq % Hkv == 0 and d % 64 == 0 and 64 <= d <= 768
        assert 2 <= kb <= 5 and vb in (2, 4, 8)
    # 3-bit keys (2-bit indices), 2-bit values in groups of 32 at head_dim 256: 64 + 32 + 2 + 2 + 64 + 32 bytes
    assert bench.algorithmic_bytes_per_token_head(256, 2, 2, 32) == 196
    assert bench.algorithmic_bytes_per_token_head(128, 2, 4, 32) == 132


def test_a_rearranged_block_table_leaves_the_lengths_alone(monkeypatch):
    """A store's block_table is the caller's to rearrange (pages swapped, another page put in); the lengths and start positions
    of later calls are numbers of their own."""
    from turboquant_amd import store as ST
    calls = []

    class Pool:
        def __init__(self, quantizer, heads, pages, *args, dtype, device):
            self.num_pages, self.dtype, self.device = pages, dtype, torch.device("cpu")

        def append(self, key, value, block_table, start_pos=None):
            calls.append((block_table.tolist(), start_pos.tolist()))

    monkeypatch.setattr(ST, "PagedKVPool", Pool)
    st = ST.CompressedKVStore(64, 1, device=torch.device("cpu"))
    x = torch.zeros(3, 1, 64)
    st.append_chunk(x, x)
    table = st.block_table
    table.copy_(table.flip(1))
    st.append_chunk(x, x)
    pages = list(range(st.pool.num_pages))
    assert calls == [([pages], [0]), ([pages[::-1]], [3])]
    assert [st.lengths(n, 1).tolist() for n in (0, 3, 63)] == [[0], [3], [63]] and st.lengths(5, 3).tolist() == [5, 5, 5]


def test_a_compressed_part_put_in_by_hand_is_taken_as_it_is():
    """The cache object's entries for fp32 read codes of the cache's own bits and shape; any other state goes the general way."""
    from turboquant_amd.kv_cache import TurboQuantKVCache
    from turboquant_amd.quantizer import ProdQuantized
    cache = TurboQuantKVCache(128, key_bits=4, value_bits=2, device=torch.device("cpu"), dtype=torch.float32)

    def u8(w):
        return torch.zeros(1, 2, 5, w, dtype=torch.uint8)

    def f32(*w):
        return torch.zeros(1, 2, 5, *w)

    keys, values = ProdQuantized(u8(64), u8(16), f32(), f32(), 3), ValueQuantized(u8(32), f32(4), f32(4), 2)

    def plain(k=keys, v=values):
        cache.key_quantized, cache.value_quantized = k, v
        return cache._compressed_plain()

    assert plain()
    assert not plain(v=ValueQuantized(u8(64), f32(4), f32(4), 4))                     # another number of bits
    assert not plain(v=values._replace(bits=4)) and not plain(v=values._replace(data=u8(16)))
    assert not plain(k=keys._replace(mse_indices=u8(32)))                             # codes of a narrower quantiser
    assert not plain(k=keys._replace(residual_norms=f32().half())) and not plain(k=keys._replace(norms=f32().half()))
    assert not plain(k=keys._replace(residual_norms=torch.zeros(1, 1, 5)))            # (the general path lets it broadcast)
    assert not plain(k=keys._replace(qjl_signs=u8(16)[:, :1])) and not plain(v=values._replace(zeros=f32(4).half()))
    assert not plain(v=values._replace(scales=f32(1))) and not plain(v=values._replace(scales=f32(4).mT.contiguous().mT))
    assert not plain(k=None) and not plain(v=None)


def test_cache_entries_refuse_what_they_cannot_index_before_any_launch():
    """With TQ_EUNSUPPORTED, on which the cache object takes its general path: code sections off a word boundary, blocks of queries and
    buffers beyond the entries' limits.  (The addresses are never read.)"""
    lib = _ffi.lib()
    ly = _ffi.TqLayer()
    ly.d, ly.mse_bits = 128, 2
    ly.Pi = ly.PiT = ly.S = ly.ST = ly.centroids = ly.thresholds = 4096
    A = 4096

    def append(sections=(A,) * 7, n_buf=128):
        return lib.tq_cache_append(A, A, 128, 128, A, A, 0, n_buf * 128, 128, 0, n_buf * 128, 128, 8, 8, n_buf, C.byref(ly), 2, 32, 100,
                                   *sections, *(A,) * 7, A, A, A, None)

    def scores(idx=A, signs=A, n_q=1, n_buf=128):
        return lib.tq_cache_scores(A, 8, 8, n_q, idx, signs, A, A, 100, C.byref(ly), A, 0, n_buf * 128, 128, n_buf, 0.1, A, A, None)

    def attend(data=A, n_q=1, n_buf=128):
        return lib.tq_cache_attend(A, 8, 8, n_q, data, A, A, 100, 128, 32, 2, A, 0, n_buf * 128, 128, n_buf, A, A, None)

    for i in range(7):
        assert append(tuple(A + (j == i) for j in range(7))) == _ffi.TQ_EUNSUPPORTED
    assert append(n_buf=(1 << 20) + 1) == _ffi.TQ_EUNSUPPORTED
    assert scores(idx=A + 1) == scores(signs=A + 2) == scores(n_q=(1 << 18) + 1) == _ffi.TQ_EUNSUPPORTED
    assert attend(data=A + 1) == attend(n_q=65536) == _ffi.TQ_EUNSUPPORTED
    assert scores(n_buf=(1 << 24) + 1) == attend(n_buf=(1 << 24) + 1) == _ffi.TQ_EUNSUPPORTED


def _paper_pool(d, heads, key_bits=4, value_bits=4):
    """A pool without memory: what the split rules read of one."""
    from types import SimpleNamespace
    from turboquant_amd.paged import PagedKVPool
    pool = object.__new__(PagedKVPool)
    pool.head_dim, pool.num_kv_heads, pool.value_bits, pool.value_group_size = d, heads, value_bits, 32
    pool.dtype, pool.quantizer = torch.bfloat16, SimpleNamespace(bits=key_bits)
    pool.page_kernel = lambda: 2 if d > 256 else 1
    return pool


@pytest.mark.parametrize("d,heads,Hq,B", [(128, 8, 32, 16), (256, 2, 16, 4), (576, 1, 8, 3), (576, 1, 64, 1), (512, 2, 40, 5), (192, 1, 4, 7)])
def test_a_step_never_leaves_the_workspace_it_is_given(d, heads, Hq, B):
    """A split count of our own is cut to what the workspace holds, a caller's count that does not fit is refused."""
    pool = _paper_pool(d, heads)
    need = _ffi.lib().tq_decode_workspace_bytes
    for held in (1, 2, 7, 64):
        for spare in (0, 4, 400):
            ws = torch.empty(need(B, Hq, d, held) // 4 + spare // 4, dtype=torch.float32, device="meta")
            for n in (1, held, held + 1, 3 * held, 500):
                got = pool._splits_within(ws, B, Hq, n, True)
                assert 1 <= got <= n and need(B, Hq, d, got) <= 4 * ws.numel() and (got == n or need(B, Hq, d, got + 1) > 4 * ws.numel())
                if need(B, Hq, d, n) <= 4 * ws.numel():
                    assert pool._splits_within(ws, B, Hq, n, False) == n
                else:
                    with pytest.raises(ValueError, match="workspace"):
                        pool._splits_within(ws, B, Hq, n, False)
    small = torch.empty(need(B, Hq, d, 1) // 4 - 1, dtype=torch.float32, device="meta")
    with pytest.raises(ValueError, match="workspace"):
        pool._splits_within(small, B, Hq, 1, True)


def test_short_contexts_of_many_heads_are_split_by_turns():
    """The kernel of sixteen heads per wavefront: a workgroup per turn of its loop in short contexts, about four turns each in long ones,
    never more workgroups than compute units (unless sequences alone are more), no split without tokens."""
    pool = _paper_pool(576, 1)
    for G, side in ((9, 3), (16, 3), (17, 2), (33, 1), (64, 1), (65, 1), (128, 1)):
        groups = -(-G // 64)
        for B in (2, 3, 16, 300):
            most = max(1, 256 // (B * groups))
            for N in (1, 31, 200, 500, 2000, 8192, 32768, 131072):
                n, turns = pool.default_splits(B, N, G), -(-N // (32 * side))
                each = -(-turns // n)
                assert 1 <= n <= min(most, turns) and (n - 1) * each < turns <= n * each
                assert each == 1 or (turns > most or turns > 40 * side) and (each <= 4 or -(-turns // most) == each)


@pytest.mark.parametrize("d,turns", [(576, 24), (512, 8)])
def test_one_sequence_of_many_heads_takes_groups_of_eight_while_they_are_short(d, turns):
    """Workgroups of 8 heads that the card holds at once, none without tokens, up to a number of turns; longer contexts of more than sixteen
    heads take so many splits that the library runs the kernel of sixteen heads per wavefront pair."""
    pool = _paper_pool(d, 1)
    for G in (9, 16, 17, 24, 32, 33, 40, 48, 57, 64, 65, 72, 80, 100, 128):
        groups = -(-G // 8)
        for N in (1, 31, 33, 64, 300, 1000, 2000, 4000, 8192, 13000, 16384, 21800, 32768, 65536, 131072):
            n, blocks = pool.default_splits(1, N, G), -(-N // 32)
            if G <= 16 or -(-blocks * groups // 256) <= turns:
                assert 1 <= n <= min(blocks, 128) and n * groups <= 256
            else:
                assert n * groups > 256
    assert pool.default_splits(1, 500, 8) == 1


@pytest.mark.parametrize("d", [64, 128, 256, 320, 512, 576])
def test_a_split_count_without_query_heads_bounds_those_with_any(d):
    """So that a workspace sized before the query heads are known holds a step at full speed."""
    for heads in (1, 2, 8):
        pool = _paper_pool(d, heads)
        for B in (1, 2, 3, 17, 64, 300):
            for N in (1, 90, 500, 3000, 8192, 20000, 32768, 131072):
                most = pool.default_splits(B, N)
                assert all(pool.default_splits(B, N, heads * per) <= most for per in (*range(1, 20), 24, 32, 33, 48, 64, 65, 80, 128))


def test_splits_of_many_heads_in_the_static_area():
    """Steps of more than 8 heads on a wide KV head take the split count of their kernel there too, cut to what the area holds."""
    for d in (512, 576):
        pool = _paper_pool(d, 1)
        ly = _ffi.TqLayer()
        ly.d, ly.mse_bits = d, 3
        pool.quantizer._layer = lambda: ly
        need = lambda B, Hq, n: _ffi.lib().tq_decode_noalloc_bytes(B, Hq, 1, n, C.byref(ly))
        for Hq in (9, 16, 17, 64, 65, 128):
            for B in (1, 2, 3, 8, 64):
                for N in (1, 500, 8192, 131072):
                    n, free = pool.default_splits(B, N, Hq, True), pool.default_splits(B, N, Hq)
                    assert n == free or 1 <= n < free and need(B, Hq, n + 1) > _ffi.NOALLOC_SCRATCH_BYTES
                    assert n == 1 or need(B, Hq, n) <= _ffi.NOALLOC_SCRATCH_BYTES
        assert pool.default_splits(1, 65536, 128, True) >= 32 and pool.default_splits(1, 8192, 128, True) >= 16


class _Evicting:
    """A native host side that has another descriptor built before it reads the one of the call (as another thread may while the call has
    given up the interpreter's lock), and says whether that one and its matrices are still there."""

    def __init__(self, rebuild, built):
        self.rebuild, self.built, self.calls = rebuild, built, []

    def __getattr__(self, name):
        def call(*args):
            self.rebuild()
            gc.collect()
            self.calls.append(name)
            assert self.built[-1]() is not None, f"{name}: the descriptor was freed under the call"
            assert all(t() is not None for t in self.built[-1].terms), f"{name}: the matrices it points to were freed under the call"
            raise _Seen
        return call


class _Seen(Exception):
    pass


def test_a_descriptor_outlives_the_native_call_that_reads_it(monkeypatch):
    """Every call of the native host side, with the quantiser's kept descriptor replaced in the middle of it."""
    from turboquant_amd.kv_cache import TurboQuantKVCache
    from turboquant_amd.paged import PagedKVPool
    from turboquant_amd.quantizer import ProdQuantized
    monkeypatch.setattr(_ffi, "require_gpu", lambda t, name: t)
    tq = TurboQuantProd(128, bits=3, device="cpu")
    built, build = [], tq._layer

    class Ref(weakref.ref):
        terms = ()

    def layer():
        ly = build()
        ref = Ref(ly)
        ref.terms = [weakref.ref(t) for t in (*tq.mse_quantizer._splits[True][1][:4], *tq.mse_quantizer._splits[True][1][4])]
        built.append(ref)
        return ly
    tq._layer = layer

    def rebuild():
        tq.S.add_(0)                                           # (a buffer that is written)
        build()
    _ffi.lib()
    host = _Evicting(rebuild, built)
    monkeypatch.setattr(_ffi, "_host", host)
    pool = PagedKVPool.__new__(PagedKVPool)
    pool.quantizer, pool.head_dim, pool.num_kv_heads, pool.value_bits, pool.value_group_size = tq, 128, 2, 4, 32
    pool.dtype, pool.device, pool.num_pages = torch.bfloat16, torch.device("cpu"), 4
    pool.layout = _ffi.make_page_layout(128, 2, 4, 32, torch.bfloat16)
    pool.data = torch.zeros(4, 2, pool.layout.page_bytes, dtype=torch.uint8)
    cache = TurboQuantKVCache(128, buffer_size=3, device="cpu", dtype=torch.float32)
    cache.key_quantizer = tq
    rows = torch.zeros(1, 2, 3, 128)
    code = ProdQuantized(torch.zeros(1, 2, 5, 32, dtype=torch.uint8), torch.zeros(1, 2, 5, 16, dtype=torch.uint8), torch.zeros(1, 2, 5), torch.zeros(1, 2, 5), 2)
    cache.key_quantized, cache.key_buffer, cache.value_buffer = code, rows, rows
    cache.value_quantized = ValueQuantized(torch.zeros(1, 2, 5, 32, dtype=torch.uint8), torch.zeros(1, 2, 5, 4), torch.zeros(1, 2, 5, 4), 2)
    kv = torch.zeros(1, 1, 2, 128, dtype=torch.bfloat16)
    q = torch.zeros(1, 4, 128, dtype=torch.bfloat16)
    table, one = torch.zeros(1, 4, dtype=torch.int32), torch.ones(1, dtype=torch.int32)
    exact = torch.zeros(4, 16, 2, 128, dtype=torch.bfloat16)
    calls = [("quantize", lambda: tq.quantize(rows)), ("dequantize", lambda: tq.dequantize(code)), ("score", lambda: tq.attention_score(rows, code)),
             ("append", lambda: pool.append(kv, kv, table)), ("append", lambda: pool._append_newest(kv, kv, table, one)),
             ("decode", lambda: pool.decode_attention(q, table, one)),
             ("decode_ring", lambda: pool.decode_attention_ring(q, table, one, exact, exact, 16)),
             ("cache_append", lambda: cache.append(rows[..., :1, :], rows[..., :1, :])), ("cache_scores", lambda: cache.attention_scores(rows))]
    for name, call in calls:
        with pytest.raises(_Seen):
            call()
        assert host.calls[-1] == name


def test_the_stages_of_a_quantiser_keep_a_descriptor_each(monkeypatch):
    """The first stage used alone, in turn with the whole and in the middle of the other's build (where it waits for the card, another
    thread may run): each has its own matrices, and neither is built again."""
    monkeypatch.setattr(_ffi, "require_gpu", lambda t, name: t)
    for other_first in (False, True):
        tq = TurboQuantProd(128, bits=3, device="cpu")
        mse, norm, inside = tq.mse_quantizer, torch.Tensor.norm, []
        if other_first:
            mse._layer()
        with monkeypatch.context() as m:
            m.setattr(torch.Tensor, "norm", lambda t, *a, **k: (inside.append(mse._layer()), norm(t, *a, **k))[1])
            ly = tq._layer()
        alone = mse._layer()
        assert inside and all(x is alone for x in inside) and tq._layer() is ly and mse._layer() is alone
        assert alone.S is None and not alone.S_split and not alone.PiT_fp6
        pi, pit, s, st, fp6 = mse._splits[True][1]
        assert (ly.Pi_split, ly.PiT_split, ly.S_split, ly.ST_split, ly.PiT_fp6) == tuple(t.data_ptr() for t in (pi, pit, s, st, fp6[0]))
        assert ly.Pi == alone.Pi and ly.S_rownorm_max > 0


def test_a_quantiser_in_use_can_be_copied_and_pickled(monkeypatch):
    """Its descriptors hold addresses of its own tensors: a copy builds its own, also of a sketch matrix that was written since."""
    monkeypatch.setattr(_ffi, "require_gpu", lambda t, name: t)
    for d in (64, 128):
        tq = TurboQuantProd(d, bits=3, device="cpu")
        tq._layer(), tq.mse_quantizer._layer()
        tq.S.neg_()
        for other in (copy.deepcopy(tq), pickle.loads(pickle.dumps(tq))):
            ly = other._layer()
            assert ly.Pi == other.mse_quantizer.Pi.data_ptr() != tq.mse_quantizer.Pi.data_ptr()
            assert torch.equal(other._ST, other.S.T) and torch.equal(other.S, tq.S) and ly.ST == other._ST.data_ptr()
            assert set(other.state_dict()) == set(tq.state_dict())


@pytest.mark.parametrize("built_for,bound", [("this", True), ("Python 3.10, torch 2.9.0 abc, library 2, interface 1", False), (None, False)])
def test_a_native_host_side_built_for_something_else_is_left_alone(monkeypatch, built_for, bound):
    """One for another torch or Python, or from before it said what it is for (whose calls may take other arguments): never called."""
    calls = []

    class Module(types.ModuleType):
        def bind(self, addresses):
            calls.append(addresses)
            if not bound:
                raise KeyError("a call that this library lacks")
    module = Module("_tq_host")
    if built_for is not None:
        module.built_for = _ffi.host_stamp() if built_for == "this" else built_for
    library = _ffi.lib()
    monkeypatch.setitem(sys.modules, "turboquant_amd._tq_host", module)
    monkeypatch.setattr(turboquant_amd, "_tq_host", module, raising=False)
    monkeypatch.setattr(_ffi, "_host", None)
    _ffi._bind_host(library)
    assert (_ffi._host is module) == bound and len(calls) == bound
    if bound:
        assert set(calls[0]) == set(_ffi._HOST_CALLS) and all(calls[0].values())


def test_the_native_host_side_is_for_this_torch():
    from turboquant_amd.build import HOST
    if not os.path.exists(HOST):
        pytest.skip("not built here")
    _ffi.lib()
    assert _ffi._host is not None and _ffi._host.built_for == _ffi.host_stamp()


@pytest.mark.parametrize("fails", [None, "host", "headers", "hipcc", "link"])
def test_a_library_is_built_with_the_native_host_side_or_without(monkeypatch, tmp_path, capsys, fails):
    """What the module alone needs (a host compiler, torch's headers) may be missing: the library stands, and a module of before is gone.
    Where the library does not build, the module of before stays beside it."""
    from turboquant_amd import build
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "LIB", str(tmp_path / "libtq_hip.so"))
    monkeypatch.setattr(build, "HOST", str(tmp_path / "_tq_host.so"))
    (tmp_path / "_tq_host.so").write_text("before")

    def run(cmd, **_):
        out = cmd[cmd.index("-o") + 1]
        kind = "host" if out.endswith("_tq_host.so") else "link" if out.endswith("libtq_hip.so") else "hipcc"
        if kind == "host" and fails == "host":
            raise FileNotFoundError("g++")
        if kind != fails:
            open(out, "w").write("now")
        return types.SimpleNamespace(returncode=int(kind == fails), stderr="")
    monkeypatch.setattr(build.subprocess, "run", run)
    if fails == "headers":
        monkeypatch.setitem(sys.modules, "torch.utils.cpp_extension", None)
    if fails in ("hipcc", "link"):
        with pytest.raises(RuntimeError, match="hipcc"):
            build.build_library()
        assert (tmp_path / "_tq_host.so").read_text() == "before"
        return
    assert build.build_library() == str(tmp_path / "libtq_hip.so") and (tmp_path / "libtq_hip.so").read_text() == "now"
    assert os.path.exists(build.HOST) == (fails is None) == ("not built" not in capsys.readouterr().err)
    assert fails or (tmp_path / "_tq_host.so").read_text() == "now"


@pytest.mark.parametrize("how", ["as it is", "subclass", "object", "class", "stand-in"])
def test_a_method_in_the_place_of_one_that_native_calls_go_past_sees_every_call(monkeypatch, how):
    """Writes and decode steps of the engine's hooks and of a store, which reach the native host side without the pool's `append`,
    `decode_attention` and `workspace` where those are the package's own."""
    from turboquant_amd import score, store as S
    from turboquant_amd.integration import batched
    from turboquant_amd.paged import PagedKVPool
    seen, native = [], []

    class Host:
        def append(self, *a):
            native.append("append")
            return True

        def decode(self, *a):
            native.append("decode_attention")
            return torch.zeros(1)

        def decode_ring(self, *a):
            native.append("decode_attention_ring")
            return torch.zeros(1)

    def spy(name, result=None):
        return lambda *a, **k: (seen.append(name), result)[1]

    class Own(PagedKVPool):
        append, decode_attention, workspace = spy("append"), spy("decode_attention", torch.zeros(1)), spy("workspace")

    class StandIn:
        __slots__ = ("dtype", "num_pages", "device")
        append, decode_attention, default_splits = spy("append"), spy("decode_attention", torch.zeros(1)), lambda *a: 1
    monkeypatch.setattr(_ffi, "require_gpu", lambda t, name: t)
    _ffi.lib()
    monkeypatch.setattr(_ffi, "_host", Host())
    tq = TurboQuantProd(128, bits=3, device="cpu")
    monkeypatch.setattr(TurboQuantProd, "_layer", lambda self: None)
    pool = {"subclass": Own, "stand-in": StandIn}.get(how, PagedKVPool)
    pool = pool.__new__(pool)
    pool.dtype, pool.device, pool.num_pages = torch.bfloat16, torch.device("cpu"), 64
    if how != "stand-in":
        pool.quantizer, pool.head_dim, pool.num_kv_heads, pool.data, pool.layout = tq, 128, 2, torch.zeros(1), None
        pool.value_bits, pool.value_group_size = 4, 32
    if how in ("object", "class"):
        for name in ("append", "decode_attention"):
            monkeypatch.setattr(pool if how == "object" else PagedKVPool, name, spy(name, torch.zeros(1)))
    meta = types.SimpleNamespace(num_actual_tokens=3, max_query_len=1, block_table=torch.zeros(3, 2, dtype=torch.int32), seq_lens=torch.ones(3, dtype=torch.int32))
    config = types.SimpleNamespace(num_kv_heads=2, head_dim=128)
    kv = torch.zeros(3, 2, 128, dtype=torch.bfloat16)
    batched.BatchedLayerState(config=config, quantizer=tq, pool=pool).write(kv, kv, meta)
    store = S.CompressedKVStore(128, 2, value_bits=4, device="cpu")
    store._pool, store._block_table, store._counts = pool, torch.arange(64, dtype=torch.int32)[None], torch.arange(1025, dtype=torch.int32)
    store._chunk_lengths, store._table_pages = [100], 64
    query = torch.zeros(1, 4, 128, dtype=torch.bfloat16)
    score.compute_hybrid_attention(query, store, None, None, 4)
    assert (seen, native) == (([], ["append", "decode_attention"]) if how == "as it is" else (["append", "decode_attention"], []))
    # a store whose lengths or pages come from elsewhere takes its step through them
    for cls in (type("Lengths", (S.CompressedKVStore,), {"lengths": lambda self, n, rows: seen.append("lengths")}),
                type("Pages", (S.CompressedKVStore,), {"ensure_pool": lambda self, dtype, n=0: (seen.append("ensure_pool"), pool)[1]})):
        store.__class__, before = cls, len(seen)
        score.compute_hybrid_attention(query, store, None, None, 4)
        assert len(seen) > before and seen[before] in ("lengths", "ensure_pool")


def test_a_workspace_of_its_own_is_taken_by_every_decode_step(monkeypatch):
    from turboquant_amd.paged import PagedKVPool

    class Asked(Exception):
        pass

    class Pool(PagedKVPool):
        def workspace(self, B, Hq, n_split):
            raise Asked
    monkeypatch.setattr(_ffi, "require_gpu", lambda t, name: t)
    _ffi.lib()
    monkeypatch.setattr(_ffi, "_host", types.SimpleNamespace(decode=lambda *a: torch.zeros(1), decode_ring=lambda *a: torch.zeros(1)))
    pool = Pool.__new__(Pool)
    pool.quantizer, pool.head_dim, pool.num_kv_heads = TurboQuantProd(128, bits=3, device="cpu"), 128, 2
    pool.value_bits, pool.value_group_size = 4, 32
    pool.dtype, pool.device, pool.num_pages, pool.data, pool.layout = torch.bfloat16, torch.device("cpu"), 4, torch.zeros(1), None
    monkeypatch.setattr(TurboQuantProd, "_layer", lambda self: None)
    q, table, one = torch.zeros(1, 4, 128, dtype=torch.bfloat16), torch.zeros(1, 4, dtype=torch.int32), torch.ones(1, dtype=torch.int32)
    exact = torch.zeros(4, 16, 2, 128, dtype=torch.bfloat16)
    for step in (lambda: pool.decode_attention(q, table, one), lambda: pool.decode_attention_ring(q, table, one, exact, exact, 16)):
        with pytest.raises(Asked):
            step()


@pytest.mark.parametrize("d,mse_bits", [(64, 1), (128, 2), (128, 3), (256, 4)])
def test_the_workspace_of_a_cache_token_holds_the_keys_codes_and_no_more(d, mse_bits):
    """Four sections (indices, signs, norms, residual norms), each begun on a 16-byte boundary, from any address: a value's codes are not among
    them."""
    for batch in (1, 3, 17, 4096):
        sections = [batch * d * (1, 1, 2, 4, 4)[mse_bits] // 8, batch * d // 8, batch * 4, batch * 4]
        at = 15
        for n in sections:
            at += (n + 15) // 16 * 16
        for value_bits, group_size in ((2, 16), (4, 32), (8, 64)):
            have = _ffi.lib().tq_cache_append_bytes(batch, d, mse_bits, value_bits, group_size)
            assert at <= have <= sum(sections) + 5 * 16
    assert _ffi.lib().tq_cache_append_bytes(1, 128, 5, 2, 32) == 0 == _ffi.lib().tq_cache_append_bytes(0, 128, 2, 2, 32)


@pytest.mark.parametrize("query", [torch.zeros(1, 4, 128), torch.zeros(1, 4, 128, dtype=torch.bfloat16), torch.zeros(2, 4, 128, dtype=torch.bfloat16),
                                   torch.zeros(1, 4, 64, dtype=torch.bfloat16)])
def test_a_step_that_the_native_host_side_leaves_is_looked_at_once_and_checked(monkeypatch, query):
    """A query on the CPU (or of another head size) raises before the library is called, and one token is offered to the native host side
    once where nothing about it changes on the way."""
    from turboquant_amd import score, store as S
    from turboquant_amd.paged import PagedKVPool
    offered = []
    library = _ffi.lib()

    class Library:
        def __getattr__(self, name):
            assert "attn" not in name, f"{name} was called"
            return getattr(library, name)
    monkeypatch.setattr(_ffi, "lib", lambda: Library())
    monkeypatch.setattr(_ffi, "_host", types.SimpleNamespace(decode=lambda *a: offered.append(a)))
    monkeypatch.setattr(TurboQuantProd, "_layer", lambda self: None)
    pool = PagedKVPool.__new__(PagedKVPool)
    pool.quantizer, pool.head_dim, pool.num_kv_heads, pool.data, pool.layout = TurboQuantProd(128, bits=3, device="cpu"), 128, 2, torch.zeros(1), None
    pool.dtype, pool.device, pool.num_pages, pool.value_bits, pool.value_group_size = torch.bfloat16, torch.device("cpu"), 64, 4, 32
    store = S.CompressedKVStore(128, 2, value_bits=4, device="cpu")
    store._pool, store._block_table, store._counts = pool, torch.arange(64, dtype=torch.int32)[None], torch.arange(1025, dtype=torch.int32)
    store._chunk_lengths, store._table_pages = [100], 64
    with pytest.raises((RuntimeError, ValueError), match="lives on cpu|Incompatible"):
        score.compute_hybrid_attention(query, store, None, None, 4)
    assert len(offered) <= 1
