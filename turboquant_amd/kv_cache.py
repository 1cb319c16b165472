"""Value group quantiser and the stand-alone TurboQuant KV cache object.

Mirrors turboquant/kv_cache.py of the reference: `ValueQuantized`,
`unpack_values`, `quantize_values`, `dequantize_values` (kv_cache.py:20-116) and
`TurboQuantKVCache` (kv_cache.py:119-349) with the same arguments, layouts and
dtypes; the arithmetic runs in libtq_hip.so.
"""

from __future__ import annotations

import ctypes as C
import math
from typing import NamedTuple, Optional

import torch

from . import _ffi
from .quantizer import ProdQuantized, TurboQuantProd, _packing


class ValueQuantized(NamedTuple):
    """Bit-packed group-quantised values."""
    data: torch.Tensor       # (..., n_tokens, d*bits/8) uint8
    scales: torch.Tensor     # (..., n_tokens, n_groups) input dtype
    zeros: torch.Tensor      # (..., n_tokens, n_groups) input dtype
    bits: int = 2


def unpack_values(vq: ValueQuantized) -> torch.Tensor:
    """One uint8 code per element (layout helper; kernels read the packed form)."""
    bits = vq.bits if len(vq) > 3 else 2
    packed = vq.data
    if bits not in (2, 4):
        return packed
    per_byte = 8 // bits
    fields = [(packed >> (bits * s)) & ((1 << bits) - 1) for s in range(per_byte)]
    return torch.stack(fields, dim=-1).reshape(*packed.shape[:-1], packed.shape[-1] * per_byte)


def quantize_values(v: torch.Tensor, bits: int = 2, group_size: int = 32) -> ValueQuantized:
    """Asymmetric per-group min/max quantisation of (..., seq_len, d) values to
    2, 4 or 8 bits, computed with the rounding of v's dtype."""
    _ffi.require_gpu(v, "v")
    d = v.shape[-1]
    assert d % group_size == 0, f"head_dim {d} must be divisible by group_size {group_size}"
    rows = v.reshape(-1, d)
    if rows.stride(-1) != 1 or (rows.shape[0] > 1 and rows.stride(0) < d):
        rows = rows.contiguous()
    n = rows.shape[0]
    stride = rows.stride(0) if n > 1 else d
    n_groups = d // group_size
    data = torch.empty(n, d * bits // 8, dtype=torch.uint8, device=v.device)
    scales = torch.empty(n, n_groups, dtype=v.dtype, device=v.device)
    zeros = torch.empty(n, n_groups, dtype=v.dtype, device=v.device)
    with torch.cuda.device(v.device):
        _ffi.check(_ffi.lib().tq_quantize_values(
            rows.data_ptr(), _ffi.dtype_tag(v.dtype), n, stride, d, group_size, bits, data.data_ptr(),
            scales.data_ptr(), zeros.data_ptr(), _ffi.stream_ptr(v.device)), "tq_quantize_values")
    lead = v.shape[:-1]
    return ValueQuantized(data=data.reshape(*lead, -1), scales=scales.reshape(*lead, n_groups),
                          zeros=zeros.reshape(*lead, n_groups), bits=bits)


def dequantize_values(vq: ValueQuantized, group_size: int = 32) -> torch.Tensor:
    """fp32 code * scale + zero, (..., seq_len, d)."""
    bits = vq.bits if len(vq) > 3 else 2
    data = _ffi.require_gpu(vq.data, "data").contiguous()
    scales, zeros = vq.scales.contiguous(), vq.zeros.contiguous()
    d = data.shape[-1] * 8 // bits
    n = data.numel() // data.shape[-1]
    out = torch.empty(*data.shape[:-1], d, dtype=torch.float32, device=data.device)
    with torch.cuda.device(data.device):
        _ffi.check(_ffi.lib().tq_dequant_values(
            data.data_ptr(), scales.data_ptr(), zeros.data_ptr(), _ffi.dtype_tag(scales.dtype), n, d, group_size, bits,
            out.data_ptr(), _ffi.stream_ptr(data.device)), "tq_dequant_values")
    return out


def _plain(*tensors) -> bool:
    """Ordinary fp32 tensors of four dimensions with contiguous channels, on which torch would run an operation as it stands."""
    if not _ffi.ordinary(*tensors):
        return False
    for t in tensors:
        if t.dtype is not torch.float32 or t.dim() != 4 or t.stride(3) != 1:
            return False
    return True


def _plain_product(*tensors) -> bool:
    """... and a product of them in fp32 (under autocast it is one of 16-bit numbers)."""
    return _plain(*tensors) and not torch.is_autocast_enabled("cuda")


class TurboQuantKVCache:
    """Self-contained cache: the newest `buffer_size` tokens stay exact, older
    ones are TurboQuant keys + group-quantised values.  Tensors are
    (batch, heads, seq, head_dim)."""

    def __init__(self, head_dim: int, key_bits: int = 3, value_bits: int = 2, value_group_size: int = 32,
                 buffer_size: int = 128, device=None, dtype: torch.dtype = torch.float16, layer_idx: int = 0):
        self.head_dim = head_dim
        self.key_bits = key_bits
        self.value_bits = value_bits
        self.value_group_size = value_group_size
        self.buffer_size = buffer_size
        self.device = device or torch.device("cuda")
        self.dtype = dtype
        self.layer_idx = layer_idx
        self.key_quantizer = TurboQuantProd(dim=head_dim, bits=key_bits, device=self.device, seed=42 + layer_idx * 7)
        self.seq_len = 0
        self.key_quantized: Optional[ProdQuantized] = None
        self.value_quantized: Optional[ValueQuantized] = None
        self.key_buffer: Optional[torch.Tensor] = None
        self.value_buffer: Optional[torch.Tensor] = None

    def _compress(self, keys: torch.Tensor, values: torch.Tensor):
        kq = self.key_quantizer.quantize(keys)
        vq = quantize_values(values, bits=self.value_bits, group_size=self.value_group_size)
        if self.key_quantized is None:
            self.key_quantized, self.value_quantized = kq, vq
            return
        old_k, old_v = self.key_quantized, self.value_quantized
        self.key_quantized = ProdQuantized(
            mse_indices=torch.cat([old_k.mse_indices, kq.mse_indices], dim=-2),
            qjl_signs=torch.cat([old_k.qjl_signs, kq.qjl_signs], dim=-2),
            residual_norms=torch.cat([old_k.residual_norms, kq.residual_norms], dim=-1),
            norms=torch.cat([old_k.norms, kq.norms], dim=-1),
            mse_bits=kq.mse_bits)
        self.value_quantized = ValueQuantized(
            data=torch.cat([old_v.data, vq.data], dim=-2),
            scales=torch.cat([old_v.scales, vq.scales], dim=-2),
            zeros=torch.cat([old_v.zeros, vq.zeros], dim=-2),
            bits=self.value_bits)

    def prefill(self, keys: torch.Tensor, values: torch.Tensor):
        """All but the newest buffer_size tokens are compressed at once."""
        total = keys.shape[-2]
        self.seq_len = total
        if total <= self.buffer_size:
            self.key_buffer, self.value_buffer = keys, values
            return
        cut = total - self.buffer_size
        self.key_buffer, self.value_buffer = keys[..., cut:, :], values[..., cut:, :]
        self.key_quantized = self.value_quantized = None
        self._compress(keys[..., :cut, :], values[..., :cut, :])

    # ---- a decode token in fp32 (the general paths below take everything else) -----------------------------------------
    # A step of the general paths is some thirty small launches and seven concatenations of the whole history: 270 us, nearly all of it
    # host time, at 4096 tokens of 8 heads of 128.  The entries below are one launch for the token (two at head_dim 64, beyond 48 MB of copies
    # and for rows off a 16-byte boundary), two for the scores and two for the values: with the softmax between them 38 us of the card, 53 of the
    # host through its native side and 101 through the Python methods.  What an entry does not take (sections that are not word-aligned,
    # buffers or blocks of queries beyond its indexes) it refuses before it launches anything, and the general path goes on.
    def _compressed_plain(self) -> bool:
        """Whether the compressed part is what this cache writes itself in fp32.  One put in its place may have other bits, 16-bit norms
        or pieces that broadcast: the entries would read those wrongly, or read past them."""
        kq, vq = self.key_quantized, self.value_quantized
        d, bits, gs = self.head_dim, self.value_bits, self.value_group_size
        if kq is None or vq is None or vq.bits != bits or d not in (64, 128, 256) or gs % 16 or kq.norms.dim() != 3:
            return False
        idx, signs, rnorms, norms = kq[:4]
        data, scales, zeros = vq[:3]
        n, groups, byte, f32, Tensor = norms.numel(), d // gs, torch.uint8, torch.float32, torch.Tensor
        for t, dtype, count in ((idx, byte, d * _packing(self.key_bits - 1)[0] // 8), (signs, byte, d // 8), (rnorms, f32, 1), (norms, f32, 1),
                                (data, byte, d * bits // 8), (scales, f32, groups), (zeros, f32, groups)):
            if type(t) is not Tensor or t.dtype is not dtype or t.numel() != n * count or not t.is_contiguous():
                return False
        return True

    def _sections(self) -> Optional[tuple]:
        """The seven tensors of the compressed part, for the native host side, which looks at each; None: not for it."""
        kq, vq = self.key_quantized, self.value_quantized
        if (_ffi.native() is None or kq is None or vq is None or vq.bits != self.value_bits or self.head_dim not in (64, 128, 256)
                or self.value_group_size % 16 or kq.norms.dim() != 3 or kq.norms.dtype is not torch.float32):
            return None
        return (*kq[:4], *vq[:3])

    def _append_spill(self, key: torch.Tensor, value: torch.Tensor) -> bool:
        """One token into a full buffer whose first row leaves for the compressed part, in one library call; False: the case is
        not that one, nothing was done."""
        kb, vb = self.key_buffer, self.value_buffer
        if kb is None or vb is None:
            return False
        part = self._sections()
        if part is not None and kb.shape[-2] == self.buffer_size:
            q = self.key_quantizer
            new = _ffi.native().cache_append(*part, key, value, kb, vb, q._layer(), self.head_dim, self.key_bits - 1,
                                             self.value_bits, self.value_group_size)
            if new is not None:
                self.key_quantized = ProdQuantized(*new[:4], self.key_quantized.mse_bits)
                self.value_quantized = ValueQuantized(*new[4:7], bits=self.value_bits)
                self.key_buffer, self.value_buffer = new[7:]
                return True
        if not self._compressed_plain() or not _plain(key, value, kb, vb):
            return False
        B, H, n_buf, d = kb.shape
        kq, vq = self.key_quantized, self.value_quantized
        n_c = kq.norms.shape[-1]
        if (n_buf != self.buffer_size or n_buf < 1 or d != self.head_dim or vb.shape != kb.shape or key.shape != (B, H, 1, d)
                or value.shape != key.shape or tuple(kq.norms.shape) != (B, H, n_c) or tuple(vq.scales.shape[:3]) != (B, H, n_c)
                or B * H > 65535 or n_c >= 1 << 20 or kq.norms.device != kb.device):
            return False
        if any(t.stride(2) != d or t.stride(1) < d or (B > 1 and t.stride(0) != H * t.stride(1)) for t in (kb, vb)):
            return False
        if B > 1 and any(t.stride(0) != H * t.stride(1) for t in (key, value)) or any(t.stride(1) < d for t in (key, value)):
            return False
        lib, dev, ly = _ffi.lib(), kb.device, self.key_quantizer._layer()
        grown = [torch.empty(B, H, n_c + 1, *t.shape[3:], dtype=t.dtype, device=dev) for t in (*kq[:4], *vq[:3])]
        nk, nv = torch.empty(B, H, n_buf, d, dtype=torch.float32, device=dev), torch.empty(B, H, n_buf, d, dtype=torch.float32, device=dev)
        work = torch.empty(lib.tq_cache_append_bytes(B * H, d, self.key_bits - 1, self.value_bits, self.value_group_size),
                           dtype=torch.uint8, device=dev)
        idx, signs, rnorms, norms = grown[:4]
        with _ffi.on_device(dev):
            rc = lib.tq_cache_append(
                key.data_ptr(), value.data_ptr(), key.stride(1), value.stride(1), kb.data_ptr(), vb.data_ptr(), *kb.stride()[:3],
                *vb.stride()[:3], B * H, H, n_buf, C.byref(ly), self.value_bits, self.value_group_size, n_c,
                kq.mse_indices.data_ptr(), kq.qjl_signs.data_ptr(), kq.norms.data_ptr(), kq.residual_norms.data_ptr(),
                vq.data.data_ptr(), vq.scales.data_ptr(), vq.zeros.data_ptr(), idx.data_ptr(), signs.data_ptr(),
                norms.data_ptr(), rnorms.data_ptr(), *[t.data_ptr() for t in grown[4:]], nk.data_ptr(), nv.data_ptr(),
                work.data_ptr(), _ffi.stream_ptr(dev))
        if rc == _ffi.TQ_EUNSUPPORTED:
            return False
        _ffi.check(rc, "tq_cache_append")
        self.key_quantized = ProdQuantized(idx, signs, rnorms, norms, kq.mse_bits)
        self.value_quantized = ValueQuantized(*grown[4:], bits=self.value_bits)
        self.key_buffer, self.value_buffer = nk, nv
        return True

    # The entries are made for the few queries of a decode step; a block of queries is two matrix products in the general paths.
    # us of a call, entry / general, buffers of 128 rows:
    #   scores: a wavefront per exact row and query, which pays while the host time of the general path or its passes over the scores of
    #   the compressed keys cost more. 8 heads of 128, 100 keys: 256 queries 35 / 63, 1024 202 / 61; 32 heads of 4096 keys: 32 queries 66 / 73,
    #   128 206 / 199; 32 heads of 64, 1000 keys: 64 queries 43 / 68, 128 83 / 68; 2 heads of 256, 4096 keys: 256 queries 63 / 96,
    #   1024 211 / 177; 8 heads of 128, 32768 keys: 128 queries 266 / 377, 2048 3953 / 5512.
    @staticmethod
    def _few_score_queries(rows: int, n_c: int, n_buf: int, d: int) -> bool:
        return rows * (n_buf * max(48, d // 2) - n_c) <= 1 << 24

    #   values: every query unpacks the history again and writes a partial per 128 tokens (within the limit 21 MB of them). 8 heads of 128, 4096 tokens:
    #   48 queries 45 / 61, 128 99 / 61, 2048 1365 / 155; 32 heads: 16 queries 58 / 62, 24 84 / 62; 8 heads, 32768 tokens: 12 queries 80 / 96,
    #   24 141 / 130; 8 heads of 64, 4096 tokens: 64 queries 42 / 64, 128 74 / 64; of 128, 100 tokens: 256 queries 31 / 64, 1024 96 / 60.
    @staticmethod
    def _few_value_queries(rows: int, n_c: int, n_buf: int, d: int) -> bool:
        return rows * (d + 32) * (n_c + 4 * n_buf) * 32768 <= (5 << 26) * (32768 + n_c)

    def append(self, key: torch.Tensor, value: torch.Tensor):
        """One decode token (batch, heads, 1, head_dim); the oldest buffered
        tokens spill into the compressed part once the buffer overflows."""
        if not self._append_spill(key, value):
            self._append(key, value)
        self.seq_len += 1

    def _append(self, key: torch.Tensor, value: torch.Tensor):
        if self.key_buffer is None:
            self.key_buffer, self.value_buffer = key, value
        else:
            self.key_buffer = torch.cat([self.key_buffer, key], dim=-2)
            self.value_buffer = torch.cat([self.value_buffer, value], dim=-2)
        extra = self.key_buffer.shape[-2] - self.buffer_size
        if extra > 0:
            spill_k, spill_v = self.key_buffer[..., :extra, :], self.value_buffer[..., :extra, :]
            self.key_buffer, self.value_buffer = self.key_buffer[..., extra:, :], self.value_buffer[..., extra:, :]
            self._compress(spill_k, spill_v)

    def attention_scores(self, query: torch.Tensor, scale: float = None) -> torch.Tensor:
        """scale * <q, k> over [compressed ; buffer]: (batch, heads, n_q, seq_len)."""
        if scale is None:
            scale = 1.0 / math.sqrt(self.head_dim)
        kb = self.key_buffer
        part = self._sections() if kb is not None and isinstance(scale, (int, float)) else None
        if part is not None and query.dim() == 4 and kb.dim() == 4:
            B, H, n_buf, d = kb.shape
            if self._few_score_queries(B * H * query.shape[2], part[3].shape[-1], n_buf, d):
                scores = _ffi.native().cache_scores(*part, query, kb, self.key_quantizer._layer(), self.head_dim, self.key_bits - 1,
                                                    self.value_bits, self.value_group_size, scale)
                if scores is not None:
                    return scores
        if kb is not None and isinstance(scale, (int, float)) and self._compressed_plain() and _plain_product(query, kb):
            kq = self.key_quantized
            B, H, n_buf, d = kb.shape
            n_c, n_q = kq.norms.shape[-1], query.shape[2]
            if (query.shape == (B, H, n_q, self.head_dim) and d == self.head_dim and tuple(kq.norms.shape) == (B, H, n_c)
                    and n_c and n_buf and n_q and B * H <= 65535 and kq.norms.device == kb.device
                    and self._few_score_queries(B * H * n_q, n_c, n_buf, d)):
                q, ly, dev = query.contiguous(), self.key_quantizer._layer(), kb.device
                scores = torch.empty(B, H, n_q, n_c + n_buf, dtype=torch.float32, device=dev)
                work = torch.empty(2 * B * H * n_q * d, dtype=torch.float32, device=dev)
                with _ffi.on_device(dev):
                    rc = _ffi.lib().tq_cache_scores(
                        q.data_ptr(), B * H, H, n_q, kq.mse_indices.data_ptr(), kq.qjl_signs.data_ptr(), kq.norms.data_ptr(),
                        kq.residual_norms.data_ptr(), n_c, C.byref(ly), kb.data_ptr(), *kb.stride()[:3], n_buf, float(scale),
                        scores.data_ptr(), work.data_ptr(), _ffi.stream_ptr(dev))
                if rc != _ffi.TQ_EUNSUPPORTED:
                    _ffi.check(rc, "tq_cache_scores")
                    return scores
        pieces = []
        if self.key_quantized is not None:
            pieces.append(self.key_quantizer.attention_score(query, self.key_quantized) * scale)
        if self.key_buffer is not None:
            kt = self.key_buffer.transpose(-2, -1)
            if kt.dtype == torch.bfloat16 or torch.is_autocast_enabled("cuda"):
                kt = kt.contiguous()         # (batched bf16 products with a transposed right operand have faulted in the library)
            pieces.append(torch.matmul(query, kt) * scale)
        return torch.cat(pieces, dim=-1)

    def attend(self, attn_weights: torch.Tensor) -> torch.Tensor:
        """softmaxed weights (batch, heads, n_q, seq_len) -> (batch, heads, n_q, head_dim)."""
        vb = self.value_buffer
        part = self._sections() if vb is not None else None
        if part is not None and attn_weights.dim() == 4 and vb.dim() == 4:
            B, H, n_buf, d = vb.shape
            if self._few_value_queries(B * H * attn_weights.shape[2], part[3].shape[-1], n_buf, d):
                out = _ffi.native().cache_attend(*part, attn_weights, vb, self.head_dim, self.key_bits - 1, self.value_bits,
                                                 self.value_group_size)
                if out is not None:
                    return out
        if vb is not None and self._compressed_plain() and _plain_product(attn_weights, vb):
            vq = self.value_quantized
            B, H, n_buf, d = vb.shape
            n_c, n_q = vq.data.shape[-2], attn_weights.shape[2]
            if (attn_weights.shape == (B, H, n_q, n_c + n_buf) and d == self.head_dim and tuple(vq.scales.shape[:3]) == (B, H, n_c)
                    and n_c and n_buf and 0 < n_q <= 65535 and B * H <= 65535 and vq.scales.device == vb.device
                    and self._few_value_queries(B * H * n_q, n_c, n_buf, d)):
                w, dev, lib = attn_weights.contiguous(), vb.device, _ffi.lib()
                out = torch.empty(B, H, n_q, d, dtype=torch.float32, device=dev)
                work = torch.empty(lib.tq_cache_attend_bytes(B * H, n_q, d, n_c, n_buf) // 4, dtype=torch.float32, device=dev)
                with _ffi.on_device(dev):
                    rc = lib.tq_cache_attend(
                        w.data_ptr(), B * H, H, n_q, vq.data.data_ptr(), vq.scales.data_ptr(), vq.zeros.data_ptr(), n_c, d,
                        self.value_group_size, self.value_bits, vb.data_ptr(), *vb.stride()[:3], n_buf, out.data_ptr(),
                        work.data_ptr(), _ffi.stream_ptr(dev))
                if rc != _ffi.TQ_EUNSUPPORTED:
                    _ffi.check(rc, "tq_cache_attend")
                    return out
        result = None
        col = 0
        if self.value_quantized is not None:
            n_c = self.value_quantized.data.shape[-2]
            dense = dequantize_values(self.value_quantized, self.value_group_size)
            result = torch.matmul(attn_weights[..., col:col + n_c], dense)
            col += n_c
        if self.value_buffer is not None:
            n_b = self.value_buffer.shape[-2]
            part = torch.matmul(attn_weights[..., col:col + n_b], self.value_buffer)
            result = part if result is None else result + part
        return result

    def memory_bytes(self) -> dict:
        """Bytes held, counting norms / scales / zeros at 2 bytes each."""
        info = {"quantized_keys": 0, "quantized_values": 0, "buffer": 0, "total": 0}
        if self.key_quantized is not None:
            kq = self.key_quantized
            info["quantized_keys"] = (kq.mse_indices.nelement() + kq.qjl_signs.nelement()
                                      + 2 * kq.residual_norms.nelement() + 2 * kq.norms.nelement())
        if self.value_quantized is not None:
            vq = self.value_quantized
            info["quantized_values"] = vq.data.nelement() + 2 * vq.scales.nelement() + 2 * vq.zeros.nelement()
        for buf in (self.key_buffer, self.value_buffer):
            if buf is not None:
                info["buffer"] += 2 * buf.nelement()
        info["total"] = info["quantized_keys"] + info["quantized_values"] + info["buffer"]
        return info

    def get_seq_length(self) -> int:
        return self.seq_len
