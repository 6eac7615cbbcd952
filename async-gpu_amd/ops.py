"""nn::ops over torch device tensors (reference: crates/core/gpu-host/src/nn/ops/*.rs).

Each function checks shapes like its reference twin, allocates the output with torch (torch is
only the allocator) and launches the HIP kernel through the C ABI on torch's current stream; for
the operators that a decode step is made of, csrc/torch_ops.cpp does these steps.
Errors surface as AgpuError with the reference's NnError meaning.
"""
import torch

from . import _lib
from ._lib import AgpuError

_ctx_cache = {}


class _Native:
    """csrc/torch_ops.cpp, loaded with the first operator that is called (importing this module needs no built library)."""

    def __getattr__(self, name):
        global _native
        _native = _lib.torch_ops(context)
        return getattr(_native, name)


_native = _Native()


def context(device=0):
    """One Context per (device, torch current stream)."""
    if not torch.cuda.is_available():
        raise AgpuError(_lib.ERR_UNSUPPORTED, "no GPU visible: the HIP path cannot run (there is no CPU fallback)")
    stream = torch.cuda.current_stream(device).cuda_stream
    key = (device, stream)
    if key not in _ctx_cache:
        _ctx_cache[key] = _lib.Context(device, stream)
    return _ctx_cache[key]


def _shape_err(expected, actual):
    raise AgpuError(_lib.ERR_SHAPE_MISMATCH, f"shape mismatch: expected {expected}, got {actual}")


def _f32(t):
    assert t.dtype == torch.float32 and t.is_cuda and t.is_contiguous(), "expects contiguous fp32 device tensors"
    return t


def int4_linear(x, packed, scales, bias=None, residual=None, group=32, flags=0, ln=None, out=None):
    """Int4Linear::forward (nn/layers/int4_linear.rs:71-133): x [*, K] -> [*, N].
    ln = (gamma, beta, eps) applies LayerNorm to the rows first."""
    return _native.int4_linear(x, packed, scales, bias, residual, group, flags, ln, out)


def int4_linear_pieces(x, packed, scales, bias=None, residual=None, group=32, flags=0, ln=None, out_gamma=None, want_pieces=False):
    """The batched decode Linear of the model driver (5 .. 16 rows) on bf16 pieces of x, as agpu_int4_linear_pieces
    describes it.  Returns y, or (y, pieces [N/32, 3, 64, 8] int16 bit patterns, stats [N/32, 16, 2]) with want_pieces."""
    M, K = x.shape
    N = packed.shape[1]
    y = torch.empty((M, N), dtype=torch.float32, device=x.device)
    pieces = stats = None
    if want_pieces:
        pieces = torch.zeros((N // 32, 3, 64, 8), dtype=torch.int16, device=x.device)
        stats = torch.zeros((N // 32, 16, 2), dtype=torch.float32, device=x.device)
    g, b, eps = ln if ln is not None else (None, None, 0.0)
    context(x.device.index or 0).call("agpu_int4_linear_pieces", _f32(x), g, b, float(eps), packed, scales, bias, residual, y, M, N, K,
                                      group, flags, out_gamma, pieces, stats)
    return (y, pieces, stats) if want_pieces else y


def int4_matmul(a, b, group=128):
    """ops::int4_matmul (nn/ops/gemm.rs:1186-1266): B [K, N] is quantized on the fly (per column, groups of 128 along
    K, the Rust quantizer's rounding; on the device here, on the host after a download in the reference), then
    A [M, K] goes through the int4 Linear."""
    if a.dim() != 2 or b.dim() != 2:
        _shape_err("2D tensors", f"a.ndim={a.dim()}, b.ndim={b.dim()}")
    if a.shape[1] != b.shape[0]:
        _shape_err(f"B with {a.shape[1]} rows", f"{b.shape[0]}")
    if a.shape[1] % 8 != 0:
        _shape_err("K divisible by 8 for INT4 packing", f"K={a.shape[1]}")
    packed, scales = int4_quantize(b, group, _lib.QUANT_RUST)
    return int4_linear(a, packed, scales, group=group)


def int4_dequantize(packed, scales, group):
    kp, N = packed.shape
    w = torch.empty((kp * 8, N), dtype=torch.float32, device=packed.device)
    context(packed.device.index or 0).call("agpu_int4_dequantize", packed, scales, w, kp * 8, N, group)
    return w


def int4_quantize(weight_t, group, mode=_lib.QUANT_RUST):
    """quantize_weight_int4 (nn/ops/quantize.rs:102-153) on the device."""
    K, N = weight_t.shape
    if K % 8 != 0:
        _shape_err("K divisible by 8", f"K = {K}")
    packed = torch.empty((K // 8, N), dtype=torch.int32, device=weight_t.device)
    scales = torch.empty(((K + group - 1) // group, N), dtype=torch.float32, device=weight_t.device)
    context(weight_t.device.index or 0).call("agpu_int4_quantize", _f32(weight_t), packed, scales, K, N, group, mode)
    return packed, scales


def int4_quantize_host(weight_t, group, mode=_lib.QUANT_RUST):
    """quantize_weight_int4 on the host CPU (numpy in, numpy out); needs no GPU."""
    import numpy as np

    w = np.ascontiguousarray(weight_t, dtype=np.float32)
    K, N = w.shape
    packed = np.empty((K // 8 if K % 8 == 0 else 0, N), np.uint32)
    scales = np.empty(((K + group - 1) // group, N), np.float32)
    rc = _lib.cdll().agpu_int4_quantize_host(w.ctypes.data, packed.ctypes.data, scales.ctypes.data, K, N, group, mode)
    if rc != 0:
        raise AgpuError(rc, "int4_quantize_host: K must be divisible by 8" if rc == -1 else "int4_quantize_host failed")
    return packed, scales


def layer_norm(x, gamma, beta, eps=1e-5):
    return _native.layer_norm(x, gamma, beta, eps)


def add_layer_norm_dual(a, b, gamma, beta, eps=1e-5, want_sum=True):
    return _native.add_layer_norm_dual(a, b, gamma, beta, eps, want_sum)


def layer_norm_residual(x, residual, gamma, beta, eps=1e-5):
    """ops::layer_norm_residual (nn/ops/norm.rs:88-237): LayerNorm(x + residual)."""
    return add_layer_norm_dual(x, residual, gamma, beta, eps, want_sum=False)


def layer_norm_residual_dual(x, residual, gamma, beta, eps=1e-5):
    """ops::layer_norm_residual_dual (nn/ops/norm.rs:248-400): (x + residual, LayerNorm(x + residual))."""
    return add_layer_norm_dual(x, residual, gamma, beta, eps, want_sum=True)


def gelu(x, mode=_lib.GELU_TANH):
    return _native.gelu(x, mode)


def add_inplace(a, b):
    return _native.add_inplace(a, b)


def bias_add(data, bias):
    return _native.bias_add(data, bias)


def softmax_rows(x):
    return _native.softmax_rows(x)


def embedding(tokens, wte, wpe, pos_offset=0):
    return _native.embedding(tokens, wte, wpe, pos_offset)


def argmax_rows(x, last_index=False):
    return _native.argmax_rows(x, last_index)


def split_qkv(qkv, n_heads, d_head):
    return _native.split_qkv(qkv, n_heads, d_head)


def concat_heads(x):
    return _native.concat_heads(x)


def attention(q, k, v, kv_len=None, q_offset=0, causal=True):
    """q [H,q_len,dh]; k,v [H,kv_stride,dh] with the first kv_len rows valid."""
    return _native.attention(q, k, v, kv_len, q_offset, causal)


def multi_head_flash_attention(q, k, v, seq_len, n_heads, d_head):
    """ops::multi_head_flash_attention (nn/ops/attention.rs:151-202): q, k, v [H*seq, dh] head-major, causal."""
    return _native.multi_head_flash_attention(q, k, v, seq_len, n_heads, d_head)


def scaled_dot_product_attention(q, k, v, causal=True):
    """ops::scaled_dot_product_attention (nn/ops/attention.rs:17-100): one head, q, k, v [seq, dh]."""
    if q.dim() != 2 or k.shape != q.shape or v.shape != q.shape:
        _shape_err("q, k, v [seq, d_head]", f"{tuple(q.shape)}, {tuple(k.shape)}, {tuple(v.shape)}")
    return attention(q[None], k[None], v[None], causal=causal)[0]


def scaled_dot_product_attention_kv(q, k, v, q_len, kv_len, q_offset):
    """ops::scaled_dot_product_attention_kv (nn/ops/attention.rs:557-606): one head, q [q_len, dh] at positions
    q_offset.., k and v [kv_stride, dh] with the first kv_len rows valid; causal."""
    if q.dim() != 2 or q.shape[0] != q_len or k.shape != v.shape or k.shape[0] < kv_len:
        _shape_err(f"q [{q_len}, dh], k and v [>= {kv_len}, dh]", f"{tuple(q.shape)}, {tuple(k.shape)}, {tuple(v.shape)}")
    return attention(q[None], k[None], v[None], kv_len=kv_len, q_offset=q_offset, causal=True)[0]


def kv_append(src, cache, write_pos):
    return _native.kv_append(src, cache, write_pos)


def gemm_f32(a, b):
    return _native.gemm_f32(a, b)


class SimpleRng:
    """SimpleRng (nn/models/gpt2.rs:1000-1023): xorshift64; next_f32 in [0, 1)."""

    def __init__(self, seed):
        import ctypes as C
        self._s = C.c_uint64(_lib.cdll().agpu_simple_rng_new(int(seed) & 0xFFFFFFFFFFFFFFFF))

    @property
    def state(self):
        return int(self._s.value)

    def next_f32(self):
        import ctypes as C
        return float(_lib.cdll().agpu_simple_rng_next_f32(C.addressof(self._s)))


def top_k(logits, k, temperature=1.0):
    """Ranked candidates of top_k_sample (gpt2.rs:1029-1039) per row: (indices [rows, k] int32 view of uint32, values)."""
    import torch

    lg = logits.contiguous().view(-1, logits.shape[-1])
    rows, n = lg.shape
    kk = min(int(k), n)
    idx = torch.empty((rows, kk), dtype=torch.int32, device=lg.device)
    val = torch.empty((rows, kk), dtype=torch.float32, device=lg.device)
    context(lg.device.index or 0).call("agpu_top_k", lg, rows, n, int(k), float(temperature), idx, val)
    return idx, val


def softmax_max_prob(logits):
    """softmax_max_prob (gpt2.rs:983-988) per row of device logits: (confidence [rows] f32, arg-max [rows] int32 view)."""
    import torch

    lg = logits.contiguous().view(-1, logits.shape[-1])
    rows, n = lg.shape
    conf = torch.empty(rows, dtype=torch.float32, device=lg.device)
    idx = torch.empty(rows, dtype=torch.int32, device=lg.device)
    context(lg.device.index or 0).call("agpu_softmax_max_prob", lg, rows, n, conf, idx)
    return conf, idx


def top_k_sample(logits, k, temperature, rng):
    """top_k_sample (gpt2.rs:1029-1058) on a device logit vector; advances rng; returns the token id."""
    import ctypes as C

    lg = logits.contiguous().view(-1)
    tok = C.c_uint32(0)
    context(lg.device.index or 0).call("agpu_top_k_sample", lg, lg.numel(), int(k), float(temperature), C.addressof(rng._s),
                                       C.addressof(tok))
    return int(tok.value)
