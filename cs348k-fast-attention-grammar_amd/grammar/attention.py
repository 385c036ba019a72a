"""Python face of the hand-written CDNA4 attention forward (gr_attn_fwd).

`flash_attention_fwd(q, k, v)` computes softmax(scale * q k^T [causal]) v for
[B, H, N, D] fp16/bf16 tensors (or fp32 ones, non-causal, on the fp32 matrix
cores) on the GPU -- the same math as the reference's
attention module contract `fn(KT, Q, V)` (pytorch-naive.py:23-65,
run_attention_search.py:169-181) and its SDPA reference point
(flash-attn2-sota.py:41-62), batched over B and H.

There is no CPU path: CPU tensors or a missing library raise.
"""
from __future__ import annotations

import ctypes
import math

from . import runtime as rt


def _strides3(t) -> "ctypes.Array":
    st = t.stride()
    return rt.strides3(st[0], st[1], st[2])


def default_tiles(N: int, D: int, dtype: str | None = None, causal: bool = False) -> tuple:
    """(block_m, block_n) of the flash body's largest tiles: the largest query
    tile of 256 / 128 / 64 dividing N, and 128 keys per tile at D = 64 when
    they divide N, else 64 or 32. With the dtype given, the same except 256 x 64
    where the two-wave body applies (fp16, D = 64, non-causal, N a multiple of
    256): what gr_attn_fwd runs for block_m = block_n = 0 once B * H * N fills
    the GPU (smaller grids take smaller query tiles and key groups)."""
    bm = 256 if N % 256 == 0 else 128 if N % 128 == 0 else 64
    if dtype == "fp16" and D == 64 and not causal and N % 256 == 0:
        return bm, 64
    bn = 128 if (D == 64 and N % 128 == 0) else 64 if N % 64 == 0 else 32
    return bm, bn


def picked_shape(B: int, H: int, N: int, D: int, dtype: str, *, causal: bool = False, k_transposed: bool = False,
                 train: bool = False) -> tuple:
    """(queries, key groups, keys per tile) of the workgroup that gr_attn_fwd (or
    gr_attn_fwd_train) runs when no tile is named; N a multiple of 64, dtype "fp16"
    (scale log2(e) <= 1) or "bf16". Host arithmetic."""
    out = (ctypes.c_int * 3)()
    rt.check(rt.lib().gr_attn_fwd_shape(rt.GR_F16 if dtype == "fp16" else rt.GR_BF16, B, H, N, D, int(k_transposed),
                                        int(causal), int(train), out), "gr_attn_fwd_shape")
    return tuple(out)


def _fwd_args(q, k, v, lse, causal, scale, k_transposed, block_m, block_n, out, stream):
    """(C arguments, out) of gr_attn_fwd, or (lse given) of gr_attn_fwd_train,
    after checking the operands."""
    import torch
    dtype = q.dtype
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not t.is_cuda:
            raise ValueError(f"flash_attention_fwd: {name} must be a GPU tensor (no CPU path)")
        if t.dtype != dtype:
            raise ValueError("flash_attention_fwd: q, k, v must share a dtype")
        if t.dim() != 4:
            raise ValueError(f"flash_attention_fwd: {name} must be 4-D")
    shape = q.shape
    B, H, N, D = shape
    if v.shape != shape:
        raise ValueError(f"flash_attention_fwd: v shape {tuple(v.shape)} != q shape {tuple(shape)}")
    want_k = (B, H, D, N) if k_transposed else shape
    if k.shape != want_k:
        raise ValueError(f"flash_attention_fwd: k shape {tuple(k.shape)} != {tuple(want_k)}")
    if q.stride(3) != 1 or v.stride(3) != 1 or k.stride(3) != 1:
        raise ValueError("flash_attention_fwd: innermost dimension must be contiguous")
    if out is None:
        out = torch.empty(shape, dtype=dtype, device=q.device)
    elif out.shape != shape or out.dtype != dtype or out.stride(3) != 1:
        raise ValueError("flash_attention_fwd: bad `out` tensor")
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr())
    if lse is not None:
        head += (lse.data_ptr(),)
    return head + (rt.dtype_code(dtype), B, H, N, D, _strides3(q), _strides3(k), _strides3(v), _strides3(out),
                   int(bool(k_transposed)), int(bool(causal)), float(scale), int(block_m), int(block_n),
                   rt._stream_ptr(stream)), out


def bind_flash_attention(q, k, v, *, causal: bool = False, scale: float | None = None,
                         k_transposed: bool = False, block_m: int = 0, block_n: int = 0,
                         out=None, stream=None):
    """Validate the operands once and return (launch, out): launch() enqueues
    gr_attn_fwd with the pre-packed C arguments (no per-call checks or
    allocation, for launch-bound loops such as a timing loop); out is the
    [B, H, N, D] result tensor it writes. Arguments as flash_attention_fwd."""
    args, out = _fwd_args(q, k, v, None, causal, scale, k_transposed, block_m, block_n, out, stream)
    fn = rt.lib().gr_attn_fwd
    keep = (q, k, v, out)   # the tensors stay alive as long as the launcher

    def launch():
        rt.check(fn(*args), "gr_attn_fwd")
        return keep[3]
    return launch, out


def flash_attention_fwd(q, k, v, *, causal: bool = False, scale: float | None = None,
                        k_transposed: bool = False, block_m: int = 0, block_n: int = 0,
                        out=None, stream=None):
    """O = softmax(scale * Q K^T [+ causal mask]) V on the MI355X.

    q, v: [B, H, N, D]; k: [B, H, N, D], or [B, H, D, N] when k_transposed.
    All three share dtype (float16 or bfloat16) and live on the GPU. Returns a
    new [B, H, N, D] tensor (or writes `out`)."""
    args, out = _fwd_args(q, k, v, None, causal, scale, k_transposed, block_m, block_n, out, stream)
    rt.check(rt.lib().gr_attn_fwd(*args), "gr_attn_fwd")
    return out


def _train_lse(q, lse):
    """The [B, H, N] float32 row log-sum-exp to write: `lse`, checked, or a new one."""
    import torch
    shape = q.shape[:3]
    if lse is None:
        return torch.empty(shape, dtype=torch.float32, device=q.device)
    if lse.shape != shape or lse.dtype != torch.float32 or not lse.is_contiguous():
        raise ValueError("flash_attention_fwd_train: bad `lse` tensor")
    return lse


def bind_flash_attention_train(q, k, v, *, causal: bool = False, scale: float | None = None,
                               block_m: int = 0, block_n: int = 0, out=None, lse=None, stream=None):
    """bind_flash_attention for gr_attn_fwd_train: returns (launch, out, lse),
    launch() enqueueing the forward that also writes the row log-sum-exp of
    the scaled scores ([B, H, N] fp32, natural log). K in [B, H, N, D]."""
    if q.dim() != 4:
        raise ValueError("flash_attention_fwd: q must be 4-D")
    lse = _train_lse(q, lse)
    args, out = _fwd_args(q, k, v, lse, causal, scale, False, block_m, block_n, out, stream)
    fn = rt.lib().gr_attn_fwd_train
    keep = (q, k, v, out, lse)

    def launch():
        rt.check(fn(*args), "gr_attn_fwd_train")
        return keep[3], keep[4]
    return launch, out, lse


def flash_attention_fwd_train(q, k, v, *, causal: bool = False, scale: float | None = None,
                              block_m: int = 0, block_n: int = 0, out=None, lse=None, stream=None):
    """flash_attention_fwd that also returns the row log-sum-exp of the scaled
    scores ([B, H, N] fp32, natural log), kept for flash_attention_bwd.
    K in [B, H, N, D] layout. Returns (out, lse)."""
    if q.dim() != 4:
        raise ValueError("flash_attention_fwd: q must be 4-D")
    lse = _train_lse(q, lse)
    args, out = _fwd_args(q, k, v, lse, causal, scale, False, block_m, block_n, out, stream)
    rt.check(rt.lib().gr_attn_fwd_train(*args), "gr_attn_fwd_train")
    return out, lse


def _bwd_args(q, k, v, o, do, lse, causal, scale, workspace, grads, stream):
    """(C arguments, gradients, workspace) of gr_attn_bwd after checking the
    operands."""
    import torch
    shape, dtype = q.shape, q.dtype
    B, H, N, D = shape
    for name, t in (("q", q), ("k", k), ("v", v), ("o", o), ("do", do)):
        if t.shape != shape or t.dtype != dtype or not t.is_cuda:
            raise ValueError(f"flash_attention_bwd: {name} must match q ({tuple(shape)}, {dtype}, GPU)")
        if not t.is_contiguous():
            raise ValueError(f"flash_attention_bwd: {name} must be contiguous")
    if lse.shape != (B, H, N) or lse.dtype != torch.float32 or not lse.is_contiguous():
        raise ValueError("flash_attention_bwd: lse must be a contiguous [B, H, N] float32 tensor")
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    need = int(rt.lib().gr_attn_bwd_workspace(B, H, N, D))
    if workspace is None:
        workspace = rt.workspace(need, q.device, stream)
    elif workspace.numel() * workspace.element_size() < need:
        raise ValueError(f"flash_attention_bwd: workspace of {need} bytes needed")
    if grads is None:
        grads = (torch.empty_like(q), torch.empty_like(q), torch.empty_like(q))
    else:
        for t in grads:
            if t.shape != shape or t.dtype != dtype or not t.is_contiguous():
                raise ValueError("flash_attention_bwd: bad gradient tensor")
    dq, dk, dv = grads
    return (q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), do.data_ptr(), lse.data_ptr(),
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), rt.dtype_code(dtype), B, H, N, D, _strides3(q),
            int(bool(causal)), float(scale), workspace.data_ptr(), need, rt._stream_ptr(stream)), grads, workspace


def bind_flash_attention_bwd(q, k, v, o, do, lse, *, causal: bool = False, scale: float | None = None,
                             workspace=None, grads=None, stream=None):
    """Validate once and return (launch, (dq, dk, dv)): launch() enqueues
    gr_attn_bwd with pre-packed C arguments. q, k, v, o, do: contiguous
    [B, H, N, D] fp16/bf16 GPU tensors of one dtype (the kernels take one
    stride set); lse: [B, H, N] float32 from the training forward; grads: an
    optional (dq, dk, dv) triple of such tensors to write."""
    args, grads, workspace = _bwd_args(q, k, v, o, do, lse, causal, scale, workspace, grads, stream)
    fn = rt.lib().gr_attn_bwd
    keep = (q, k, v, o, do, lse, workspace, grads)

    def launch():
        rt.check(fn(*args), "gr_attn_bwd")
        return keep[7]
    return launch, grads


def flash_attention_bwd(q, k, v, o, do, lse, *, causal: bool = False, scale: float | None = None,
                        workspace=None, stream=None):
    """dQ, dK, dV of sum(O * dO) for the attention forward that produced o and
    lse (flash_attention_fwd_train). q, k, v, o, do: [B, H, N, D] fp16/bf16
    on the GPU (made contiguous here: the kernel takes one stride set)."""
    q, k, v, o, do, lse = (rt.contiguous(t, stream) for t in (q, k, v, o, do, lse))
    args, grads, workspace = _bwd_args(q, k, v, o, do, lse, causal, scale, workspace, None, stream)
    rt.check(rt.lib().gr_attn_bwd(*args), "gr_attn_bwd")
    return grads


def _autograd_function():
    import torch

    class FlashAttention(torch.autograd.Function):
        @staticmethod
        def forward(ctx, q, k, v, causal, scale):
            q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
            o, lse = flash_attention_fwd_train(q, k, v, causal=causal, scale=scale)
            ctx.save_for_backward(q, k, v, o, lse)
            ctx.causal, ctx.scale = causal, scale
            return o

        @staticmethod
        def backward(ctx, do):
            q, k, v, o, lse = ctx.saved_tensors
            dq, dk, dv = flash_attention_bwd(q, k, v, o, do, lse, causal=ctx.causal, scale=ctx.scale)
            return dq, dk, dv, None, None
    return FlashAttention


_FLASH_FN = None


def flash_attention(q, k, v, *, causal: bool = False, scale: float | None = None):
    """Differentiable attention on the MI355X kernels: forward through
    gr_attn_fwd_train, backward through gr_attn_bwd (torch.autograd)."""
    global _FLASH_FN
    if _FLASH_FN is None:
        _FLASH_FN = _autograd_function()
    return _FLASH_FN.apply(q, k, v, causal, scale)


def decode_splits(B: int, H: int, Nq: int, N: int, cu_count: int = 256, *, D: int = 64, groups: bool = True) -> int:
    """Key parts per query tile for gr_attn_decode, by the kernel that runs
    (lines measured over B H 1-512, N 128-16384, both head dims, every count of
    parts; in brackets the time over the best count's, geometric mean):
    1 query (streaming kernel): as many parts as fit one workgroup per compute
    unit, of at least 256 keys; up to 512 keys one launch is faster than two (D
    64 N 512: 5.0 us against 7.2) [1.02].
    With heads for a third of the units the second launch pays from 1,024 keys
    on (B H 128, N 768, D 64: 7.2 us in one part, 8.6 in two).
    2 to 4 queries (the same kernel for 2 or 4, more arithmetic per key): up to
    1.5 workgroups per compute unit for 2, 2 for 4 and with heads for more than
    half the units. Parts pay by their work, queries x keys x D: above 2^16,
    at least half of that a part (B H 8, N 3104, 4 queries, D 64: 12.6 us at 32
    parts, 20.6 at 6); with heads for more than half the units from 2^18 on (B H
    255, N 512, 4 queries, D 64: 12.3 us in one part, 17.6 in three) [1.03].
    5 to 64 queries (flash body, four key groups per workgroup): one workgroup
    per compute unit, at most 16 parts of at least 256 keys (B H 16, N 8192: 13.2
    us at 16 parts, 15.9 at 32). Heads for more than half the units take one part,
    except where two to four long ones take three quarters of its rounds of
    resident workgroups or less (two per unit at D 64, one at D 128: B H 150, N
    8192, D 128 137 us in one part, 121 in three; N 2048 31 and 37) [1.02].
    More, and the kernel without key groups (groups=False: fp16 with scale
    log2(e) > 1): two workgroups per compute unit, each part keeping at least
    four 64-key tiles (without groups B H 129, N 8192, D 64: 52 us in four parts,
    153 in one)."""
    heads = B * H
    many = 2 * heads > cu_count
    if Nq == 1:
        if N <= 512 or (3 * heads > cu_count and N < 1024):
            return 1
        return max(1, min(cu_count // heads, N // 256, 32))
    if Nq <= 4:
        slots = 2 if Nq == 2 else 4
        work = slots * N * D
        if work <= 1 << 16 or (many and work < 1 << 18):
            return 1
        per_unit = 3 if slots == 2 and not many else 4          # workgroups, in halves
        return max(1, min(per_unit * cu_count // (2 * heads), work >> 15, 32))
    if Nq <= 64 and groups:
        if N <= 512:
            return 1
        if not many:
            return min(cu_count // heads, N // 256, 16)
        resident = cu_count * (2 if D == 64 else 1)
        for s in (2, 3, 4):
            if N * D >= s << 18 and 4 * -(-heads * s // resident) <= 3 * s * -(-heads // resident):
                return s
        return 1
    tiles_q = heads * -(-Nq // 128)
    want = -(-2 * cu_count // tiles_q)
    return max(1, min(want, N // 256 if N >= 256 else 1))


def _key_groups(dtype, scale) -> bool:
    """Whether decode launches of 5 to 64 queries have key groups: not where fp16
    keeps Q as given (launch_decode's rule)."""
    return rt.dtype_code(dtype) != rt.GR_F16 or float(scale) * math.log2(math.e) <= 1.0


def decode_splits_noalloc(B: int, H: int, Nq: int, N: int, D: int, cu_count: int = 256, *, groups: bool = True) -> int:
    """decode_splits, lowered until the key parts' partials fit the library's
    scratch array (rt.DECODE_SCRATCH_BYTES), which gr_attn_decode_noalloc
    cannot grow. One part needs no scratch."""
    L = rt.lib()
    s = decode_splits(B, H, Nq, N, cu_count, D=D, groups=groups)
    while s > 1 and int(L.gr_attn_decode_workspace(B, H, Nq, D, s)) > rt.DECODE_SCRATCH_BYTES:
        s -= 1
    return s


def _decode_args(q, k, v, scale, splits, out, workspace, stream):
    """(C arguments, out, workspace) of gr_attn_decode after checking the operands."""
    import torch
    dtype = q.dtype
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not t.is_cuda:
            raise ValueError(f"flash_attention_decode: {name} must be a GPU tensor (no CPU path)")
        if t.dtype != dtype or t.dim() != 4 or t.stride(3) != 1:
            raise ValueError(f"flash_attention_decode: {name} must be 4-D, q's dtype, unit stride on D")
    B, H, Nq, D = q.shape
    N = k.shape[2]
    if k.shape != (B, H, N, D) or v.shape != (B, H, N, D):
        raise ValueError(f"flash_attention_decode: k {tuple(k.shape)} / v {tuple(v.shape)} do not match q {tuple(q.shape)}")
    if out is None:
        out = torch.empty((B, H, Nq, D), dtype=dtype, device=q.device)
    elif out.shape != (B, H, Nq, D) or out.dtype != dtype or out.stride(3) != 1:
        raise ValueError("flash_attention_decode: bad `out` tensor")
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    if splits <= 0:
        splits = decode_splits(B, H, Nq, N, rt.cu_count(q.device.index or 0), D=D, groups=_key_groups(dtype, scale))
        if workspace is not None and splits > 1:      # sized by the caller: the most parts that fit, from two on
            fit = workspace.numel() * workspace.element_size() // (int(rt.lib().gr_attn_decode_workspace(B, H, Nq, D, 2)) // 2)
            splits = fit if 2 <= fit < splits else splits
    need = int(rt.lib().gr_attn_decode_workspace(B, H, Nq, D, splits)) if splits > 1 else 0
    if need and workspace is None:
        workspace = rt.workspace(need, q.device, stream)
    elif need and workspace.numel() * workspace.element_size() < need:
        raise ValueError(f"flash_attention_decode: workspace of {need} bytes needed")
    return (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), rt.dtype_code(dtype), B, H, Nq, N, D,
            _strides3(q), _strides3(k), _strides3(v), _strides3(out), float(scale), int(splits),
            workspace.data_ptr() if need else None, need, rt._stream_ptr(stream)), out, workspace


def bind_flash_attention_decode(q, k, v, *, scale: float | None = None, splits: int = 0, out=None,
                                workspace=None, stream=None):
    """Validate once and return (launch, out) for gr_attn_decode, arguments
    pre-packed (as bind_flash_attention); see flash_attention_decode."""
    args, out, workspace = _decode_args(q, k, v, scale, splits, out, workspace, stream)
    fn = rt.lib().gr_attn_decode
    keep = (q, k, v, out, workspace)

    def launch():
        rt.check(fn(*args), "gr_attn_decode")
        return keep[3]
    return launch, out


def bind_flash_attention_decode_noalloc(q, k, v, *, scale: float | None = None, splits: int = 0, out=None,
                                        stream=None):
    """(launch, out) for gr_attn_decode_noalloc: the decode launch with its
    key-split partials in the library's per-device scratch array, so neither
    the binding (given `out`) nor a launch allocates device memory. Launches
    that overlap on one device race on that array. Raises if the split needs
    more than rt.DECODE_SCRATCH_BYTES; splits = 0 picks the largest split
    decode_splits allows that fits it (decode_splits_noalloc)."""
    import torch
    for name, t in (("q", q), ("k", k), ("v", v)):
        if not t.is_cuda:
            raise ValueError(f"flash_attention_decode_noalloc: {name} must be a GPU tensor (no CPU path)")
        if t.dtype != q.dtype or t.dim() != 4 or t.stride(3) != 1:
            raise ValueError(f"flash_attention_decode_noalloc: {name} must be 4-D, q's dtype, unit stride on D")
    B, H, Nq, D = q.shape
    N = k.shape[2]
    if tuple(k.shape) != (B, H, N, D) or tuple(v.shape) != (B, H, N, D):
        raise ValueError("flash_attention_decode_noalloc: k / v do not match q")
    if out is None:
        out = torch.empty((B, H, Nq, D), dtype=q.dtype, device=q.device)
    elif tuple(out.shape) != (B, H, Nq, D) or out.dtype != q.dtype or out.stride(3) != 1:
        raise ValueError("flash_attention_decode_noalloc: bad `out` tensor")
    if scale is None:
        scale = 1.0 / math.sqrt(D)
    L = rt.lib()
    if splits <= 0:
        splits = decode_splits_noalloc(B, H, Nq, N, D, rt.cu_count(q.device.index or 0),
                                       groups=_key_groups(q.dtype, scale))
    fn = L.gr_attn_decode_noalloc
    args = (ctypes.c_void_p(q.data_ptr()), ctypes.c_void_p(k.data_ptr()), ctypes.c_void_p(v.data_ptr()),
            ctypes.c_void_p(out.data_ptr()), rt.dtype_code(q.dtype), B, H, Nq, N, D,
            _strides3(q), _strides3(k), _strides3(v), _strides3(out), float(scale), int(splits),
            rt._stream_ptr(stream))
    keep = (q, k, v, out)

    def launch():
        rt.check(fn(*args), "gr_attn_decode_noalloc")
        return keep[3]
    return launch, out


def flash_attention_decode(q, k, v, *, scale: float | None = None, splits: int = 0, out=None,
                           workspace=None, stream=None):
    """O = softmax(scale * Q K^T) V for Nq queries against N keys (non-causal):
    q [B, H, Nq, D], k and v [B, H, N, D] (N a multiple of 32), fp16/bf16 on
    the GPU. splits = 0 picks the key split (decode_splits; with a workspace
    given, at most the parts it holds); the workspace it needs is allocated
    here unless given."""
    args, out, workspace = _decode_args(q, k, v, scale, splits, out, workspace, stream)
    rt.check(rt.lib().gr_attn_decode(*args), "gr_attn_decode")
    return out


def attention_flops(B: int, H: int, N: int, D: int, causal: bool = False) -> int:
    """Algorithmic FLOPs of attention forward: 4*B*H*N^2*D (two GEMMs), halved
    for a causal mask (old/benchmark.py:354-355 defines the 4*B*H*S^2*D count)."""
    f = 4 * B * H * N * N * D
    return f // 2 if causal else f


def attention_io_bytes(B: int, H: int, N: int, D: int, elem_bytes: int = 2) -> int:
    """Minimal HBM traffic: read Q, K, V once and write O once."""
    return 4 * B * H * N * D * elem_bytes


def mfma32_selftest(a, b):
    """D = A[32,16] @ B[16,32] through one 32x32x16 MFMA with the operand and
    accumulator layout the kernels assume (fp16 in, fp32 out)."""
    import torch
    if a.shape != (32, 16) or b.shape != (16, 32) or a.dtype != torch.float16 or b.dtype != torch.float16:
        raise ValueError("mfma32_selftest: need fp16 A[32,16] and B[16,32]")
    a = a.contiguous()
    b = b.contiguous()
    d = torch.empty((32, 32), dtype=torch.float32, device=a.device)
    rt.check(rt.lib().gr_selftest_mfma32(ctypes.c_void_p(a.data_ptr()), ctypes.c_void_p(b.data_ptr()),
                                         ctypes.c_void_p(d.data_ptr()), rt._stream_ptr(None)),
             "gr_selftest_mfma32")
    return d
