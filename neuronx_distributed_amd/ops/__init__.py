"""Hand-written CDNA4 HIP kernels — python wrappers + autograd.

The native library (``libnxd_ops.so``, built in-tree by ``ops/build.py``)
replaces the reference's NKI kernels: RMSNorm, RoPE,
SwiGLU, flash attention, fused AdamW.  On a GPU box the HIP path is
MANDATORY — if the library is missing, GPU calls raise instead of silently
falling back to eager torch.  CPU tensors use plain-torch reference
implementations (the numerics baseline the GPU kernels are tested against).
"""

import ctypes
import functools
import math
import os
import warnings
from typing import Optional

import torch

_LIB = None
_LIB_ERR = None


def _load():
    global _LIB, _LIB_ERR
    if _LIB is not None or _LIB_ERR is not None:
        return _LIB
    from .build import LIB

    if not os.path.exists(LIB):
        _LIB_ERR = f"{LIB} not built — run neuronx_distributed_amd.ops.build"
        return None
    try:
        lib = ctypes.CDLL(LIB)
    except OSError as e:  # pragma: no cover
        _LIB_ERR = str(e)
        return None
    _declare_flash(lib)
    if hasattr(lib, "embedding_work"):
        lib.embedding_work.restype = ctypes.c_long
    _LIB = lib
    return _LIB


def _declare_flash(lib):
    """Argument types of the flash entry points, so that numbers go in as they
    are: a short sequence waits for its launches, not for the kernels."""
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    shape = [i] * 4
    for name, args in (
            ("flash_attn_fwd_strided", [p] * 5 + shape + [f, i, i, p, p]),
            ("flash_attn_bwd_strided", [p] * 10 + shape + [i, f, i, i, p, p]),
            ("flash_attn_bwd_reduce", [p] * 4 + shape + [p, p])):
        if hasattr(lib, name):
            getattr(lib, name).argtypes = args


def is_available() -> bool:
    return _load() is not None


def _require_lib():
    lib = _load()
    if lib is None:
        raise RuntimeError(
            f"nxd_ops HIP library unavailable on a GPU tensor: {_LIB_ERR}. "
            "The MI355X-native kernels are mandatory on GPU — build with "
            "python -m neuronx_distributed_amd.ops.build")
    return lib


def _stream() -> ctypes.c_void_p:
    # the current stream's handle alone (0.3 us, with the object around it 2.9)
    return ctypes.c_void_p(
        torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice()))


def _ptr(t: torch.Tensor) -> ctypes.c_void_p:
    return ctypes.c_void_p(t.data_ptr())


# ---------------------------------------------------------------------------
# RMSNorm
# ---------------------------------------------------------------------------

def _bf16_rows(x, *beside) -> bool:
    """May the norm kernels run: everything that they read is bf16, in rows of
    whole 16-byte words.  (A 32-bit weight beside bf16 rows takes the composed
    form, which reads it as it is.)"""
    return x.is_cuda and x.shape[-1] % 8 == 0 and \
        x.dtype == torch.bfloat16 and all(t.dtype == x.dtype for t in beside)


def _rmsnorm_bwd(x, weight, dy, rstd, dpass=None):
    """dx (+ dpass) and dw of contiguous bf16 rows x."""
    lib = _require_lib()
    H = x.shape[-1]
    rows = x.numel() // H
    # named, so that copies live until the launch
    w, dy = weight.contiguous(), dy.contiguous()
    dpass = None if dpass is None else dpass.contiguous()
    dx = torch.empty_like(x)
    dw = torch.empty(H, dtype=weight.dtype, device=x.device)
    part = torch.empty(lib.rmsnorm_bwd_parts(rows), H, dtype=torch.float32,
                       device=x.device)
    lib.rmsnorm_bwd(_ptr(x), _ptr(w), _ptr(dy), _ptr(rstd),
                    None if dpass is None else _ptr(dpass), _ptr(dx),
                    _ptr(part), _ptr(dw), rows, H, _stream())
    return dx, dw


class _RMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        ctx.eps = eps
        if _bf16_rows(x, weight):
            lib = _require_lib()
            x2 = x.contiguous()
            rows = x2.numel() // x2.shape[-1]
            out = torch.empty_like(x2)
            rstd = torch.empty(rows, dtype=torch.float32, device=x.device)
            lib.rmsnorm_fwd(_ptr(x2), _ptr(weight.contiguous()), _ptr(out),
                            _ptr(rstd), ctypes.c_int(rows),
                            ctypes.c_int(x2.shape[-1]), ctypes.c_float(eps),
                            _stream())
            ctx.save_for_backward(x2, weight, rstd)
            return out
        # composed form (fp32 math like the kernel)
        xf = x.float()
        rstd = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
        ctx.save_for_backward(x, weight, rstd.squeeze(-1).reshape(-1))
        return (xf * rstd * weight.float()).to(x.dtype)

    @staticmethod
    def backward(ctx, dy):
        x, weight, rstd = ctx.saved_tensors
        H = x.shape[-1]
        if _bf16_rows(x, weight):
            return (*_rmsnorm_bwd(x, weight, dy, rstd), None)
        xf = x.float()
        dyf = dy.float()
        wf = weight.float()
        r = rstd.reshape(x.shape[:-1]).unsqueeze(-1).to(torch.float32)
        dot = (dyf * wf * xf).sum(-1, keepdim=True)
        dx = r * wf * dyf - r.pow(3) / H * xf * dot
        dw = (dyf * xf * r).reshape(-1, H).sum(0)
        return dx.to(x.dtype), dw.to(weight.dtype), None


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6):
    return _RMSNormFn.apply(x, weight, eps)


def add_rmsnorm_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "add_rmsnorm_fwd")


def add_rmsnorm(residual: torch.Tensor, delta: torch.Tensor,
                weight: torch.Tensor, eps: float = 1e-6):
    """Fused ``res_out = residual + delta; normed = rmsnorm(res_out)*w``
    (inference only, no autograd).  GPU rows; the kernel takes bf16 rows and
    weight of H % 8 == 0."""
    lib = _require_lib()
    if not _bf16_rows(residual, delta, weight):
        return _add_rmsnorm_composed(residual, delta, weight, eps)[:2]
    H = residual.shape[-1]
    rows = residual.numel() // H
    r = residual.contiguous()
    d = delta.contiguous()
    res_out = torch.empty_like(r)
    normed = torch.empty_like(r)
    lib.add_rmsnorm_fwd(_ptr(r), _ptr(d), _ptr(weight.contiguous()),
                        _ptr(res_out), _ptr(normed), rows, H,
                        ctypes.c_float(eps), _stream())
    return res_out, normed


def _add_rmsnorm_composed(res, delta, weight, eps):
    """(h, normed, rstd) in fp32 math, norm stats on the rounded sum: matches
    the kernel and an unfused bf16 add -> rmsnorm chain."""
    h = (delta.float() + res.float()).to(delta.dtype)
    hf = h.float()
    rstd = torch.rsqrt(hf.pow(2).mean(-1, keepdim=True) + eps)
    return h, (hf * rstd * weight.float()).to(delta.dtype), rstd


class _AddRMSNormFn(torch.autograd.Function):
    """Training fused residual-add + RMSNorm: (delta, res) -> (h, normed)
    with h = bf16(delta + res), normed = rmsnorm(h) * w.  The backward
    folds the residual fork's pass-through gradient dh into the RMSNorm
    backward pass, so the fused site costs one
    kernel in each direction instead of norm + a 3-pass eager add
    (CUDAFunctor_add was ~2%% of the training step)."""

    @staticmethod
    def forward(ctx, delta, res, weight, eps):
        ctx.eps = eps
        if _bf16_rows(delta, res, weight):
            lib = _require_lib()
            H = delta.shape[-1]
            rows = delta.numel() // H
            dc, rc = delta.contiguous(), res.contiguous()
            h = torch.empty_like(dc)
            normed = torch.empty_like(dc)
            rstd = torch.empty(rows, dtype=torch.float32,
                               device=delta.device)
            lib.add_rmsnorm_fwd_train(_ptr(rc), _ptr(dc),
                                      _ptr(weight.contiguous()), _ptr(h),
                                      _ptr(normed), _ptr(rstd), rows, H,
                                      ctypes.c_float(eps), _stream())
            ctx.save_for_backward(h, weight, rstd)
            return h, normed
        h, normed, rstd = _add_rmsnorm_composed(res, delta, weight, eps)
        ctx.save_for_backward(h, weight, rstd.squeeze(-1).reshape(-1))
        return h, normed

    @staticmethod
    def backward(ctx, dh, dnormed):
        h, weight, rstd = ctx.saved_tensors
        H = h.shape[-1]
        if dnormed is None:
            # normed output unused: the op reduces to the residual add —
            # grads pass straight through, no weight grad
            return dh, dh, None, None
        if _bf16_rows(h, weight):
            dx, dw = _rmsnorm_bwd(h, weight, dnormed, rstd, dh)
            return dx, dx, dw, None
        hf = h.float()
        dyf = dnormed.float()
        wf = weight.float()
        r = rstd.reshape(h.shape[:-1]).unsqueeze(-1).to(torch.float32)
        dot = (dyf * wf * hf).sum(-1, keepdim=True)
        dx = r * wf * dyf - r.pow(3) / H * hf * dot
        if dh is not None:
            dx = dx + dh.float()
        dw = (dyf * hf * r).reshape(-1, H).sum(0)
        dxc = dx.to(h.dtype)
        return dxc, dxc, dw.to(weight.dtype), None


def add_rmsnorm_train(delta: torch.Tensor, res: torch.Tensor,
                      weight: torch.Tensor, eps: float = 1e-6):
    """Autograd fused ``h = delta + res; normed = rmsnorm(h) * w`` —
    returns (h, normed); d delta == d res == rmsnorm_bwd + dh (fused)."""
    return _AddRMSNormFn.apply(delta, res, weight, eps)


def add_rmsnorm_train_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "add_rmsnorm_fwd_train")


# ---------------------------------------------------------------------------
# RoPE (neox rotate-half), in-place on clones
# ---------------------------------------------------------------------------

def _rope_torch(x, cos, sin, sign=1.0):
    # x (B,S,h,D); cos/sin (S, D/2) f32
    half = x.shape[-1] // 2
    x0 = x[..., :half].float()
    x1 = x[..., half:].float()
    c = cos.view(1, cos.shape[0], 1, half)
    s = sin.view(1, sin.shape[0], 1, half) * sign
    o0 = x0 * c - x1 * s
    o1 = x1 * c + x0 * s
    return torch.cat([o0, o1], dim=-1).to(x.dtype)


class _RoPEFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, cos, sin, pos_offset):
        # bounds-check HERE: an out-of-range position would be an
        # out-of-bounds global read inside the HIP kernel (GPU fault)
        S = q.shape[1]
        off = int(pos_offset) if not isinstance(pos_offset, torch.Tensor) \
            else 0  # device-tensor positions are decode-path (S == 1)
        if off + S > cos.shape[0]:
            raise ValueError(
                f"RoPE table too short: seq {off}+{S} > table "
                f"{cos.shape[0]} (raise max_position_embeddings)")
        ctx.pos_offset = pos_offset
        ctx.save_for_backward(cos, sin)
        if q.is_cuda and q.dtype == torch.bfloat16:
            lib = _require_lib()
            B, S, Hq, D = q.shape
            Hk = k.shape[2]
            qc, kc = q.contiguous(), k.contiguous()
            qo = torch.empty_like(qc)
            ko = torch.empty_like(kc)
            lib.rope_fwd(_ptr(qc), _ptr(kc), _ptr(qo), _ptr(ko), _ptr(cos),
                         _ptr(sin),
                         ctypes.c_int(B), ctypes.c_int(S), ctypes.c_int(Hq),
                         ctypes.c_int(Hk), ctypes.c_int(D),
                         ctypes.c_int(pos_offset), ctypes.c_int(0), _stream())
            return qo, ko
        S = q.shape[1]
        c = cos[pos_offset:pos_offset + S]
        s = sin[pos_offset:pos_offset + S]
        return _rope_torch(q, c, s), _rope_torch(k, c, s)

    @staticmethod
    def backward(ctx, dq, dk):
        cos, sin = ctx.saved_tensors
        off = ctx.pos_offset
        if dq.is_cuda and dq.dtype == torch.bfloat16:
            lib = _require_lib()
            B, S, Hq, D = dq.shape
            Hk = dk.shape[2]
            dqc, dkc = dq.contiguous(), dk.contiguous()
            dqo = torch.empty_like(dqc)
            dko = torch.empty_like(dkc)
            lib.rope_fwd(_ptr(dqc), _ptr(dkc), _ptr(dqo), _ptr(dko),
                         _ptr(cos), _ptr(sin),
                         ctypes.c_int(B), ctypes.c_int(S), ctypes.c_int(Hq),
                         ctypes.c_int(Hk), ctypes.c_int(D), ctypes.c_int(off),
                         ctypes.c_int(1), _stream())
            return dqo, dko, None, None, None
        S = dq.shape[1]
        c = cos[off:off + S]
        s = sin[off:off + S]
        return (_rope_torch(dq, c, s, -1.0), _rope_torch(dk, c, s, -1.0),
                None, None, None)


def apply_rotary_pos_emb(q, k, cos, sin, pos_offset: int = 0):
    """q (B,S,Hq,D), k (B,S,Hk,D); cos/sin (S_max, D/2) fp32 tables."""
    return _RoPEFn.apply(q, k, cos, sin, pos_offset)


def _llama3_scale_freqs(inv_freqs: torch.Tensor, scaling: dict):
    """Llama-3.1 long-context frequency scaling (reference
    attention/utils.py apply_scaling): high-frequency components (short
    wavelength vs the original context) pass through, low-frequency ones
    divide by ``factor``, the band between interpolates smoothly."""
    import math as _math

    factor = float(scaling["factor"])
    lo = float(scaling.get("low_freq_factor", 1.0))
    hi = float(scaling.get("high_freq_factor", 4.0))
    orig = float(scaling.get("original_max_position_embeddings", 8192))
    wavelen = 2 * _math.pi / inv_freqs
    smooth = ((orig / wavelen - lo) / (hi - lo)).clamp(0.0, 1.0)
    blended = (1.0 - smooth) * inv_freqs / factor + smooth * inv_freqs
    return torch.where(wavelen < orig / hi, inv_freqs,
                       torch.where(wavelen > orig / lo, inv_freqs / factor,
                                   blended))


def precompute_rope_freqs(seq_len: int, dim: int, theta: float = 10000.0,
                          device=None, rope_scaling: dict = None):
    """cos/sin tables (S, D/2) fp32 (reference attention/utils.py
    precompute_freqs_cis; ``rope_scaling`` with rope_type \"llama3\"
    applies the 3.1 long-context wavelength interpolation)."""
    inv = 1.0 / (theta ** (torch.arange(0, dim, 2, device=device,
                                        dtype=torch.float32) / dim))
    if rope_scaling:
        rt = rope_scaling.get("rope_type", rope_scaling.get("type",
                                                            "llama3"))
        if rt == "llama3":
            inv = _llama3_scale_freqs(inv, rope_scaling)
        elif rt == "linear":
            inv = inv / float(rope_scaling["factor"])
        else:
            raise NotImplementedError(f"rope_scaling type {rt!r}")
    t = torch.arange(seq_len, device=device, dtype=torch.float32)
    freqs = torch.outer(t, inv)
    return freqs.cos(), freqs.sin()


def apply_rotary_polar_compatible(query, key, freqs):
    """Meta-llama INTERLEAVED rotary (reference attention/utils.py:50
    apply_rotary_polar_compatible): dims pair as (2i, 2i+1) complex
    components — used for Meta-format checkpoints, whereas the model
    stack and HIP kernel use the HF neox rotate-half pairing.
    query/key (B, S, H, D); freqs (S, D/2) fp32 angles."""
    if freqs.dtype != torch.float32:
        raise ValueError("freqs must be fp32 for accuracy")
    phase = torch.polar(torch.ones_like(freqs), freqs)  # e^{i*theta}
    phase = phase.view(1, freqs.shape[0], 1, freqs.shape[1])

    def rot(x):
        xc = torch.view_as_complex(
            x.float().reshape(*x.shape[:-1], x.shape[-1] // 2, 2))
        return torch.view_as_real(xc * phase).reshape(x.shape).to(x.dtype)

    return rot(query), rot(key)


# ---------------------------------------------------------------------------
# weight gradients
# ---------------------------------------------------------------------------

def turn_rule(T: int, N: int, K: int):
    """Which operands of dy^T x, dy (T, N) and x (T, K), are turned first, so that
    the library reads them along T: (dy, x).  It reaches 1.05 PFLOP/s with none,
    1.23 with one and up to 1.55 with both; turning runs at 5.7 TB/s.  Its forms, and
    so the gain, jump with the sizes; lines were drawn over 870 of them where next to
    none is slower (8 by 2 % to 8 %; gains, with the turning):

    - both of wide ones (from 8192: 1.15 to 1.23), and below 2600 rows, where the
      library has no good form for one (1200, 32000 x 4096: 342 -> 278 us, with one
      364), unless a side is below 4096 (2048, 3584 x 18944: 275 -> 302, with one 259)
      or the weight is small (6144 x 4096: 0.87 to 1.00, 8200 x 4096: 0.86 to 1.05;
      4096 x 11008: 1100 and 1200 0.97, 1400 to 2600 1.08 to 1.27; 800, 22016 x 4096:
      162 -> 205);
    - else the smaller one, from 1600 rows: of weights from 55 million 1.02 to 1.25
      (8192, 22016 x 4096: 1430 -> 1222; but 1800, 3584 x 18944: 0.96); of smaller
      ones with a side below 3584 1.00 to 1.41 (8192 x 3072, 22016 x 2048, of which
      3300 and 5000 rows 0.92; but dy of many rows for weights below 30 million: 2048
      x 11008: 3300 1.23, from 5000 on 0.97, 2560 x 9728: 0.95 to 1.03); of others up
      to 9216 rows (5120 x 5120: 1.04 to 1.45, 10752 0.78; 3584 x 8192: 1.03 to 1.6,
      9728 0.90), with a side from 4096 to 5119 not below 40 million (4096 x 6144:
      0.87 to 1.02), and not from 3073 to 8191 rows (4096 x 11008: 3072 1.02, 3300
      0.90, 5000 0.91, 7168 0.98, from 8192 on 0.98 to 1.08; 11008 x 4096: 0.89 to
      1.16)."""
    least, size = min(N, K), N * K
    if T < 1100 or size < 20_000_000:
        return False, False
    if least >= 8192:
        return True, True
    large, square = size >= 55_000_000, 4096 <= least < 5120
    if T < 2600 and least >= 4096:
        both = large or not square or size >= 40_000_000 and T >= 1400
        return both, both
    if T < 1600 or not large and (
            square and (size < 40_000_000 or 3072 < T < 8192) or
            not square and least >= 3584 and T > 9216 or
            N < K and size < 30_000_000 and T > 3500):
        return False, False
    return N <= K, N > K


def _turned(x: torch.Tensor) -> torch.Tensor:
    """x (T, K) as a view of its columns laid out in rows: a copy as large as x, which
    lives as long as the product that reads it; x itself where there is no room for
    one.  64 words beside the rows keep those of a power of two off one memory channel
    (8192 rows of 4096: 23.3 us, without 24.6; the product of it 204, without 225)."""
    T, K = x.shape
    pitch = (T + 63) // 64 * 64 + 64
    try:
        out = torch.empty(K, pitch, dtype=x.dtype, device=x.device)
    except torch.OutOfMemoryError:
        return x
    if _require_lib().transpose_words(
            _ptr(x), ctypes.c_long(x.stride(0)), _ptr(out), ctypes.c_long(pitch),
            T, K, _stream()):
        raise RuntimeError("transpose_words failed")
    return out[:, :T].t()


def _turns(t: torch.Tensor) -> bool:
    """May these rows be turned: bf16, whole 16-byte words?"""
    return t.is_cuda and t.dtype == torch.bfloat16 and t.stride(1) == 1 and \
        not (t.shape[1] | t.stride(0)) & 7 and not t.data_ptr() & 15


def weight_grads(grads, x: torch.Tensor):
    """[dy^T x for dy in grads] of dy (T, N) and x (T, K)."""
    T, K = x.shape
    if T < 1100 or not x.is_cuda:              # as in the rule, for all
        return [g.t().matmul(x) for g in grads]
    from .serving import unseen

    ways = [(False, False)] * len(grads)
    if _turns(x) and unseen(x, *grads) and \
            x.get_device() == torch._C._cuda_getDevice():
        ways = [turn_rule(T, g.shape[1], K) for g in grads]
        # x is turned once for all of them
        if turn_rule(T, sum(g.shape[1] for g in grads), K)[1]:
            ways = [(dy, True) for dy, _ in ways]
    if any(way for _, way in ways):
        xt = _turned(x)
    return [(_turned(g) if dy and _turns(g) else g).t().matmul(xt if way else x)
            for g, (dy, way) in zip(grads, ways)]


def turn_weight_rule(T: int, N: int, K: int) -> bool:
    """Is w (N, K) turned for dy w of T rows?  As above, 1.01 to 1.32 times as fast
    with the turning where the library's tiles of 256 rows are whole sixteens (8192
    rows, 32000 x 4096: 1545 -> 1367 us; 4096 x 4096: 198 -> 185, so from 7937 rows
    on; 12288: 1.03 to 1.10; 16384: 391 -> 352), and of any 24576 rows and more (1.06
    to 1.18).  Others jump (4096 x 4096: 7872 rows 1.08, 11776 0.87, 12544 0.93, 13568
    1.10, 20000 0.96; 32000 x 4096: 6656 0.82, 7168 1.30, 7680 0.85, 7872 0.93, 8256
    0.99, 10240 0.93).  Not below (6144, 4096 x 11008: 449 -> 493), and of the largest
    weights only for many (8192, 27648 x 5120: 2279 -> 2349, 16384: 3429 -> 2982)."""
    tiles = -(-T // 256)
    return tiles >= 32 and (tiles % 16 == 0 or T >= 24576) and \
        16_000_000 < N * K < (140_000_000 if T < 16384 else 1 << 31)


def input_weight(dy: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """w (N, K), laid out as dy (..., N) times it is the fastest."""
    if dy.is_cuda and w.dim() == 2 and dy.shape[-1] and \
            turn_weight_rule(dy.numel() // dy.shape[-1], *w.shape):
        from .serving import unseen

        if _turns(w) and dy.dtype == w.dtype and unseen(dy, w) and \
                dy.get_device() == w.get_device() == torch._C._cuda_getDevice():
            return _turned(w)
    return w


def input_grad(dy: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """dy (..., N) w, w (N, K).  With a turned weight it is one product of all rows:
    torch makes a batch of them where the strides of dy's dimensions of one do not
    follow from the others (one sequence, tokens first) and nobody differentiates the
    second operand."""
    laid = input_weight(dy, w)
    if laid is w:
        return dy.matmul(w)
    return dy.reshape(-1, w.shape[0]).mm(laid).view(*dy.shape[:-1], w.shape[1])


# ---------------------------------------------------------------------------
# embedding
# ---------------------------------------------------------------------------

def embedding_rule(T: int, V: int, W: int) -> bool:
    """Is ``_EmbeddingFn`` the faster one for T tokens and a table (V, W)?  Over 400
    calls, of tokens evenly and unevenly spread, far apart, of one row and of padding
    (torch's and this, us): from 2048 tokens on, below which the host takes longer than
    the device (32000 x 4096: 512 tokens 78, 71, 2048 187, 66; 256 x 512: 512 40, 68,
    1536 66, 68, 2048 85, 68), up to 32768 (32000 x 4096: 1000, 143; 40 words of 8192 x
    768: 146, 130, of 65536 tokens 197, 247), of rows from 1 KB and tables up to 2^18
    (32768 tokens, 262144 x 512: 240, 130; 10^6 x 512, 3073 tokens 222, 240; 10^6 x 64:
    102, 176)."""
    return 2048 <= T <= 32768 and W >= 512 and W % 8 == 0 and 0 < V <= 1 << 18


class _EmbeddingFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ids, weight, padding_idx):
        ctx.save_for_backward(ids)
        ctx.rows, ctx.skip = weight.shape[0], padding_idx
        return torch.nn.functional.embedding(ids, weight, padding_idx)

    @staticmethod
    def backward(ctx, dy):
        from .serving import unseen

        (ids,) = ctx.saved_tensors
        skip = -1 if ctx.skip is None else ctx.skip % ctx.rows
        T, W = ids.numel(), dy.shape[-1]
        if not (unseen(dy, ids) and dy.is_cuda
                and dy.get_device() == torch._C._cuda_getDevice()):
            return None, torch.ops.aten.embedding_dense_backward(
                dy, ids, ctx.rows, skip, False), None
        rows, ids = dy.contiguous(), ids.contiguous()
        if rows.data_ptr() & 15:
            rows = rows.clone()
        out = torch.empty(ctx.rows, W, dtype=dy.dtype, device=dy.device)
        lib = _require_lib()
        work = torch.empty(lib.embedding_work(T, ctx.rows, W), dtype=torch.int32,
                           device=dy.device)
        if lib.embedding_bwd(_ptr(ids), _ptr(rows), _ptr(out), _ptr(work),
                             T, ctx.rows, W, skip, _stream()):
            raise RuntimeError("embedding_bwd failed")
        return None, out, None


def embedding(ids: torch.Tensor, weight: torch.Tensor,
              padding_idx: Optional[int] = None) -> torch.Tensor:
    """``torch.nn.functional.embedding``, with its gradient in one pass over the
    table where that is bf16 and nobody traces or transforms the call."""
    from .serving import _plain, _unwatched

    if torch.is_grad_enabled() and _plain(weight) and _plain(ids) and \
            weight.is_cuda and weight.requires_grad and \
            weight.dtype == torch.bfloat16 and ids.dtype == torch.int64 and \
            weight.dim() == 2 and embedding_rule(ids.numel(), *weight.shape) and \
            _unwatched():
        return _EmbeddingFn.apply(ids, weight, padding_idx)
    return torch.nn.functional.embedding(ids, weight, padding_idx)


# ---------------------------------------------------------------------------
# SwiGLU
# ---------------------------------------------------------------------------

def _swiglu(x: torch.Tensor) -> torch.Tensor:
    I = x.shape[-1] // 2
    if x.is_cuda and x.dtype == torch.bfloat16 and I % 8 == 0:
        lib = _require_lib()
        x2 = x.contiguous()
        N = x2.numel() // x2.shape[-1]
        out = torch.empty(x2.shape[:-1] + (I,), dtype=x2.dtype,
                          device=x2.device)
        lib.swiglu_fwd(_ptr(x2), _ptr(out), ctypes.c_long(N),
                       ctypes.c_int(I), _stream())
        return out
    g, u = x[..., :I].float(), x[..., I:].float()
    return (torch.nn.functional.silu(g) * u).to(x.dtype)


class _SwiGLUFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return _swiglu(x)

    @staticmethod
    def backward(ctx, dy):
        (x,) = ctx.saved_tensors
        I = x.shape[-1] // 2
        if x.is_cuda and x.dtype == torch.bfloat16 and I % 8 == 0:
            lib = _require_lib()
            dy2 = dy.contiguous()
            N = x.numel() // x.shape[-1]
            dx = torch.empty_like(x)
            lib.swiglu_bwd(_ptr(x), _ptr(dy2), _ptr(dx), ctypes.c_long(N),
                           ctypes.c_int(I), _stream())
            return dx
        g, u = x[..., :I].float(), x[..., I:].float()
        dyf = dy.float()
        sig = torch.sigmoid(g)
        s = g * sig
        dg = dyf * u * (sig + s * (1 - sig))
        du = dyf * s
        return torch.cat([dg, du], dim=-1).to(x.dtype)


def swiglu(x: torch.Tensor) -> torch.Tensor:
    """x = [gate; up] on the last dim -> silu(gate)*up."""
    from .serving import unseen

    return _swiglu(x) if unseen(x) else _SwiGLUFn.apply(x)


# ---------------------------------------------------------------------------
# Flash attention (MFMA kernel in csrc/flash_attn.hip)
# ---------------------------------------------------------------------------

def flash_attn_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "flash_attn_fwd")


def _fa_ok_layout(t) -> bool:
    """The flash kernels take any (batch, head, seq) strides with a DENSE
    last dim — transpose views of BSHD activations go in with no copy.  Rows
    are moved in 16-byte words, so the strides are whole numbers of them; 31
    rows are less than 2 GB."""
    b, h, s, d = t.stride()
    if d != 1 or s >= 1 << 25:
        return False
    return not (b | h | s) & 7 or not any(
        st & 7 for st, n in zip((b, h, s), t.shape) if n > 1)


def _fa_operand(t):
    """``t`` in a layout that the kernels take, at a 16-byte boundary."""
    if not _fa_ok_layout(t):
        t = t.contiguous()
    return t.clone() if t.data_ptr() & 15 else t


def _fa_strides(*tensors):
    vals = [st for t in tensors for st in t.stride()[:3]]
    return (ctypes.c_long * len(vals))(*vals)


def _fa_alloc_like(t):
    """Allocate an empty tensor with t's LAYOUT (so a BSHD-view input
    produces a BSHD-view output and the downstream reshape stays a view)."""
    B, H, S, D = t.shape
    if t.stride(1) == D and t.stride(2) == H * D:  # BSHD transpose view
        return torch.empty(B, S, H, D, dtype=t.dtype,
                           device=t.device).permute(0, 2, 1, 3)
    return torch.empty_like(t, memory_format=torch.contiguous_format)


@functools.lru_cache(maxsize=256)         # (1.2 to 4.4 us otherwise)
def _fa_dkv_heads(B: int, Hq: int, Hkv: int, S: int, causal: bool,
                  window: int) -> int:
    """Heads of dK and dV that the kernel writes: a workgroup adds up the q heads
    of one, as many as do not leave CUs idle.  256 workgroups run at a time.  With
    a window, or none of causality, all last as long; else the first block's lasts
    longest and short ones fill the gaps.  Backward, together with delta inside
    the dQ kernel: 2 x 3001 of 32/8 heads, window 1024, in twos: 397 -> 370 us;
    8192 of 32/8, all four: 1823 -> 1790."""
    blocks, rep = -(-S // 128), Hq // Hkv
    even = not causal or 0 < window < S

    def cost(n):
        if even:
            return -(-B * Hq // n * blocks // 256) * n
        return max(n * blocks, B * Hq * blocks * (blocks + 1) / 512)

    return Hq // max((n for n in range(1, rep + 1) if rep % n == 0),
                     key=lambda n: (-cost(n), n))


def _fa_alloc_dkv(k, v, heads):
    """dk/dv as the kernel writes them: in the layout of k and v if they have
    as many heads, else (B,heads,S,D) for ``_fa_sum_replicas``."""
    if heads == k.shape[1]:
        return _fa_alloc_like(k), _fa_alloc_like(v)
    B, _, S, D = k.shape
    return (torch.empty(B, heads, S, D, dtype=k.dtype, device=k.device),
            torch.empty(B, heads, S, D, dtype=v.dtype, device=v.device))


def _fa_sum_replicas(dk_pq, dv_pq, k, v):
    """GQA replicas cover distinct Q heads: 32-bit SUM, in one pass (the
    casts, sums and casts back of both took 137 us where this takes 33, at
    8192 tokens, 32/8 heads)."""
    B, heads, S, _ = dk_pq.shape
    Hkv = k.shape[1]
    if heads == Hkv:
        return dk_pq, dv_pq
    dk, dv = _fa_alloc_like(k), _fa_alloc_like(v)
    _require_lib().flash_attn_bwd_reduce(
        dk_pq.data_ptr(), dv_pq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B,
        heads, Hkv, S, _fa_strides(dk, dv), _stream())
    return dk, dv


class _FlashAttnFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, causal, scale, window=0):
        lib = _require_lib()
        B, Hq, S, D = q.shape
        Hkv = k.shape[1]
        assert D == 128, "flash kernel supports D=128"
        assert q.dtype == torch.bfloat16
        q, k, v = _fa_operand(q), _fa_operand(k), _fa_operand(v)
        out = _fa_alloc_like(q)
        lse = torch.empty(B, Hq, S, dtype=torch.float32, device=q.device)
        lib.flash_attn_fwd_strided(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
            lse.data_ptr(), B, Hq, Hkv, S, scale, 1 if causal else 0,
            window or 0, _fa_strides(q, k, v, out), _stream())
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.causal = causal
        ctx.scale = scale
        ctx.window = window or 0
        return out

    @staticmethod
    def backward(ctx, dout):
        q, k, v, out, lse = ctx.saved_tensors
        lib = _require_lib()
        if not hasattr(lib, "flash_attn_bwd"):
            raise RuntimeError("flash_attn_bwd kernel not built")
        B, Hq, S, D = q.shape
        Hkv = k.shape[1]
        dout = _fa_operand(dout)
        delta = torch.empty(B, Hq, S, dtype=torch.float32, device=q.device)
        # grads are allocated in their producer's LAYOUT so autograd's
        # accumulation into BSHD views stays copy-free
        dq = _fa_alloc_like(q)
        window = getattr(ctx, "window", 0)
        heads = _fa_dkv_heads(B, Hq, Hkv, S, ctx.causal, window)
        dk_pq, dv_pq = _fa_alloc_dkv(k, v, heads)
        lib.flash_attn_bwd_strided(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
            dout.data_ptr(), lse.data_ptr(), delta.data_ptr(), dq.data_ptr(),
            dk_pq.data_ptr(), dv_pq.data_ptr(), B, Hq, Hkv, heads, S,
            ctx.scale, 1 if ctx.causal else 0, window,
            _fa_strides(q, k, v, out, dout, dq, dk_pq, dv_pq), _stream())
        dk, dv = _fa_sum_replicas(dk_pq, dv_pq, k, v)
        return dq, dk, dv, None, None, None


@functools.lru_cache(maxsize=1)
def _native_flash():
    """``_FlashAttnFn`` in csrc/host/flash_autograd.cpp; None where it is not built for
    this torch and these kernels, or does not load: calls are Python's then, on the same
    kernels."""
    from .build import host_lib, host_libs

    why = None
    try:
        lib = host_lib()
        if os.path.exists(lib):
            _require_lib()            # its kernels
            torch.ops.load_library(lib)
            return torch.ops.nxd_host.flash_attention.default
        if host_libs():
            why = f"{host_libs()} built for another torch or from other sources"
    except (OSError, AttributeError) as e:
        why = f"the native autograd library does not load ({e})"
    if why:
        warnings.warn(f"{why}: short attention takes its host up to 1.5 times as long")
    return None


def _fa_native(q, k, v) -> bool:
    """May the native function take these: plain bf16 tensors that nobody traces or
    transforms?  Python's takes the others, and refuses what neither takes."""
    from .serving import _plain, _unwatched

    bf16 = torch.bfloat16
    return q.dtype == k.dtype == v.dtype == bf16 and q.is_cuda and k.is_cuda and \
        v.is_cuda and q.dim() == k.dim() == v.dim() == 4 and \
        q.shape[3] == k.shape[3] == v.shape[3] == 128 and \
        _plain(q) and _plain(k) and _plain(v) and _unwatched()


def flash_attn(q, k, v, causal=True, softmax_scale=None, window=0):
    """q (B,Hq,S,D=128), k/v (B,Hkv,S,D) bf16 on GPU.  window > 0:
    sliding-window causal (Mistral), fwd AND bwd on the MFMA kernels."""
    scale = softmax_scale or 1.0 / math.sqrt(q.shape[-1])
    native = _native_flash()
    if native is not None and _fa_native(q, k, v):
        B, Hq, S, _ = q.shape
        window = int(window or 0)
        return native(q, k, v, bool(causal), scale, window,
                      _fa_dkv_heads(B, Hq, k.shape[1], S, bool(causal), window))
    return _FlashAttnFn.apply(q, k, v, causal, scale, window)


def flash_attn_window_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "flash_attn_fwd_window")


def flash_attn_windowed(q, k, v, window: int, softmax_scale=None):
    """Sliding-window causal flash attention (inference/no-grad): q row i
    attends kv rows [i-window+1, i].  q (B,Hq,S,128), k/v (B,Hkv,S,128)
    bf16; out-of-band tiles are skipped entirely (Mistral-style)."""
    lib = _require_lib()
    B, Hq, S, D = q.shape
    Hkv = k.shape[1]
    assert D == 128 and q.dtype == torch.bfloat16
    scale = softmax_scale or 1.0 / math.sqrt(D)
    q, k, v = (_fa_operand(t.contiguous()) for t in (q, k, v))
    out = torch.empty_like(q)
    lse = torch.empty(B, Hq, S, dtype=torch.float32, device=q.device)
    lib.flash_attn_fwd_window(_ptr(q), _ptr(k), _ptr(v), _ptr(out),
                              _ptr(lse), ctypes.c_int(B), ctypes.c_int(Hq),
                              ctypes.c_int(Hkv), ctypes.c_int(S),
                              ctypes.c_float(scale), ctypes.c_int(window),
                              _stream())
    return out


# ---------------------------------------------------------------------------
# Fused AdamW (ZeRO-1 master-shard update; csrc/adamw.hip)
# ---------------------------------------------------------------------------

def adamw_step(master: torch.Tensor, m: torch.Tensor, v: torch.Tensor,
               grad_bf16: torch.Tensor, param_bf16: torch.Tensor,
               clip: Optional[torch.Tensor], lr: float, beta1: float,
               beta2: float, eps: float, weight_decay: float, step: int):
    """One fused pass: bf16 grad -> fp32 m/v/master update -> bf16 param."""
    lib = _require_lib()
    n = master.numel()
    assert m.numel() == n and v.numel() == n and grad_bf16.numel() == n
    assert grad_bf16.dtype == torch.bfloat16 and param_bf16.dtype == torch.bfloat16
    inv_bc1 = 1.0 / (1.0 - beta1 ** step)
    inv_bc2 = 1.0 / (1.0 - beta2 ** step)
    lib.adamw_step(ctypes.c_long(n), _ptr(master), _ptr(m), _ptr(v),
                   _ptr(grad_bf16), _ptr(param_bf16),
                   _ptr(clip) if clip is not None else None,
                   ctypes.c_float(lr), ctypes.c_float(beta1),
                   ctypes.c_float(beta2), ctypes.c_float(eps),
                   ctypes.c_float(weight_decay), ctypes.c_float(inv_bc1),
                   ctypes.c_float(inv_bc2), _stream())


# ---------------------------------------------------------------------------
# Fused MoE decode (K9 parity; csrc/moe_decode.hip)
# ---------------------------------------------------------------------------

_MOE_MB = 16


def moe_decode_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "moe_decode_glu")


def moe_decode_glu(hidden: torch.Tensor, gate_up_w: torch.Tensor,
                   down_w: torch.Tensor, expert_affinities: torch.Tensor,
                   expert_index: torch.Tensor) -> torch.Tensor:
    """Fused decode MoE (inference): hidden (T,H) bf16, gate_up_w
    (E,H,2I) fused [gate|up], down_w (E,I,H), affinities (T,E) float,
    expert_index (T,k) long -> (T,H) bf16 (TP-partial, like ExpertMLPs).

    Slots (token, expert hit) are grouped per expert into blocks of 16 so
    each block streams its expert's weights once; gather, SwiGLU, affinity
    scaling and the scatter-add all happen inside the two kernels."""
    lib = _require_lib()
    T, H = hidden.shape
    E, _, twoI = gate_up_w.shape
    I = twoI // 2
    assert H % 64 == 0 and I % 64 == 0, (H, I)
    k = expert_index.shape[1]
    dev = hidden.device

    flat_e = expert_index.reshape(-1)
    order = torch.argsort(flat_e, stable=True)
    sorted_e = flat_e[order].to(torch.long)
    sorted_tok = (order // k).to(torch.int32)

    counts = torch.bincount(flat_e, minlength=E)
    blocks_per_e = (counts + _MOE_MB - 1) // _MOE_MB
    nb = int(blocks_per_e.sum().item())
    if nb == 0:
        return hidden.new_zeros(T, H)
    blockbase = torch.cumsum(torch.nn.functional.pad(blocks_per_e, (1, 0)),
                             0)  # (E+1,)
    countbase = torch.cumsum(torch.nn.functional.pad(counts, (1, 0)), 0)

    within = torch.arange(T * k, device=dev) - countbase[sorted_e]
    padded_idx = (blockbase[sorted_e] + within // _MOE_MB) * _MOE_MB + \
        within % _MOE_MB

    slot_token = torch.zeros(nb * _MOE_MB, dtype=torch.int32, device=dev)
    slot_token[padded_idx] = sorted_tok
    aff = torch.zeros(nb * _MOE_MB, dtype=torch.float32, device=dev)
    aff[padded_idx] = expert_affinities.float()[
        sorted_tok.long(), sorted_e]

    block_expert = torch.repeat_interleave(
        torch.arange(E, device=dev), blocks_per_e).to(torch.int32)
    bi = torch.arange(nb, device=dev)
    block_ord = bi - blockbase[block_expert.long()]
    block_len = torch.clamp(counts[block_expert.long()] -
                            _MOE_MB * block_ord, 0, _MOE_MB).to(torch.int32)

    act = torch.empty(nb * _MOE_MB, I, dtype=torch.bfloat16, device=dev)
    out = torch.zeros(T, H, dtype=torch.float32, device=dev)
    hidden = hidden.contiguous()
    gate_up_w = gate_up_w.contiguous()
    down_w = down_w.contiguous()
    lib.moe_decode_glu(_ptr(hidden), _ptr(gate_up_w), _ptr(down_w),
                       _ptr(slot_token), _ptr(block_expert), _ptr(block_len),
                       _ptr(aff), _ptr(act), _ptr(out), nb, H, I, _stream())
    return out.to(hidden.dtype)


# ---------------------------------------------------------------------------
# Skinny-M decode GEMM (csrc/serving/stream_linear.hip)
# ---------------------------------------------------------------------------

def skinny_gemm_available() -> bool:
    from . import serving as sv

    return sv.available()


def skinny_linear(x2: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x2 (M<=32, K) bf16 @ w (N, K)^T -> (M, N) bf16 via the
    weight-streaming kernel, which reads words of 16 bytes: of a K that is no
    multiple of 8, or rows that start elsewhere, it reads a copy."""
    from . import serving as sv

    def words(t):
        t = torch.nn.functional.pad(t, (0, -t.shape[1] % 8))
        if t.stride(1) != 1 or t.stride(0) & 7:
            t = t.contiguous()
        return t.clone() if t.data_ptr() & 15 else t

    return sv.stream_linear(words(x2), words(w))


def use_skinny_linear(inp: torch.Tensor, weight: torch.Tensor,
                      sequence_parallel_enabled: bool = False) -> bool:
    """Is ``skinny_linear`` faster than the library for the rows of ``inp`` (other
    kernels than that may be: ``skinny_or_none``), and
    nobody in its way (autograd, tracing, modes, NXDA_SKINNY_GEMM=0)?"""
    from . import serving as sv

    return not sequence_parallel_enabled and \
        sv.stream_how(inp, weight, rings=False) is not None


def skinny_or_none(inp: torch.Tensor, weight: torch.Tensor,
                   sequence_parallel_enabled: bool = False,
                   glu: bool = False):
    """inp (.., K) @ weight (N, K)^T, or with ``glu`` silu(gate) * up of
    weight = [gate; up], by the weight-streaming kernels where they beat the
    library (a few rows; ``serving.stream_how``), else None."""
    if torch.is_grad_enabled() or sequence_parallel_enabled:
        return None
    from . import serving as sv

    return sv.streamed(inp, weight, glu=glu)


# ---------------------------------------------------------------------------
# Fused decode attention (csrc/decode_attn.hip)
# ---------------------------------------------------------------------------

def decode_attn_available() -> bool:
    lib = _load()
    return lib is not None and hasattr(lib, "decode_attn")


def decode_attn_step(q2: torch.Tensor, k2: torch.Tensor, v2: torch.Tensor,
                     kcache: torch.Tensor, vcache: torch.Tensor,
                     cos: torch.Tensor, sin: torch.Tensor,
                     pos_t: torch.Tensor, Hq: int, Hkv: int,
                     scale: float) -> torch.Tensor:
    """One fused decode-attention step: RoPE(q,k) + cache append at the
    device position ``pos_t`` + flash-decode over the cache + GQA.
    q2 (B, Hq*128), k2/v2 (B, Hkv*128) bf16 pre-rope; kcache/vcache
    (B, Hkv, Smax, 128); cos/sin (Smax, 64) fp32 -> out (B, Hq*128).

    q2/k2/v2 may be row-strided views (e.g. slices of one fused-QKV GEMM
    output): only the last dim must be dense (stride 1)."""
    lib = _require_lib()
    B = q2.shape[0]
    Smax = kcache.shape[2]
    assert Hq // Hkv in (1, 2, 4, 8), "GQA rep must be 1/2/4/8"
    assert cos.dtype == torch.float32 and pos_t.dtype == torch.int64
    assert cos.shape[0] >= Smax, (
        f"RoPE table ({cos.shape[0]}) shorter than KV cache ({Smax})")
    assert q2.stride(1) == 1 and k2.stride(1) == 1 and v2.stride(1) == 1
    assert k2.stride(0) == v2.stride(0)
    rep = Hq // Hkv
    # split-KV workspace (4 splits; see decode_attn.hip) — cached-alloc
    # tensors with static shapes, so the pair of launches is
    # hipGraph-capturable
    part_o = torch.empty(B * Hkv * 4, rep, 128, dtype=torch.float32,
                         device=q2.device)
    part_ml = torch.empty(B * Hkv * 4, rep, 2, dtype=torch.float32,
                          device=q2.device)
    out = torch.empty(B, Hq * 128, dtype=torch.bfloat16, device=q2.device)
    lib.decode_attn(_ptr(q2), _ptr(k2), _ptr(v2), _ptr(kcache), _ptr(vcache),
                    _ptr(cos), _ptr(sin), _ptr(pos_t), _ptr(part_o),
                    _ptr(part_ml), _ptr(out), B, Hq, Hkv,
                    Smax, ctypes.c_float(scale), int(q2.stride(0)),
                    int(k2.stride(0)), _stream())
    return out
