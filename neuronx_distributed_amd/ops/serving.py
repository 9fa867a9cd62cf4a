"""Serving kernels: ragged batches over a paged KV cache and state slots.

Python wrappers of ``libnxd_serving.so`` (``csrc/serving/*.hip``).  They run
on the GPU only — there is no eager substitute, a CPU tensor or a missing
library raises.  Activations and weights are bfloat16, or float32 in the
32-bit mode; the residual stream, attention scores and weights, norms,
gates and recurrent state are 32-bit in both.
"""

import ctypes
import math
import os
from bisect import bisect_left
from dataclasses import dataclass, replace
from functools import lru_cache
from typing import Optional, Sequence, Union

import torch

PAGE_SIZE = 64
MAX_HEAD_DIM = 512          # attention q/k and v size, recurrent q/k size
MAX_LATENT_ROW = 1024       # latents and shared key columns of a cached row
MAX_EXPERTS = 512
MAX_TAPS = 65               # of a short convolution
EXPAND_MIN_TOKENS = 32      # shorter portions attend in the latent space
CHUNK = 256                 # tokens of one chunk of a matrix memory

_LIB = None


def library():
    global _LIB
    if _LIB is None:
        from .build import SERVING_LIB

        if not os.path.exists(SERVING_LIB):
            raise RuntimeError(
                f"{SERVING_LIB} is not built — run "
                "python -m neuronx_distributed_amd.ops.build")
        _LIB = ctypes.CDLL(SERVING_LIB)
    return _LIB


def available() -> bool:
    """Is the library there, with the products of few rows (one that was built
    before they came has none, and layers then use torch's)?"""
    if _LIB is None:
        from .build import SERVING_LIB

        if not os.path.exists(SERVING_LIB):
            return False
    return hasattr(library(), "sv_stream_linear")


def ensure_built():
    """Compile the serving library if it is missing or out of date (and
    nothing else)."""
    from .build import build_group

    build_group("serving", verbose=False)


def _stream():
    # the current stream's handle alone (0.3 us, with the object around it 2.9)
    return ctypes.c_void_p(
        torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice()))


def _p(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _f32(t: torch.Tensor) -> int:
    if not t.is_cuda:
        raise RuntimeError("serving kernels run on the GPU only")
    if t.dtype not in (torch.bfloat16, torch.float32):
        raise TypeError(f"serving kernels take bfloat16 or float32, "
                        f"not {t.dtype}")
    return int(t.dtype == torch.float32)


def _check(status: int, what: str):
    if status:
        raise RuntimeError(f"{what}: launch failed with status {status}")


def _fields(names, ctype):
    return [(n, ctype) for n in names.split()]


class _BranchArgs(ctypes.Structure):
    _fields_ = (_fields("delta coef plus gate", ctypes.c_void_p)
                + _fields("gst", ctypes.c_long)
                + _fields("bias", ctypes.c_void_p)
                + _fields("parts", ctypes.c_long))


class _ResidualNormArgs(ctypes.Structure):
    _fields_ = (_fields("x delta delta2 w1 w2 coef vec x_out h w cat x0 "
                        "index", ctypes.c_void_p)
                + _fields("table", ctypes.c_long)
                + _fields("conv ring singles hc", ctypes.c_void_p)
                + _fields("rows_out W delta_f32 parts groups p_groups taps "
                          "conv_row", ctypes.c_int)
                + _fields("eps scale w_base p_base h_scale", ctypes.c_float)
                + _fields("branches", ctypes.c_int)
                + [("br", _BranchArgs * 2)])


class _StreamArgs(ctypes.Structure):
    _fields_ = (_fields("x", ctypes.c_void_p) + _fields("xst", ctypes.c_long)
                + _fields("w", ctypes.c_void_p) + _fields("wst", ctypes.c_long)
                + _fields("out", ctypes.c_void_p)
                + _fields("T N K", ctypes.c_int)
                + _fields("res delta res_out weight", ctypes.c_void_p)
                + _fields("eps", ctypes.c_float)
                + _fields("row", ctypes.c_void_p) + _fields("rows", ctypes.c_long))


class _WideArgs(ctypes.Structure):
    _fields_ = (_fields("x", ctypes.c_void_p) + _fields("xst", ctypes.c_long)
                + _fields("w", ctypes.c_void_p) + _fields("wst", ctypes.c_long)
                + _fields("out", ctypes.c_void_p)
                + _fields("T N K splits g", ctypes.c_int))


class _ConvArgs(ctypes.Structure):
    _fields_ = (_fields("x", ctypes.c_void_p) + _fields("xst", ctypes.c_long)
                + _fields("w bias out", ctypes.c_void_p)
                + _fields("ost", ctypes.c_long)
                + _fields("ring seg chunks", ctypes.c_void_p)
                + _fields("n_chunks chunk C taps silu add", ctypes.c_int))


class _QkvArgs(ctypes.Structure):
    _fields_ = (_fields("q k v", ctypes.c_void_p)
                + _fields("qst kst vst", ctypes.c_long)
                + _fields("freq qw kw first", ctypes.c_void_p)
                + _fields("fst", ctypes.c_long)
                + _fields("mix kc vc pos seq bt", ctypes.c_void_p)
                + _fields("MB T H G D E rot norm temp_every", ctypes.c_int)
                + _fields("temp_coef eps", ctypes.c_float))


class _ScoreArgs(ctypes.Structure):
    _fields_ = (_fields("temp sink slope gate", ctypes.c_void_p)
                + _fields("gst", ctypes.c_long)
                + _fields("cap", ctypes.c_float))


class _RowsArgs(ctypes.Structure):
    _fields_ = (_fields("q k v", ctypes.c_void_p)
                + _fields("qst kst vst", ctypes.c_long)
                + _fields("kc vc", ctypes.c_void_p)
                + _fields("kcs vcs", ctypes.c_long)
                + _fields("pos seq bt part out", ctypes.c_void_p)
                + _fields("MB rows H G D E splits append window keep",
                          ctypes.c_int)
                + _fields("scale", ctypes.c_float) + [("mod", _ScoreArgs)]
                + _fields("cos sin", ctypes.c_void_p))


class _TilesArgs(ctypes.Structure):
    _fields_ = (_fields("q", ctypes.c_void_p) + _fields("qst", ctypes.c_long)
                + _fields("kc vc kr", ctypes.c_void_p)
                + _fields("kpage khead krow vpage vhead vrow rrow",
                          ctypes.c_long)
                + _fields("gate", ctypes.c_void_p)
                + _fields("gst", ctypes.c_long)
                + _fields("tiles bt out", ctypes.c_void_p)
                + _fields("MB H G D E DS window keep", ctypes.c_int)
                + _fields("scale", ctypes.c_float) + [("mod", _ScoreArgs)])


class _LatentAppendArgs(ctypes.Structure):
    _fields_ = (_fields("q", ctypes.c_void_p)
                + _fields("qst qh", ctypes.c_long)
                + _fields("qr", ctypes.c_void_p)
                + _fields("qrst qrh", ctypes.c_long)
                + _fields("kv", ctypes.c_void_p)
                + _fields("kvst", ctypes.c_long)
                + _fields("w freq cache pos seq bt", ctypes.c_void_p)
                + _fields("MB H R P rot", ctypes.c_int)
                + _fields("eps amp", ctypes.c_float)
                + _fields("pairs", ctypes.c_int))


class _HeadLinearArgs(ctypes.Structure):
    _fields_ = (_fields("x", ctypes.c_void_p)
                + _fields("xst xh", ctypes.c_long)
                + _fields("w out", ctypes.c_void_p)
                + _fields("ost oh", ctypes.c_long)
                + _fields("gate", ctypes.c_void_p)
                + _fields("gst gh", ctypes.c_long)
                + _fields("T H N K", ctypes.c_int))


class _LatentRowsArgs(ctypes.Structure):
    _fields_ = (_fields("q cache pos seq bt part out", ctypes.c_void_p)
                + _fields("MB rows H R P splits window", ctypes.c_int)
                + _fields("scale", ctypes.c_float)
                + _fields("sink", ctypes.c_void_p))


class _LatentStepArgs(ctypes.Structure):
    _fields_ = [("append", _LatentAppendArgs), ("absorb", _HeadLinearArgs),
                ("rows", _LatentRowsArgs), ("values", _HeadLinearArgs)]


class _MoePlanArgs(ctypes.Structure):
    _fields_ = (_fields("z bias idx coef order tiles", ctypes.c_void_p)
                + _fields("T E top tile_rows max_tiles kind groups keep best",
                          ctypes.c_int))


class _MoeGemmArgs(ctypes.Structure):
    _fields_ = (_fields("x", ctypes.c_void_p) + _fields("xst", ctypes.c_long)
                + _fields("w out order tiles", ctypes.c_void_p)
                + _fields("top N K max_tiles", ctypes.c_int)
                + _fields("alpha limit shift", ctypes.c_float)
                + _fields("rows", ctypes.c_int))


class _MemoryArgs(ctypes.Structure):
    _fields_ = (_fields("q k v", ctypes.c_void_p)
                + _fields("qst kst vst", ctypes.c_long)
                + _fields("gates ib fb decay log2_decay S n m seg out",
                          ctypes.c_void_p)
                + _fields("H D E", ctypes.c_int)
                + _fields("gate_cap qscale", ctypes.c_float)
                + _fields("G", ctypes.c_int)
                + _fields("skip z", ctypes.c_void_p)
                + _fields("zst", ctypes.c_long)
                + _fields("cw cb ring", ctypes.c_void_p)
                + _fields("taps C kch qch", ctypes.c_int)
                + _fields("freq", ctypes.c_void_p)
                + _fields("rot", ctypes.c_int)
                + _fields("amp kscale", ctypes.c_float))


class _ChunkArgs(ctypes.Structure):
    _fields_ = ([("a", _MemoryArgs)] + _fields("chunks first", ctypes.c_void_p)
                + _fields("n_chunks n_seg T", ctypes.c_int)
                + _fields("b i c tot cend U N P mst VT KA QA", ctypes.c_void_p)
                + _fields("norm_eps", ctypes.c_float))


# ---------------------------------------------------------------------------
# matrix products with a 32-bit result
# ---------------------------------------------------------------------------

def stream_rule(T: int, N: int, K: int, f32: bool = False,
                glu: bool = False) -> Optional[int]:
    """How T rows x (T, K) meet a large weight (N, K) without rings: 0 every workgroup
    streams its weight rows and all of x, 1 workgroups stay with x in registers,
    None the library's product is as fast.  The library reads weights at 2.5 to
    6 TB/s, by their sizes; the lines were drawn where it was not the faster one
    in 220 sizes (N 8..201088, K 512..28672, 1..32 rows, both results; two are
    left where it is, by 4 and 7%).  Below, us here and the library's.  512
    streaming workgroups, of 16 weight rows each, run at a time:

    - more than one such round: the last must not be nearly empty (13824 x 5120
      of 32 bits, 1 row: 30, 27) and K long enough to be worth a workgroup's
      start (151936 x 896, 1 row: 64, 53).  All of them read x, so streaming
      ends at 4 rows (at 3 of a large weight: 61344 x 3200, 4 rows: 75, 70; at
      one of a long K: 64000 x 7168, 4 rows: 171, 152).  Then staying, for a K
      that gives all 8 waves columns and leaves them registers (54784 x 1536, 8
      rows: 40, 34; 64000 x 7168, 16 rows: 168, 153);
    - one round in which some CUs have a second workgroup: the shorter K, the
      more rows before that shows (5632 x 2048, 12 rows: 9.7, 11.8; 4608 x 3584,
      8 rows: 14.3, 12.2);
    - a workgroup a CU or fewer: of a long K the library takes pieces, which few
      workgroups do not keep up with (1152 x 7168, 1 row: 10, 8.4), and of a
      multiple of 1024 those of one on nearly every CU (3136 x 10240, 4 rows:
      18, 16.7; 4096 x 14336: 24.6, 25.3; 4096 x 11008: 22, 37);
      a gate's weight is too small to share x (64 x 4096 of 32 bits, 4 rows:
      6.7, 5.9), and 16 rows are as much to read as the weight (2048 x 4096 of
      32 bits, 16 rows: 9.4, 8.5);
    - gates: staying takes two and more tiles a CU; with 17..32 rows the library
      is as fast where 5 or 6 of the 8 waves have columns (K = 3072: 35.5, 34).
      Two of 37 sizes are left where it is 5% faster (K = 5120, 25600 gates, 12
      rows on; K = 640, 32 rows)."""
    if glu:
        stay = N % 32 == 0 and K <= 8192 and N // 32 >= 640
        return 1 if stay and (
            T <= 16 or T <= 32 and (K <= 2048 or 3584 < K <= 4096)) else None
    tiles, long = -(-N // 16), K > 4096
    if tiles > 512:
        uneven = f32 or long and tiles <= 1024
        if K < 1536:
            return None
        if tiles >= (441 if uneven else 384) * -(-tiles // 512) and \
                T <= (1 if long else 4 if tiles < 2048 else 3) and \
                not (f32 and long and tiles < 1024):
            return 0
        return 1 if N % 16 == 0 and tiles >= 1024 and 2048 <= K <= 6144 and \
            T <= (4 if f32 and long else 16) else None
    if tiles > 256:
        if tiles < 384:
            most = 12 if K <= 2048 else 4 if K <= 3072 else 0
        elif N * K <= 4096 * 4096:
            most = 16
        else:
            most = 4 if not long else 0 if f32 else 1
    elif N < 512:
        most = 8 if K <= (2048 if f32 else 3072) else \
            4 if not (f32 or long) else 0
    elif long:
        if tiles <= 120:
            most = 4 if K <= 4864 else 0
        elif K % 1024 == 0 and tiles <= 224:
            most = 1
        else:
            most = min(2 if tiles <= 160 and K > 4864 else 4, 4 * 14336 // K)
    else:
        most = 8 if f32 and K > 2048 and N < 2560 else 16
    return 0 if T <= most else None


def ring_rule(T: int, N: int, K: int, f32: bool = False,
              glu: bool = False) -> Optional[int]:
    """The same for weights that come through rings in LDS, whole cache lines of a
    row at a time that no cache keeps: 2 workgroups stay with x in registers, 3 x
    flows too, None neither is the faster one.  Drawn over 982 sizes (N
    512..151936, K 512..28672, 1, 4, 16 and 32 rows) against the faster of the
    library and what ``stream_rule`` takes; us here, that and the rings':

    - x is little up to 8 rows, and read once where a CU has one tile of 16 weight
      rows: there it flows (16 rows of 4096 x 4096: staying 9.4, flowing 8.8);
      elsewhere staying saves its way through the L2 (28672 x 4096 gated, 16 rows:
      flowing 44.0, staying 41.3; 32 rows: 61, 43), but of short rows, whose
      workgroups have begun when x is there (7168 x 1024, 16 rows: 10.2, 9.0);
    - short rows of small weights are streamed with 16 waves a workgroup, which
      begin and end sooner (2048 x 2048, 1 row: 4.7, 5.0; 8192 x 2048: 7.5, 8.7;
      32000 x 2048: 21.8, 23.7; 4096 x 2560, 6 rows 6.5, 7.1), and of 17 rows and
      more are the library's (512 x 768: 5.0, 6.0; 1024 x 896: 5.9, 5.4);
    - 17 rows and more stay in registers up to K = 4096 (not of small weights where
      only 5 blocks of 64 columns a wave cover the start: 6144 x 2560, 32 rows: 11.4,
      12.0), and flow for one tile a CU (4096 x 11008, 32 rows: 31.5, 26.5); else
      the library's are faster (32000 x 5120, 32 rows: 48, 73), as of a K that it
      takes in even pieces (3072 x 14336: 28.6, 30.6)."""
    if K % 64 or K < 512 or glu and N % 32:
        return None
    tiles = -(-N // 16)                  # 256 a round
    if T <= 16:
        if not glu and (T <= 4 and K <= 2048 and (
                N <= 8192 or T == 1 and K > 1536) or
                T == 1 and K <= 3584 and N <= 8192 or
                T <= 8 and K <= 3072 and 2048 < N <= 4096 and
                stream_rule(T, N, K, f32) == 0 or
                T <= 4 and K <= 3072 and N <= 4096 or
                T > 4 and K <= 1536 and N <= 8192):
            return None
        if T <= 8 or tiles <= 256 or K <= 1024 and tiles <= 1024 or \
                K <= 2048 and tiles <= 512:
            return 3
        return 2 if K <= 8192 else None if K >= 14336 else 3
    if tiles <= 512 and K <= 2048:
        return 3 if glu or N > 1024 or K >= 1024 else None
    if K <= 4096:
        return None if N < 1024 or 2048 < K < 3072 and 2048 < N < 8192 else 2
    return None if glu or tiles > 256 or \
        K < 16384 and K % 2048 == 0 and N > 2048 else 3


def wide_rule(T: int, N: int, K: int, f32: bool = False,
              glu: bool = False) -> Optional[int]:
    """Into how many shares of K ``wide_linear`` cuts the product of T rows with a
    weight (N, K), or None where the library or ``stream_how`` is the faster one.
    As many shares as leave no CU without a workgroup of 128 weight rows, of 256
    columns at least; of many rows no more than 16, whose sums are as much to write
    as the weights (1024 x 8192, 128 rows: 14.5 us, by 32 19.3), and of few columns
    no more than for 200 CUs (4096 x 4096, 128 rows: by 8 23.6, 6 21.1); of gates of
    512 columns, and no more than 8 (1024 x 8192, 28 rows: 15.7, by 32 23.8), since
    their merge has half the threads for as many sums.  Drawn over 7200
    calls of 9 to 128 rows, 1.04 to 1.25 times as fast; us here, there and here:

    - up to 32 rows only a K beyond the registers of ``ring_rule`` (4096 x 14336, 17
      rows: 29, 24; fewer than 17 of a very long one: 6144 x 18944, 9 rows 110, 42),
      and weights of many rows;
    - up to 64 rows are the weights'; more are also bound by their way through LDS,
      and the library is faster where rounds of fewer rows a workgroup leave too
      little to each (gated 37888 x 3584, 48 rows: 62.5, 55.0, 100 rows: 72.3, 73.3;
      43008 x 4096, 100 rows: 97.7, 88.2; 50304 x 2560, 112 rows: 70.7, 62.5), and rings up to 32 rows there (34816 x
      4096, 32 rows: 54.0, 56.9; 22016 x 4096, of one round: 36.5, 33.7);
    - short K under few weight rows has too little to hide a merge behind (4096 x
      2048, 40 rows: 9.9, 9.1; 2560 x 3072, 48: 12.5, 10.4, 3584 x 3584, 56: 14.0,
      12.5; 8192 x 3072, 96: 19.2, 21.4), all the more of gates (3072 x 4096 gated, 48
      rows: 17.3, 15.8, 5120 15.3, 16.5), and where the library cuts K evenly (4096 x
      8192 gated, 20 rows: 21.8, 20.2; 1024 x 8192, 128 rows: 16.4, 14.8);
    - 4096 x 4096 is the library's between the batches of captured steps (100 rows:
      19.3, 17.0; 64: 15.9, 15.6; 128: 21.1, 24.8), where a prompt waits for the host,
      whose call of it costs 20 us more."""
    if K % 64 or K < 512 or N % 8 or not 0 < T <= 128 or N <= 0 or glu and N % 32:
        return None
    tiles, many = -(-N // 128), T > 64
    target = 200 if many and not glu and K <= 4096 and tiles <= 64 else 256
    splits = max(1, min(target // tiles, K // (512 if glu else 256),
                        8 if glu else 16 if many else 64))
    idle = 1 - tiles * splits / (256 * -(-tiles * splits // 256))
    if tiles > 256 and (idle > 0.15 if T <= 32 else many and idle > 0.38):
        return None
    if T <= 32:
        if K <= 4096:
            take = T >= 17 and N >= 20000 and K >= 1536
        elif glu and N < 4500:
            take = T >= 17 and (K >= 5120 and K % 8192 > 0 if N >= 2500 else
                                K > 8192 and K % 2048 > 0)
        else:
            take = T >= 17 or T >= 9 and N >= 5120 and (
                K >= 14336 if T < 13 else K >= 11008)
    elif tiles >= 168:
        take = K >= 1536 and (not many or glu or
                              idle < (0.2 if tiles > 256 else 0.3))
    elif N >= 4500:
        take = K >= (4096 if many else 3072)
    elif glu:
        take = K >= (6144 if many and N < 3072 else 5120) if N >= 2500 else \
            K > 8192 and K % 2048 > 0
    elif many:
        take = K >= (8256 if N < 2500 else 7168 if N < 3072 else 4096)
    else:
        take = K >= (4096 if N < 2048 or N >= 3072 else 5120)
    return splits if take else None


def wide_linear(x: torch.Tensor, w: torch.Tensor, splits: int = 1,
                f32: bool = False, glu: bool = False) -> torch.Tensor:
    """As ``stream_linear``, for up to 128 rows, with K in ``splits`` shares."""
    T, K = x.shape
    N = w.shape[0]
    assert x.dtype == w.dtype == torch.bfloat16 and w.shape[1] == K
    assert x.is_cuda and x.stride(1) == 1 and w.stride(1) == 1
    assert _words(x) and _words(w) and not (f32 and glu)
    out = torch.empty(T, N // 2 if glu else N, device=x.device,
                      dtype=torch.float32 if f32 else torch.bfloat16)
    part = torch.empty(splits * T * N, dtype=torch.float32,
                       device=x.device) if splits > 1 else None
    a = _WideArgs(x=x.data_ptr(), xst=x.stride(0), w=w.data_ptr(),
                  wst=w.stride(0), out=out.data_ptr(), T=T, N=N, K=K,
                  splits=splits)
    _check(library().sv_wide_linear(
        ctypes.byref(a), ctypes.c_void_p(_p(part)), 2 if glu else int(f32),
        _stream()), "wide_linear")
    return out


def stream_linear(x: torch.Tensor, w: torch.Tensor, stay: int = 0,
                  f32: bool = False, glu: bool = False) -> torch.Tensor:
    """x (T, K) @ w (N, K)^T, bfloat16, with the sums rounded once or not at
    all (``f32``); ``glu``: silu(gate) * up of w = [gate; up]."""
    T, K = x.shape
    N = w.shape[0]
    assert x.dtype == w.dtype == torch.bfloat16 and w.shape[1] == K
    assert x.is_cuda and x.stride(1) == 1 and w.stride(1) == 1
    assert _words(x) and _words(w) and not (f32 and glu)
    out = torch.empty(T, N // 2 if glu else N, device=x.device,
                      dtype=torch.float32 if f32 else torch.bfloat16)
    a = _StreamArgs(x=x.data_ptr(), xst=x.stride(0), w=w.data_ptr(),
                    wst=w.stride(0), out=out.data_ptr(), T=T, N=N, K=K)
    _check(library().sv_stream_linear(
        ctypes.byref(a), 2 if glu else int(f32), stay, _stream()),
        "stream_linear")
    return out


def _words(t: torch.Tensor) -> bool:
    """Does every row start at a 16-byte word and hold a whole number?"""
    return not (t.stride(0) | t.shape[1]) & 7 and not t.data_ptr() & 15


def _plain(t) -> bool:
    return type(t) in (torch.Tensor, torch.nn.Parameter)


def _few_rows(x: torch.Tensor, w: torch.Tensor, rule) -> Optional[tuple]:
    """(rows of x (..., K), what ``rule`` (T, N, K, far) says of them) for the
    kernels of few rows; None where it says None, under autograd, and where somebody
    else watches the operations (tracing, dispatch modes, autocast).  ``far``: the
    rows are 2^22 elements apart or more.  NXDA_SKINNY_GEMM=0 keeps every product on
    the library."""
    if torch.is_grad_enabled() or not (_plain(x) and _plain(w)) or \
            not x.is_cuda:
        return None
    shape, size = x.shape, w.shape
    if len(shape) < 2 or len(size) != 2:
        return None
    K = shape[-1]
    T = shape[0] if len(shape) == 2 else x.numel() // K if K else 0
    if not 0 < T <= 128 or not K or K != size[1] or not size[0] or \
            x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or \
            w.stride(1) != 1 or \
            x.get_device() != torch._C._cuda_getDevice() or \
            w.get_device() != x.get_device() or \
            os.environ.get("NXDA_SKINNY_GEMM", "1") != "1":
        return None
    how = rule(T, size[0], K, False)
    if how is None or not available() or not _unwatched():
        return None
    rows = x if len(shape) == 2 else x.reshape(T, K)
    if rows.stride(0) >= 1 << 22:        # (of the last tokens of long prompts)
        how = rule(T, size[0], K, True)
        if how is None:
            return None
    if rows.stride(1) != 1 or not (_words(rows) and _words(w)):
        return None
    return rows, how


def _near(w: torch.Tensor) -> bool:
    """Are all offsets in w bytes of 31 bits, also a tile past its end (and the
    kernels there that count on it)?"""
    return w.stride(0) * (w.shape[0] + 128) < 1 << 30 and \
        hasattr(library(), "sv_wide_linear")


def stream_how(x: torch.Tensor, w: torch.Tensor, f32: bool = False,
               glu: bool = False, rings: bool = True) -> Optional[int]:
    """How ``stream_linear`` takes the rows of x (..., K) where it is the faster
    one (by ``ring_rule``, if ``rings``, or ``stream_rule``); else None."""
    def rule(T, N, K, far):
        if T > 32:
            return None
        how = ring_rule(T, N, K, f32, glu) if rings and available() and \
            _near(w) else None
        return stream_rule(T, N, K, f32, glu) if how is None else how

    took = _few_rows(x, w, rule)
    return took and took[1]


def streamed(x: torch.Tensor, w: torch.Tensor, f32: bool = False,
             glu: bool = False) -> Optional[torch.Tensor]:
    """The product of the rows of x (..., K) by ``wide_linear`` where
    ``wide_rule`` takes it, or ``stream_linear`` by ``stream_how``, or None."""
    def rule(T, N, K, far):
        near = available() and _near(w)
        splits = wide_rule(T, N, K, f32, glu) if near and not far else None
        if splits is not None:
            return True, splits
        how = None
        if T <= 32:
            how = ring_rule(T, N, K, f32, glu) if near else None
            if how is None:
                how = stream_rule(T, N, K, f32, glu)
        return None if how is None else (False, how)

    took = _few_rows(x, w, rule)
    if took is None:
        return None
    rows, (wide, how) = took
    out = wide_linear(rows, w, how, f32, glu) if wide else \
        stream_linear(rows, w, how, f32, glu)
    return out if x.dim() == 2 else out.view(*x.shape[:-1], -1)


def _unwatched() -> bool:
    return not (torch.jit.is_tracing() or torch.compiler.is_compiling()
                or torch.is_autocast_enabled("cuda")
                or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack()
                or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def unseen(*tensors) -> bool:
    """May a call on these go past its autograd function: nobody differentiates,
    traces or transforms it?"""
    if torch.is_grad_enabled():
        return False
    for t in tensors:
        if t is not None and not _plain(t):
            return False
    return _unwatched()


def linear_f32(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """x (T, K) @ w (N, K)^T with a float32 result (no rounding to the
    activation type): gate logits, vocabulary logits, residual projections."""
    if x.dtype == torch.float32:
        return torch.mm(x, w.t())
    out = streamed(x, w, f32=True)
    return torch.mm(x, w.t(), out_dtype=torch.float32) if out is None else out


# ---------------------------------------------------------------------------
# residual + norm
# ---------------------------------------------------------------------------

@dataclass
class Pending:
    """A sublayer result that has not been added to the residual yet: one
    tensor, or two branches that are RMS-normed with their own weights and
    summed; ``scale`` times that.  One tensor is RMS-normed when ``w1`` is
    given, over ``groups`` equal parts each.  ``coef`` (rows, parts) makes a row the weighted sum of ``parts``
    rows of ``delta`` (rows * parts, W).  ``centred``: w1 and w2 are stored as
    their distance from one.  ``vec`` is a row added to every token.  Instead
    of ``delta``, up to two gated ``branches`` may be pending.  ``rows``: delta is
    a table, of which these rows (int32) are pending, and nothing else is."""
    delta: Optional[torch.Tensor] = None
    delta2: Optional[torch.Tensor] = None
    w1: Optional[torch.Tensor] = None
    w2: Optional[torch.Tensor] = None
    scale: float = 1.0
    vec: Optional[torch.Tensor] = None
    coef: Optional[torch.Tensor] = None
    centred: bool = False
    groups: int = 1
    branches: Sequence["Branch"] = ()
    rows: Optional[torch.Tensor] = None

    def count(self) -> int:
        """Of rows of one pending tensor."""
        return (self.delta if self.rows is None else self.rows).shape[0]


@dataclass
class Branch:
    """A gated sublayer result: the rows of ``delta``, or with ``coef`` (rows,
    parts) their weighted sums; plus ``plus`` (rows, W); times sigmoid(gate +
    bias) of ``gate`` (rows, W) and ``bias`` (W,)."""
    delta: torch.Tensor
    coef: Optional[torch.Tensor] = None
    plus: Optional[torch.Tensor] = None
    gate: Optional[torch.Tensor] = None
    bias: Optional[torch.Tensor] = None

    @property
    def rows(self) -> int:
        return (self.delta if self.coef is None else self.coef).shape[0]

    def args(self, rows: int, W: int, dtype) -> _BranchArgs:
        parts = 1 if self.coef is None else self.coef.shape[1]
        assert self.delta.shape == (rows * parts, W)
        assert self.delta.is_contiguous() and self.delta.dtype == dtype
        a = _BranchArgs(delta=_p(self.delta), parts=parts)
        if self.coef is not None:
            assert self.coef.shape[0] == rows and self.coef.is_contiguous()
            assert self.coef.dtype == torch.float32
            a.coef = _p(self.coef)
        if self.plus is not None:
            assert self.plus.shape == (rows, W) and self.plus.dtype == dtype
            assert self.plus.is_contiguous()
            a.plus = _p(self.plus)
        if self.gate is not None:
            assert self.gate.shape == (rows, W) and self.gate.dtype == dtype
            assert self.gate.stride(1) == 1
            a.gate, a.gst = _p(self.gate), self.gate.stride(0)
        if self.bias is not None:
            assert self.bias.shape == (W,) and self.bias.dtype == dtype
            assert self.gate is not None and self.bias.is_contiguous()
            a.bias = _p(self.bias)
        return a


@dataclass
class ShortConv:
    """A causal convolution over time, one filter a channel, with the last
    inputs of every request: ``ring`` (slots, taps, C) holds the input at
    position p in place p % taps."""
    w: torch.Tensor            # (taps, C); the last row weighs the token itself
    ring: torch.Tensor
    bias: Optional[torch.Tensor] = None

    def check(self, C, dtype):
        assert self.w.shape[1] == C and self.w.is_contiguous()
        assert self.ring.shape[1:] == self.w.shape
        assert self.ring.is_contiguous() and self.w.shape[0] <= MAX_TAPS
        assert self.w.dtype == self.ring.dtype == dtype
        assert self.bias is None or (self.bias.shape == (C,)
                                     and self.bias.dtype == dtype)


def short_conv(x, conv: ShortConv, seg, chunks, silu: bool = False,
               add: bool = False,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Convolve the rows of prompt portions x (T, C) and keep their last
    inputs: silu(y), or x + y, of y = bias + conv(x).  ``seg`` lists the
    portions (slot, first row, rows, context), ``chunks`` is the device form of
    ``chunk_table``."""
    T, C = x.shape
    conv.check(C, x.dtype)
    assert x.stride(1) == 1
    out = _out(out, T, C, x)
    a = _ConvArgs(x=_p(x), xst=x.stride(0), w=_p(conv.w), bias=_p(conv.bias),
                  out=_p(out), ost=C, ring=_p(conv.ring), seg=_p(seg),
                  chunks=_p(chunks), n_chunks=chunks.shape[0], chunk=CHUNK,
                  C=C, taps=conv.w.shape[0], silu=int(silu), add=int(add))
    _check(library().sv_short_conv(ctypes.byref(a),
                                   int(_aligned((C,), x, out)), _f32(x),
                                   _stream()), "short_conv")
    return out


def _plain_norm(x, pending, eps, weight, index, centred, scale):
    """``residual_norm`` of one tensor or sum that is neither normed nor gated, as
    between a decoder's products: the same with fewer questions."""
    d, coef = pending.delta, pending.coef
    rows, W = d.shape
    parts = table = 0
    if pending.rows is not None:
        assert index is None and x is None and coef is None
        index, table = pending.rows, rows
        assert index.dtype == torch.int32 and index.is_contiguous() \
            and index.is_cuda
    if coef is not None:
        assert coef.is_contiguous() and coef.dtype == torch.float32
        assert coef.numel() == rows and d.dtype == weight.dtype
        rows, parts = coef.shape
    dtype = weight.dtype
    f32 = _f32(d) if dtype == torch.float32 else 0
    assert d.is_contiguous() and d.dtype in (dtype, torch.float32)
    out_rows = rows if index is None else index.shape[0]
    x_new = torch.empty(out_rows, W, dtype=torch.float32, device=d.device)
    h = torch.empty(out_rows, W, dtype=dtype, device=d.device)
    a = _ResidualNormArgs(
        x=_p(x), delta=d.data_ptr(), coef=_p(coef), x_out=x_new.data_ptr(),
        h=h.data_ptr(), w=weight.data_ptr(), index=_p(index),
        table=table, rows_out=out_rows, W=W, parts=parts, groups=1, p_groups=1,
        eps=eps, scale=pending.scale, w_base=centred, p_base=pending.centred,
        h_scale=scale,
        delta_f32=not f32 and d.dtype == torch.float32)
    _check(library().sv_residual_norm(ctypes.byref(a), f32, _stream()),
           "residual_norm")
    return x_new, h, None


def residual_norm(x: Optional[torch.Tensor], pending: Optional[Pending],
                  eps: float, weight: Optional[torch.Tensor] = None,
                  x0: Optional[torch.Tensor] = None, keep_x: bool = True,
                  index: Optional[torch.Tensor] = None, dtype=None,
                  centred: bool = False, copy: bool = False, groups: int = 1,
                  scale: float = 1.0, conv: Optional[ShortConv] = None,
                  batch=None):
    """Add ``pending`` to the float32 residual ``x`` (None: zero) and return
    (new x or None, RMS-normed row * weight or None, [new x; x0] or None).
    ``centred``: the weight is stored as its distance from one.  ``copy``: the
    second result is the new x itself, rounded to ``dtype``.  ``groups``: every
    one of so many equal parts is normed on its own.  ``scale`` multiplies the
    second result.  ``conv``: the second result is h + conv(h) of the rows h of
    ``batch``."""
    if x0 is None and keep_x and conv is None and not copy and \
            pending is not None and weight is not None and groups == 1 and \
            not (dtype or pending.branches or pending.delta2 is not None or
                 pending.w1 is not None or pending.vec is not None or
                 pending.groups != 1):
        return _plain_norm(x, pending, eps, weight, index, centred, scale)
    assert pending is None or pending.rows is None
    branches = () if pending is None else pending.branches
    src = x if pending is None else \
        branches[0].delta if branches else pending.delta
    rows, W = src.shape
    if branches:
        assert pending.delta is None and pending.coef is None and \
            pending.w1 is None and len(branches) <= 2
        rows = branches[0].rows
        assert x is None or x.shape == (rows, W)
    if pending is not None and pending.coef is not None:
        assert pending.coef.is_contiguous() and \
            pending.coef.dtype == torch.float32
        assert pending.delta2 is None and \
            pending.coef.numel() == rows
        rows = pending.coef.shape[0]
    dtype = dtype or (weight if weight is not None else x0).dtype
    f32 = _f32(src) if dtype == torch.float32 else 0
    out_rows = rows if index is None else index.shape[0]
    dev = src.device
    x_new = torch.empty(out_rows, W, dtype=torch.float32, device=dev) \
        if keep_x else None
    h = torch.empty(out_rows, W, dtype=dtype, device=dev) \
        if weight is not None or copy else None
    cat = torch.empty(out_rows, 2 * W, dtype=dtype, device=dev) \
        if x0 is not None else None
    a = _ResidualNormArgs(rows_out=out_rows, W=W, eps=eps, groups=groups,
                          p_groups=1, h_scale=scale)
    a.x, a.x_out, a.h, a.w = _p(x), _p(x_new), _p(h), _p(weight)
    a.cat, a.x0, a.index = _p(cat), _p(x0), _p(index)
    a.w_base, a.scale = float(centred), 1.0
    for i, b in enumerate(branches):
        a.br[i] = b.args(rows, W, dtype)
    a.branches = len(branches)
    if pending is not None and pending.vec is not None:
        a.vec = _p(pending.vec)
    if pending is not None and not branches:
        d = pending.delta
        assert d.is_contiguous() and d.dtype in (dtype, torch.float32)
        assert pending.delta2 is None or (
            d.dtype == dtype and pending.delta2.is_contiguous()
            and pending.delta2.shape == d.shape)
        a.delta, a.delta2 = _p(d), _p(pending.delta2)
        a.w1, a.w2 = _p(pending.w1), _p(pending.w2)
        a.coef, a.scale = _p(pending.coef), pending.scale
        a.p_groups = pending.groups
        assert pending.groups == 1 or (pending.w1 is not None
                                       and pending.delta2 is None)
        if pending.coef is not None:
            a.parts = pending.coef.shape[1]
            assert d.dtype == dtype
        a.p_base = float(pending.centred)
        a.delta_f32 = int(d.dtype == torch.float32 and
                          dtype != torch.float32)
    hc = None
    if conv is not None:
        assert weight is not None and index is None
        conv.check(W, dtype)
        hc = torch.empty_like(h)
        n = batch.portion_tokens
        assert out_rows - n == batch.singles.shape[0] and conv.bias is None
        a.conv, a.ring, a.hc = _p(conv.w), _p(conv.ring), _p(hc)
        a.singles, a.taps, a.conv_row = _p(batch.singles), conv.w.shape[0], n
    _check(library().sv_residual_norm(ctypes.byref(a), f32, _stream()),
           "residual_norm")
    if hc is not None:
        if n:
            short_conv(h[:n], conv, batch.portions, batch.chunks, add=True,
                       out=hc[:n])
        h = hc
    return x_new, h, cat


def gated_norm(o: torch.Tensor, weight: Optional[torch.Tensor],
               gate: Optional[torch.Tensor], group: int,
               eps: float, silu: bool = False,
               out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """o (T, N): every ``group`` elements divided by their root mean square,
    times weight (N,) if there is one, times sigmoid(gate (T, N)), or
    silu(gate), if there is a gate.  ``out`` may be o."""
    T, N = o.shape
    assert N % group == 0 and o.is_contiguous()
    out = _out(out, T, N, o)
    vec4 = int(group % 4 == 0)
    if gate is not None:
        assert gate.shape == o.shape and gate.stride(1) == 1
        vec4 = int(vec4 and gate.stride(0) % 4 == 0
                   and gate.storage_offset() % 4 == 0)
    _check(library().sv_gated_norm(
        ctypes.c_void_p(_p(o)), ctypes.c_void_p(_p(weight)),
        ctypes.c_void_p(_p(gate)),
        ctypes.c_long(0 if gate is None else gate.stride(0)),
        ctypes.c_void_p(_p(out)), T, N // group, group, ctypes.c_float(eps),
        int(silu), vec4, _f32(o), _stream()), "gated_norm")
    return out


def poly_norm(x: torch.Tensor, act: torch.Tensor, eps: float) -> torch.Tensor:
    """x (T, n) -> a N(x) + b N(x^2) + c N(x^3) + e of act = (a, b, c, e),
    powers element by element; N divides a row by its root mean square."""
    T, n = x.shape
    assert x.stride(1) == 1 and act.shape == (4,) and act.is_contiguous()
    assert act.dtype == x.dtype
    out = torch.empty(T, n, dtype=x.dtype, device=x.device)
    _check(library().sv_poly_norm(
        ctypes.c_void_p(_p(x)), ctypes.c_long(x.stride(0)),
        ctypes.c_void_p(_p(act)), ctypes.c_void_p(_p(out)), T, n,
        ctypes.c_float(eps), _vec4((n,), x), _f32(x), _stream()),
        "poly_norm")
    return out


def silu_mul(x: torch.Tensor) -> torch.Tensor:
    """x (T, 2 n) = [gate | up] -> silu(gate) * up (T, n)."""
    T, n = x.shape[0], x.shape[1] // 2
    assert x.stride(1) == 1 and x.shape[1] == 2 * n
    out = torch.empty(T, n, dtype=x.dtype, device=x.device)
    _check(library().sv_silu_mul(
        ctypes.c_void_p(_p(x)), ctypes.c_long(x.stride(0)),
        ctypes.c_void_p(_p(out)), T, n, _vec4((n,), x), _f32(x),
        _stream()), "silu_mul")
    return out


def relu_squared_(x: torch.Tensor) -> torch.Tensor:
    assert x.is_contiguous()
    _check(library().sv_relu_squared(ctypes.c_void_p(_p(x)),
                                     ctypes.c_long(x.numel()), _f32(x),
                                     _stream()), "relu_squared")
    return x


def gelu_tanh_(x: torch.Tensor) -> torch.Tensor:
    assert x.is_contiguous()
    _check(library().sv_gelu_tanh(ctypes.c_void_p(_p(x)),
                                  ctypes.c_long(x.numel()), _f32(x),
                                  _stream()), "gelu_tanh")
    return x


def gelu_rows_(x: torch.Tensor, table: torch.Tensor, tokens: torch.Tensor,
               at: int) -> torch.Tensor:
    """x (T, n) <- gelu(x), in its tanh form, times the columns [at, at + n)
    of table (vocab, columns) in the rows ``tokens`` (T,) int32."""
    T, n = x.shape
    assert x.is_contiguous() and table.stride(1) == 1
    assert x.dtype == table.dtype and 0 <= at <= table.shape[1] - n
    assert tokens.dtype == torch.int32 and tokens.shape == (T,)
    _check(library().sv_gelu_rows(
        ctypes.c_void_p(_p(x)), ctypes.c_void_p(_p(table)),
        ctypes.c_long(table.stride(0)), ctypes.c_void_p(_p(tokens)),
        ctypes.c_long(T), n, at, _f32(x), _stream()), "gelu_rows")
    return x


def softcap_(x: torch.Tensor, cap: float) -> torch.Tensor:
    assert x.is_contiguous() and x.dtype == torch.float32 and x.is_cuda
    _check(library().sv_softcap(ctypes.c_void_p(_p(x)),
                                ctypes.c_long(x.numel()),
                                ctypes.c_float(cap), _stream()), "softcap")
    return x


# ---------------------------------------------------------------------------
# paged attention
# ---------------------------------------------------------------------------

def _aligned(sizes, *tensors) -> bool:
    """Can rows be read in 16-byte pieces of 8 bf16 (or 2 x 4 f32)?"""
    return not _low_bits(sizes, tensors) & 7


def _vec4(sizes, *tensors) -> int:
    return int(not _low_bits(sizes, tensors) & 3)


def _low_bits(sizes, tensors) -> int:
    bits = 0
    for s in sizes:
        bits |= s
    for t in tensors:
        bits |= t.stride(0) | t.storage_offset()
    return bits


def _check_cache(q, k, v, kc, vc, H):
    n, G, page, D = kc.shape
    m, g, size, E = vc.shape
    assert n == m and G == g and page == size == PAGE_SIZE
    assert kc.is_contiguous() and vc.is_contiguous() and H % G == 0
    assert q.shape[1] == H * D and k.shape[1] == G * D and \
        v.shape[1] == G * E
    assert q.stride(1) == k.stride(1) == v.stride(1) == 1
    assert q.dtype == k.dtype == v.dtype == kc.dtype == vc.dtype
    if max(D, E) > MAX_HEAD_DIM:
        raise ValueError(f"head size {max(D, E)} > {MAX_HEAD_DIM}")
    return G, D, E


def _out(out, rows, cols, like):
    if out is None:
        return torch.empty(rows, cols, dtype=like.dtype, device=like.device)
    assert out.shape == (rows, cols) and out.is_contiguous() and \
        out.dtype == like.dtype
    return out


def kv_append(k, v, kc, vc, pos, seq, block_table):
    """Write k (T, G*D) and v (T, G*E) at positions ``pos`` of the requests
    ``seq`` (int32, row of the block table)."""
    G, D, E = kc.shape[1], kc.shape[3], vc.shape[3]
    T = k.shape[0]
    assert pos.shape[0] == T and seq.shape[0] == T
    _check(library().sv_kv_append(
        ctypes.c_void_p(_p(k)), ctypes.c_void_p(_p(v)),
        ctypes.c_long(k.stride(0)), ctypes.c_long(v.stride(0)),
        ctypes.c_void_p(_p(kc)), ctypes.c_void_p(_p(vc)),
        ctypes.c_void_p(_p(pos)), ctypes.c_void_p(_p(seq)),
        ctypes.c_void_p(_p(block_table)), block_table.shape[1], T, G, D, E,
        int(_aligned((D, E), k, v)), _f32(k), _stream()), "kv_append")


@dataclass
class QkvPrep:
    """What happens to queries, keys and values before they are attended and
    cached: the first elements of a head turn in neighbouring pairs, queries
    and keys are RMS-normed a head, queries grow with their position, values
    take a share of another layer's."""
    freq: Optional[torch.Tensor] = None    # (dims / 2,) float64 rad a position
    norm: bool = False
    q_norm: Optional[torch.Tensor] = None  # (D,) weights of the norm
    k_norm: Optional[torch.Tensor] = None
    eps: float = 0.0
    temp_coef: float = 0.0                 # q *= 1 + coef ln(floor((p + 1) /
    temp_every: int = 0                    #   every) + 1), if every > 0
    first: Optional[torch.Tensor] = None   # (T, G * E)
    mix: Optional[torch.Tensor] = None     # one number: v + mix (first - v)


@dataclass
class ScoreMod:
    """Of the scores s = q.k scale and their softmax: s *= temp[h];
    s = cap tanh(s / cap); s -= slope[h] distance; exp(sink[h]) joins the
    denominator; the output is multiplied by sigmoid(gate[row, h])."""
    temp: Optional[torch.Tensor] = None    # (H,)
    cap: float = 0.0
    slope: Optional[torch.Tensor] = None   # (H,) float32
    sink: Optional[torch.Tensor] = None    # (H,)
    gate: Optional[torch.Tensor] = None    # (T, H)

    def rows(self, a, b):
        """The same for rows [a, b) of the batch."""
        return self if self.gate is None else replace(self,
                                                      gate=self.gate[a:b])


def _score_args(mod: Optional[ScoreMod], q, H) -> _ScoreArgs:
    if mod is None:
        return _ScoreArgs()
    for t in (mod.temp, mod.sink):
        assert t is None or (t.shape == (H,) and t.dtype == q.dtype
                             and t.is_cuda and t.is_contiguous())
    assert mod.slope is None or (mod.slope.shape == (H,) and mod.slope.is_cuda
                                 and mod.slope.dtype == torch.float32)
    a = _ScoreArgs(temp=_p(mod.temp), sink=_p(mod.sink), slope=_p(mod.slope),
                   cap=mod.cap)
    if mod.gate is not None:
        assert mod.gate.shape == (q.shape[0], H) and mod.gate.stride(1) == 1
        assert mod.gate.dtype == q.dtype
        a.gate, a.gst = _p(mod.gate), mod.gate.stride(0)
    return a


def qkv_append(q, k, v, kc, vc, pos, seq, block_table, heads: int,
               prep: QkvPrep):
    """Prepare q (T, H*D) in place and write the prepared k and v at positions
    ``pos`` of the requests ``seq``."""
    G, D, E = _check_cache(q, k, v, kc, vc, heads)
    T = q.shape[0]
    assert pos.shape[0] == seq.shape[0] == T
    a = _QkvArgs(q=_p(q), k=_p(k), v=_p(v), qst=q.stride(0), kst=k.stride(0),
                 vst=v.stride(0), kc=_p(kc), vc=_p(vc), pos=_p(pos),
                 seq=_p(seq), bt=_p(block_table), MB=block_table.shape[1],
                 T=T, H=heads, G=G, D=D, E=E, norm=int(prep.norm),
                 temp_every=prep.temp_every, temp_coef=prep.temp_coef,
                 eps=prep.eps)
    tensors = [q, k, v]
    if prep.freq is not None:
        assert prep.freq.dtype == torch.float64 and prep.freq.is_cuda
        a.freq, a.rot = _p(prep.freq), 2 * prep.freq.shape[0]
    for name, w in (("qw", prep.q_norm), ("kw", prep.k_norm)):
        if w is not None:
            assert w.shape == (D,) and w.dtype == q.dtype and prep.norm
            setattr(a, name, _p(w))
    if prep.first is not None:
        f = prep.first
        assert f.shape == v.shape and f.stride(1) == 1 and f.dtype == v.dtype
        assert prep.mix.numel() == 1 and prep.mix.dtype == v.dtype
        a.first, a.fst, a.mix = _p(f), f.stride(0), _p(prep.mix)
        tensors.append(f)
    _check(library().sv_qkv_append(
        ctypes.byref(a), int(_aligned((D, E), *tensors)), _f32(q), _stream()),
        "qkv_append")


def _row_splits(target: int, units: int, max_keys: int, per: int) -> int:
    """Workgroups that share a row: enough for ``target`` of them, each with
    about ``per`` keys or more."""
    return max(1, min(target // max(1, units), -(-max_keys // per), 64))


# Workgroups of the first form of ``rows_kernel`` to aim at, where up to so many
# (row, key head) meet keys up to 256, 700, 1200, 2500, 5000 and more; 0 shares
# no row.  One a CU (256) or less while rows are short: more meet on one CU and
# read no faster.  Longer rows fill all 512 places, and of many rows there are
# several rounds, so that unequal ones end together; up to 320 leave few CUs
# with a second workgroup, which all wait for.  Over 1100 sizes of 1 to 128 rows
# of 32/32, 32/8 and 28/4 heads of 128 and 64, up to 12000 keys, equal and
# unequal, 2.4% over the best number, where 1024 to 2048 above 700 keys were
# 8.6% (us then and now: 8 rows of 32/8 heads, 4000 keys 26.4, 21.3; 32, 1000:
# 26.6, 18.8; 32 of up to 4096, in eight and in four 62.5, 61.5; 64, 2000: 54.0,
# 52.8; 128 rows of 28/4, 1000: 37.5, 28.4).  Equal rows of a few more than 256
# are up to 12% over it between 700 and 1200 keys (34 of 16/8, 1195: 33.0,
# 37.1), where unequal ones gain as much.
_SHARED_KEYS = (256, 700, 1200, 2500, 5000)
_SHARED_UNITS = (64, 128, 256, 320)
_SHARED_ROWS = ((0, 256, 256, 256, 512, 512), (0, 512, 512, 512, 512, 768),
                (0, 0, 0, 512, 1024, 2048), (0, 0, 0, 1024, 2048, 2048),
                (0, 0, 0, 0, 2048, 2048))


@lru_cache(maxsize=1024)
def rows_kernel(rows: int, heads: int, groups: int, D: int, max_keys: int,
                modified: bool = False):
    """Form (2 on matrix cores, 1 on vectors) and workgroups a row of
    ``attn_rows``, for bf16 heads of D = 64 or 128.  Of the first form 512
    workgroups run at a time, each for one key head of a row, and each takes 4
    to 7 us: with more of them, heads to themselves or in pairs, and short
    contexts the second is the faster one (64 rows of 32/32 heads of 128, 64
    keys: 18 and 12 us, 200: 26 and 23; 128 of 32/16, 64: 18.5 and 16.6; 128 of
    32/32 of 64, 20: 14.2 and 12.6; 32 of 32/32 with modified scores, 100: 12.4
    and 11.5).  Over 2300 sizes 0.65 of the second form's time; up to 8% over it
    are left with modified scores of heads to themselves (96 rows of 16/16 of 64,
    300 keys: 16.6 and 15.8).

    Sharing a row costs a merge, and partial results: ``_SHARED_ROWS``."""
    units, rep = rows * groups, heads // groups
    if D == 64:
        short = 64 if rep == 1 and units > (1024 if modified else 2048) else 0
    elif rep == 1:
        short = 200 if modified or units > 1024 else 64
    else:
        short = 0 if rep > 2 else \
            100 if units > (1024 if modified else 2048) else 64
    if units > 512 and 0 < max_keys <= short:
        return 1, _row_splits(1024, units, max_keys, 128)
    target = _SHARED_ROWS[bisect_left(_SHARED_UNITS, units)][
        bisect_left(_SHARED_KEYS, max_keys)]
    return 2, _row_splits(target, units, max_keys, 128)


def attn_rows(q, k, v, kc, vc, pos, seq, block_table, heads: int,
              scale: float, window: int = 0, keep: int = 0,
              append: bool = True, max_keys: int = 0,
              out: Optional[torch.Tensor] = None,
              mod: Optional[ScoreMod] = None,
              rotary=None) -> torch.Tensor:
    """One query row per request row: decoding.  ``append`` also writes the
    row's own k/v into the cache (without it they must be there already).
    ``max_keys`` bounds the visible keys of any row (it only chooses the kernel
    and how many workgroups share a row).  ``rotary`` (cos, sin) as in
    ``rope_rows_``, in the kernel where it has a form for that, else in place."""
    G, D, E = _check_cache(q, k, v, kc, vc, heads)
    rows = q.shape[0]
    assert pos.shape[0] == rows and seq.shape[0] == rows
    if rotary is not None:
        _check_rotary(*rotary, q, k, pos, D, max_keys)
    if window > 0:
        max_keys = min(max_keys, window + keep) if max_keys else window + keep
    vec = int(_aligned((D, E), q, k, v))
    if vec and q.dtype == torch.bfloat16 and D == E and D in (64, 128):
        vec, splits = rows_kernel(rows, heads, G, D, max_keys,
                                  mod is not None)
    else:
        splits = _row_splits(1024, rows * G, max_keys, 128)
    if rotary is not None and (vec != 2 or mod is not None or not append or
                               any(t.data_ptr() & 15 for t in rotary)):
        rope_rows_(q, k, *rotary, pos, D, 0)
        rotary = None
    out = _out(out, rows, heads * E, q)
    part = torch.empty(rows * heads * splits * (E + 2), dtype=torch.float32,
                       device=q.device) if splits > 1 else None
    a = _RowsArgs(q=_p(q), k=_p(k), v=_p(v), qst=q.stride(0),
                  kst=k.stride(0), vst=v.stride(0), kc=_p(kc), vc=_p(vc),
                  kcs=D, vcs=E,
                  pos=_p(pos), seq=_p(seq), bt=_p(block_table),
                  part=_p(part), out=_p(out), MB=block_table.shape[1],
                  rows=rows, H=heads, G=G, D=D, E=E, splits=splits,
                  append=int(append), window=window, keep=keep, scale=scale)
    if mod is not None:
        a.mod = _score_args(mod, q, heads)
    if rotary is not None:
        a.cos, a.sin = map(_p, rotary)
    _check(library().sv_attn_rows(ctypes.byref(a), vec, _f32(q), _stream()),
           "attn_rows")
    return out


def attn_tiles_supported(q, kc, vc) -> bool:
    D, E = kc.shape[3], vc.shape[3]
    return (q.dtype == torch.bfloat16 and max(D, E) <= 256
            and _aligned((D, E), q))


def attn_portions(q, k, v, kc, vc, pos, seq, block_table, tiles, heads: int,
                  scale: float, window: int = 0, keep: int = 0,
                  append: bool = True, max_keys: int = 0,
                  out: Optional[torch.Tensor] = None,
                  mod: Optional[ScoreMod] = None) -> torch.Tensor:
    """Prompt portions: append k/v (unless they are there), then causal
    attention of every row over its request's cache.  ``tiles`` (n, 4) int32
    lists (request, first row, rows <= 128, position of the first row)."""
    G, D, E = _check_cache(q, k, v, kc, vc, heads)
    if append:
        kv_append(k, v, kc, vc, pos, seq, block_table)
    if not attn_tiles_supported(q, kc, vc):
        return attn_rows(q, k, v, kc, vc, pos, seq, block_table, heads,
                         scale, window, keep, append=False,
                         max_keys=max_keys, out=out, mod=mod)
    out = _out(out, q.shape[0], heads * E, q)
    a = _TilesArgs(q=_p(q), qst=q.stride(0), kc=_p(kc), vc=_p(vc),
                   kpage=G * PAGE_SIZE * D, khead=PAGE_SIZE * D, krow=D,
                   vpage=G * PAGE_SIZE * E, vhead=PAGE_SIZE * E, vrow=E,
                   tiles=_p(tiles), bt=_p(block_table), out=_p(out),
                   MB=block_table.shape[1], H=heads, G=G, D=D, E=E, DS=D,
                   window=window, keep=keep, scale=scale)
    if mod is not None:
        a.mod = _score_args(mod, q, heads)
    _check(library().sv_attn_tiles(ctypes.byref(a), tiles.shape[0],
                                   _stream()), "attn_tiles")
    return out


def ragged_attention(q, k, v, batch, pool, heads: int, scale: float,
                     window: int = 0, keep: int = 0,
                     prep: Optional[QkvPrep] = None,
                     mod: Optional[ScoreMod] = None,
                     rotary=None) -> torch.Tensor:
    """Attention of a packed batch over its cache pool: portions first, then
    single tokens, into one (T, heads * E) tensor.  ``prep`` changes q in
    place, ``rotary`` (cos, sin) turns q and k as ``rope_rows_`` does and may."""
    kc, vc = pool
    T, n = q.shape[0], batch.portion_tokens
    if rotary is not None:
        assert prep is None
        if n:
            rope_rows_(q, k, *rotary, batch.pos, kc.shape[3], batch.max_keys)
            rotary = None
    out = torch.empty(T, heads * vc.shape[3], dtype=q.dtype, device=q.device)
    append = prep is None
    if prep is not None:
        qkv_append(q, k, v, kc, vc, batch.pos, batch.seq, batch.block_table,
                   heads, prep)
    parts = ((0, T),) if n in (0, T) else ((0, n), (n, T))
    for a, b in parts:
        at = (q, k, v, batch.pos, batch.seq, out)
        if b - a < T:                    # (a slice costs the host 1 us)
            at = [t[a:b] for t in at]
        qa, ka, va, pos, seq, oa = at
        ma = mod and mod.rows(a, b)
        if a < n:
            attn_portions(qa, ka, va, kc, vc, pos, seq, batch.block_table,
                          batch.tiles, heads, scale, window, keep, append,
                          batch.max_keys, oa, ma)
        elif a < T:
            attn_rows(qa, ka, va, kc, vc, pos, seq, batch.block_table, heads,
                      scale, window, keep, append, batch.max_keys, oa, ma,
                      rotary)
    return out


def _check_rotary(cos, sin, q, k, pos, dim: int, max_pos: int):
    rows = min(cos.shape[0], sin.shape[0])
    if max_pos > rows:
        raise ValueError(f"position {max_pos - 1} is outside the rotary "
                         f"table of {rows}")
    assert cos.dtype == sin.dtype == torch.float32 and cos.is_contiguous()
    assert sin.is_contiguous() and cos.shape[1] * 2 == dim
    assert sin.shape[1] == cos.shape[1]
    assert q.stride(1) == k.stride(1) == 1 and pos.shape[0] == q.shape[0]


def rope_rows_(q, k, cos, sin, pos, dim: int, max_pos: int):
    """Rotate the heads of q and k (rotate-half) in place, each row at its
    own position; cos/sin (positions, dim / 2) float32."""
    _check_rotary(cos, sin, q, k, pos, dim, max_pos)
    vp, lg = ctypes.c_void_p, ctypes.c_long
    _check(library().sv_rope_rows(
        vp(_p(q)), lg(q.stride(0)), q.shape[1] // dim, vp(_p(k)),
        lg(k.stride(0)), k.shape[1] // dim, vp(_p(cos)), vp(_p(sin)),
        vp(_p(pos)), q.shape[0], dim, _f32(q), _stream()), "rope_rows")


# ---------------------------------------------------------------------------
# recurrent matrix memories
# ---------------------------------------------------------------------------

@dataclass
class DecayGate:
    """S <- decay S + k v^T; q, k and v pass through silu."""
    decay: torch.Tensor        # (H,) float32
    log2_decay: torch.Tensor   # (H,) float32


@dataclass
class ExpGate:
    """Exponential input and forget gates with a running maximum."""
    raw: torch.Tensor          # (T, 2H) float32: i then f projections
    i_bias: torch.Tensor       # (H,)
    f_bias: torch.Tensor       # (H,)
    cap: float
    qscale: float


@dataclass
class TimeGate:
    """A time step from a projection: dt = softplus(raw + bias), S <-
    exp(-exp(A_log) dt) S + dt k v^T; o = (S^T q + skip v) silu(z).  Heads share
    q and k in groups.  ``conv``: q, k and v of single tokens have not passed
    their convolution and silu yet; its channels are v's, then k's, then q's."""
    raw: torch.Tensor          # (T, H) float32
    bias: torch.Tensor         # (H,)
    A_log: torch.Tensor        # (H,)
    skip: torch.Tensor         # (H,)
    z: torch.Tensor            # (T, H * E)
    conv: Optional[ShortConv] = None


@dataclass
class TurnGate:
    """S <- decay S + kscale k v^T, with q and k rotated at their position:
    elements i and i + dims / 2 of a head turn together."""
    decay: torch.Tensor        # (H,) float32
    log2_decay: torch.Tensor   # (H,) float32
    kscale: float
    freq: torch.Tensor         # (dims / 2,) float64 rad a position
    amplitude: float = 1.0     # of cos and sin

    @staticmethod
    def norm_fits(dtype, D: int, E: int, *tensors) -> bool:
        """Can the chunk kernels norm and gate the heads as well?"""
        return (dtype == torch.bfloat16 and D <= 256
                and E <= (128 if D <= 128 else 64)
                and _aligned((D, E), *tensors))


_GATINGS = {DecayGate: 0, ExpGate: 1, TimeGate: 2, TurnGate: 3}


def chunk_table(segments):
    """Chunks of prompt portions: rows (segment, first row, rows, does a
    state come in) and the first chunk of every segment, from rows (slot,
    first row, rows, context)."""
    rows, first = [], [0]
    for i, (_, r0, n, ctx) in enumerate(segments):
        for at in range(0, n, CHUNK):
            rows.append((i, r0 + at, min(CHUNK, n - at),
                         int(at > 0 or ctx > 0)))
        first.append(len(rows))
    return rows, first


def memory_carries(chunks: int, segments: int, state: int) -> bool:
    """Are the states of a timed memory of 64 keys (``state`` elements a segment)
    carried from chunk to chunk, not made for all chunks at once and scanned?  A chunk
    of the longest segment takes a workgroup 4 us; at once, 4096 elements of a
    chunk's state take 0.018 us of the device, and two launches more.  The
    longest segment is at most as long as all but one chunk a segment.
    Whole calls of heads of 64 keys, at once and carried, over 140 sizes (0.3 % from
    the better one in the mean, 8 % at most): 128 heads of 64, 60 tokens 18.5 and 13.9,
    1472 66.5 and 70.8, 3237 beside 51 124.7 and 138.2; of 128, 1445 and 924 tokens 176
    and 161; 16 heads of 64, 3409 tokens 39.9 and 74.8."""
    return chunks - segments + 1 <= chunks * (state // 4096) / 217 + 2


def memory_pass(chunks: int, segments: int, columns: int) -> bool:
    """Does a timed memory of 128 keys go through its segments in one pass, a
    workgroup for 64 of all heads' ``columns``?  A chunk of the longest segment
    takes it 8.3 us, 12.4 where all CUs have one; states of all chunks at once and
    outputs after them take 0.062 us for 64 columns of a chunk and 9 in all.  Whole
    calls, those and one pass, over 223 sizes (1.37 in the mean): 64 heads of 64,
    1500 tokens 54.5 and 55.1, 3000 82.7 and 100.8; 128 heads, 2 x 2048 181 and 105,
    200 tokens 36 and 20; 16 heads, 1500 tokens 34.8 and 52.2.  The longest segment
    is at most as long as all but one chunk a segment."""
    return chunks - segments + 1 <= chunks * (columns // 64) / 80 + 2


def single_pass(chunks: int, segments: int, columns: int, gated: bool) -> bool:
    """The same for a decayed or a gated memory.  A chunk of the longest segment takes
    one pass 11.9 us (gated 11.3) behind 5 for the call; the launches and passes it
    stands for take 17 to 44 (21 to 50) up to a chunk or two and 0.08 us more for every
    64 columns of a chunk: 64 x 64 columns, 1000 tokens in one segment 51 and 52 (55 and
    47), 1300 58 and 65, 1500 66 and 77 (66 and 67).  A segment's last chunk is half full
    in the mean, and of many segments half of a chunk each is not there (16 x 256 columns,
    2192 tokens beside 9 short segments 96 and 105, counted as whole ones).  4664 random
    calls of 1 to 128 heads and up to 40 segments, this over those in the 3090 where it is
    chosen: 0.41 in the mean, none slower by more than 2 %."""
    full = chunks - (segments - 1) / 2
    return chunks - segments + 1 <= full * (columns // 64) / 140 + 2 + gated


def memory_mix(q, k, v, gate, S, n, m, seg, heads: int,
               chunks: Optional[torch.Tensor] = None,
               chunk_first: Optional[torch.Tensor] = None,
               out: Optional[torch.Tensor] = None,
               silu_gate: Optional[torch.Tensor] = None,
               eps: float = 0.0) -> torch.Tensor:
    """Run a matrix memory over segments of a ragged batch.  q, k (T, H*D),
    v (T, H*E) — q, k (T, G*D) for a TimeGate; S (slots, H, D, E) float32; n (slots, H, ceil(E/32), D) and
    m (slots, H, ceil(E/32)) float32 for an ExpGate.  ``seg`` (n, 4) int32
    lists (slot, first row, rows, context); rows count from the start of
    the tensors, so portions and single tokens of one batch can be run by
    two calls into one ``out``.  With the device form of
    ``chunk_table`` the 256-token MFMA kernels run where they apply; with a
    TurnGate that ``norm_fits`` they also divide every head of the output by
    its root mean square and multiply it by silu(``silu_gate`` (T, H*E))."""
    D, E = S.shape[2], S.shape[3]
    T = q.shape[0]
    assert q.shape[1] == k.shape[1] and v.shape[1] == heads * E
    assert q.stride(1) == k.stride(1) == v.stride(1) == 1
    assert S.is_contiguous() and S.dtype == torch.float32
    assert S.shape[1] == heads
    if D > MAX_HEAD_DIM:
        raise ValueError(f"key size {D} > {MAX_HEAD_DIM}")
    out = _out(out, T, heads * E, q)
    a = _MemoryArgs(q=_p(q), k=_p(k), v=_p(v), qst=q.stride(0),
                    kst=k.stride(0), vst=v.stride(0), S=_p(S), seg=_p(seg),
                    out=_p(out), H=heads, D=D, E=E, gate_cap=1.0, qscale=1.0,
                    G=q.shape[1] // D)
    assert q.shape[1] == a.G * D and heads % a.G == 0
    gating = _GATINGS[type(gate)]
    gated, timed = isinstance(gate, ExpGate), isinstance(gate, TimeGate)
    turned = isinstance(gate, TurnGate)
    assert timed or a.G == heads
    strided = [q, k, v]
    if timed:
        for t in (gate.bias, gate.A_log, gate.skip):
            assert t.shape == (heads,) and t.dtype == q.dtype
        assert gate.raw.shape == (T, heads) and gate.raw.is_contiguous() \
            and gate.raw.dtype == torch.float32
        assert gate.z.shape == v.shape and gate.z.stride(1) == 1 \
            and gate.z.dtype == v.dtype
        a.gates, a.ib, a.fb = _p(gate.raw), _p(gate.bias), _p(gate.A_log)
        a.skip, a.z, a.zst = _p(gate.skip), _p(gate.z), gate.z.stride(0)
        strided.append(gate.z)
        if gate.conv is not None:
            assert chunks is None      # one token a segment
            a.kch, a.qch = heads * E, heads * E + k.shape[1]
            a.C, a.taps = a.qch + q.shape[1], gate.conv.w.shape[0]
            gate.conv.check(a.C, q.dtype)
            a.cw, a.cb = _p(gate.conv.w), _p(gate.conv.bias)
            a.ring = _p(gate.conv.ring)
    elif gated:
        nt = (E + 31) // 32
        assert n.shape[1:] == (heads, nt, D) and m.shape[1:] == (heads, nt)
        assert gate.raw.shape == (T, 2 * heads) and \
            gate.raw.is_contiguous() and gate.raw.dtype == torch.float32
        assert gate.i_bias.dtype == gate.f_bias.dtype == q.dtype
        a.gates, a.ib, a.fb = _p(gate.raw), _p(gate.i_bias), _p(gate.f_bias)
        a.n, a.m = _p(n), _p(m)
        a.gate_cap, a.qscale = gate.cap, gate.qscale
    else:
        assert gate.decay.shape == (heads,)
        a.decay, a.log2_decay = _p(gate.decay), _p(gate.log2_decay)
    if turned:
        assert gate.freq.dtype == torch.float64 and gate.freq.is_cuda
        a.freq, a.rot = _p(gate.freq), 2 * gate.freq.shape[0]
        a.amp, a.kscale = gate.amplitude, gate.kscale
        if a.rot > D:
            raise ValueError(f"{a.rot} of {D} elements turn")
    if silu_gate is not None:
        assert turned and chunks is not None
        assert gate.norm_fits(q.dtype, D, E, q, k, v, silu_gate)
        assert silu_gate.shape == v.shape and silu_gate.stride(1) == 1 \
            and silu_gate.dtype == v.dtype
        a.z, a.zst = _p(silu_gate), silu_gate.stride(0)
    lib = library()
    if (chunks is not None and q.dtype == torch.bfloat16 and D <= 256
            and _aligned((D, E), *strided)):
        nc = chunks.shape[0]
        assert chunk_first.shape[0] == seg.shape[0] + 1
        f32 = dict(dtype=torch.float32, device=q.device)
        whole = D in (64, 128) and E % 64 == 0 and \
            max(t.stride(0) for t in strided) < 1 << 22
        tiled, decayed = timed and whole, isinstance(gate, DecayGate)
        # one pass writes 16 bytes of the results at once, and of the normaliser
        once = whole and D == 128 and _aligned((), out) and \
            (not gated or n.data_ptr() % 16 == 0) and (
            timed and memory_pass(nc, seg.shape[0], heads * E) or
            (decayed or gated) and single_pass(nc, seg.shape[0], heads * E,
                                               gated))
        U = None if once or tiled and D == 64 and memory_carries(
            nc, seg.shape[0], heads * D * E) \
            else torch.empty(nc, heads, E, D, **f32)
        P = None if once else torch.empty(nc, heads, 3, E, D,
                                          dtype=torch.bfloat16, device=q.device)
        VT = None if tiled or once else \
            torch.empty(nc, heads, E, CHUNK, dtype=torch.bfloat16,
                        device=q.device)
        KA = torch.empty(T, heads * D, dtype=q.dtype, device=q.device) \
            if decayed and not once else None
        if turned:
            KA, QA = torch.empty(2, 2, T, heads * D, dtype=q.dtype,
                                 device=q.device)
        x = _ChunkArgs(a=a, chunks=_p(chunks), first=_p(chunk_first),
                       n_chunks=nc, n_seg=seg.shape[0], T=T, U=_p(U),
                       P=_p(P), VT=_p(VT), KA=_p(KA), norm_eps=eps)
        if turned:
            x.QA = _p(QA)
        if timed and not once:
            bic = torch.empty(2, heads, T, **f32)
            small = torch.empty(nc, heads, 4, **f32)
            x.b, x.i, x.tot = _p(bic[0]), _p(bic[1]), _p(small)
        elif gated and not once:
            bic = torch.empty(3, heads, T, **f32)
            small = torch.empty(nc, heads, 6 + D, **f32)
            x.b, x.i, x.c = (_p(t) for t in bic)
            flat, nh = small.view(-1), nc * heads
            x.tot, x.cend = _p(flat), _p(flat[4 * nh:])
            x.mst, x.N = _p(flat[5 * nh:]), _p(flat[6 * nh:])
        st = lib.sv_memory_chunks(ctypes.byref(x), gating, _stream())
    else:
        st = lib.sv_memory_steps(ctypes.byref(a), seg.shape[0], gating,
                                 _f32(q), _stream())
    _check(st, "memory_mix")
    return out


def decay_gate(decay, device) -> DecayGate:
    d = torch.tensor([float(x) for x in decay], dtype=torch.float64)
    # finite for a decay of zero: 0 tokens apart must still weigh 2^0
    log2 = torch.log2(d).clamp(min=-1e4)
    return DecayGate(d.float().to(device), log2.float().to(device))


# ---------------------------------------------------------------------------
# latent attention
# ---------------------------------------------------------------------------

@dataclass
class KeySpans:
    """The keys that the prompt portions of a step see, gathered page after
    page into a workspace."""
    pages: torch.Tensor        # (n,) cache page of every workspace page
    table: torch.Tensor        # (portions, width) position / 64 -> its page


def key_spans(portions, block_table, window: int):
    """Host form of KeySpans: (pages, table) as lists of int from portions
    (slot, first row, rows, context) and their block-table rows."""
    pages, table = [], []
    for (_, _, n, ctx), row in zip(portions, block_table):
        a = max(0, ctx - window + 1) // PAGE_SIZE if window > 0 else 0
        b = (ctx + n - 1) // PAGE_SIZE
        places = [0] * len(row)
        for p in range(a, b + 1):
            places[p] = len(pages)
            pages.append(int(row[p]))
        table.append(places)
    return pages, table


def rotary_frequencies(base: float, dims: int, device,
                       scaling: Optional[dict] = None) -> torch.Tensor:
    """Radians a position of every rotated pair, float64.  ``scaling`` (factor,
    low, high, original): a pair that turns less than ``low`` times in
    ``original`` positions is slowed by ``factor``, one that turns more than
    ``high`` times is kept, those between are interpolated."""
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = torch.pow(torch.tensor(base, dtype=torch.float64), -2.0 * i / dims)
    if scaling:
        low, high = scaling["low"], scaling["high"]
        turns = scaling["original"] * f / (2.0 * math.pi)
        keep = ((turns - low) / (high - low)).clamp(0.0, 1.0) \
            if high > low else (turns > low).double()
        f = f * (keep + (1.0 - keep) / scaling["factor"])
    return f.to(device)


def yarn_frequencies(base: float, dims: int, device, scaling: dict):
    """Radians a position of every rotated pair, float64, and the amplitude
    of cos and sin.  ``scaling`` (factor, original, fast, slow): pairs that turn
    more than ``fast`` times in ``original`` positions are kept, those that turn
    less than ``slow`` times are slowed by ``factor``; between them, pair by
    pair, linearly from one to the other."""
    f = rotary_frequencies(base, dims, "cpu")

    def pair(turns):
        return dims * math.log(scaling["original"] / (2 * math.pi * turns)) \
            / (2 * math.log(base))

    lo = max(math.floor(pair(scaling["fast"])), 0)
    hi = min(math.ceil(pair(scaling["slow"])), dims - 1)
    i = torch.arange(dims // 2, dtype=torch.float64)
    slow = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    f = f / scaling["factor"] * slow + f * (1.0 - slow)
    return f.to(device), 0.1 * math.log(scaling["factor"]) + 1.0


@dataclass
class LatentWeights:
    norm: torch.Tensor         # (rank,) of the latents
    absorb: torch.Tensor       # (H, rank, dim): query -> latent space
    expand: torch.Tensor       # (H * dim + H * vdim, rank): keys, values
    freq: torch.Tensor         # (rot / 2,) float64 rad a position
    amplitude: float = 1.0     # of cos and sin
    pairs: bool = False        # neighbours turn together, not halves
    sink: Optional[torch.Tensor] = None   # (H,) joins the denominator


def _append_args(q, rot_at, q_step, qr, qr_at, qr_step, kv, w, cache, pos, seq,
                 block_table, heads, eps):
    P = cache.shape[2] - w.norm.shape[0]
    assert qr.stride(1) == 1 and q.dtype == qr.dtype
    assert (heads - 1) * q_step + rot_at + P <= q.shape[1]
    assert (heads - 1) * qr_step + qr_at + P <= qr.shape[1]
    assert q.shape[0] == qr.shape[0]
    return _append_of(_p(q), q.stride(0), rot_at, q_step, _p(qr), qr.stride(0),
                      qr_at, qr_step, kv, w, cache, pos, seq, block_table, heads,
                      eps, q)


def _append_of(q, qst, rot_at, q_step, qr, qrst, qr_at, qr_step, kv, w, cache,
               pos, seq, block_table, heads, eps, like):
    """Of addresses and pitches; ``like``: the queries."""
    T, R = like.shape[0], w.norm.shape[0]
    P = cache.shape[2] - R
    half = w.freq.shape[0]
    assert kv.shape == (T, R + P) and cache.shape[1] == PAGE_SIZE
    assert cache.is_contiguous() and 2 * half <= P
    assert w.freq.dtype == torch.float64 and w.freq.is_cuda
    assert like.stride(1) == kv.stride(1) == 1
    assert like.dtype == kv.dtype == cache.dtype == w.norm.dtype
    assert pos.shape[0] == seq.shape[0] == T
    size = like.element_size()
    return _LatentAppendArgs(
        q=q + rot_at * size, qst=qst, qh=q_step, qr=qr + qr_at * size,
        qrst=qrst, qrh=qr_step, kv=_p(kv), kvst=kv.stride(0), w=_p(w.norm),
        freq=_p(w.freq), cache=_p(cache), pos=_p(pos), seq=_p(seq),
        bt=_p(block_table), MB=block_table.shape[1], H=heads, R=R, P=P,
        rot=2 * half, eps=eps, amp=w.amplitude, pairs=int(w.pairs))


def latent_append(q, rot_at: int, q_step: int, qr, qr_at: int, qr_step: int,
                  kv, w: LatentWeights, cache, pos, seq, block_table,
                  heads: int, eps: float):
    """Norm the latents of kv (T, rank + P), rotate the shared key, write
    both into the cache (pages, 64, rank + P); rotate columns [rot_at, + P) of
    every head of q (heads ``q_step`` apart) into those at ``qr_at`` of qr."""
    a = _append_args(q, rot_at, q_step, qr, qr_at, qr_step, kv, w, cache, pos,
                     seq, block_table, heads, eps)
    _check(library().sv_latent_append(ctypes.byref(a), q.shape[0], _f32(q),
                                      _stream()), "latent_append")


def _linear_args(x, x_step, w, out, out_step, gate):
    """Arguments, and whether the form on matrix cores takes them."""
    H, N, K = w.shape
    T = x.shape[0]
    assert w.is_contiguous() and x.stride(1) == out.stride(1) == 1
    assert x.dtype == w.dtype == out.dtype and out.shape[0] == T
    assert (H - 1) * x_step + K <= x.shape[1]
    assert (H - 1) * out_step + N <= out.shape[1]
    a = _HeadLinearArgs(x=_p(x), xst=x.stride(0), xh=x_step, w=_p(w),
                        out=_p(out), ost=out.stride(0), oh=out_step,
                        T=T, H=H, N=N, K=K)
    mfma = x.dtype == torch.bfloat16 and K >= 8 and N >= 4 and N % 4 == 0 \
        and _aligned((K, x_step, out_step), x, out)
    if gate is not None:
        assert gate.shape == (T, H * N) and gate.stride(1) == 1
        assert gate.dtype == x.dtype
        a.gate, a.gst, a.gh = _p(gate), gate.stride(0), N
        mfma = mfma and _aligned((), gate)
    return a, mfma


def normed_linear(x: Optional[torch.Tensor], pending: Pending, eps: float,
                  weight: torch.Tensor, w: torch.Tensor, glu: bool = False):
    """``residual_norm`` of one row and the product of its result with w (N, K)
    in one launch: (new x, h w^T, or with ``glu`` silu(gate) * up of w = [gate;
    up]); None where they are two: other rows, pending things, types and sizes,
    and where ``stream_how`` leaves the product to the library.  Every workgroup
    norms the row, 32 KB of a K of 4096, while its weights are on their way; of
    more than one such round of them (512) the later ones have nothing to hide
    that behind."""
    d, row = pending.delta, pending.rows
    table = 0
    if row is not None and row.shape[0] == 1 and x is None and d.shape[0] and \
            row.dtype == torch.int32 and row.is_cuda:
        table, d = d.shape[0], d[:1]
    if d is None or d.shape[0] != 1 or (row is not None and not table) or \
            d.dtype != torch.bfloat16 or not d.is_contiguous() or pending.scale != 1.0 or any(
                t is not None for t in (pending.delta2, pending.w1, pending.w2,
                                        pending.vec, pending.coef)):
        return None
    K = d.shape[1]
    if K > 4096 or not (glu or w.shape[0] <= 512 * 16) or \
            not (_plain(weight) and weight.dtype == d.dtype) or \
            not _aligned((K,), d) or weight.data_ptr() & 15 or \
            weight.shape != (K,) or not weight.is_contiguous() or \
            not (x is None or x.dtype == torch.float32 and x.is_contiguous()
                 and x.shape == d.shape and not x.data_ptr() & 15):
        return None
    how = stream_how(d, w, glu=glu)
    if how is None:
        return None
    N = w.shape[0]
    x_new = torch.empty(1, K, dtype=torch.float32, device=d.device)
    out = torch.empty(1, N // 2 if glu else N, dtype=d.dtype, device=d.device)
    a = _StreamArgs(w=w.data_ptr(), wst=w.stride(0), out=out.data_ptr(), T=1,
                    N=N, K=K, res=_p(x), delta=d.data_ptr(),
                    res_out=x_new.data_ptr(), weight=weight.data_ptr(), eps=eps,
                    row=_p(row), rows=table)
    _check(library().sv_stream_linear(ctypes.byref(a), 2 if glu else 0, how,
                                      _stream()), "normed_linear")
    return x_new, out


def head_linear(x, x_step: int, w, out, out_step: int,
                gate: Optional[torch.Tensor] = None):
    """out[t, h * out_step + n] = sum_k x[t, h * x_step + k] w[h, n, k], times
    sigmoid(gate[t, h * N + n])."""
    a, mfma = _linear_args(x, x_step, w, out, out_step, gate)
    _check(library().sv_head_linear(ctypes.byref(a), int(mfma), _f32(x),
                                    _stream()), "head_linear")
    return out


def latent_rows_supported(dtype, rank: int, shared: int) -> bool:
    return (dtype == torch.bfloat16 and rank % 8 == 0 and shared % 8 == 0
            and rank <= 512 and shared <= 64)


def _latent_shares(rows, heads, rank, max_keys, device):
    """Shares of a row and the workspace for them.  Workgroups of 64 keys
    while CUs have none (1 row of 1000 keys: the whole step 28.1 us with 128,
    24.9 with 64), then of 128 (8 of 4096: 32.5, with 64 35.7).  A merge is not
    worth its launch up to 128 keys (43 rows of 82: 23.6, in two 28.7), of more
    than 32 workgroups up to 256 (94 rows of 192, 64 heads, no values behind
    them: 17.6, in two 28.1; 58 of 178, 8 heads 25.2, in three 23.1)."""
    units = rows * -(-heads // 32)
    splits = 1 if max_keys <= (256 if units > 32 else 128) else max(
        _row_splits(512, units, max_keys, 128),
        _row_splits(256, units, max_keys, 64))
    # sums, maxima and totals of every share; of every row, its shares
    return splits, torch.empty(
        rows * heads * splits * (rank + 2) + 2 * rows, dtype=torch.float32,
        device=device) if splits > 1 else None


def _latent_rows_args(q, cache, rank, pos, seq, block_table, heads, scale,
                      window, max_keys, sink, out):
    """Arguments and the workspace that they point to."""
    rows, D = q.shape[0], cache.shape[2]
    splits, part = _latent_shares(rows, heads, rank, max_keys, q.device)
    return _LatentRowsArgs(
        q=_p(q), cache=_p(cache), pos=_p(pos), seq=_p(seq),
        bt=_p(block_table), part=_p(part), out=_p(out),
        MB=block_table.shape[1], rows=rows, H=heads, R=rank, P=D - rank,
        splits=splits, window=window, scale=scale, sink=sink), part


def latent_rows(q, cache, rank: int, pos, seq, block_table, heads: int,
                scale: float, window: int = 0, max_keys: int = 0,
                sink: Optional[torch.Tensor] = None):
    """Absorbed queries q (rows, H * (rank + P)) over the cached rows, which
    hold the rows' own keys already -> (rows, H * rank) sums of latents.
    exp(sink[h]) joins the denominator."""
    rows, D = q.shape[0], cache.shape[2]
    assert q.is_contiguous() and q.shape[1] == heads * D
    assert cache.is_contiguous() and cache.shape[1] == PAGE_SIZE
    assert q.dtype == cache.dtype and pos.shape[0] == seq.shape[0] == rows
    if D > MAX_LATENT_ROW:
        raise ValueError(f"latent row of {D} > {MAX_LATENT_ROW}")
    mod = _score_args(ScoreMod(sink=sink), q, heads)
    if window > 0:
        max_keys = min(max_keys, window) if max_keys else window
    out = torch.empty(rows, heads * rank, dtype=q.dtype, device=q.device)
    fast = latent_rows_supported(q.dtype, rank, D - rank)
    if fast:
        a, part = _latent_rows_args(q, cache, rank, pos, seq, block_table,
                                    heads, scale, window, max_keys, mod.sink,
                                    out)
        _check(library().sv_latent_rows(ctypes.byref(a), _stream()),
               "latent_rows")
        return out
    splits = _row_splits(1024, rows, max_keys, 128)
    part = torch.empty(rows * heads * splits * (rank + 2),
                       dtype=torch.float32, device=q.device) \
        if splits > 1 else None
    # one key/value head whose value is the front of its key
    a = _RowsArgs(q=_p(q), k=_p(q), v=_p(q), qst=q.stride(0),
                  kst=q.stride(0), vst=q.stride(0), kc=_p(cache),
                  vc=_p(cache), kcs=D, vcs=D, pos=_p(pos), seq=_p(seq),
                  bt=_p(block_table), part=_p(part), out=_p(out),
                  MB=block_table.shape[1], rows=rows, H=heads, G=1, D=D,
                  E=rank, splits=splits, append=0, window=window, keep=0,
                  scale=scale, mod=mod)
    _check(library().sv_attn_rows(ctypes.byref(a),
                                  int(_aligned((D, rank), q)), _f32(q),
                                  _stream()), "attn_rows")
    return out


def latent_tiles_supported(q, gate, dim, vdim, rank, shared) -> bool:
    return (q.dtype == torch.bfloat16 and dim + shared <= 256
            and vdim <= 256
            and _aligned((dim, vdim, rank, shared), q)
            and (gate is None or _aligned((), gate)))


def expand_rule(rows: int, N: int, R: int) -> bool:
    """Are keys and values (rows, N) of a latent cache made by a kernel that reads its
    pages where they lie, not by a copy and a library product?  Both within a call, over
    7161 sizes of rank 64 to 1536, us, copy and product | kernel.  Yes where its tiles of
    128 x 128 are one round of workgroups and the rank is not so long that the library's
    larger ones gain (128 x 8192, R 64 7.9 | 5.0, R 512 13.9 | 9.2; 128 x 2048 of R 1536
    11.0 | 15.2); past that where the library's tiles of 256 x 256 leave CUs idle and the
    rank is neither so short that the results alone decide nor so long (R 512: 1344 x 8192
    39 | 23, 2048 x 10240 49 | 36, 2048 x 12288 45.5 | 41.7), but not where they fill them
    or nearly (4096 x 4096 28.1 | 29.9, 3136 x 4096 25.5 | 29.6; R 64, 2240 x 12288 22.3 |
    29.0), nor for large products (5184 x 8192 63.1 | 70.4).  Of the 4283 that it takes 3
    lose more than 3 % and 0.5 us, 6 % at most: 128 tokens of two long ranks, and 768 x
    32768 of 512, 45.1 | 47.4; the mean is 1.37 of the speed."""
    own = -(-rows // 128) * -(-N // 128)
    tiles = -(-rows // 256) * -(-N // 256)
    whole = tiles >= 216 and not 0 < tiles % 256 < 216
    if R % 64 or N * R >= 1 << 30 or rows * N > 28_000_000 or whole:
        return False
    if own <= 512:
        return R <= 640 or R <= 1024 and own <= 256
    return 256 <= R <= 512 and (172 <= tiles <= 192 or 256 < tiles < 384 or
                                R >= 384 and own >= 1440)


def _expandable(cache, expand, pages, R: int, P: int) -> bool:
    return cache.is_contiguous() and expand.is_contiguous() and \
        pages.is_contiguous() and pages.dtype == torch.int32 and \
        cache.dtype == expand.dtype == torch.bfloat16 and \
        cache.shape[1:] == (PAGE_SIZE, R + P) and expand.shape[1] == R and \
        cache.device == expand.device == pages.device and \
        not (expand.shape[0] | P) & 7 and \
        not (cache.data_ptr() | expand.data_ptr()) & 15


def latent_portions(q, gate, cache, w: LatentWeights, batch,
                    spans: KeySpans, heads: int, dim: int, vdim: int,
                    scale: float, window: int, out):
    """Prompt portions with rotated queries q (T, H * (dim + P)): gather the
    visible rows, make all heads' keys and values with one product, attend."""
    R = w.norm.shape[0]
    P = cache.shape[2] - R
    n = spans.pages.shape[0]
    N = w.expand.shape[0]
    if n and P and expand_rule(n * PAGE_SIZE, N, R) and \
            _expandable(cache, w.expand, spans.pages, R, P):
        kv = torch.empty(n * PAGE_SIZE, N, dtype=q.dtype, device=q.device)
        ws = torch.empty(n * PAGE_SIZE, P, dtype=q.dtype, device=q.device)
        _check(library().sv_latent_expand(
            ctypes.c_void_p(_p(cache)), ctypes.c_void_p(_p(spans.pages)), n,
            ctypes.c_void_p(_p(w.expand)), ctypes.c_void_p(_p(kv)),
            ctypes.c_void_p(_p(ws)), R, P, N, _stream()), "latent_expand")
    else:
        ws = torch.empty(n * PAGE_SIZE, R + P, dtype=q.dtype, device=q.device)
        _check(library().sv_latent_gather(
            ctypes.c_void_p(_p(cache)), ctypes.c_void_p(_p(ws)),
            ctypes.c_void_p(_p(spans.pages)), n,
            PAGE_SIZE * (R + P) * q.element_size(), _stream()), "latent_gather")
        kv = torch.mm(ws[:, :R], w.expand.t())
    return expanded_attention(q, gate, kv, ws, batch.tiles, spans, heads,
                              dim, vdim, scale, window, out, w.sink)


def expanded_attention(q, gate, kv, ws, tiles, spans: KeySpans, heads: int,
                       dim: int, vdim: int, scale: float, window: int, out,
                       sink: Optional[torch.Tensor] = None):
    """Query tiles over keys and values kv (rows, H * dim + H * vdim) of the
    workspace rows ws (rows, rank + P), whose last columns end every key."""
    P = q.shape[1] // heads - dim
    R = ws.shape[1] - P
    assert q.shape[1] == heads * (dim + P) and q.stride(1) == 1
    assert kv.shape == (spans.pages.shape[0] * PAGE_SIZE,
                        heads * (dim + vdim)) and kv.is_contiguous()
    assert ws.shape[0] == kv.shape[0] and ws.is_contiguous()
    assert out.shape == (q.shape[0], heads * vdim) and out.is_contiguous()
    row, size = kv.shape[1], q.element_size()
    a = _TilesArgs(q=_p(q), qst=q.stride(0), kc=_p(kv),
                   vc=_p(kv) + heads * dim * size, kr=_p(ws) + R * size,
                   kpage=PAGE_SIZE * row, khead=dim, krow=row,
                   vpage=PAGE_SIZE * row, vhead=vdim, vrow=row, rrow=R + P,
                   tiles=_p(tiles), bt=_p(spans.table), out=_p(out),
                   MB=spans.table.shape[1], H=heads, G=heads, D=dim + P,
                   E=vdim, DS=dim, window=window, keep=0, scale=scale,
                   mod=_score_args(ScoreMod(sink=sink), q, heads))
    if gate is not None:
        assert gate.shape == out.shape and gate.stride(1) == 1
        a.gate, a.gst = _p(gate), gate.stride(0)
    _check(library().sv_attn_tiles(ctypes.byref(a), tiles.shape[0],
                                   _stream()), "attn_tiles")
    return out


def latent_attention(q, kv, gate, batch, cache, w: LatentWeights, heads: int,
                     dim: int, vdim: int, scale: float, eps: float,
                     window: int = 0) -> torch.Tensor:
    """Latent attention of a packed batch.  q (T, H * (dim + P)) head by head
    [unrotated | rotated], kv (T, rank + P), gate (T, H * vdim) or None ->
    (T, H * vdim), times sigmoid(gate)."""
    T, R = q.shape[0], w.norm.shape[0]
    D = cache.shape[2]
    P = D - R
    out = torch.empty(T, heads * vdim, dtype=q.dtype, device=q.device)
    n = batch.portion_tokens
    spans = batch.spans.get(window)
    if spans is None or not latent_tiles_supported(q, gate, dim, vdim, R, P):
        n = 0
    if n:
        g = None if gate is None else gate[:n]
        latent_append(q[:n], dim, dim + P, q[:n], dim, dim + P, kv[:n], w,
                      cache, batch.pos[:n], batch.seq[:n], batch.block_table,
                      heads, eps)
        latent_portions(q[:n], g, cache, w, batch, spans, heads, dim, vdim,
                        scale, window, out[:n])
    if n < T:
        one = (batch.pos, batch.seq)
        if n:
            q, kv, gate = (t if t is None else t[n:] for t in (q, kv, gate))
            one = [t[n:] for t in one]
        at = (*one, batch.block_table)
        to = out[n:] if n else out
        if _latent_step(q, kv, gate, *at, batch.max_keys, cache, w, heads, dim,
                        vdim, scale, eps, window, to):
            return out
        ql = torch.empty(T - n, heads * D, dtype=q.dtype, device=q.device)
        latent_append(q, dim, dim + P, ql, R, D, kv, w, cache, *at, heads, eps)
        head_linear(q, dim + P, w.absorb, ql, D)
        lat = latent_rows(ql, cache, R, *at, heads, scale, window,
                          batch.max_keys, w.sink)
        head_linear(lat, R, w.expand[heads * dim:].view(heads, vdim, R),
                    to, vdim, gate)
    return out


def _latent_step(q, kv, gate, pos, seq, block_table, max_keys, cache,
                 w: LatentWeights, heads, dim, vdim, scale, eps, window,
                 out) -> bool:
    """Single tokens in one call, on matrix cores: rows that are appended, queries
    taken into the latent space, attention, values into ``out``.  False where one
    of them has no such form."""
    rows, R, D = q.shape[0], w.norm.shape[0], cache.shape[2]
    P = D - R
    if not (latent_rows_supported(q.dtype, R, P) and dim >= 8 and
            _aligned((dim, vdim, R, P), q) and
            (gate is None or _aligned((), gate))):
        return False
    assert w.absorb.shape == (heads, R, dim) and w.absorb.is_contiguous()
    assert w.expand.shape == (heads * (dim + vdim), R)
    assert w.expand.is_contiguous() and q.stride(1) == out.stride(1) == 1
    assert q.dtype == w.absorb.dtype == w.expand.dtype == out.dtype
    assert q.shape[1] >= heads * (dim + P) and out.shape[1] == heads * vdim
    if window > 0:
        max_keys = min(max_keys, window) if max_keys else window
    # absorbed queries, then merged rows: a workspace that only kernels see
    work = torch.empty(rows * heads * (D + R), dtype=q.dtype, device=q.device)
    ql = work.data_ptr()
    lat = ql + rows * heads * D * 2
    values = w.expand.data_ptr() + heads * dim * R * 2
    sink = w.sink
    assert sink is None or (sink.shape == (heads,) and sink.is_contiguous()
                            and sink.dtype == q.dtype and sink.is_cuda)
    qp, qst = q.data_ptr(), q.stride(0)
    splits, part = _latent_shares(rows, heads, R, max_keys, q.device)
    a = _LatentStepArgs(
        append=_append_of(qp, qst, dim, dim + P, ql, heads * D, R, D, kv, w,
                          cache, pos, seq, block_table, heads, eps, q),
        absorb=_HeadLinearArgs(x=qp, xst=qst, xh=dim + P, w=w.absorb.data_ptr(),
                               out=ql, ost=heads * D, oh=D, T=rows, H=heads,
                               N=R, K=dim),
        rows=_LatentRowsArgs(
            q=ql, cache=cache.data_ptr(), pos=pos.data_ptr(),
            seq=seq.data_ptr(), bt=block_table.data_ptr(), part=_p(part),
            out=lat, MB=block_table.shape[1], rows=rows, H=heads, R=R, P=P,
            splits=splits, window=window, scale=scale, sink=_p(sink)),
        values=_HeadLinearArgs(x=lat, xst=heads * R, xh=R, w=values,
                               out=out.data_ptr(), ost=out.stride(0), oh=vdim,
                               T=rows, H=heads, N=vdim, K=R))
    if gate is not None:
        assert gate.shape == (rows, heads * vdim) and gate.stride(1) == 1
        assert gate.dtype == q.dtype
        v = a.values
        v.gate, v.gst, v.gh = gate.data_ptr(), gate.stride(0), vdim
    _check(library().sv_latent_step(ctypes.byref(a), _stream()), "latent_step")
    return True


# ---------------------------------------------------------------------------
# mixture of experts
# ---------------------------------------------------------------------------

# kernels of the grouped products, and the most slots of their tiles
MOE_PLAIN, MOE_STREAM = 0, 1
MOE_TILES = (2, 3, 4, 5)
MOE_TILE_ROWS = (32, 32, 32, 64, 128, 256)


def moe_kernel(pairs: int, experts: int, width: int, ff: int) -> int:
    """The fastest kernel for ``pairs`` spread over ``experts`` of ff x width
    (measured): streaming up to 24 rows an expert where workgroups can stay with
    their rows (width and ff up to 4096), 16 where only the gates' can; else the
    rows are read again and again, and tiles are faster from 4 on (256 experts
    7168 x 2048, 4 rows: 3.64 ms, streamed 4.21), as where less than half of the
    columns that a staying workgroup covers are there and the tiles of 256 gates
    and projections fill the CUs (8 rows of 128 experts 2048 x 768: 238 us,
    streamed 254; of 64 of 2048 x 512: 104, 96).  Tiles of 64 slots and more
    read weights two steps ahead where width and ff are multiples of 64, and are
    the faster ones from 16 rows on (8 experts 4096 x 14336, 16 rows: 32 slots 549
    us, 64 516; 256 of 7168 x 2048: 3930, 3774), those of 128 from 24 (64 experts
    2048 x 1408, 24 rows: 64 slots 212, 128 215, 64 rows: 260, 235), with long rows
    from 48 (8 experts 4096 x 14336, 32 rows: 504, 526, 48: 595, 520), those of 256
    from 112 (96 rows: 128 slots 582, 256 664, 112: 774, 679).  The mean rows are all
    that the host knows: 32 rows that go to the same 6 of 64 experts stay as well,
    528 units on 512 workgroups (58 us; 71 before staying came).  One size is
    slower than it was: 64 experts 4096 x 2048 of 24 to 32 rows, 777 to 796 us
    where tiles of 64 took 732 to 760 before the XCDs shared the tiles that have
    rows."""
    rows = pairs / experts
    stay = width <= 4096 and (min(width, ff) > 960 or
                              experts * ff <= 256 * 128)
    if rows < ((24 if ff <= 4096 else 16) if stay else 4):
        return MOE_STREAM
    if rows >= 16 and not (width | ff) & 63:
        if rows < 24 or rows < 48 and max(width, ff) > 4096:
            return MOE_TILES[1]
        return MOE_TILES[2 if rows < 112 else 3]
    return MOE_TILES[sum(rows >= r for r in (24, 112, 160))]


@dataclass
class Routing:
    """How logits choose experts.  Plain: the largest z + bias, weights a
    softmax over the chosen.  ``sigmoid``: the largest sigmoid(z) + bias,
    weights the chosen sigmoids over their sum.  ``softmax``: the largest z +
    bias, weights a softmax over all experts, not scaled to a sum of one.  With
    several ``groups`` of neighbours only the experts of the ``keep`` best can
    be chosen; a group counts the sum of its ``best`` (one or two) largest."""
    top: int
    sigmoid: bool = False
    groups: int = 1
    keep: int = 1
    softmax: bool = False
    best: int = 2

    @property
    def kind(self) -> int:
        return 2 if self.softmax else int(self.sigmoid)

    def check(self, experts: int):
        g = self.groups
        if experts > MAX_EXPERTS or not 1 <= self.top <= min(64, experts):
            raise ValueError(f"{self.top} of {experts} experts")
        if not 1 <= g <= 64 or experts % g or not 1 <= self.keep <= g or \
                self.keep * (experts // g) < self.top:
            raise ValueError(f"{self.top} experts from {self.keep} of {g} "
                             f"groups of {experts}")
        if self.best not in (1, 2) or (self.sigmoid and self.softmax):
            raise ValueError(f"routing {self}")


@dataclass
class MoePlan:
    coef: torch.Tensor         # (T, top) float32 weights of the chosen
    idx: torch.Tensor          # (T, top) int32 chosen experts
    order: torch.Tensor        # (T * top,) pairs, expert by expert
    tiles: torch.Tensor        # (n, 4) expert, first slot, slots
    how: int                   # kernel of the grouped products


def moe_plan(z: torch.Tensor, bias: Optional[torch.Tensor],
             routing: Union[int, Routing], how: int) -> MoePlan:
    """Choose the experts of every row from its logits z (plainly, if
    ``routing`` is just their number), and group the pairs."""
    T, E = z.shape
    if isinstance(routing, int):
        routing = Routing(routing)
    assert z.dtype == torch.float32 and z.is_contiguous() and z.is_cuda
    routing.check(E)
    top = routing.top
    pairs, rows = T * top, MOE_TILE_ROWS[how]
    n = min(pairs, pairs // rows + E)
    ints = torch.empty(2 * pairs + 4 * n, dtype=torch.int32, device=z.device)
    p = MoePlan(torch.empty(T, top, dtype=torch.float32, device=z.device),
                ints[4 * n:4 * n + pairs].view(T, top), ints[4 * n + pairs:],
                ints[:4 * n].view(n, 4), how)
    a = _MoePlanArgs(z=_p(z), bias=_p(bias), idx=_p(p.idx), coef=_p(p.coef),
                     order=_p(p.order), tiles=_p(p.tiles), T=T, E=E, top=top,
                     tile_rows=rows, max_tiles=n,
                     kind=routing.kind, groups=routing.groups,
                     keep=routing.keep, best=routing.best)
    _check(library().sv_moe_plan(
        ctypes.byref(a), 0 if bias is None else _f32(bias), _stream()),
        "moe_plan")
    return p


def moe_gemm(x: torch.Tensor, w: torch.Tensor, plan: MoePlan, gated: bool,
             alpha: float = 1.0, limit: float = float("inf"),
             shift: float = 0.0) -> torch.Tensor:
    """Grouped product over w (E, rows, K).  ``gated``: rows of x (T, K) ->
    min(g, limit) sigmoid(alpha g) (clamp(u, limit) + shift) of w = [gate;
    up], in slot order.  Else: slots x (T * top, K) -> pairs."""
    pairs = plan.order.shape[0]
    _, rows, K = w.shape
    T, cols = x.shape
    N = rows // 2 if gated else rows
    assert x.stride(1) == 1 and cols == K and w.is_contiguous()
    assert x.dtype == w.dtype and rows == (2 * N if gated else N)
    assert T == (plan.coef.shape[0] if gated else pairs)
    out = torch.empty(pairs, N, dtype=x.dtype, device=x.device)
    a = _MoeGemmArgs(x=x.data_ptr(), xst=x.stride(0), w=w.data_ptr(),
                     out=out.data_ptr(), order=plan.order.data_ptr(),
                     tiles=plan.tiles.data_ptr(),
                     top=plan.coef.shape[1] if gated else 0, N=N, K=K,
                     max_tiles=plan.tiles.shape[0], alpha=alpha, limit=limit,
                     shift=shift, rows=T)
    assert plan.how == MOE_PLAIN or (x.dtype == torch.bfloat16
                                     and _aligned((N, K), x))
    _check(library().sv_moe_gemm(ctypes.byref(a), plan.how, int(gated),
                                 _f32(x), _stream()), "moe_gemm")
    return out


def moe_mlp(h, z, bias, gate_up, down, routing: Union[int, Routing],
            alpha: float, limit: float, shift: float) -> Pending:
    """Gated experts on h (T, W) with router logits z (T, E): a pending sum
    of the chosen experts' outputs."""
    if isinstance(routing, int):
        routing = Routing(routing)
    E, W, ff = down.shape
    pairs = h.shape[0] * routing.top
    fast = h.dtype == torch.bfloat16 and _aligned((W, ff), h)
    plan = moe_plan(z, bias, routing,
                    moe_kernel(pairs, E, W, ff) if fast else MOE_PLAIN)
    act = moe_gemm(h, gate_up, plan, True, alpha, limit, shift)
    return Pending(moe_gemm(act, down, plan, False), coef=plan.coef)
