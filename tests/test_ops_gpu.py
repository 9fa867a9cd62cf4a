"""GPU numerics: every HIP kernel vs the plain-torch fp32 reference
(the CPU fallback implementations in ops/__init__.py and kernels/)."""

import ctypes
import math
import os

import pytest
import torch

pytestmark = pytest.mark.gpu

from neuronx_distributed_amd import ops
from neuronx_distributed_amd.kernels.flash_attn import _torch_reference


@pytest.fixture(scope="module", autouse=True)
def _require_lib():
    assert torch.cuda.is_available()
    ops.build = __import__("neuronx_distributed_amd.ops.build",
                           fromlist=["build"])
    ops.build.build()
    assert ops.is_available(), ops._LIB_ERR


def _cmp(a, b, atol, rtol=2e-2, name=""):
    a = a.float().cpu()
    b = b.float().cpu()
    err = (a - b).abs().max().item()
    ref = b.abs().max().item()
    assert err <= atol + rtol * ref, f"{name}: max err {err} (ref max {ref})"


def test_rmsnorm_fwd_bwd():
    torch.manual_seed(0)
    for rows, H in ((128, 512), (1024, 4096), (64, 8192)):
        x = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
        w = torch.randn(H, dtype=torch.bfloat16, device="cuda")
        xg = x.clone().requires_grad_(True)
        wg = w.clone().requires_grad_(True)
        out = ops.rmsnorm(xg, wg, 1e-5)
        xr = x.clone().float().requires_grad_(True)
        wr = w.clone().float().requires_grad_(True)
        ref = xr * torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + 1e-5) * wr
        _cmp(out, ref, atol=3e-2, name=f"rmsnorm fwd {H}")
        dy = torch.randn_like(out)
        out.backward(dy)
        ref.backward(dy.float())
        _cmp(xg.grad, xr.grad, atol=5e-2, name=f"rmsnorm dx {H}")
        _cmp(wg.grad, wr.grad, atol=5e-1, name=f"rmsnorm dw {H}")


def test_rope_fwd_bwd():
    torch.manual_seed(1)
    B, S, Hq, Hk, D = 2, 64, 4, 2, 128
    cos, sin = ops.precompute_rope_freqs(128, D, device="cuda")
    q = torch.randn(B, S, Hq, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    k = torch.randn(B, S, Hk, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    qo, ko = ops.apply_rotary_pos_emb(q, k, cos, sin, pos_offset=3)
    from neuronx_distributed_amd.ops import _rope_torch

    qr = _rope_torch(q.detach(), cos[3:3 + S].cpu().cuda(), sin[3:3 + S])
    kr = _rope_torch(k.detach(), cos[3:3 + S], sin[3:3 + S])
    _cmp(qo, qr, atol=2e-2, name="rope q")
    _cmp(ko, kr, atol=2e-2, name="rope k")
    (qo.float().pow(2).sum() + ko.float().pow(2).sum()).backward()
    # rotation is orthogonal: grad check via rotation-transpose property
    qg = q.grad.clone()
    q.grad = None
    k.grad = None
    q2 = q.detach().clone().requires_grad_(True)
    qr2 = _rope_torch(q2, cos[3:3 + S], sin[3:3 + S])
    qr2.float().pow(2).sum().backward()
    _cmp(qg, q2.grad, atol=5e-2, name="rope dq")


def test_swiglu_fwd_bwd():
    torch.manual_seed(2)
    x = torch.randn(512, 2048, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    out = ops.swiglu(x)
    xr = x.detach().float().requires_grad_(True)
    I = 1024
    ref = torch.nn.functional.silu(xr[..., :I]) * xr[..., I:]
    _cmp(out, ref, atol=3e-2, name="swiglu fwd")
    dy = torch.randn_like(out)
    out.backward(dy)
    ref.backward(dy.float())
    _cmp(x.grad, xr.grad, atol=5e-2, name="swiglu dx")


@pytest.mark.parametrize("B,Hq,Hkv,S,causal", [
    (1, 4, 4, 256, True),
    (2, 8, 2, 512, True),
    (1, 4, 4, 300, True),    # ragged S
    (1, 2, 2, 1024, False),
    (1, 32, 8, 2048, True),
    (1, 32, 8, 4096, True),  # llama2-7b/llama3-8b production shape
    (1, 8, 8, 8192, True),   # seq-8192 long-context shape
])
def test_flash_attn_fwd(B, Hq, Hkv, S, causal):
    torch.manual_seed(3)
    D = 128
    q = torch.randn(B, Hq, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    k = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    v = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    out = ops.flash_attn(q, k, v, causal=causal)
    ref = _torch_reference(q.float(), k.float(), v.float(), causal=causal)
    _cmp(out, ref, atol=3e-2, rtol=3e-2, name=f"flash fwd S={S}")


def test_flash_attn_lse():
    torch.manual_seed(4)
    B, H, S, D = 1, 2, 256, 128
    q = torch.randn(B, H, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    k = torch.randn(B, H, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    v = torch.randn_like(k)
    qg = q.requires_grad_(False)
    out = ops._FlashAttnFn.apply(q, k, v, True, 1.0 / math.sqrt(D))
    # recompute lse reference
    scores = (q.float() @ k.float().transpose(-1, -2)) / math.sqrt(D)
    mask = torch.ones(S, S, dtype=torch.bool, device="cuda").tril()
    scores = scores.masked_fill(~mask, float("-inf"))
    lse_ref = torch.logsumexp(scores, dim=-1)
    # pull lse out of the autograd ctx by re-running the raw kernel
    import ctypes
    from neuronx_distributed_amd.ops import _ptr, _require_lib, _stream

    lib = _require_lib()
    o2 = torch.empty_like(q)
    lse = torch.empty(B, H, S, dtype=torch.float32, device="cuda")
    lib.flash_attn_fwd(_ptr(q), _ptr(k), _ptr(v), _ptr(o2), _ptr(lse),
                       ctypes.c_int(B), ctypes.c_int(H), ctypes.c_int(H),
                       ctypes.c_int(S), ctypes.c_float(1.0 / math.sqrt(D)),
                       ctypes.c_int(1), _stream())
    torch.cuda.synchronize()
    _cmp(lse, lse_ref, atol=2e-3, name="lse")


@pytest.mark.parametrize("B,Hq,Hkv,S,causal", [
    (1, 2, 2, 256, True),
    (1, 4, 1, 512, True),
    (1, 2, 2, 512, False),
    (1, 32, 8, 4096, True),  # production GQA 32/8 at seq 4096
    (1, 8, 2, 2048, True),
])
def test_flash_attn_bwd(B, Hq, Hkv, S, causal):
    from neuronx_distributed_amd.ops import _load

    if not hasattr(_load(), "flash_attn_bwd"):
        pytest.skip("bwd kernel not built yet")
    torch.manual_seed(5)
    D = 128
    q = torch.randn(B, Hq, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    k = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    v = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    out = ops.flash_attn(q * 0.5, k * 0.5, v * 0.5, causal=causal)
    dy = torch.randn_like(out)
    out.backward(dy)

    qr = (q.detach() * 0.5).float().requires_grad_(True)
    kr = (k.detach() * 0.5).float().requires_grad_(True)
    vr = (v.detach() * 0.5).float().requires_grad_(True)
    ref = _torch_reference(qr, kr, vr, causal=causal)
    ref.backward(dy.float())
    _cmp(q.grad, qr.grad * 0.5, atol=5e-2, rtol=5e-2, name="dq")
    _cmp(k.grad, kr.grad * 0.5, atol=5e-2, rtol=5e-2, name="dk")
    _cmp(v.grad, vr.grad * 0.5, atol=5e-2, rtol=5e-2, name="dv")


@pytest.mark.parametrize("Hq,Hkv,heads", [(4, 1, 1), (4, 1, 2), (4, 1, 4),
                                          (6, 2, 2), (6, 2, 6)])
@pytest.mark.parametrize("S,causal,window,scale", [
    (1, True, 0, 0.09), (64, True, 0, -0.09), (129, True, 0, 0.09),
    (333, True, 70, 0.09), (700, True, 130, -0.09), (290, False, 0, 0.09)])
def test_flash_attn_bwd_sums_heads_in_a_workgroup(monkeypatch, Hq, Hkv, heads,
                                                  S, causal, window, scale):
    """dK and dV of one, some or all q heads of a kv head from a workgroup."""
    monkeypatch.setattr(ops, "_fa_dkv_heads", lambda *a: heads)
    torch.manual_seed(S)
    B, D = 2, 128
    leaves = [torch.randn(B, S, h, D, device="cuda").bfloat16().requires_grad_()
              for h in (Hq, Hkv, Hkv)]
    dy = torch.randn(B, S, Hq, D, device="cuda").bfloat16().transpose(1, 2)
    out = ops.flash_attn(*(t.transpose(1, 2) for t in leaves), causal, scale,
                         window)
    got = torch.autograd.grad(out, leaves, dy)
    exact = [t.detach().double().cpu().requires_grad_() for t in leaves]
    ref = _torch_reference(*(t.transpose(1, 2) for t in exact), causal, scale,
                           window or None)
    want = torch.autograd.grad(ref, exact, dy.double().cpu())
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        # P, dS and the results are rounded to bf16 once each, 2^-9 relative
        err = (a.double().cpu() - b).norm() / b.norm().clamp(min=1e-3)
        assert err < 3 * 2 ** -8, (name, err)


@pytest.mark.parametrize("pitch", [(1 << 25) - 8, 1 << 25])
def test_flash_attn_of_rows_far_apart(pitch):
    """Rows as far apart as 31 bits of bytes reach, and one word further, where
    they are copied: the same bits as of rows that follow each other."""
    torch.manual_seed(3)
    S, D = 40, 128
    near = [torch.randn(1, 1, S, D, device="cuda").bfloat16() for _ in range(4)]
    # all four in the gaps of one another
    room = torch.empty((S - 1) * pitch + 4 * D, dtype=torch.bfloat16,
                       device="cuda")
    far = []
    for i, t in enumerate(near):
        view = room[i * D:].as_strided((1, 1, S, D), (8, 8, pitch, 1))
        far.append(view.copy_(t))

    def run(q, k, v, dy):
        q, k, v = (t.detach().requires_grad_() for t in (q, k, v))
        out = ops.flash_attn(q, k, v, True, 0.09, 0)
        return (out, *torch.autograd.grad(out, (q, k, v), dy))

    for a, b in zip(run(*far), run(*near)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("row", [75, 199])
@pytest.mark.parametrize("bad", [math.nan, math.inf, -math.inf])
@pytest.mark.parametrize("causal,window", [(True, None), (True, 70),
                                           (False, None)])
def test_flash_attn_bwd_of_a_row_without_weights(causal, window, bad, row):
    """A row whose lse is no number reaches the keys that it sees, and nothing
    else: all other gradients are the same bits."""
    from neuronx_distributed_amd.kernels.ring_attn import _block_bwd, _block_fwd

    torch.manual_seed(7)
    B, Hq, Hkv, S, D, head = 1, 4, 2, 200, 128, 1
    q, dout = (torch.randn(B, Hq, S, D, device="cuda").bfloat16()
               for _ in range(2))
    k, v = (torch.randn(B, Hkv, S, D, device="cuda").bfloat16()
            for _ in range(2))
    out, lse = _block_fwd(q, k, v, causal, 0.09, window)
    out = out.bfloat16()
    want = _block_bwd(q, k, v, out, dout, lse, causal, 0.09, window)
    lse = lse.clone()
    lse[0, head, row] = bad
    dq, dk, dv = _block_bwd(q, k, v, out, dout, lse, causal, 0.09, window)
    alone = torch.ones(B, Hq, S, dtype=torch.bool)
    alone[0, head, row] = False
    assert torch.equal(dq[alone.cuda()], want[0][alone.cuda()])
    unseen = torch.ones(B, Hkv, S, dtype=torch.bool)
    unseen[0, 0, row - window + 1 if window else 0:
           row + 1 if causal else S] = False
    for got, w in ((dk, want[1]), (dv, want[2])):
        assert torch.equal(got[unseen.cuda()], w[unseen.cuda()])
        if math.isnan(bad):
            assert got[~unseen.cuda()].isnan().all()


def test_flash_attn_bwd_heads_of_a_workgroup():
    """They divide the group, and no CU is left idle for them."""
    for B, Hq, Hkv, S, causal, window, n in (
            (2, 32, 8, 3001, True, 1024, 2), (1, 32, 8, 8192, True, 0, 4),
            (1, 32, 8, 4096, True, 0, 2), (1, 28, 4, 300, True, 0, 1),
            (1, 40, 40, 5000, True, 0, 1), (2, 32, 8, 2000, False, 0, 4)):
        assert ops._fa_dkv_heads(B, Hq, Hkv, S, causal, window) * n == Hq


@pytest.mark.parametrize("B,Hq,Hkv,S", [
    (2, 8, 2, 512),
    (1, 32, 8, 2048),   # production GQA shape
])
def test_flash_attn_strided_bshd_matches_contiguous(B, Hq, Hkv, S):
    """BSHD transpose views (the model's native activation layout) must
    produce bit-identical results to the contiguous-BHSD path, fwd AND
    bwd — validates the stride-parametrized kernels and the
    layout-preserving output allocation (no hidden .contiguous())."""
    torch.manual_seed(7)
    D = 128

    def mk(h, grad):
        t = torch.randn(B, S, h, D, dtype=torch.bfloat16, device="cuda")
        t = t * 0.5
        return t.requires_grad_(grad)

    q_b, k_b, v_b = mk(Hq, True), mk(Hkv, True), mk(Hkv, True)
    # strided path: transpose VIEWS go straight into the kernel
    qv, kv, vv = (t.transpose(1, 2) for t in (q_b, k_b, v_b))
    assert not qv.is_contiguous()
    out_s = ops.flash_attn(qv, kv, vv, causal=True)
    # the output comes back in BSHD storage: downstream reshape is a view
    assert out_s.transpose(1, 2).is_contiguous()
    dy = torch.randn_like(out_s)
    out_s.backward(dy)
    gq_s, gk_s, gv_s = (t.grad.clone() for t in (q_b, k_b, v_b))
    for t in (q_b, k_b, v_b):
        t.grad = None

    # contiguous path on identical values
    qc = q_b.detach().transpose(1, 2).contiguous().requires_grad_(True)
    kc = k_b.detach().transpose(1, 2).contiguous().requires_grad_(True)
    vc = v_b.detach().transpose(1, 2).contiguous().requires_grad_(True)
    out_c = ops.flash_attn(qc, kc, vc, causal=True)
    out_c.backward(dy.contiguous())
    torch.cuda.synchronize()
    assert torch.equal(out_s.contiguous(), out_c), "fwd strided != contig"
    assert torch.equal(gq_s.transpose(1, 2), qc.grad), "dq mismatch"
    assert torch.equal(gk_s.transpose(1, 2), kc.grad), "dk mismatch"
    assert torch.equal(gv_s.transpose(1, 2), vc.grad), "dv mismatch"


@pytest.mark.parametrize("B,Hq,Hkv,pos", [
    (32, 32, 8, 1023),   # llama3-8b decode shape, batch 32
    (4, 8, 8, 511),      # MHA
    (1, 4, 1, 63),       # extreme GQA, tiny batch
])
def test_decode_attn_numerics(B, Hq, Hkv, pos):
    """Fused decode attention (RoPE + cache append + flash-decode + GQA)
    vs a plain fp32 torch reference over the same cache."""
    if not ops.decode_attn_available():
        pytest.skip("decode_attn kernel not built")
    torch.manual_seed(11)
    D, Smax = 128, pos + 65
    dev = "cuda"
    cos, sin = ops.precompute_rope_freqs(Smax, D, device=dev)
    kcache = torch.randn(B, Hkv, Smax, D, dtype=torch.bfloat16, device=dev) * 0.5
    vcache = torch.randn(B, Hkv, Smax, D, dtype=torch.bfloat16, device=dev) * 0.5
    kcache[:, :, pos:] = 0
    vcache[:, :, pos:] = 0
    kc_ref = kcache.clone()
    vc_ref = vcache.clone()
    q2 = torch.randn(B, Hq * D, dtype=torch.bfloat16, device=dev) * 0.5
    k2 = torch.randn(B, Hkv * D, dtype=torch.bfloat16, device=dev) * 0.5
    v2 = torch.randn(B, Hkv * D, dtype=torch.bfloat16, device=dev) * 0.5
    pos_t = torch.tensor([pos], dtype=torch.int64, device=dev)
    scale = 1.0 / math.sqrt(D)

    out = ops.decode_attn_step(q2, k2, v2, kcache, vcache, cos, sin, pos_t,
                               Hq, Hkv, scale)
    torch.cuda.synchronize()

    # ---- torch fp32 reference -----------------------------------------
    def rope(x, p):  # x (B, H, D)
        c = cos[p].float()  # (D/2,)
        s = sin[p].float()
        x = x.float()
        x1, x2 = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1)

    q = rope(q2.view(B, Hq, D), pos)
    k_new = rope(k2.view(B, Hkv, D), pos)
    kc = kc_ref.float()
    vc = vc_ref.float()
    kc[:, :, pos] = k_new
    vc[:, :, pos] = v2.view(B, Hkv, D).float()
    rep = Hq // Hkv
    kx = kc[:, :, : pos + 1].repeat_interleave(rep, dim=1)
    vx = vc[:, :, : pos + 1].repeat_interleave(rep, dim=1)
    att = torch.softmax((q.unsqueeze(2) @ kx.transpose(-1, -2)) * scale, -1)
    ref = (att @ vx).squeeze(2).reshape(B, Hq * D)
    _cmp(out, ref, atol=3e-2, name=f"decode_attn B{B} Hq{Hq}")
    # the kernel must also have appended to the cache
    _cmp(kcache[:, :, pos].float(), k_new, atol=2e-2, name="cache k append")
    _cmp(vcache[:, :, pos].float(), v2.view(B, Hkv, D).float(), atol=1e-3,
         name="cache v append")


def test_add_rmsnorm_matches_unfused():
    """Fused residual-add + RMSNorm vs the unfused bf16 add -> rmsnorm."""
    if not ops.add_rmsnorm_available():
        pytest.skip("add_rmsnorm not built")
    torch.manual_seed(6)
    for rows, H in ((32, 4096), (128, 1024), (7, 512)):
        r = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
        d = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
        w = torch.randn(H, dtype=torch.bfloat16, device="cuda")
        res_out, normed = ops.add_rmsnorm(r, d, w, 1e-5)
        ref_res = r + d  # bf16 rounding like the kernel
        ref = ref_res.float() * torch.rsqrt(
            ref_res.float().pow(2).mean(-1, keepdim=True) + 1e-5) * w.float()
        _cmp(res_out, ref_res, atol=1e-6, name=f"add_rmsnorm res {H}")
        _cmp(normed, ref, atol=2e-2, name=f"add_rmsnorm out {H}")


def test_fused_adamw_matches_torch():
    torch.manual_seed(7)
    n = 10007
    master = torch.randn(n, dtype=torch.float32, device="cuda")
    m = torch.randn(n, device="cuda").abs() * 0.01
    v = torch.randn(n, device="cuda").abs() * 0.001
    grad = torch.randn(n, dtype=torch.bfloat16, device="cuda")
    param = torch.zeros(n, dtype=torch.bfloat16, device="cuda")
    clip = torch.tensor([0.7], device="cuda")

    mm, vv, ww = m.clone(), v.clone(), master.clone()
    lr, b1, b2, eps, wd, t = 1e-3, 0.9, 0.95, 1e-8, 0.1, 3
    g = grad.float() * clip
    mm = b1 * mm + (1 - b1) * g
    vv = b2 * vv + (1 - b2) * g * g
    ww = ww * (1 - lr * wd)
    ww = ww - lr * (mm / (1 - b1 ** t)) / ((vv / (1 - b2 ** t)).sqrt() + eps)

    ops.adamw_step(master, m, v, grad, param, clip, lr, b1, b2, eps, wd, t)
    torch.cuda.synchronize()
    _cmp(master, ww, atol=1e-5, rtol=1e-4, name="fused adamw master")
    _cmp(m, mm, atol=1e-6, name="fused adamw m")
    _cmp(v, vv, atol=1e-7, name="fused adamw v")
    _cmp(param, ww.to(torch.bfloat16), atol=1e-6, name="fused adamw param")


def test_fused_cross_entropy():
    import torch.distributed as dist
    import os

    os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
    os.environ.setdefault("MASTER_PORT", "29755")
    if not dist.is_initialized():
        dist.init_process_group("nccl", rank=0, world_size=1)
    from neuronx_distributed_amd.parallel import parallel_state as ps
    from neuronx_distributed_amd.parallel.loss_functions import (
        parallel_cross_entropy)

    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(tensor_model_parallel_size=1)
    torch.manual_seed(0)
    B, S, V = 2, 64, 1024
    logits = (torch.randn(B, S, V, device="cuda") * 2).to(torch.bfloat16)
    logits.requires_grad_(True)
    target = torch.randint(0, V, (B, S), device="cuda")
    loss = parallel_cross_entropy(logits, target)

    ref_in = logits.detach().float().requires_grad_(True)
    ref = torch.nn.functional.cross_entropy(
        ref_in.reshape(-1, V), target.reshape(-1),
        reduction="none").reshape(B, S)
    _cmp(loss, ref, atol=1e-2, name="fused CE fwd")
    g = torch.randn(B, S, device="cuda")
    loss.backward(g)
    ref.backward(g)
    _cmp(logits.grad, ref_in.grad, atol=2e-3, rtol=5e-2, name="fused CE bwd")


def test_fp8_scaled_linear_matches_bf16():
    """W8A8 fp8 MFMA GEMM (torch._scaled_mm) vs bf16 reference: per-channel
    weight scales + dynamic per-token activation scales keep relative
    error within fp8 e4m3 resolution."""
    from neuronx_distributed_amd.quantization.quantization_config import (
        QuantizationConfig, QuantizedDtype)
    from neuronx_distributed_amd.quantization.quantization_utils import (
        fp8_scaled_linear, quantize_symmetric)

    torch.manual_seed(0)
    M, N, K = 512, 256, 512
    x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * 0.05
    cfg = QuantizationConfig(quantized_dtype=QuantizedDtype.F8E4M3,
                             quantize_activation=True)
    q, s = quantize_symmetric(w, cfg)
    out = fp8_scaled_linear(x, q, s, torch.bfloat16)
    ref = x.float() @ w.float().t()
    rel = (out.float() - ref).norm() / ref.norm()
    assert rel < 0.05, f"rel err {rel}"


def test_fp8_quantized_layer_forward():
    """QuantizedColumnParallel.from_float with quantize_activation runs the
    scaled_mm path on GPU and stays close to the float layer."""
    import torch.distributed as dist
    from neuronx_distributed_amd.parallel import parallel_state as ps
    from neuronx_distributed_amd.parallel.layers import ColumnParallelLinear
    from neuronx_distributed_amd.quantization.quantization_config import (
        QuantizationConfig, QuantizedDtype)
    from neuronx_distributed_amd.quantization.quantization_layers import (
        QuantizedColumnParallel)

    if not dist.is_initialized():
        import os
        os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
        os.environ.setdefault("MASTER_PORT", "29541")
        dist.init_process_group("nccl", rank=0, world_size=1)
    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(tensor_model_parallel_size=1)
    torch.manual_seed(0)
    fl = ColumnParallelLinear(256, 128, bias=False, gather_output=False,
                              dtype=torch.bfloat16).cuda()
    cfg = QuantizationConfig(quantized_dtype=QuantizedDtype.F8E4M3,
                             quantize_activation=True)
    ql = QuantizedColumnParallel.from_float(fl, cfg).cuda()
    x = torch.randn(64, 256, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        out = ql(x)
        ref = fl(x)
    rel = (out.float() - ref.float()).norm() / ref.float().norm()
    assert out.dtype == torch.bfloat16
    assert rel < 0.06, f"rel err {rel}"


def test_moe_decode_fused_matches_reference():
    """Fused decode MoE kernels (moe_decode_glu) vs the dense all-experts
    computation on random routing."""
    torch.manual_seed(0)
    T, H, I, E, k = 24, 256, 192, 8, 2
    dev = "cuda"
    x = torch.randn(T, H, device=dev, dtype=torch.bfloat16)
    w_gu = torch.randn(E, H, 2 * I, device=dev, dtype=torch.bfloat16) * 0.05
    w_d = torch.randn(E, I, H, device=dev, dtype=torch.bfloat16) * 0.05
    logits = torch.randn(T, E, device=dev)
    aff_full = torch.softmax(logits, -1)
    vals, idx = torch.topk(aff_full, k, dim=-1)
    aff = torch.zeros_like(aff_full).scatter(-1, idx, vals)

    out = ops.moe_decode_glu(x, w_gu, w_d, aff, idx)

    # reference: dense per-expert MLP, affinity-combined in fp32
    ref = torch.zeros(T, H, device=dev, dtype=torch.float32)
    xf = x.float()
    for e in range(E):
        gu = xf @ w_gu[e].float()
        act = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
        ref += (act @ w_d[e].float()) * aff[:, e:e + 1].float()
    _cmp(out, ref.to(torch.bfloat16), atol=2e-2, name="moe_decode")


def test_moe_decode_imbalanced_routing():
    """All tokens on one expert (multiple blocks) + empty experts."""
    torch.manual_seed(1)
    T, H, I, E, k = 40, 128, 64, 4, 1
    dev = "cuda"
    x = torch.randn(T, H, device=dev, dtype=torch.bfloat16)
    w_gu = torch.randn(E, H, 2 * I, device=dev, dtype=torch.bfloat16) * 0.05
    w_d = torch.randn(E, I, H, device=dev, dtype=torch.bfloat16) * 0.05
    idx = torch.full((T, k), 2, dtype=torch.long, device=dev)
    aff = torch.zeros(T, E, device=dev)
    aff[:, 2] = 1.0

    out = ops.moe_decode_glu(x, w_gu, w_d, aff, idx)
    gu = x.float() @ w_gu[2].float()
    act = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    ref = act @ w_d[2].float()
    _cmp(out, ref.to(torch.bfloat16), atol=2e-2, name="moe_decode_imb")


def test_skinny_gemm_matches_matmul():
    """Products of few rows vs torch matmul (fp32 reference)."""
    torch.manual_seed(0)
    for M, N, K in [(32, 4096, 4096), (8, 1024, 11008), (1, 512, 256),
                    (32, 1000, 4096)]:
        x = torch.randn(M, K, device="cuda", dtype=torch.bfloat16)
        w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16) * 0.05
        out = ops.skinny_linear(x, w)
        ref = (x.float() @ w.float().t())
        _cmp(out, ref.to(torch.bfloat16), atol=2e-2,
             name=f"skinny_{M}x{N}x{K}")


@pytest.mark.parametrize("K,at,pitch", [(256, 1, 256), (256, 0, 257),
                                        (250, 0, 250), (7, 3, 9)])
def test_skinny_linear_of_rows_off_the_words(K, at, pitch):
    torch.manual_seed(K + at)

    def rows(n):
        return torch.randn(n * pitch + 8, device="cuda").bfloat16()[
            at:at + n * pitch].view(n, pitch)[:, :K]

    x, w = rows(5), rows(33)
    ref = x.double() @ w.double().t()
    # rounded once to 8 bits; K products of 32 bits
    torch.testing.assert_close(ops.skinny_linear(x, w).double(), ref,
                               rtol=2.0 ** -8, atol=K * 2.0 ** -22)


@pytest.mark.parametrize("bias", [False, True])
def test_layers_of_few_rows_match_64_bits(bias):
    """What the layers dispatch: own products of few rows, the library's of
    more rows, under autograd and with a bias."""
    from neuronx_distributed_amd.parallel.layers import \
        linear_with_async_allreduce

    torch.manual_seed(1)
    x = torch.randn(40, 1, 4096, device="cuda").bfloat16()
    w = torch.randn(6144, 4096, device="cuda").div(64).bfloat16()
    b = torch.randn(6144, device="cuda").bfloat16() if bias else None
    for rows in (1, 4, 5, 32, 40):
        with torch.no_grad():
            assert ops.use_skinny_linear(x[:rows], w) == (rows <= 4)
            out = linear_with_async_allreduce(x[:rows], w, b)
        ref = x[:rows].double() @ w.double().t()
        ref = ref + b.double() if bias else ref
        # sums of about 1 rounded once to 8 bits, with a bias twice
        torch.testing.assert_close(out.double(), ref, rtol=2.0 ** -7,
                                   atol=4096 * 2.0 ** -22)
    assert not ops.use_skinny_linear(x[:1], w)         # under autograd


def test_ring_block_primitives_gpu():
    """The ring-attention per-block fwd/bwd (HIP flash kernels + global-lse
    decomposition) match the CPU torch implementations on one block."""
    import math as _math

    from neuronx_distributed_amd.kernels.ring_attn import (_block_bwd,
                                                           _block_fwd)

    torch.manual_seed(0)
    B, H, S, D = 1, 4, 256, 128
    scale = 1.0 / _math.sqrt(D)
    q = torch.randn(B, H, S, D, dtype=torch.bfloat16)
    k = torch.randn(B, H, S, D, dtype=torch.bfloat16)
    v = torch.randn(B, H, S, D, dtype=torch.bfloat16)
    o_cpu, lse_cpu = _block_fwd(q, k, v, True, scale)
    o_gpu, lse_gpu = _block_fwd(q.cuda(), k.cuda(), v.cuda(), True, scale)
    _cmp(o_gpu, o_cpu, atol=3e-2, name="ring_block_fwd")
    _cmp(lse_gpu, lse_cpu, atol=2e-3, name="ring_block_lse")

    do = torch.randn_like(q)
    dq_c, dk_c, dv_c = _block_bwd(q, k, v, o_cpu, do, lse_cpu, True, scale)
    dq_g, dk_g, dv_g = _block_bwd(q.cuda(), k.cuda(), v.cuda(), o_gpu,
                                  do.cuda(), lse_gpu, True, scale)
    _cmp(dq_g, dq_c, atol=5e-2, name="ring_block_dq")
    _cmp(dk_g, dk_c, atol=5e-2, name="ring_block_dk")
    _cmp(dv_g, dv_c, atol=5e-2, name="ring_block_dv")


def test_fused_ce_ignore_index():
    """Fused CE path zeroes loss AND grad at ignore_index targets
    (mask-multiply routes zero grad_output into ce_bwd)."""
    import torch.distributed as dist
    from neuronx_distributed_amd.parallel import parallel_state as ps
    from neuronx_distributed_amd.parallel.loss_functions import (
        parallel_cross_entropy)

    if not dist.is_initialized():
        os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
        os.environ.setdefault("MASTER_PORT", "29553")
        dist.init_process_group("nccl", rank=0, world_size=1)
    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(tensor_model_parallel_size=1)
    torch.manual_seed(0)
    logits = torch.randn(6, 64, device="cuda", dtype=torch.bfloat16,
                         requires_grad=True)
    tgt = torch.tensor([1, 3, -100, 7, -100, 12], device="cuda")
    loss = parallel_cross_entropy(logits, tgt)
    assert float(loss[2]) == 0.0 and float(loss[4]) == 0.0
    (loss.sum() / 4).backward()
    g = logits.grad.float()
    assert g[2].abs().max().item() == 0.0
    assert g[4].abs().max().item() == 0.0
    assert torch.isfinite(loss).all()


@pytest.mark.parametrize("B,Hq,Hkv,S,W", [
    (1, 4, 4, 1024, 256),
    (2, 8, 2, 2048, 512),   # GQA + window smaller than seq
    (1, 2, 2, 512, 4096),   # window larger than seq == plain causal
])
def test_flash_attn_sliding_window(B, Hq, Hkv, S, W):
    """Sliding-window MFMA kernel vs the fp32 composed reference."""
    if not ops.flash_attn_window_available():
        pytest.skip("window kernel not built")
    torch.manual_seed(9)
    D = 128
    q = torch.randn(B, Hq, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    k = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    v = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda") * 0.5
    out = ops.flash_attn_windowed(q, k, v, W)
    ref = _torch_reference(q.float(), k.float(), v.float(), causal=True,
                           window=W)
    _cmp(out, ref, atol=3e-2, rtol=3e-2, name=f"window S={S} W={W}")


@pytest.mark.parametrize("S,window,causal", [
    (1, 0, True), (31, 0, True), (64, 0, True), (65, 0, True),
    (127, 0, False), (128, 0, True), (129, 0, True), (191, 0, False),
    (257, 0, True), (300, 33, True), (513, 64, True), (640, 200, True),
])
@pytest.mark.parametrize("Hq,Hkv,scale,offset", [
    (4, 2, None, 0), (2, 2, -0.05, 0), (3, 1, 0.2, 1)])
def test_flash_attn_tile_edges(S, window, causal, Hq, Hkv, scale, offset):
    """Forward and backward at the edges of the 32-row waves, 64-key tiles and
    128-row workgroups; a scale of either sign; rows that start between two
    16-byte words (``offset`` elements into their storage)."""
    torch.manual_seed(S + Hq)
    B, D = 2, 128

    def make(h):
        n = B * S * h * D
        t = torch.randn(n + offset, device="cuda").bfloat16()[offset:]
        return t.view(B, S, h, D).transpose(1, 2).requires_grad_(True)

    q, k, v = make(Hq), make(Hkv), make(Hkv)
    dy = make(Hq).detach()
    out = ops.flash_attn(q, k, v, causal, scale, window)
    got = (out, *torch.autograd.grad(out, (q, k, v), dy))
    qr, kr, vr = (t.detach().float().requires_grad_(True) for t in (q, k, v))
    ref = _torch_reference(qr, kr, vr, causal, scale, window or None)
    want = (ref, *torch.autograd.grad(ref, (qr, kr, vr), dy.float()))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        # weights, their gradients and the result are rounded to bf16, 2^-9
        # each; gradients that vanish leave the rounding of their summands
        bound = 3 * 2.0 ** -9 * (b.norm() + 0.05 * b.numel() ** 0.5)
        assert (a.float() - b).norm() <= bound, name


@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (16, 16), (24, 6), (40, 8), (20, 4)])
def test_flash_attn_heads_go_to_their_xcd(Hq, Hkv):
    """Every head is taken once, with the keys of its group, where heads are a
    multiple of the XCDs and where they are not."""
    torch.manual_seed(Hq)
    B, S, D = 2, 193, 128
    q, k, v = (torch.randn(B, h, S, D, device="cuda").bfloat16().requires_grad_(True)
               for h in (Hq, Hkv, Hkv))
    dy = torch.randn(B, Hq, S, D, device="cuda").bfloat16()
    out = ops.flash_attn(q, k, v)
    got = (out, *torch.autograd.grad(out, (q, k, v), dy))
    qr, kr, vr = (t.detach().float().requires_grad_(True) for t in (q, k, v))
    ref = _torch_reference(qr, kr, vr)
    want = (ref, *torch.autograd.grad(ref, (qr, kr, vr), dy.float()))
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        # as above, of every head by itself
        bound = 3 * 2.0 ** -9 * (b.norm(dim=(2, 3)) + 0.05 * (S * D) ** 0.5)
        assert ((a.float() - b).norm(dim=(2, 3)) <= bound).all(), name


@pytest.mark.parametrize("B,Hq,Hkv,S,causal,window,layout", [
    (1, 4, 4, 1, True, 0, "bshd"), (2, 8, 2, 193, True, 0, "bshd"),
    (2, 6, 2, 300, True, 70, "bhsd"), (1, 4, 1, 129, False, 0, "bhsd"),
    (1, 4, 2, 140, True, 0, "odd"), (1, 4, 2, 140, True, 0, "between")])
def test_native_flash_attn_is_pythons(monkeypatch, B, Hq, Hkv, S, causal, window,
                                      layout):
    """The native autograd function and Python's: the same bits and strides, with
    saved tensors that a hook takes through the host."""
    torch.manual_seed(S)
    assert ops._native_flash() is not None

    def make(h):
        if layout == "bshd":
            t = torch.randn(B, S, h, 128, device="cuda").bfloat16().transpose(1, 2)
        elif layout == "odd":              # rows of 129 elements
            t = torch.randn(B, h, S, 129, device="cuda").bfloat16()[..., :128]
        elif layout == "between":          # rows that start between two words
            t = torch.randn(B * h * S * 128 + 3, device="cuda").bfloat16()[3:]
            t = t.view(B, h, S, 128)
        else:
            t = torch.randn(B, h, S, 128, device="cuda").bfloat16()
        return t.detach().requires_grad_(True)

    q, k, v, dy = make(Hq), make(Hkv), make(Hkv), make(Hq).detach()
    moved, got = [], []

    def pack(t):
        moved.append(t.shape)
        return t.cpu()

    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_native_flash", lambda: None)
        with torch.no_grad():
            plain = ops.flash_attn(q, k, v, causal, None, window)
        out = ops.flash_attn(q, k, v, causal, None, window)
        grads = torch.autograd.grad(out, (q, k, v), dy)
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
            again = ops.flash_attn(q, k, v, causal, None, window)
        hooked = torch.autograd.grad(again, (q, k, v), dy)
        for a, b in zip(grads, hooked):
            assert torch.equal(a, b)
        got.append((plain, out.detach(), *grads))
    assert len(moved) == 10
    for a, b in zip(*got):
        assert torch.equal(a, b) and a.stride() == b.stride()


def test_native_flash_attn_leaves_others_to_python():
    q = torch.randn(1, 2, 64, 128, device="cuda").bfloat16()

    class Seen(torch.Tensor):
        pass

    assert ops._fa_native(q, q, q)
    for t in (q.float(), q[..., :64], q[0], q.as_subclass(Seen)):
        assert not ops._fa_native(t, t, t) and not ops._fa_native(q, t, q)
    with torch.autograd.forward_ad.dual_level():
        assert not ops._fa_native(q, q, q)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not ops._fa_native(q, q, q)
    with pytest.raises(AssertionError):
        ops.flash_attn(q.float(), q.float(), q.float())


def test_native_flash_attn_leaves_watched_calls_to_python():
    """Transforms, and dispatch and function modes: what they see is Python's function,
    which functorch refuses as it did."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    q = torch.randn(1, 2, 64, 128, device="cuda").bfloat16()
    seen = []

    def look(x):
        seen.append(ops._fa_native(x, x, x))
        return x.float().sum()

    torch.func.grad(look)(q)
    torch.func.vmap(look)(q[None])
    torch.func.jvp(look, (q,), (q,))
    assert seen == [False] * 3
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda x: ops.flash_attn(x, x, x).float().sum())(q)

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    want = ops.flash_attn(q, q, q)
    for mode in (Dispatch, Function):
        with mode():
            assert not ops._fa_native(q, q, q)
            got = ops.flash_attn(q, q, q)
        assert torch.equal(got, want)
    with torch.inference_mode():
        assert ops._fa_native(q, q, q)
        assert torch.equal(ops.flash_attn(q, q, q), want)


@pytest.mark.parametrize("how", ["stream", "checkpoint", "twice", "create_graph"])
def test_native_flash_attn_in_a_program(monkeypatch, how):
    """On a stream of its own, recomputed, differentiated twice from one graph, and by a
    graph of the gradients, which ends there: as Python's."""
    from torch.utils.checkpoint import checkpoint

    torch.manual_seed(3)
    q, k, v = (torch.randn(1, 200, h, 128, device="cuda").bfloat16().transpose(1, 2)
               .requires_grad_(True) for h in (4, 2, 2))
    dy = torch.randn(1, 4, 200, 128, device="cuda").bfloat16()
    side, got = torch.cuda.Stream(), []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(ops, "_native_flash", lambda: None)
        torch.cuda.synchronize()
        if how == "stream":
            with torch.cuda.stream(side):
                x = [t * 2 for t in (q, k, v)]       # (what the call has to wait for)
                out = ops.flash_attn(*x) * 2
                grads = torch.autograd.grad(out, (q, k, v), dy)
            side.synchronize()
        elif how == "checkpoint":
            out = checkpoint(lambda *x: ops.flash_attn(*x) * 2, q, k, v,
                             use_reentrant=False)
            grads = torch.autograd.grad(out, (q, k, v), dy)
        else:
            out = ops.flash_attn(q, k, v)
            grads = torch.autograd.grad(out, (q, k, v), dy, retain_graph=True,
                                        create_graph=how == "create_graph")
            if how == "twice":
                again = torch.autograd.grad(out, (q, k, v), dy)
                assert all(torch.equal(a, b) for a, b in zip(grads, again))
                with pytest.raises(RuntimeError):    # the graph is freed
                    torch.autograd.grad(out, (q, k, v), dy)
        got.append((out.detach(), *grads))
    for a, b in zip(*got):
        assert torch.equal(a, b) and a.requires_grad == b.requires_grad


def test_add_rmsnorm_train_matches_unfused_autograd():
    """Training fused add+RMSNorm (fwd + the dpass-folding backward) vs
    the unfused bf16 add -> ops.rmsnorm chain: forward outputs equal and
    gradients equal (the kernel computes norm stats on the rounded sum,
    so the chains are arithmetically identical)."""
    torch.manual_seed(11)
    rows, H = 512, 1024
    delta = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
    res = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(H, dtype=torch.bfloat16, device="cuda")

    d1 = delta.clone().requires_grad_(True)
    r1 = res.clone().requires_grad_(True)
    w1 = w.clone().requires_grad_(True)
    h1, n1 = ops.add_rmsnorm_train(d1, r1, w1, 1e-5)
    # both outputs used downstream (residual carried + normed consumed),
    # like a decoder layer
    loss1 = (n1.float().pow(2).sum() + 0.5 * h1.float().sum())
    loss1.backward()

    d2 = delta.clone().requires_grad_(True)
    r2 = res.clone().requires_grad_(True)
    w2 = w.clone().requires_grad_(True)
    h2 = d2 + r2
    n2 = ops.rmsnorm(h2, w2, 1e-5)
    loss2 = (n2.float().pow(2).sum() + 0.5 * h2.float().sum())
    loss2.backward()
    torch.cuda.synchronize()

    assert torch.equal(h1, h2)
    _cmp(n1, n2, atol=1e-3, name="normed")
    _cmp(d1.grad, d2.grad, atol=2e-2, rtol=2e-2, name="ddelta")
    _cmp(r1.grad, r2.grad, atol=2e-2, rtol=2e-2, name="dres")
    _cmp(w1.grad, w2.grad, atol=2e-1, rtol=2e-2, name="dw")


def test_add_rmsnorm_train_final_norm_no_dh():
    """Final-norm use: the carried h output is dropped (dh is None) —
    the backward must fall back to the plain rmsnorm_bwd kernel."""
    torch.manual_seed(12)
    rows, H = 64, 512
    delta = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda",
                        requires_grad=True)
    res = torch.randn(rows, H, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(H, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    _, normed = ops.add_rmsnorm_train(delta, res, w, 1e-5)
    normed.float().pow(2).sum().backward()

    d2 = delta.detach().clone().requires_grad_(True)
    w2 = w.detach().clone().requires_grad_(True)
    n2 = ops.rmsnorm(d2 + res, w2, 1e-5)
    n2.float().pow(2).sum().backward()
    torch.cuda.synchronize()
    _cmp(delta.grad, d2.grad, atol=2e-2, rtol=2e-2, name="ddelta")
    _cmp(w.grad, w2.grad, atol=2e-1, rtol=2e-2, name="dw")


@pytest.mark.parametrize("B,Hq,Hkv,S,W", [
    (1, 4, 2, 512, 128),
    (1, 2, 2, 448, 200),    # ragged S, window not a tile multiple
    (2, 8, 2, 1024, 256),
])
def test_flash_attn_windowed_bwd(B, Hq, Hkv, S, W):
    """Sliding-window flash TRAINING path (fwd band masks + windowed
    dkdv/dq backward) vs the composed windowed reference."""
    torch.manual_seed(13)
    D = 128
    q = torch.randn(B, Hq, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    k = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    v = torch.randn(B, Hkv, S, D, dtype=torch.bfloat16, device="cuda",
                    requires_grad=True)
    out = ops.flash_attn(q * 0.5, k * 0.5, v * 0.5, causal=True, window=W)
    ref_in = [(t.detach() * 0.5).float().requires_grad_(True)
              for t in (q, k, v)]
    ref = _torch_reference(*ref_in, causal=True, window=W)
    _cmp(out, ref, atol=3e-2, rtol=3e-2, name=f"win fwd W={W}")
    dy = torch.randn_like(out)
    out.backward(dy)
    ref.backward(dy.float())
    _cmp(q.grad, ref_in[0].grad * 0.5, atol=5e-2, rtol=5e-2, name="win dq")
    _cmp(k.grad, ref_in[1].grad * 0.5, atol=5e-2, rtol=5e-2, name="win dk")
    _cmp(v.grad, ref_in[2].grad * 0.5, atol=5e-2, rtol=5e-2, name="win dv")


def _one_rank():
    import torch.distributed as dist
    from neuronx_distributed_amd.parallel import parallel_state as ps

    if not dist.is_initialized():
        os.environ.setdefault("MASTER_ADDR", "127.0.0.1")
        os.environ.setdefault("MASTER_PORT", "29553")
        dist.init_process_group("nccl", rank=0, world_size=1)
    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(tensor_model_parallel_size=1)


@pytest.mark.parametrize("N,V", [(1, 8), (3, 2040), (5, 2048), (2, 8200),
                                 (2100, 16376)])
def test_fused_ce_in_one_pass(N, V):
    """Loss and gradient against 64 bits; rows that rise, that hold -inf and
    that are far out; an ignored row of NaN stays out of both."""
    from neuronx_distributed_amd.parallel.loss_functions import (
        parallel_cross_entropy)

    _one_rank()
    torch.manual_seed(0)
    x = torch.randn(N, V, device="cuda")
    tgt = torch.randint(0, V, (N,), device="cuda")
    if N > 2:
        x[0] = torch.linspace(-30, 30, V)
        x[1] -= 3e4
        x[2, 1::2] = float("-inf")
        tgt[2] = 4
    if N > 4:
        x[3] = float("nan")
        tgt[3] = -100
    x = x.bfloat16().requires_grad_()
    loss = parallel_cross_entropy(x, tgt)
    (loss * torch.arange(1, N + 1, device="cuda")).sum().backward()
    keep = tgt != -100
    d = x.detach().double()[keep].requires_grad_()
    ref = torch.nn.functional.cross_entropy(d, tgt[keep], reduction="none")
    (ref * torch.arange(1, N + 1, device="cuda")[keep]).sum().backward()
    # V exponentials of 2 ulp summed in 32 bits, each thread V / 256 of them
    torch.testing.assert_close(loss[keep].double(), ref.detach(), rtol=1e-5,
                               atol=2.0 ** -23 * (8 + V / 256))
    torch.testing.assert_close(x.grad[keep].double(), d.grad, rtol=2.0 ** -7,
                               atol=1e-6 * N)
    assert (loss[~keep] == 0).all() and (x.grad[~keep] == 0).all()


def test_next_token_loss_ignores_the_last_position():
    from neuronx_distributed_amd.parallel.loss_functions import (
        next_token_cross_entropy, parallel_cross_entropy)

    _one_rank()
    torch.manual_seed(1)
    x = torch.randn(2, 37, 512, device="cuda").bfloat16()
    labels = torch.randint(0, 512, (2, 37), device="cuda")
    labels[0, 5:9] = -100
    a, b = (x.clone().requires_grad_() for _ in range(2))
    want = parallel_cross_entropy(a[:, :-1].contiguous(),
                                  labels[:, 1:].contiguous())
    got = next_token_cross_entropy(b, labels)
    assert torch.equal(got[:, :-1], want) and (got[:, -1] == 0).all()
    want.sum().backward()
    got.sum().backward()
    assert torch.equal(a.grad, b.grad)
    assert next_token_cross_entropy(x.float(), labels) is None
    assert next_token_cross_entropy(x.cpu(), labels.cpu()) is None


def test_ce_shards_meet_at_the_common_max():
    """What ranks all-reduce, for two halves of the vocabulary in one process;
    one half all -inf in a row."""
    from neuronx_distributed_amd.parallel import loss_functions as lf

    torch.manual_seed(2)
    x = torch.randn(6, 512, device="cuda").mul(4).bfloat16()
    x[2, :256] = float("-inf")
    tgt = torch.tensor([0, 255, 300, 511, -100, 256], device="cuda")
    parts = []
    for i in range(2):
        half = x[:, i * 256:(i + 1) * 256].contiguous()
        st = torch.empty(3, 6, device="cuda")
        ops._require_lib().ce_stats(
            ops._ptr(half), ops._ptr(tgt), ops._ptr(st[0]), ops._ptr(st[1]),
            ops._ptr(st[2]), ctypes.c_long(6), ctypes.c_int(256),
            ctypes.c_long(256 * i), ops._stream())
        parts.append(st)
    top = torch.maximum(parts[0][0], parts[1][0])
    both = sum(lf._over(top, *p, (tgt >= 256 * i) & (tgt < 256 * i + 256))
               for i, p in enumerate(parts))
    loss = (both[0].log() - both[1]).double()
    ref = torch.nn.functional.cross_entropy(x.double(), tgt.clamp(min=0),
                                            reduction="none")
    keep = tgt >= 0
    torch.testing.assert_close(loss[keep], ref[keep], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("rows,H", [(1, 8), (2, 2048), (511, 2056),
                                    (513, 4096), (1025, 4104), (3, 6152),
                                    (1030, 8192), (515, 8200), (0, 64)])
@pytest.mark.parametrize("forked", [False, True])
def test_rmsnorm_rows_and_widths(rows, H, forked):
    """Forward and backward against 64 bits around the rows of a round of
    workgroups and the columns of a thread."""
    torch.manual_seed(rows + H)
    x, r = (torch.randn(rows, H, device="cuda").bfloat16().requires_grad_()
            for _ in range(2))
    w = torch.randn(H, device="cuda").bfloat16().requires_grad_()
    gy, gh = (torch.randn(rows, H, device="cuda").bfloat16()
              for _ in range(2))
    if forked:
        h, y = ops.add_rmsnorm_train(x, r, w, 1e-5)
        torch.autograd.backward([h, y], [gh, gy])
    else:
        y = ops.rmsnorm(x, w, 1e-5)
        y.backward(gy)
    d = (x + r if forked else x).detach().double().requires_grad_()
    wd = w.detach().double().requires_grad_()
    ref = d * torch.rsqrt(d.pow(2).mean(-1, keepdim=True) + 1e-5) * wd
    ref.backward(gy.double())
    # rounded once to 8 bits; 32-bit sums of H columns or of the rows
    for got, want in ((y, ref), (x.grad, d.grad + (gh if forked else 0))):
        torch.testing.assert_close(got.double(), want, rtol=2.0 ** -7,
                                   atol=1e-4)
    torch.testing.assert_close(w.grad.double(), wd.grad, rtol=2.0 ** -7,
                               atol=1e-4 * max(rows, 1) ** 0.5)
    if forked:
        assert torch.equal(x.grad, r.grad)


@pytest.mark.parametrize("form", ["plain", "forked", "inference"])
def test_norms_read_a_32_bit_weight_as_it_is(form):
    """bf16 rows beside a float32 weight, against 64 bits."""
    torch.manual_seed(3)
    x, r, gy, gh = (torch.randn(5, 512, device="cuda").bfloat16()
                    for _ in range(4))
    w = torch.randn(512, device="cuda")
    wd = w.double().requires_grad_()
    xd = (x if form == "plain" else x + r).double().requires_grad_()
    ref = xd * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5) * wd
    if form == "inference":
        h, y = ops.add_rmsnorm(r, x, w, 1e-5)
        assert torch.equal(h, x + r)
    else:
        x.requires_grad_()
        w.requires_grad_()
        if form == "plain":
            y = ops.rmsnorm(x, w, 1e-5)
            y.backward(gy)
        else:
            h, y = ops.add_rmsnorm_train(x, r, w, 1e-5)
            torch.autograd.backward([h, y], [gh, gy])
        ref.backward(gy.double())
        # rounded once to 8 bits; sums of 512 columns, of 5 rows in 32 bits
        torch.testing.assert_close(
            x.grad.double(), xd.grad + (gh if form == "forked" else 0),
            rtol=2.0 ** -7, atol=1e-4)
        assert w.grad.dtype == torch.float32
        torch.testing.assert_close(w.grad.double(), wd.grad, rtol=1e-5,
                                   atol=1e-5)
    assert y.dtype == torch.bfloat16
    torch.testing.assert_close(y.double(), ref, rtol=2.0 ** -8, atol=1e-5)


@pytest.mark.parametrize("T,K,pitch", [
    (1, 8, 8), (7, 72, 80), (8, 64, 64), (65, 136, 136), (257, 520, 1024),
    (1111, 4096, 4096)])
def test_turned_rows(T, K, pitch):
    """Remainders of the 8 x 8 words of a lane and of the tiles of a workgroup."""
    x = torch.randn(T, pitch, device="cuda", dtype=torch.bfloat16)[:, :K]
    xt = ops._turned(x)
    assert torch.equal(xt, x) and xt.t().stride(1) == 1


@pytest.mark.parametrize("T,K,widths,aligned", [
    (1111, 4096, (14344,), True),            # both operands
    (2601, 2048, (8192, 1024, 1024), True),  # x for all of them
    (2601, 11008, (2056,), True),            # dy
    (2600, 8200, (8192,), True),             # both, of wide ones
    (2601, 2044, (12288,), False),           # rows that are not whole words
    (300, 64, (32,), True)])                 # as they are
def test_weight_gradients(T, K, widths, aligned):
    x = torch.randn(T, K, device="cuda", dtype=torch.bfloat16)
    grads = [torch.randn(T, n, device="cuda", dtype=torch.bfloat16)
             for n in widths]
    got = ops.weight_grads(grads, x)
    assert not aligned or any(ops.turn_rule(T, sum(widths), K)) == (T > 1000)
    for g, w in zip(grads, got):
        want = g.float().t() @ x.float()
        # rounded to 8 bits; sums of T terms in float32, in any order
        bound = want.abs() * 2 ** -8 + 2 * T * 2 ** -24 * \
            (g.float().abs().t() @ x.float().abs())
        assert w.shape == want.shape and w.is_contiguous()
        assert ((w.float() - want).abs() <= bound).all()
    # a backward that is differentiated itself does without
    with torch.enable_grad():
        gx = grads[0].clone().requires_grad_()
        (w,) = ops.weight_grads([gx], x)
        assert w.requires_grad


def test_turned_weight_of_an_input_gradient():
    dy = torch.randn(2, 4096, 4096, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(4096, 4096, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        wt = ops.input_weight(dy, w)
        assert torch.equal(wt, w) and wt.stride(0) == 1
        got, want = dy.matmul(wt)[0, :64], dy[0, :64].float() @ w.float()
    # rounded to 8 bits; sums of 4096 terms in float32, in any order
    bound = want.abs() * 2 ** -8 + 2 * 4096 * 2 ** -24 * \
        (dy[0, :64].float().abs() @ w.float().abs())
    assert ((got.float() - want).abs() <= bound).all()
    assert ops.input_weight(dy, w) is w                # under autograd
    with torch.no_grad():
        assert ops.input_weight(dy[:, :100], w) is w


@pytest.mark.parametrize("T,V,W,skip,kind", [
    (1, 5, 8, None, "any"), (8, 3, 24, 1, "any"), (9, 1, 8, None, "one"),
    (300, 40, 520, -1, "any"), (700, 5000, 2056, 0, "any"),
    (2000, 32000, 4096, None, "any"), (1500, 900, 1032, 3, "few"),
    (8192, 100, 512, None, "one")])
def test_embedding_gradient(monkeypatch, T, V, W, skip, kind):
    """Rows without tokens, of one, two, up to eight and more; of all."""
    monkeypatch.setattr(ops, "embedding_rule", lambda *sizes: True)
    ids = torch.randint(V, (T,), device="cuda")
    if kind == "one":
        ids[:] = V // 2
    elif kind == "few":
        ids[::3] = 7
        ids[1::3] %= 40
    w = torch.randn(V, W, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(T, W, device="cuda", dtype=torch.bfloat16)
    out = ops.embedding(ids, w, skip)
    assert torch.equal(out, w[ids])
    (got,) = torch.autograd.grad(out, w, dy, retain_graph=True)
    (again,) = torch.autograd.grad(out, w, dy)
    assert torch.equal(got, again)
    want = torch.zeros(V, W, device="cuda", dtype=torch.float64)
    want.index_add_(0, ids, dy.double())
    size = torch.zeros_like(want).index_add_(0, ids, dy.double().abs())
    if skip is not None:
        want[skip % V] = 0
    # rounded to 8 bits; sums of up to T terms in float32
    bound = want.abs() * 2 ** -8 + 2 * T * 2 ** -24 * size
    assert ((got.double() - want).abs() <= bound).all()
    # a backward that is differentiated itself
    out = ops.embedding(ids, w, skip)
    dy.requires_grad_()
    (g,) = torch.autograd.grad(out, w, dy, create_graph=True)
    assert g.requires_grad


@pytest.mark.parametrize("each,V,W", [
    (1, 9000, 8), (3, 70, 8), (8, 900, 520), (9, 1900, 2056), (16, 600, 512),
    (17, 500, 1032), (256, 20, 64), (257, 20, 520), (1000, 9, 64), (6000, 3, 1032)])
def test_embedding_gradient_of_rows_far_apart(monkeypatch, each, V, W):
    """Every row's tokens lie over all of them: as many as a wave and a workgroup take
    and one more, parts of rows; more rows than waves and workgroups at once."""
    monkeypatch.setattr(ops, "embedding_rule", lambda *sizes: True)
    T = each * V
    ids = torch.arange(T, device="cuda") % V
    if each == 1000:
        ids[::2] = ids[::2] // 3 * 3       # unequal ones, some without
        ids[:3000] = 4                     # and parts that have more than others
    w = torch.randn(V, W, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(T, W, device="cuda", dtype=torch.bfloat16)
    out = ops.embedding(ids, w)
    (got,) = torch.autograd.grad(out, w, dy, retain_graph=True)
    (again,) = torch.autograd.grad(out, w, dy)
    assert torch.equal(got, again)
    want = torch.zeros(V, W, device="cuda", dtype=torch.float64)
    want.index_add_(0, ids, dy.double())
    size = torch.zeros_like(want).index_add_(0, ids, dy.double().abs())
    # rounded to 8 bits; sums of up to T terms in float32
    bound = want.abs() * 2 ** -8 + 2 * T * 2 ** -24 * size
    assert ((got.double() - want).abs() <= bound).all()
