"""Serving kernels on the GPU, each against the plain implementation in
``voletar_oracle`` (float64), one mechanism at a time."""

import math
import types

import pytest
import torch

import voletar_oracle as vo

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module", autouse=True)
def sv():
    from neuronx_distributed_amd.ops import serving

    serving.ensure_built()
    return serving


def _close(got, want, dtype, scale=1.0, what=""):
    got, want = got.detach().double().cpu(), want.double()
    assert torch.isfinite(got).all(), what
    tol = (3e-6 if dtype == torch.float32 else 6e-3) * scale
    err = (got - want).abs() / want.abs().amax(dim=-1, keepdim=True).clamp(
        min=1e-3)
    assert err.max().item() < tol, (what, err.max().item(), tol)


def _rand(*shape, dtype, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


# ---------------------------------------------------------------------------
# attention
# ---------------------------------------------------------------------------

class Paged:
    """Requests of given lengths over scattered pages of a cache that is
    full of large stale values."""

    def __init__(self, lengths, G, D, E, dtype, seed=0):
        gen = torch.Generator().manual_seed(seed)
        per = [-(-n // 64) for n in lengths]
        pages = sum(per) + 2
        perm = torch.randperm(pages, generator=gen).int()
        self.bt = torch.full((len(lengths), max(per) + 1), int(perm[-1]),
                             dtype=torch.int32)
        at = 0
        for r, n in enumerate(per):
            self.bt[r, :n] = perm[at:at + n]
            at += n
        self.bt = self.bt.cuda()
        self.kc = torch.full((pages, G, 64, D), 77.0, dtype=dtype).cuda()
        self.vc = torch.full((pages, G, 64, E), -55.0, dtype=dtype).cuda()


ATTN = [
    # H, G, D, E, window, keep
    (4, 2, 56, 64, 90, 21),
    (6, 2, 40, 24, 70, 5),
    (3, 1, 20, 12, 33, 0),        # sizes that are no multiple of 8
    (8, 8, 128, 96, 130, 130),
    (16, 2, 96, 128, 64, 64),
    (2, 2, 200, 256, 65, 1),
    (4, 4, 32, 48, 0, 0),         # plain causal
    (10, 2, 16, 16, 1, 3),
]


def _attn_case(H, G, D, E, window, keep, T, dtype, seed=1):
    q = _rand(T, H * D, dtype=dtype, seed=seed)
    k = _rand(T, G * D, dtype=dtype, seed=seed + 1)
    v = _rand(T, G * E, dtype=dtype, seed=seed + 2)
    mask = {"size": window, "keep_first": keep} if window else None
    want = vo.windowed_attention(
        q.double().view(T, H, D), k.double().view(T, G, D),
        v.double().view(T, G, E), 0.11, mask).reshape(T, H * E)
    return q, k, v, want


def _portions(sv, c, q, k, v, cuts, H, window, keep, req=0):
    """Feed one request in portions; a portion of one token decodes."""
    outs, at = [], 0
    for n in cuts:
        qs, ks, vs = (t[at:at + n].cuda() for t in (q, k, v))
        pos = torch.arange(at, at + n, dtype=torch.int32).cuda()
        seq = torch.full((n,), req, dtype=torch.int32).cuda()
        kw = dict(heads=H, scale=0.11, window=window, keep=keep,
                  max_keys=at + n)
        if n == 1:
            o = sv.attn_rows(qs, ks, vs, c.kc, c.vc, pos, seq, c.bt, **kw)
        else:
            tiles = torch.tensor(
                [(req, s, min(128, n - s), at + s) for s in range(0, n, 128)],
                dtype=torch.int32).cuda()
            o = sv.attn_portions(qs, ks, vs, c.kc, c.vc, pos, seq, c.bt,
                                 tiles, **kw)
        outs.append(o)
        at += n
    assert at == q.shape[0]
    return torch.cat(outs)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", ATTN)
def test_attention_prompt_portions_and_decoding(sv, case, dtype):
    H, G, D, E, window, keep = case
    T = 290
    q, k, v, want = _attn_case(*case, T, dtype)
    for cuts in ([T], [2, 62, 64, 3, 129, 30], [130] + [1] * 160,
                 [1, 1, 2, 1, 63, 2, 200, 20]):
        c = Paged([T], G, D, E, dtype, seed=len(cuts))
        got = _portions(sv, c, q, k, v, cuts, H, window, keep)
        _close(got, want, dtype, what=(case, cuts[:4]))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,window", [
    (8, 2, 128, 0), (3, 3, 128, 0), (17, 1, 128, 40), (14, 2, 64, 0),
    (8, 8, 64, 100), (6, 2, 32, 0)])
def test_single_rows_turned_in_the_kernel(sv, H, G, D, window, dtype):
    """Queries and keys turned beside the attention, or before it where it has
    no form for that: first and last places of tiles, pages and rows."""
    torch.manual_seed(H + D)
    at = [0, 31, 32, 63, 64, 95, 127, 300, 701]
    need = [p // 64 + 1 for p in at]
    table = torch.zeros(len(at), max(need), dtype=torch.int32)
    place = torch.randperm(sum(need)).int()
    for i, n in enumerate(need):
        table[i, :n] = place[sum(need[:i]):sum(need[:i + 1])]
    cache = [torch.randn(sum(need), G, 64, D, device="cuda").to(dtype)
             for _ in "kv"]
    proj = torch.randn(len(at), (H + 2 * G) * D, device="cuda").to(dtype)
    angle = torch.rand(702, D // 2, device="cuda") * 6
    cos, sin = angle.cos(), angle.sin()
    pos = torch.tensor(at, dtype=torch.int32, device="cuda")
    seq = torch.arange(len(at), dtype=torch.int32, device="cuda")
    got = []
    for turned in (False, True):
        q, k, v = proj.clone().split([H * D, G * D, G * D], 1)
        kc, vc = (c.clone() for c in cache)
        if turned:
            sv.rope_rows_(q, k, cos, sin, pos, D, 702)
        out = sv.attn_rows(q, k, v, kc, vc, pos, seq, table.cuda(), H, D ** -0.5,
                           window, max_keys=702,
                           rotary=None if turned else (cos, sin))
        got.append((out.float(), kc.float(), vc.float()))
    (out, kc, vc), (want, kw, vw) = got
    # a product may be fused with the other's sum: then an element is rounded
    # to the other side, and the scores of one key move by 2 ** -9 of a part
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22
    torch.testing.assert_close(kc, kw, rtol=eps, atol=2 * eps)
    torch.testing.assert_close(out, want, rtol=eps, atol=2 * eps)
    assert torch.equal(vc, vw)
    with pytest.raises(ValueError):
        sv.attn_rows(q, k, v, kc.to(dtype), vc.to(dtype), pos, seq,
                     table.cuda(), H, D ** -0.5, window, max_keys=703,
                     rotary=(cos, sin))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window,keep", [(92, 22), (64, 64), (70, 3),
                                         (33, 0), (128, 65)])
def test_attention_edges_show(sv, window, keep, dtype):
    """One key stands out; queries just inside see it, just outside do not.
    The planted places: the last kept token, the first that is not kept,
    page borders, and the window's edge of several queries."""
    H, G, D, E, T = 4, 2, 64, 32, 330
    spots = sorted({0, max(keep - 1, 0), keep, keep + 1, 63, 64, 65, 127,
                    128, 200})
    mask = {"size": window, "keep_first": keep}
    for s in spots:
        q = _rand(T, H * D, dtype=dtype, seed=3)
        k = _rand(T, G * D, dtype=dtype, seed=4, scale=0.3)
        v = _rand(T, G * E, dtype=dtype, seed=5)
        q[:, 0::D] = 8.0                       # first dim of every head
        k[:, 0::D] = 0.0
        k[s, 0::D] = 14.0                      # score + 12 at this key
        v[s] = 6.0
        want = vo.windowed_attention(
            q.double().view(T, H, D), k.double().view(T, G, D),
            v.double().view(T, G, E), 0.11, mask)
        seen = torch.tensor([vo.visible(i, s, mask) for i in range(T)])
        assert (want.mean((1, 2))[seen] > 5).all()       # it shows
        if (~seen).any():
            assert (want.mean((1, 2))[~seen] < 2).all()
        for cuts in ([T], [keep + 2] + [1] * (T - keep - 2)):
            c = Paged([T], G, D, E, dtype, seed=s)
            got = _portions(sv, c, q, k, v, cuts, H, window, keep)
            _close(got, want.reshape(T, H * E), dtype,
                   what=(window, keep, s, cuts[0]))


def _sized_values(v, kind):
    """v (T, G * E) of one page beside the next, and within a page."""
    v = v.clone()
    page = torch.arange(v.shape[0]) // 64
    if kind == "wide":                     # a page of 2^33 beside usual ones
        v[70] *= 2.0 ** 20
        v[71] *= 2.0 ** -13
    elif kind == "pages":                  # every page is 2^7 of the next one
        v *= (2.0 ** (-7 * page.double()))[:, None].to(v.dtype)
    elif kind == "zeros":
        v[64:128] = 0
        v[::3, ::5] = 0
    elif kind == "ends":                   # 2^29 apart everywhere
        v[:] = v.sign() * 2.0 ** -29
        v[::2, 1::3] = 1.9921875
    elif kind == "tiny":                   # some of them too small for bf16
        v *= 2.0 ** -120
    elif kind == "large":
        v *= 2.0 ** 100
    return v


@pytest.mark.parametrize("kind", ["plain", "wide", "pages", "zeros", "ends",
                                  "tiny", "large"])
@pytest.mark.parametrize("H,G,D,E,window,keep", [
    (4, 2, 128, 128, 0, 0), (3, 1, 64, 64, 90, 21), (2, 2, 96, 40, 64, 64),
    (4, 1, 24, 72, 0, 0)])
def test_values_of_all_sizes(sv, kind, H, G, D, E, window, keep):
    """Values that differ by page, that nearly leave the range of the type or are
    zero, against 64 bits; tiles in any order."""
    dtype, lens, first = torch.bfloat16, [290, 133, 200], [0, 130, 75]
    mask = {"size": window, "keep_first": keep} if window else None
    data, bounds = [], []
    for i, n in enumerate(lens):
        q, k, v, _ = _attn_case(H, G, D, E, window, keep, n, dtype, seed=40 + n)
        v = _sized_values(v, kind)
        qkv = [t.double().view(n, -1, s) for t, s in ((q, D), (k, D), (v, E))]
        want = vo.windowed_attention(*qkv, 0.11, mask).reshape(n, H * E)
        size = vo.windowed_attention(*qkv[:2], qkv[2].abs(), 0.11, mask)
        data.append((q, k, v, want))
        # the result is rounded to bf16; weights and sums have 32 bits
        bounds.append(2.0 ** -8 * want.abs() +
                      2.0 ** -20 * size.reshape(n, H * E))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    c = Paged(lens, G, D, E, dtype)
    rows = [(r, p) for r, n in enumerate(lens) for p in range(n)]
    seq, pos = i32([r for r, _ in rows]), i32([p for _, p in rows])
    _, k, v = (torch.cat([d[i] for d in data]).cuda() for i in range(3))
    sv.kv_append(k, v, c.kc, c.vc, pos, seq, c.bt)
    q = torch.cat([d[0][a:] for d, a in zip(data, first)]).cuda()
    tiles, at = [], 0
    for r, (n, a) in enumerate(zip(lens, first)):
        for p in range(a, n, 128):
            tiles.append((r, at + p - a, min(128, n - p), p))
        at += n - a
    for order in (1, -1):
        got = sv.attn_portions(
            q, k[:q.shape[0]], v[:q.shape[0]], c.kc, c.vc, pos, seq, c.bt,
            i32(tiles[::order]), H, 0.11, window, keep, append=False,
            max_keys=290)
        at = 0
        for d, a, bound in zip(data, first, bounds):
            n = d[3].shape[0] - a
            err = (got[at:at + n].double().cpu() - d[3][a:]).abs()
            assert (err <= bound[a:] + 2.0 ** -133).all(), (
                order, (err / bound[a:]).max())
            at += n


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_batch_of_unequal_requests(sv, dtype):
    H, G, D, E, window, keep = 6, 3, 48, 32, 50, 7
    lens = [3, 140, 64, 257]
    c = Paged(lens, G, D, E, dtype)
    data = [_attn_case(H, G, D, E, window, keep, n, dtype, seed=20 + n)
            for n in lens]
    kw = dict(heads=H, scale=0.11, window=window, keep=keep, max_keys=257)
    # all but the last token of every request in one call, then one each
    q, k, v = (torch.cat([d[i][:-1] for d in data]).cuda() for i in range(3))
    pos, seq, tiles, at = [], [], [], 0
    for r, n in enumerate(lens):
        for s in range(0, n - 1, 128):
            tiles.append((r, at + s, min(128, n - 1 - s), s))
        pos += range(n - 1)
        seq += [r] * (n - 1)
        at += n - 1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    got = sv.attn_portions(q, k, v, c.kc, c.vc, i32(pos), i32(seq), c.bt,
                           i32(tiles), **kw)
    _close(got, torch.cat([d[3][:-1] for d in data]), dtype)
    q, k, v = (torch.cat([d[i][-1:] for d in data]).cuda() for i in range(3))
    got = sv.attn_rows(q, k, v, c.kc, c.vc, i32([n - 1 for n in lens]),
                       i32(range(4)), c.bt, **kw)
    _close(got, torch.cat([d[3][-1:] for d in data]), dtype)


@pytest.mark.parametrize("H,G,D,n", [(8, 8, 128, 64), (8, 8, 128, 201),
                                     (16, 8, 128, 64), (16, 8, 128, 65),
                                     (24, 8, 128, 20), (8, 8, 64, 64)])
def test_decoding_of_many_short_requests(sv, H, G, D, n):
    """More rows and heads than run at a time, around the lengths at which
    another kernel takes them."""
    B, dtype = 300, torch.bfloat16
    q, k, v, want = _attn_case(H, G, D, D, 0, 0, n, dtype)
    lens = [n - i % 5 for i in range(B)]
    c = Paged(lens, G, D, D, dtype)
    at = [(r, p) for r, m in enumerate(lens) for p in range(m - 1)]
    seq, pos = (torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*at))
    sv.kv_append(k.cuda()[pos.long()], v.cuda()[pos.long()], c.kc, c.vc, pos,
                 seq, c.bt)
    last = torch.tensor(lens) - 1
    rows = torch.arange(B, dtype=torch.int32).cuda()
    got = sv.attn_rows(q[last].cuda(), k[last].cuda(), v[last].cuda(), c.kc,
                       c.vc, last.int().cuda(), rows, c.bt, H, 0.11,
                       max_keys=n)
    _close(got, want[last], dtype)


def test_attention_weights_keep_32_bits(sv):
    """Two far apart values under nearly equal weights: bf16 weights would
    lose the small one's contribution to the sum of many."""
    H, G, D, E, T = 1, 1, 32, 32, 128
    q = torch.zeros(T, D, dtype=torch.bfloat16)
    q[:, 0] = 1
    k = torch.zeros(T, D, dtype=torch.bfloat16)
    k[:, 0] = (torch.arange(T) % 7).to(torch.bfloat16) * 0.37
    v = torch.full((T, E), 1.0, dtype=torch.bfloat16)
    v[1::2] = -1.0
    want = vo.windowed_attention(q.double()[:, None], k.double()[:, None],
                                 v.double()[:, None], 0.11, None)[:, 0]
    c = Paged([T], G, D, E, torch.bfloat16)
    got = _portions(sv, c, q, k, v, [T], 1, 0, 0).double().cpu()
    # rows where the signs nearly cancel: the error of the weights decides
    small = want[:, 0].abs() < 0.02
    assert small.sum() > 20
    assert ((got - want).abs()[small] <
            2e-5 + 4e-3 * want.abs()[small]).all()


def test_small_weights_keep_32_bits(sv):
    """A key without a value takes nearly all the weight, by 2^8 to 2^22 in the eight
    groups of heads, and one that nobody looks at has a value of 2^9 times the others':
    what is left, equal weights of the many, keeps its bits.  (Weights of 16 bits, also
    two of them, end at a fixed distance from the largest.)"""
    H, G, D, T, bf = 32, 8, 128, 3200, torch.bfloat16
    q = torch.zeros(T, H, D, dtype=bf, device="cuda")
    q[:, :, 0] = 8.0
    k = torch.zeros(T, G, D, dtype=bf, device="cuda")
    k[0, :, 0] = torch.arange(8.0, 24.0, 2.0) * (math.log(2.0) / 0.88)
    k[1, :, 0] = -k[0, :, 0]
    v = 1 + torch.rand(T, G, D, device="cuda").to(bf)
    v[0], v[1] = 0.0, 2.0 ** 9
    c = Paged([T], G, D, D, bf)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    batch = types.SimpleNamespace(
        portion_tokens=T, pos=i32(range(T)), seq=i32([0] * T), block_table=c.bt,
        tiles=i32([(0, s, min(128, T - s), s) for s in range(0, T, 128)]),
        portions=i32([(0, 0, T, 0)]), max_keys=T)
    got = sv.ragged_attention(q.view(T, -1), k.view(T, -1), v.view(T, -1), batch,
                              (c.kc, c.vc), H, 0.11).view(T, H, D)
    for g in range(G):
        # the same query everywhere: running sums of weights and of weighted values
        w = (0.11 * 8.0 * (k[:, g, 0] - k[0, g, 0]).double()).exp()
        want = (w[:, None] * v[:, g].double()).cumsum(0) / w.cumsum(0)[:, None]
        err = (got[:, 4 * g:4 * g + 4].double() - want[:, None]).abs()
        # rounded to bf16 once; sums of 32 bits
        assert (err <= (2.0 ** -8 + 2.0 ** -15) * want[:, None]).all(), (
            g, (err / want[:, None])[1:].max().item())


# ---------------------------------------------------------------------------
# matrix memories
# ---------------------------------------------------------------------------

MEM = [(4, 56, 40), (3, 48, 72), (2, 20, 12), (2, 128, 96), (1, 256, 40),
       (5, 8, 8), (1, 300, 34)]


def _mem_inputs(H, D, E, T, dtype, seed=0):
    # one fused projection, read as strided slices
    pad = 8 - (2 * H * D + H * E) % 8
    p = _rand(T, 2 * H * D + H * E + pad, dtype=dtype, seed=seed)
    return p[:, :H * D], p[:, H * D:2 * H * D], p[:, 2 * H * D:][:, :H * E], p


def _tables(sv, seg, chunked):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    return (i32(seg), *map(i32, sv.chunk_table(seg))) if chunked \
        else (i32(seg),)


def _run_memory(sv, proj, sizes, cuts, H, gate_of, S, n, m, slot):
    outs, at = [], 0
    for c in cuts:
        part = proj[at:at + c].cuda()
        a, b, w = sizes
        q, k, v = part[:, :a], part[:, a:a + b], part[:, a + b:a + b + w]
        seg = [(slot, 0, c, at)]
        outs.append(sv.memory_mix(q, k, v, gate_of(at, c), S, n, m,
                                  *_tables(sv, seg, c > 1)[:1], H,
                                  *_tables(sv, seg, c > 1)[1:]))
        at += c
    return torch.cat(outs)


T_MEM = 600
CUTS = ([T_MEM], [64, 2, 190, 3, 257, 84], [500] + [1] * 100,
        [1, 1, 2, 256, 128, 212], [255, 256, 89])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,D,E", MEM)
def test_decayed_memory(sv, H, D, E, dtype):
    T = T_MEM
    decay = [0.0, 1.0, 0.97, 0.6, 0.999][:H] if H > 2 else [0.998, 0.5][:H]
    q, k, v, p = _mem_inputs(H, D, E, T, dtype, seed=7)
    d = lambda t, s: vo.silu(t.double()).view(T, H, s)
    if dtype == torch.bfloat16:   # activations may round to bf16
        d = lambda t, s: vo.silu(t.double()).to(dtype).double().view(T, H, s)
    want, S_want = vo.decayed_memory(d(q, D), d(k, D), d(v, E),
                                     torch.tensor(decay).double())
    gate = sv.decay_gate(decay, "cuda")
    for cuts in CUTS:
        S = torch.full((3, H, D, E), 1e4).cuda()   # a slot used before
        got = _run_memory(sv, p, (H * D, H * D, H * E), cuts, H,
                          lambda at, c: gate, S, None, None, slot=2)
        _close(got, want.reshape(T, H * E), dtype, 2.0, (H, D, E, cuts[:4]))
        err = (S[2].double().cpu() - S_want).abs().max() / S_want.abs().max()
        assert err < (2e-5 if dtype == torch.float32 else 5e-3), err
        assert (S[:2] == 1e4).all()                # other slots untouched


def _gates(H, T, i_scale, f_shift, seed=0):
    raw = _rand(T, 2 * H, dtype=torch.float32, seed=seed, scale=i_scale)
    raw[:, H:] += f_shift
    return raw


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("i_scale,f_shift", [(1.0, 3.0), (6.0, 6.0),
                                             (3.0, -8.0), (0.1, 12.0)])
@pytest.mark.parametrize("H,D,E", MEM)
def test_gated_memory(sv, H, D, E, i_scale, f_shift, dtype):
    T, cap = T_MEM, 5.0 if H == 3 else 15.0
    q, k, v, p = _mem_inputs(H, D, E, T, dtype, seed=9)
    raw = _gates(H, T, i_scale, f_shift, seed=H)
    raw[37] = 40.0                 # one input stands out and is carried on
    ib, fb = (_rand(H, dtype=dtype, seed=s) for s in (1, 2))
    x = raw.double()
    gi = cap * torch.tanh((x[:, :H] + ib.double()) / cap)
    gf = vo.log_sigmoid(cap * torch.tanh((x[:, H:] + fb.double()) / cap))
    f = lambda t, s: t.double().view(T, H, s)
    want, (S_w, n_w, m_w) = vo.gated_memory(f(q, D) * D ** -0.5, f(k, D),
                                            f(v, E), gi, gf)
    # o = S^T q / |n . q|: how far the division amplifies rounding
    cond, ns, ms = torch.zeros(T, H).double(), 0.0, torch.zeros(H).double()
    for t in range(T):
        mt = torch.maximum(gf[t] + ms, gi[t])
        ns = (torch.exp(gf[t] + ms - mt)[:, None] * ns
              + torch.exp(gi[t] - mt)[:, None] * f(k, D)[t])
        ms, qn = mt, f(q, D)[t] * D ** -0.5 * ns
        cond[t] = qn.abs().sum(1) / torch.maximum(
            qn.sum(1).abs(), torch.exp(-ms)) + 1.0
    want = want.reshape(T, H, E)
    nt = -(-E // 32)
    for cuts in CUTS:
        S = torch.full((2, H, D, E), -3e3).cuda()
        n = torch.full((2, H, nt, D), 9e3).cuda()
        m = torch.full((2, H, nt), 50.0).cuda()

        def gate(at, c):
            return sv.ExpGate(raw[at:at + c].cuda().contiguous(), ib.cuda(),
                              fb.cuda(), cap, D ** -0.5)

        got = _run_memory(sv, p, (H * D, H * D, H * E), cuts, H, gate, S, n,
                          m, slot=1)
        c = cond.unsqueeze(2)
        got = got.double().cpu().view(T, H, E)
        _close(want + (got - want) / c, want, torch.float32, 20.0,
               (H, D, E, cuts[:4])) if dtype == torch.float32 else \
            _close(got, want, dtype, 2.0, (H, D, E, cuts[:4]))
        assert (m[1].double().cpu() - m_w.view(H, 1)).abs().max() < 2e-3
        for got_s, w in ((S[1], S_w), (n[1], n_w.unsqueeze(1))):
            err = (got_s.double().cpu() - w).abs().max() / w.abs().max()
            assert err < 2e-4, err


@pytest.mark.parametrize("H,E", [(3, 64), (2, 128), (5, 192)])
@pytest.mark.parametrize("far", [False, True])
def test_decayed_memory_in_one_pass(sv, monkeypatch, H, E, far):
    """Segments that end at, before and behind the 16 tokens of a wave and the 64 of
    a piece, from empty and from filled slots, of adjacent and of distant rows;
    against the oracle, and against chunks."""
    D, bf = 128, torch.bfloat16
    lens, more = [1, 15, 17, 63, 64, 65, 128, 130, 193, 449], [70, 1, 300, 64, 2, 33,
                                                              65, 192, 5, 16]
    decay = [0.97, 0.0, 1.0, 0.6, 0.999][:H]
    gate = sv.decay_gate(decay, "cuda")
    assert sv.single_pass(10, 10, H * E, False)
    cases = [_mem_inputs(H, D, E, a + b, bf, seed=40 + i)[3]
             for i, (a, b) in enumerate(zip(lens, more))]
    sizes = H * D, H * D, H * E
    got = {}
    for once in (True, False):
        monkeypatch.setattr(sv, "single_pass", lambda *a: once)
        S = torch.full((10, H, D, E), 7.0).cuda()
        out = []
        for at, n in (([0] * 10, lens), (lens, more)):
            rows = torch.cat([p[a:a + k, :sum(sizes)] for p, a, k in zip(cases, at, n)])
            # among elements that nothing may see, 748 of the rows 2 MB apart
            pitch = 1 << 20 if far and at[0] else rows.shape[1] + 8
            wide = torch.full((len(rows) + 1, pitch), float("nan"), dtype=bf,
                              device="cuda")
            x = wide[:len(rows), :rows.shape[1]]
            x.copy_(rows)
            seg, *tab = _tables(sv, [(9 - i, sum(n[:i]), k, a) for i, (a, k) in
                                     enumerate(zip(at, n))], True)
            out.append(sv.memory_mix(*x.split(sizes, dim=1), gate, S, None, None, seg,
                                     H, *tab).split(n))
        got[once] = [torch.cat([o[i] for o in out]) for i in range(10)], S
    silu = lambda t, s: vo.silu(t.double()).to(bf).double().view(len(t), H, s)
    for i, p in enumerate(cases):
        q, k, v = p[:, :sum(sizes)].split(sizes, dim=1)
        want, S_want = vo.decayed_memory(silu(q, D), silu(k, D), silu(v, E),
                                         torch.tensor(decay).double())
        want = want.reshape(len(p), H * E)
        _close(got[True][0][i], want, bf, 2.0, i)
        off = [(got[way][0][i].cpu().double() - want).norm() for way in got]
        assert off[0] <= 1.05 * off[1] + 1e-6 * want.norm()
        err = [(got[way][1][9 - i].cpu().double() - S_want).norm() for way in got]
        assert err[0] <= 1.05 * err[1] + 1e-6 * S_want.norm()


@pytest.mark.parametrize("gated", [False, True])
def test_results_where_one_pass_cannot_write(sv, gated):
    """Results and normalisers that begin 8 bytes behind the 16 that are written at
    once: the same as elsewhere, by chunks."""
    H, D, E, T, bf = 2, 128, 64, 70, torch.bfloat16
    q, k, v, p = _mem_inputs(H, D, E, T, bf, seed=5)
    q, k, v = (t.cuda() for t in (q.contiguous(), k.contiguous(), v.contiguous()))
    raw, b = _gates(H, T, 1.0, 2.0).cuda(), torch.zeros(H, dtype=bf).cuda()
    gate = sv.ExpGate(raw, b, b, 15.0, 0.2) if gated else \
        sv.decay_gate([0.9, 0.99], "cuda")
    seg, *tab = _tables(sv, [(0, 0, T, 0)], True)
    outs, normalisers = [], []
    for out_at, n_at in ((0, 0), (4, 0), (0, 2)):
        S = torch.zeros(1, H, D, E).cuda()
        n = torch.zeros(H * 2 * D + 2).cuda()[n_at:n_at + H * 2 * D].view(1, H, 2, D)
        m = torch.zeros(1, H, 2).cuda()
        out = torch.full((T * H * E + 8,), 3.0, dtype=bf).cuda()
        sv.memory_mix(q, k, v, gate, S, n, m, seg, H, *tab,
                      out=out[out_at:out_at + T * H * E].view(T, H * E))
        assert (out[:out_at] == 3.0).all() and (out[out_at + T * H * E:] == 3.0).all()
        outs.append(out[out_at:out_at + T * H * E].float().cpu().view(T, -1))
        normalisers.append(n.cpu())
    for got, n in zip(outs[1:], normalisers[1:]):
        _close(got, outs[0], bf, 2.0)
        assert (n - normalisers[0]).abs().max() <= 1e-5 * normalisers[0].abs().max()


@pytest.mark.parametrize("H,E,i_scale,f_shift", [
    (3, 64, 1.0, 3.0), (2, 128, 6.0, 6.0), (4, 192, 3.0, -8.0), (1, 256, 0.1, 12.0)])
def test_gated_memory_in_one_pass(sv, monkeypatch, H, E, i_scale, f_shift):
    """Segments that end at, before and behind the 16 tokens of a wave and the 64 of
    a piece, from empty and from filled slots; gates that forget at once, that keep
    all, and inputs that stand out; against the oracle, and against chunks."""
    D, bf, cap = 128, torch.bfloat16, 15.0
    lens, more = [1, 15, 17, 63, 64, 65, 128, 130, 193, 449], [70, 1, 300, 64, 2, 33,
                                                              65, 192, 5, 16]
    assert sv.single_pass(10, 10, H * E, True)
    ib, fb = (_rand(H, dtype=bf, seed=s) for s in (1, 2))
    cases, raws = [], []
    for i, (a, b) in enumerate(zip(lens, more)):
        cases.append(_mem_inputs(H, D, E, a + b, bf, seed=60 + i)[3])
        raws.append(_gates(H, a + b, i_scale, f_shift, seed=80 + i))
        raws[-1][min(9, a + b - 1)] = 40.0
    sizes, nt = (H * D, H * D, H * E), E // 32
    got = {}
    for once in (True, False):
        monkeypatch.setattr(sv, "single_pass", lambda *a: once)
        S = torch.full((10, H, D, E), 7.0).cuda()
        n, m = torch.full((10, H, nt, D), 9e3).cuda(), torch.full((10, H, nt), 50.0).cuda()
        out = []
        for at, ln in (([0] * 10, lens), (lens, more)):
            rows = torch.cat([p[a:a + k] for p, a, k in zip(cases, at, ln)]).cuda()
            raw = torch.cat([r[a:a + k] for r, a, k in zip(raws, at, ln)]).cuda()
            seg, *tab = _tables(sv, [(9 - i, sum(ln[:i]), k, a) for i, (a, k) in
                                     enumerate(zip(at, ln))], True)
            gate = sv.ExpGate(raw, ib.cuda(), fb.cuda(), cap, D ** -0.5)
            out.append(sv.memory_mix(*rows[:, :sum(sizes)].split(sizes, dim=1), gate, S,
                                     n, m, seg, H, *tab).split(ln))
        got[once] = [torch.cat([o[i] for o in out]) for i in range(10)], S, n, m
    for i, (p, raw) in enumerate(zip(cases, raws)):
        x, T = raw.double(), len(p)
        gi = cap * torch.tanh((x[:, :H] + ib.double()) / cap)
        gf = vo.log_sigmoid(cap * torch.tanh((x[:, H:] + fb.double()) / cap))
        q, k, v = (t.double().view(T, H, -1) for t in
                   p[:, :sum(sizes)].split(sizes, dim=1))
        want, (S_w, n_w, m_w) = vo.gated_memory(q * D ** -0.5, k, v, gi, gf)
        want = want.reshape(T, H * E)
        _close(got[True][0][i], want, bf, 2.0, i)
        off = [(got[way][0][i].cpu().double() - want).norm() for way in got]
        assert off[0] <= 1.05 * off[1] + 1e-6 * want.norm()
        # as they count, times e^m; gates and maxima of 8 to 15 are rounded by 2^-21,
        # each way's its own, and so is what they weigh
        for at, w in ((1, S_w), (2, n_w.unsqueeze(1).expand(H, nt, D))):
            err = [((got[way][3][9 - i].cpu().double()[:, :1] - m_w.view(H, 1)).exp()
                    .unsqueeze(2) * got[way][at][9 - i].cpu().double() - w).norm()
                   for way in got]
            assert err[0] <= 1.05 * err[1] + 2.0 ** -21 * w.norm(), (i, at)
        assert (got[True][3][9 - i].cpu().double() - m_w.view(H, 1)).abs().max() < 2e-3


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("dtype", DTYPES)
def test_memory_batch_and_slots(sv, dtype, gated):
    """Segments of unequal length in one call equal each alone, whatever
    slots they use."""
    H, D, E = 2, 32, 48
    lens, slots = [70, 2, 529, 64], [3, 0, 4, 1]
    T = sum(lens)
    q, k, v, p = _mem_inputs(H, D, E, T, dtype, seed=11)
    raw = _gates(H, T, 1.0, 2.0).cuda()
    b = torch.zeros(H, dtype=dtype).cuda()
    mk = lambda: (torch.full((5, H, D, E), 5.0).cuda(),
                  torch.full((5, H, 2, D), 5.0).cuda(),
                  torch.full((5, H, 2), 5.0).cuda())

    def gate(a, e):
        if not gated:
            return sv.decay_gate([0.9, 0.99], "cuda")
        return sv.ExpGate(raw[a:e].contiguous(), b, b, 15.0, 0.2)

    starts = [sum(lens[:i]) for i in range(4)]
    pc = p.cuda()
    cut = lambda t: (t[:, :H * D], t[:, H * D:2 * H * D],
                     t[:, 2 * H * D:2 * H * D + H * E])
    seg, *tab = _tables(sv, [(s, a, n, 0) for s, a, n in
                             zip(slots, starts, lens)], True)
    S, n, m = mk()
    both = sv.memory_mix(*cut(pc), gate(0, T), S, n, m, seg, H, *tab)
    for s, a, ln in zip(slots, starts, lens):
        S1, n1, m1 = mk()
        one, *tab = _tables(sv, [(0, 0, ln, 0)], True)
        alone = sv.memory_mix(*cut(pc[a:a + ln]), gate(a, a + ln), S1, n1,
                              m1, one, H, *tab)
        assert torch.equal(alone, both[a:a + ln])
        assert torch.equal(S1[0], S[s])


# ---------------------------------------------------------------------------
# norms and pointwise steps
# ---------------------------------------------------------------------------

@pytest.mark.parametrize("W", [2048, 2052, 4096, 4100, 8192, 8196, 16384, 16388])
@pytest.mark.parametrize("pending,parts", [
    ("rows", 0), ("rows", 1), ("rows", 6), ("rows", 8), ("rows", 9),
    ("rows32", 0), (None, 0)])
def test_residual_norm_of_few_rows(sv, W, parts, pending):
    """A row a workgroup, one word after the other or a sum of rows; with and
    without a residual, some rows only."""
    T, eps, bf = 7, 0.03, torch.bfloat16
    x = _rand(T, W, dtype=torch.float32)
    d = _rand(T * max(1, parts), W, dtype=bf, seed=1, scale=3.0)
    w = _rand(W, dtype=bf, seed=2)
    coef = _rand(T, parts, dtype=torch.float32, seed=3) if parts else None
    if pending == "rows32":
        d = d.float() * 1.01
    index = torch.tensor([5, 0, 5, 2], dtype=torch.int32)
    y = d.double().view(T, -1, W)
    y = (y * coef.double()[:, :, None] if parts else y).sum(1)
    for res in (True, False):
        if pending is None and not res:
            continue
        p = None if pending is None else sv.Pending(
            d.cuda(), scale=0.7,
            coef=coef.cuda() if parts else None)
        base = x.double() if res else 0.0
        want = base + 0.7 * y if p is not None else base
        normed = want * (want.pow(2).mean(-1, keepdim=True) + eps).rsqrt() * \
            (1.0 + w.double()) * 1.3
        for ix in (None, index):
            got, h, _ = sv.residual_norm(
                x.cuda() if res else None, p, eps, w.cuda(), centred=True,
                scale=1.3, index=None if ix is None else ix.cuda())
            rows = slice(None) if ix is None else ix.long()
            # 32-bit sums of up to 10 terms, then one rounding to bf16
            torch.testing.assert_close(got.cpu().double(), want[rows],
                                       rtol=2e-6, atol=2e-5)
            torch.testing.assert_close(h.cpu().double(), normed[rows],
                                       rtol=2 ** -8, atol=2e-5)


@pytest.mark.parametrize("parts", [1, 3, 8, 9])
def test_an_infinite_part_of_a_sum_stays_infinite(sv, parts):
    """Also in the last part, which stands in for those that are not there."""
    T, W, bf = 3, 4096, torch.bfloat16
    d = _rand(T * parts, W, dtype=bf)
    for t in range(T):
        d[t * parts + parts - 1, 5 + t] = math.inf
    coef = torch.ones(T, parts, dtype=torch.float32)
    want = d.double().view(T, parts, W).sum(1)
    got, _, _ = sv.residual_norm(None, sv.Pending(d.cuda(), coef=coef.cuda()),
                                 1e-5, _rand(W, dtype=bf).cuda())
    assert torch.equal(got.isinf().cpu(), want.isinf())
    assert not got.isnan().any()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W", [64, 100, 97, 1000, 4096])
def test_residual_norm(sv, W, dtype):
    T, eps = 9, 0.03
    x = _rand(T, W, dtype=torch.float32)
    a, b, x0 = (_rand(T, W, dtype=dtype, seed=s, scale=3.0)
                for s in (1, 2, 3))
    w, wa, wb, vec = (_rand(W, dtype=dtype, seed=s) for s in (4, 5, 6, 7))
    y = _rand(T, W, dtype=torch.float32, seed=8)
    d = lambda t: t.double()
    c = lambda t: t.cuda()
    cases = [
        (None, sv.Pending(c(a)), d(a)),
        (x, sv.Pending(c(a)), d(x) + d(a)),
        (x, None, d(x)),
        (None, sv.Pending(c(y), vec=c(vec)), d(y) + d(vec)),
        (x, sv.Pending(c(a), c(b), c(wa), c(wb), 0.5),
         d(x) + 0.5 * (vo.rms_norm(d(a), d(wa), eps)
                       + vo.rms_norm(d(b), d(wb), eps))),
    ]
    for res, pend, want in cases:
        r = None if res is None else res.cuda()
        nx, h, cat = sv.residual_norm(r, pend, eps, c(w), x0=c(x0))
        _close(nx, want, torch.float32)
        _close(h, vo.rms_norm(want, d(w), eps), dtype)
        _close(cat[:, :W], want, dtype)
        assert torch.equal(cat[:, W:].cpu(), x0)
        idx = torch.tensor([7, 0, 7], dtype=torch.int32).cuda()
        nx, h, _ = sv.residual_norm(r, pend, eps, c(w), keep_x=False,
                                    index=idx)
        assert nx is None
        _close(h, vo.rms_norm(want, d(w), eps)[[7, 0, 7]], dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("groups,gs", [(1, 96), (3, 40), (2, 33), (1, 2048),
                                       (4, 1500), (5, 512)])
def test_gated_norm(sv, groups, gs, dtype):
    T, N, eps = 7, groups * gs, 0.02
    o = _rand(T, N, dtype=dtype)
    w = _rand(N, dtype=dtype, seed=1)
    fused = _rand(T, N + 24, dtype=dtype, seed=2)
    g = fused.cuda()[:, 24:]
    want = (vo.rms(o.double().view(T, groups, gs), eps).reshape(T, N)
            * w.double() * torch.sigmoid(fused[:, 24:].double()))
    _close(sv.gated_norm(o.cuda(), w.cuda(), g, gs, eps), want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_pointwise(sv, dtype):
    x = _rand(13, 37, dtype=dtype, scale=4.0)
    _close(sv.relu_squared_(x.cuda()), vo.relu_squared(x.double()), dtype)
    y = _rand(5, 33, dtype=torch.float32, scale=60.0)
    _close(sv.softcap_(y.cuda(), 12.0),
           12.0 * torch.tanh(y.double() / 12.0), torch.float32)


def test_cpu_tensors_are_refused(sv):
    with pytest.raises(RuntimeError):
        sv.relu_squared_(torch.zeros(4, 4))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,W", [(1, 2049), (1, 4096), (512, 2052),
                                    (513, 2052), (3, 9004), (256, 2052),
                                    (257, 2052), (512, 4100), (513, 4100)])
def test_residual_norm_of_wide_rows(sv, rows, W, dtype):
    """Long and ordinary workgroups; the last words of a row ragged."""
    eps = 0.03
    x = _rand(rows, W, dtype=torch.float32)
    a, w1, w = (_rand(*n, dtype=dtype, seed=s, scale=3.0)
                for s, n in ((1, (rows, W)), (2, (W,)), (3, (W,))))
    for pend, want in (
            (sv.Pending(a.cuda()), x.double() + a.double()),
            (sv.Pending(a.cuda(), w1=w1.cuda()),
             x.double() + vo.rms_norm(a.double(), w1.double(), eps))):
        nx, h, _ = sv.residual_norm(x.cuda(), pend, eps, w.cuda())
        _close(nx, want, torch.float32)
        _close(h, vo.rms_norm(want, w.double(), eps), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,window", [(17, 0), (40, 70)])
def test_single_rows_that_several_workgroups_read(sv, H, window, dtype):
    """The same of heads of 64 whose group several workgroups share."""
    test_single_rows_turned_in_the_kernel(sv, H, 1, 64, window, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,shift", [(1, 0, 2, 0), (3, 1, 24, 0),
                                         (5, 2, 36, 0), (32, 8, 128, 0),
                                         (32, 8, 128, 1), (7, 7, 64, 4)])
@pytest.mark.parametrize("T", [1, 33, 257])
def test_rope_rows(sv, T, H, G, D, shift, dtype):
    """Every pair of every head is turned once: words and single pairs, heads
    that start between words, the last workgroup ragged."""
    half = D // 2
    qkv = _rand(T, (H + G) * D + shift + 8 * (shift == 4), dtype=dtype).cuda()
    q, k = qkv[:, shift:shift + H * D], qkv[:, shift + H * D:][:, :G * D]
    angle = torch.arange(64)[:, None] * torch.rand(half)[None]
    cos, sin = angle.cos().cuda(), angle.sin().cuda()
    pos = torch.randint(0, 64, (T,), dtype=torch.int32)
    before = qkv.clone()
    sv.rope_rows_(q, k, cos, sin, pos.cuda(), D, 64)
    n = (H + G) * D
    x, y = before[:, shift:shift + n].double().view(T, -1, 2, half).unbind(2)
    c, s = (t[pos.cuda()].double()[:, None] for t in (cos, sin))
    want = torch.stack((x * c - y * s, y * c + x * s), 2).view(T, n)
    got = qkv[:, shift:shift + n].double()
    # two products and a sum in 32 bits of factors that reach 4 and 1, and
    # half a unit of the type's 8 or 24 bits: 2 ** -8 or 2 ** -24 of the value
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert ((got - want).abs() <= want.abs() * unit * 1.01
            + (x.abs() + y.abs()).max() * 2.0 ** -23).all()
    assert torch.equal(qkv[:, :shift], before[:, :shift])
    assert torch.equal(qkv[:, shift + n:], before[:, shift + n:])


@pytest.mark.parametrize("rows,W", [(257, 3072), (600, 3068), (513, 4100),
                                    (1100, 8192), (513, 16384)])
@pytest.mark.parametrize("wide", [False, True])
def test_residual_norm_of_many_rows(sv, rows, W, wide):
    """All words of a row at first, and one after the other below 3072 columns; what
    is pending of 32 bits, or nothing."""
    eps, bf = 0.03, torch.bfloat16
    x, w = _rand(rows, W, dtype=torch.float32), _rand(W, dtype=bf, seed=1)
    for d in (_rand(rows, W, dtype=torch.float32 if wide else bf, seed=2), None):
        new = x if d is None else x + d.float()
        want = new.double() * torch.rsqrt(
            new.double().pow(2).mean(1, keepdim=True) + eps) * w.double()
        got, h, _ = sv.residual_norm(
            x.cuda(), None if d is None else sv.Pending(d.cuda()), eps, w.cuda())
        assert torch.equal(got.cpu(), new)
        torch.testing.assert_close(h.cpu().double(), want, rtol=2.0 ** -8 + W * 2.0 ** -24,
                                   atol=1e-30)


@pytest.mark.parametrize("rows,W", [(1, 2048), (257, 3068), (257, 3072), (600, 4096),
                                    (300, 4100)])
@pytest.mark.parametrize("parts", [1, 2, 3])
def test_residual_norm_of_many_sums(sv, rows, W, parts):
    """Sums of one and two rows by the kernel of many rows, and of more."""
    eps, bf = 0.03, torch.bfloat16
    x, w = _rand(rows, W, dtype=torch.float32), _rand(W, dtype=bf, seed=1)
    d = _rand(rows * parts, W, dtype=bf, seed=2)
    coef = _rand(rows, parts, dtype=torch.float32, seed=3)
    terms = d.view(rows, parts, W).double() * coef.double()[..., None]
    new = x.double() + terms.sum(1)
    size = x.double().abs() + terms.abs().sum(1)
    got, h, _ = sv.residual_norm(x.cuda(), sv.Pending(d.cuda(), coef=coef.cuda()), eps,
                                 w.cuda())
    assert ((got.cpu().double() - new).abs() <= size * (parts + 1) * 2.0 ** -23).all()
    mine = got.cpu().double()
    want = mine * torch.rsqrt(mine.pow(2).mean(1, keepdim=True) + eps) * w.double()
    torch.testing.assert_close(h.cpu().double(), want, rtol=2.0 ** -8 + W * 2.0 ** -24,
                               atol=1e-30)


@pytest.mark.parametrize("T,V,W", [(1, 5, 4096), (7, 300, 4096), (3, 9, 72),
                                   (300, 40, 2048), (700, 1000, 3584)])
def test_norms_of_rows_of_a_table(sv, T, V, W):
    """The first norm takes its rows from the table, as after a look-up; and a single
    one in the product behind it."""
    bf, eps = torch.bfloat16, 1e-3
    table, w = _rand(V, W, dtype=bf).cuda(), _rand(W, dtype=bf, seed=1).cuda()
    rows = (torch.arange(T) * 7919 % V).int().cuda()
    rows[-1], rows[0] = 0, V - 1
    found = sv.Pending(table[rows.long()])
    x, h, _ = sv.residual_norm(None, found, eps, w)
    got, g, _ = sv.residual_norm(None, sv.Pending(table, rows=rows), eps, w)
    assert torch.equal(got, x) and torch.equal(g, h)
    with torch.no_grad():
        p = _rand(6144, W, dtype=bf, seed=2).cuda()
        one = sv.normed_linear(None, sv.Pending(table, rows=rows), eps, w, p)
        ref = sv.normed_linear(None, found, eps, w, p)
    assert (one is None) == (ref is None) and (one is not None) == (T == 1)
    if one:
        assert torch.equal(one[0], ref[0]) and torch.equal(one[1], ref[1])
