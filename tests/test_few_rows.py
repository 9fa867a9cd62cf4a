"""Decoding: which kernels take products of a few rows, attention of single
rows and experts of few rows."""

import os
import shutil
import subprocess
import types

import pytest
import torch

from neuronx_distributed_amd.ops import build, serving as sv


def test_a_library_without_the_products_is_not_used(monkeypatch):
    """One that was built before they came is there, but has none."""
    monkeypatch.setattr(sv, "_LIB", types.SimpleNamespace())
    assert not sv.available()
    monkeypatch.setattr(sv, "_LIB",
                        types.SimpleNamespace(sv_stream_linear=None))
    assert sv.available()


@pytest.mark.parametrize("rows,N,R,kernel", [
    # one round of workgroups, up to ranks of 640 and 1024
    (64, 8, 64, True), (2048, 4096, 640, True), (2048, 4096, 704, False),
    (2048, 2048, 1024, True), (2112, 2048, 1024, False), (64, 8, 1088, False),
    # two and more: 172 to 192 of the library's tiles, 257 to 383, and full ones of our own
    (2112, 4096, 512, False), (1344, 8192, 512, True), (1344, 8192, 192, False),
    (1344, 8192, 576, False), (3136, 4096, 512, False), (2048, 10240, 256, True),
    (2048, 10240, 192, False), (2048, 12288, 512, True), (2048, 12288, 320, False),
    (1408, 16384, 512, False), (6592, 4096, 576, False), (2240, 12288, 64, False)])
def test_latents_are_expanded_in_place_where_that_was_faster(rows, N, R, kernel):
    assert sv.expand_rule(rows, N, R) == kernel


@pytest.mark.parametrize("chunks,segments,columns,gated,once", [
    (1, 1, 128, False, True), (10, 10, 128, True, True), (4, 1, 8192, False, True),
    (6, 1, 4096, False, False), (4, 1, 4096, True, True),
    # segments of less than a chunk beside a long one
    (18, 10, 4096, False, False), (36, 26, 2048, True, False),
    (47, 38, 1536, True, False), (12, 5, 4096, True, False),
    (15, 7, 6144, False, True), (33, 22, 4096, False, True)])
def test_memories_go_through_their_segments_at_once_where_that_was_faster(
        chunks, segments, columns, gated, once):
    assert sv.single_pass(chunks, segments, columns, gated) == once


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_every_word_of_a_streamed_row_lies_in_it(tmp_path):
    """Rows of all K up to 4200 in the turns of 16 waves: words past the end are
    read from the row too, also of rows shorter than the 32 columns that four
    groups of lanes read at once."""
    source = tmp_path / "words.cpp"
    source.write_text("""
        #include <cstdio>
        #include "words.h"
        int main() {
          for (int K = 8; K <= 4200; K += 8)
            for (int turn = 0; turn < K + 1024; turn += 32)
              for (int grp = 0; grp < 4; ++grp) {
                const int at = word_column(turn, grp, K), own = turn + grp * 8;
                if (at < 0 || at + 8 > K || (own < K && at != own)) {
                  printf("K %d, columns %d, group %d: %d", K, turn, grp, at);
                  return 1;
                }
              }
          return 0;
        }
    """)
    program = tmp_path / "words"
    subprocess.run(["g++", "-std=c++17", "-I",
                    os.path.join(build.CSRC, "serving"), str(source), "-o",
                    str(program)], check=True)
    run = subprocess.run([str(program)], stdout=subprocess.PIPE, text=True)
    assert run.returncode == 0, run.stdout


SIZES = (8, 16, 24, 64, 248, 512, 576, 896, 1000, 1408, 2048, 2880, 3072,
         3584, 4096, 4104, 4864, 5120, 6144, 8192, 8200, 14336, 28672, 32000,
         50000, 50257, 151936)


@pytest.mark.parametrize("f32,glu", [(False, False), (True, False),
                                     (False, True)])
def test_every_choice_is_one_that_the_launcher_takes(f32, glu):
    """Streaming is for plain products; staying takes whole tiles of weight
    rows, and 8192 columns of 16 rows or 4096 of 32 in registers."""
    taken = set()
    for T in range(1, 34):
        for N in SIZES:
            for K in SIZES:
                how = sv.stream_rule(T, N, K, f32, glu)
                taken.add(how)
                assert how in (None, 0, 1)
                if how == 0:
                    assert not glu
                if how == 1:
                    assert N % (32 if glu else 16) == 0
                    assert K <= (8192 if T <= 16 else 4096 if T <= 32 else 0)
    assert taken == ({None, 1} if glu else {None, 0, 1})


@pytest.mark.parametrize("T,N,K,f32,how", [
    # where the library is faster, and the neighbours where it is not
    (1, 151936, 896, False, None), (1, 33792, 1792, False, 0),
    (8, 54784, 1536, False, None), (8, 32000, 2048, False, 1),
    (4, 61344, 3200, False, 1), (4, 32000, 4096, True, 0),
    (1, 13824, 5120, True, None), (1, 27648, 5120, False, 0),
    (4, 64000, 7168, False, None), (1, 64000, 7168, False, 0),
    (4, 27648, 5120, False, 1), (4, 28672, 4096, True, 0),
    (5, 28672, 4096, True, 1), (17, 28672, 4096, False, None),
    (8, 4608, 3584, False, None), (8, 5632, 2048, False, 0),
    (16, 5504, 2560, False, None), (2, 7680, 5120, False, None),
    (4, 6144, 4096, False, 0), (5, 6144, 4096, False, None),
    (1, 1152, 7168, False, None), (4, 4096, 11008, False, 0),
    (5, 4096, 11008, False, None), (4, 4096, 14336, False, 0),
    (4, 64, 4096, True, None), (4, 64, 4096, False, 0),
    (8, 256, 2048, True, 0), (9, 256, 2048, True, None),
    (16, 2048, 4096, True, None), (16, 2048, 4096, False, 0),
    (16, 4096, 4096, True, 0), (17, 4096, 4096, False, None)])
def test_lines_of_the_rule(T, N, K, f32, how):
    assert sv.stream_rule(T, N, K, f32) == how


@pytest.mark.parametrize("rows,heads,groups,D,keys,modified,want", [
    # 32 unequal rows of up to 3729 keys: 4 workgroups each 50.0 us, 8 51.8; of up
    # to 2658 37.6 and 40.7; 33 equal ones of 4000 1.07 and 1.01 of the best number
    (32, 32, 8, 128, 4097, False, (2, 4)), (32, 32, 8, 64, 300, False, (2, 1)),
    (1, 32, 8, 128, 4097, False, (2, 33)), (1, 32, 8, 128, 300, False, (2, 3)),
    (16, 32, 8, 128, 300, False, (2, 3)), (17, 32, 8, 128, 300, False, (2, 1)),
    # many workgroups of short rows
    (16, 32, 32, 128, 64, False, (2, 1)), (17, 32, 32, 128, 64, False, (1, 1)),
    (17, 32, 32, 128, 65, False, (2, 1)),
    (33, 32, 32, 128, 200, False, (1, 1)),
    (33, 32, 32, 128, 201, False, (2, 1)),
    (17, 32, 32, 128, 200, True, (1, 1)),
    (33, 32, 16, 128, 64, False, (1, 1)), (33, 32, 16, 128, 65, False, (2, 1)),
    (129, 32, 16, 128, 100, False, (1, 1)),
    (129, 24, 8, 128, 20, False, (2, 1)),
    (64, 32, 32, 64, 64, False, (2, 1)), (65, 32, 32, 64, 64, False, (1, 1)),
    (33, 32, 32, 64, 64, True, (1, 1)), (65, 64, 32, 64, 64, False, (2, 1)),
    # a bound that nobody gave
    (65, 32, 32, 128, 0, False, (2, 1))])
def test_kernel_of_single_rows(rows, heads, groups, D, keys, modified, want):
    assert sv.rows_kernel(rows, heads, groups, D, keys, modified) == want


@pytest.mark.parametrize("rows,groups,keys,want", [
    # each line of the table, and past it
    (8, 8, 256, 1), (8, 8, 257, 3), (8, 8, 2500, 4), (8, 8, 2501, 8),
    (9, 8, 700, 6), (16, 8, 2501, 4), (16, 8, 5001, 6), (17, 8, 700, 1),
    (17, 8, 701, 1), (17, 8, 1201, 3), (17, 8, 2501, 7), (32, 8, 1200, 1),
    (32, 8, 1201, 2), (31, 8, 2501, 4), (32, 8, 2501, 4), (33, 8, 2501, 7),
    (31, 8, 5001, 8), (32, 8, 5001, 8), (33, 8, 1200, 1), (33, 8, 1201, 3),
    (40, 8, 1201, 3), (41, 8, 1201, 1), (65, 8, 1200, 1), (65, 8, 1201, 1),
    (65, 8, 2501, 3), (512, 8, 9000, 1), (1, 8, 100000, 64)])
def test_workgroups_that_share_a_row(rows, groups, keys, want):
    assert sv.rows_kernel(rows, 4 * groups, groups, 128, keys) == (2, want)


@pytest.mark.parametrize("rows,width,ff,want", [
    # streaming, to the line of each size and past it
    (1, 2048, 1408, 1), (23, 2048, 1408, 1), (24, 2048, 1408, 4),
    (23, 4096, 4096, 1), (15, 4096, 4104, 1), (16, 4096, 4104, 2),
    (3, 4104, 2048, 1), (4, 4104, 2048, 2), (23, 1000, 2760, 1),
    (23, 4104, 2048, 2), (24, 4104, 2048, 3), (23, 4096, 896, 1),
    # tiles of sizes that are read two steps ahead
    (24, 4096, 14336, 3), (47, 4096, 14336, 3), (48, 4096, 14336, 4),
    (111, 2048, 1408, 4), (112, 2048, 1408, 5), (24, 5120, 2048, 3),
    # and of others
    (24, 1000, 2760, 3), (111, 2048, 1416, 3), (112, 2048, 1416, 4),
    (159, 2048, 1416, 4), (160, 2048, 1416, 5)])
def test_kernel_of_the_experts(rows, width, ff, want):
    assert sv.moe_kernel(rows * 8, 8, width, ff) == want


@pytest.mark.parametrize("rows,experts,width,ff,want", [
    (3, 128, 2048, 768, 1), (4, 128, 2048, 768, 2), (4, 64, 768, 2048, 2),
    (4, 64, 2048, 520, 2), (4, 64, 2048, 512, 1), (4, 64, 2048, 968, 1)])
def test_kernel_of_many_small_experts(rows, experts, width, ff, want):
    assert sv.moe_kernel(rows * experts, experts, width, ff) == want


def test_a_choice_without_the_sizes_is_refused():
    with pytest.raises(TypeError):
        sv.moe_kernel(64, 8)


def test_rotary_tables_hold_every_position():
    """Of two tables the shorter one counts; the longer one may be so."""
    cos, sin = torch.zeros(90, 32), torch.zeros(100, 32)
    q, k = torch.zeros(2, 256), torch.zeros(2, 64)
    pos = torch.zeros(2, dtype=torch.int32)
    for pair in ((cos, sin), (sin, cos), (cos, cos)):
        sv._check_rotary(*pair, q, k, pos, 64, 90)
        with pytest.raises(ValueError, match="position 90"):
            sv._check_rotary(*pair, q, k, pos, 64, 91)
    with pytest.raises(AssertionError):
        sv._check_rotary(cos, torch.zeros(90, 64), q, k, pos, 64, 90)


@pytest.mark.parametrize("rows,heads,keys,want", [
    # none merged: short rows, up to 256 keys of more than 32 workgroups
    (1, 32, 128, 1), (1, 32, 129, 3), (32, 32, 256, 4), (33, 32, 256, 1),
    (17, 64, 256, 1), (9, 128, 200, 1), (33, 8, 257, 5), (200, 64, 9000, 1),
    # workgroups of 64 keys, then of 128
    (1, 32, 1000, 16), (8, 32, 4096, 32), (32, 32, 4096, 16),
    (256, 32, 9000, 2), (257, 32, 9000, 1)])
def test_workgroups_of_a_latent_row(rows, heads, keys, want):
    R, P = 64, 64
    q = torch.zeros(rows, heads * (R + P), dtype=torch.bfloat16)
    cache = torch.zeros(1, 64, R + P, dtype=torch.bfloat16)
    i = torch.zeros(rows, dtype=torch.int32)
    a, part = sv._latent_rows_args(q, cache, R, i, i, i.view(-1, 1), heads, 1.0,
                                   0, keys, None, q)
    assert a.splits == want
    # the launcher takes no more workgroups of 32 heads, nor the workspace less
    assert want == 1 or rows * want <= 512 and part.numel() == \
        rows * want * heads * (R + 2) + 2 * rows


def test_every_ring_is_one_that_the_launcher_takes():
    """Blocks of 64 columns, one a wave at least; x in registers up to 8192
    columns of 16 rows or 4096 of 32; whole words of gated results."""
    taken = set()
    for T in range(1, 33):
        for N in SIZES:
            for K in SIZES + (512 + 64, 4096 + 64, 11008):
                for f32, glu in ((False, False), (True, False), (False, True)):
                    how = sv.ring_rule(T, N, K, f32, glu)
                    taken.add(how)
                    if how is None:
                        continue
                    assert K % 64 == 0 and K >= 512 and not (glu and N % 8)
                    if how == 2:
                        assert K <= (8192 if T <= 16 else 4096)
    assert taken == {None, 2, 3}


def test_every_cut_is_one_that_the_launcher_takes():
    """Shares of K of 256 columns at least, whole words of gated results, and none
    of what the kernels of fewer rows are there for."""
    taken = set()
    for T in range(1, 130, 3):
        for N in SIZES:
            for K in SIZES + (512 + 64, 11008):
                for f32, glu in ((False, False), (True, False), (False, True)):
                    splits = sv.wide_rule(T, N, K, f32, glu)
                    if splits is None:
                        continue
                    taken.add(splits)
                    assert 9 <= T <= 128 and K % 64 == 0 and N % 8 == 0
                    assert 1 <= splits <= K // 256 and not (glu and N % 32)
                    assert splits == 1 or splits * -(-N // 128) <= 256
    assert 1 in taken and len(taken) > 5


@pytest.mark.parametrize("T,N,K,glu,want", [
    # each line of a few weight rows, and past it; us by the library, and by shares
    (28, 1024, 8192, True, None),            # 13.7, 15.7
    (28, 1024, 11008, True, 8), (28, 1024, 14336, True, None),
    (20, 4096, 8192, True, None),            # 20.2, 21.8
    (20, 4096, 5120, True, 8), (48, 2496, 5120, True, None),
    (48, 3072, 4096, True, None),            # 15.8, 17.3
    (48, 3072, 5120, True, 8), (72, 2560, 5120, True, None),
    (72, 2560, 6144, True, 8), (48, 4544, 3072, True, 6),
    (48, 2560, 3072, False, None),           # 10.4, 12.5
    (48, 2560, 4096, False, None), (48, 2560, 5120, False, 12),
    (48, 3584, 3584, False, None), (48, 3584, 4096, False, 9),
    (48, 1536, 4096, False, 16), (48, 1536, 3584, False, None),
    (100, 4096, 3072, False, None), (100, 4096, 4096, False, 6),
    (64, 4096, 4096, False, 8), (100, 4096, 4160, False, 8),
    (128, 1024, 8192, False, None),          # 14.8, 16.4
    (128, 1024, 11008, False, 16), (112, 2560, 7168, False, 12),
    (112, 50304, 2560, False, None),         # 62.5, 70.7
    (112, 24576, 3072, False, 1), (64, 50304, 2560, False, 1),
    (100, 8192, 4096, False, 3), (100, 8200, 4096, False, 3)])
def test_lines_of_the_shares(T, N, K, glu, want):
    assert sv.wide_rule(T, N, K, False, glu) == want


@pytest.mark.parametrize("T,N,K,f32,want", [
    (24, 512, 768, False, None), (24, 1024, 960, False, None),   # 5.0, 6.0
    (24, 1024, 1024, False, 3), (24, 1040, 768, False, 3),
    (6, 4096, 2560, False, None), (9, 4096, 2560, False, 3),     # streamed 6.5, 7.1
    (8, 2064, 3072, False, None), (8, 2048, 3072, False, 3),
    (8, 4112, 3072, False, 3)])
def test_lines_of_the_rings(T, N, K, f32, want):
    assert sv.ring_rule(T, N, K, f32) == want


class _OnDevice(torch.Tensor):
    """Rows that say they are on device 0."""
    is_cuda = True

    def get_device(self):
        return 0


@pytest.fixture
def taken(monkeypatch):
    """What ``streamed`` hands to the kernels: (kernel, rows, how)."""
    calls = []
    monkeypatch.setattr(sv, "_LIB", types.SimpleNamespace(
        sv_stream_linear=None, sv_wide_linear=None))
    monkeypatch.setattr(sv, "_plain", lambda t: True)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    for name in ("wide_linear", "stream_linear"):
        def kernel(x, w, how, f32=False, glu=False, name=name):
            calls.append((name, x, how))
            return torch.empty(x.shape[0], w.shape[0] // (2 if glu else 1))
        monkeypatch.setattr(sv, name, kernel)
    return calls


def _on_device(*shape):
    return torch.empty(*shape, dtype=torch.bfloat16).as_subclass(_OnDevice)


@pytest.mark.parametrize("B,S,K,N,glu,want", [
    # beyond the 31 bits of 256 rows' offsets: another kernel, or none
    (20, 1024, 4096, 32000, False, "stream_linear"), (40, 1024, 4096, 32000, False, None),
    (32, 1024, 4096, 28672, True, "stream_linear"), (40, 400, 11008, 4096, False, None),
    # below them
    (20, 1023, 4096, 32000, False, "wide_linear"), (40, 380, 11008, 4096, False, "wide_linear"),
    (1, 1024, 4096, 32000, False, "stream_linear")])
def test_rows_far_apart(taken, B, S, K, N, glu, want):
    """Last tokens of prompts: a view of rows that lie a prompt apart, whatever the
    stride of its middle dimension of one."""
    x, w = _on_device(B, S, K)[:, -1:], _on_device(N, K)
    with torch.no_grad():
        out = sv.streamed(x, w, glu=glu)
    assert [c[0] for c in taken] == ([want] if want else [])
    if want:
        assert out.shape == (B, 1, N // 2 if glu else N)
        assert taken[0][1].stride(0) < 1 << 22 or want == "stream_linear"
    else:
        assert out is None


def test_a_middle_dimension_of_one_counts_for_nothing(taken):
    """Its stride may be anything."""
    x = _on_device(40, 4096).as_strided((40, 1, 4096), (4096, 1 << 23, 1))
    with torch.no_grad():
        sv.streamed(x, _on_device(32000, 4096))
    assert [c[0] for c in taken] == ["wide_linear"]


@pytest.mark.parametrize("T", [1, 16, 40, 128])
def test_weights_without_rows_are_the_library_s(taken, T):
    """There is nothing to share among workgroups."""
    with torch.no_grad():
        for glu in (False, True):
            assert sv.streamed(_on_device(T, 4096), _on_device(0, 4096), glu=glu) is None
            assert sv.stream_how(_on_device(T, 4096), _on_device(0, 4096),
                                 glu=glu) is None
    assert not taken


def test_nobody_is_passed_by(monkeypatch):
    """Calls go past an autograd function only where nobody would miss it."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from neuronx_distributed_amd.ops import swiglu

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    x = torch.randn(3, 16)
    assert not sv.unseen(x)
    want = swiglu(x.clone().requires_grad_())
    assert want.requires_grad
    with torch.no_grad():
        assert sv.unseen(x, None, torch.nn.Parameter(x))
        assert torch.equal(swiglu(x), want)
        assert not sv.unseen(x, x.as_subclass(Sub))
        with Mode():
            assert not sv.unseen(x)
        with torch.autograd.forward_ad.dual_level():
            assert not sv.unseen(x)
        seen = []
        torch.vmap(lambda t: seen.append(sv.unseen(t)) or t)(x)
        assert seen == [False]
        with torch.autocast("cuda"):
            # (there is none without a card)
            assert sv.unseen(x) == (not torch.cuda.is_available())
        enabled = torch.is_autocast_enabled
        monkeypatch.setattr(torch, "is_autocast_enabled",
                            lambda kind=None: kind == "cuda" or enabled(kind))
        assert not sv.unseen(x)
        monkeypatch.undo()
    with torch.inference_mode():
        assert sv.unseen(x)


@pytest.mark.parametrize("T,N,K,want", [
    (1099, 32000, 4096, (False, False)), (1100, 32000, 4096, (True, True)),
    (2600, 32000, 4096, (False, True)), (1599, 3584, 18944, (False, False)),
    (1600, 3584, 18944, (True, False)), (8192, 4096, 4096, (False, False)),
    (8192, 4096, 11008, (True, False)), (16384, 8192, 8192, (True, True))])
def test_operands_of_a_weight_gradient(T, N, K, want):
    from neuronx_distributed_amd.ops import turn_rule

    assert turn_rule(T, N, K) == want


@pytest.mark.parametrize("T,N,K,want", [
    (8192, 32000, 4096, True), (7680, 32000, 4096, False),
    (9000, 4096, 4096, False), (8192, 2048, 5632, False),
    (8192, 27648, 5120, False), (16384, 27648, 5120, True)])
def test_weights_of_an_input_gradient(T, N, K, want):
    from neuronx_distributed_amd.ops import turn_weight_rule

    assert turn_weight_rule(T, N, K) is want


@pytest.mark.parametrize("T,N,K,want", [
    # each line of the rule, and past it
    (2599, 6144, 4096, (False, False)), (1399, 4096, 11008, (False, False)),
    (1400, 4096, 11008, (True, True)), (1100, 4096, 14336, (True, True)), (1100, 5120, 5120, (True, True)),
    (3500, 2560, 9728, (True, False)), (3501, 2560, 9728, (False, False)),
    (3501, 8192, 3072, (False, True)), (3501, 2560, 12288, (True, False)),
    (3072, 11008, 4096, (False, True)), (3073, 11008, 4096, (False, False)),
    (8191, 11008, 4096, (False, False)), (8192, 11008, 4096, (False, True)),
    (9216, 5120, 5120, (True, False)), (9217, 5120, 5120, (False, False)),
    (9217, 3584, 8192, (False, False)), (9217, 8192, 3072, (False, True)),
    (8192, 6144, 4096, (False, False)), (5000, 22016, 4096, (False, True))])
def test_operands_that_are_not_turned(T, N, K, want):
    from neuronx_distributed_amd.ops import turn_rule

    assert turn_rule(T, N, K) == want


@pytest.mark.parametrize("T,want", [
    (7936, False), (7937, True), (8192, True), (8193, False), (8704, False),
    (12032, False), (12288, True), (15872, False), (24575, True), (24577, True),
    (24320, False), (30000, True)])
def test_weights_are_turned_for_whole_rounds(T, want):
    from neuronx_distributed_amd.ops import turn_weight_rule

    assert turn_weight_rule(T, 4096, 4096) is want


@pytest.mark.parametrize("shape,stride", [
    ((8, 1, 6), (6, 48, 1)), ((1, 8, 6), (6, 6, 1)), ((8, 1, 6), (6, 6, 1)),
    ((2, 4, 6), (24, 6, 1)), ((8, 6), (6, 1))])
@pytest.mark.parametrize("overlapped", [False, True])
def test_input_gradients_are_one_product(monkeypatch, shape, stride, overlapped):
    """Also of gradients that are contiguous with any stride of a dimension of one:
    one sequence, tokens first.  Not a batch of products with a turned weight."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from neuronx_distributed_amd import ops
    from neuronx_distributed_amd.parallel import layers

    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            seen.append(str(f))
            return f(*args, **(kwargs or {}))

    turned = []

    def turn(dy, w):
        turned.append(w)
        return w.detach().t().contiguous().t()

    for module in (ops, layers):
        monkeypatch.setattr(module, "input_weight", turn, raising=False)
    monkeypatch.setattr(layers.ps, "get_group_info",
                        lambda name: types.SimpleNamespace(size=1, group=None))
    monkeypatch.setattr(layers.comm, "all_gather", lambda t, dim, group: t)
    dy = torch.randn(8, 6).as_strided(shape, stride)
    assert dy.is_contiguous()
    x, w = torch.randn(*shape[:-1], 4), torch.randn(6, 4).requires_grad_()
    ctx = types.SimpleNamespace(
        saved_tensors=(x, w), compute_weight_gradient=True, use_bias=False,
        sequence_parallel_enabled=False, async_grad_allreduce=False)
    function = layers._RPLOverlappedLinearRS if overlapped else \
        layers.LinearWithAsyncCommunication
    with torch.no_grad(), Watch():
        dx, dw = function.backward(ctx, dy)[:2]
    assert turned and not any("bmm" in f for f in seen)
    rows = dy.reshape(8, 6)
    torch.testing.assert_close(dx, (rows @ w).view(x.shape))
    torch.testing.assert_close(dw, rows.t() @ x.reshape(8, 4))


@pytest.mark.parametrize("grad", [False, True])
def test_embeddings_are_traced_symbolically(monkeypatch, grad):
    """Nothing is asked of a proxy that steers the program."""
    from neuronx_distributed_amd.parallel import layers

    monkeypatch.setattr(layers.ps, "get_tensor_model_parallel_size", lambda: 1)
    embed = layers.ParallelEmbedding.__new__(layers.ParallelEmbedding)
    torch.nn.Module.__init__(embed)
    embed.weight = torch.nn.Parameter(torch.randn(16, 8))
    embed.padding_idx, embed.shard_along_embedding = None, False
    with torch.set_grad_enabled(grad):
        traced = torch.fx.symbolic_trace(torch.nn.Sequential(embed))
    ids = torch.randint(16, (3, 5))
    out = traced(ids)
    assert torch.equal(out, embed.weight[ids])
    (g,) = torch.autograd.grad(out.sum(), embed.weight)
    assert g.shape == embed.weight.shape


def test_an_embedding_without_a_weight_is_called():
    """A served model's look-up may be any module."""
    from neuronx_distributed_amd.models import llama

    class Twice(torch.nn.Module):
        def forward(self, tokens):
            return 2.0 * tokens[:, None]

    pending = llama._embedded(Twice(), torch.tensor([3, 4]))
    assert pending.rows is None
    assert torch.equal(pending.delta, torch.tensor([[6.0], [8.0]]))


@pytest.mark.parametrize("shift,rows", [(0, True), (8, True), (4, False), (1, False)])
def test_rows_of_a_table_start_at_whole_words(taken, monkeypatch, shift, rows):
    """A table inside a larger buffer may start anywhere; its norm reads words."""
    from neuronx_distributed_amd.models import llama
    from neuronx_distributed_amd.parallel import layers

    monkeypatch.setattr(llama.ps, "get_tensor_model_parallel_size", lambda: 1)
    embed = layers.ParallelEmbedding.__new__(layers.ParallelEmbedding)
    torch.nn.Module.__init__(embed)
    embed.__dict__.update(
        weight=_on_device(5 * 16 + 8)[shift:shift + 80].view(5, 16),
        padding_idx=None, shard_along_embedding=False)
    tokens = torch.tensor([1, 4], dtype=torch.int32)
    with torch.no_grad():
        pending = llama._embedded(embed, tokens)
    assert (pending.rows is tokens) == rows
    assert (pending.delta is embed.weight) == rows


@pytest.mark.parametrize("T,V,W,own", [
    (2048, 1 << 18, 512, True), (2048, (1 << 18) + 1, 512, False),
    (2047, 32000, 4096, False),
    (32768, 32000, 4096, True), (32769, 32000, 4096, False),
    (8192, 32000, 504, False), (8192, 32000, 516, False)])
def test_embedding_gradients_at_their_lines(taken, monkeypatch, T, V, W, own):
    from neuronx_distributed_amd import ops

    went = []
    monkeypatch.setattr(ops._EmbeddingFn, "apply",
                        lambda ids, w, skip: went.append(True) or w[:1])
    weight = _on_device(V, W).requires_grad_()
    assert ops.embedding_rule(T, V, W) is own
    ops.embedding(torch.zeros(T, dtype=torch.int64), weight)
    assert bool(went) == own


@pytest.mark.parametrize("short", [0, 1, 8])
def test_a_latent_step_reads_whole_queries(monkeypatch, short):
    """Queries whose last head's turned columns are not all there are refused."""
    H, dim, P, R, vdim, T = 2, 16, 8, 16, 8, 3
    calls = []
    monkeypatch.setattr(sv, "_LIB", types.SimpleNamespace(
        sv_latent_step=lambda *a: calls.append(a) or 0))
    monkeypatch.setattr(sv, "_stream", lambda: None)
    def rand(*shape):
        return torch.randn(*shape, dtype=torch.bfloat16)
    w = sv.LatentWeights(rand(R), rand(H, R, dim), rand(H * (dim + vdim), R),
                         torch.ones(P // 2, dtype=torch.float64).as_subclass(_OnDevice))
    ints = torch.zeros(T, dtype=torch.int32)
    batch = types.SimpleNamespace(portion_tokens=0, spans={}, pos=ints, seq=ints,
                                  block_table=ints.view(-1, 1), max_keys=64)
    q = rand(T, H * (dim + P) + 8)[:, :H * (dim + P) - short]
    step = lambda: sv.latent_attention(q, rand(T, R + P), None, batch,  # noqa: E731
                                       rand(1, 64, R + P), w, H, dim, vdim, 0.1, 1e-5)
    if short:
        with pytest.raises(AssertionError):
            step()
    else:
        step()
    assert len(calls) == (not short)


def test_a_card_without_room_turns_nothing(monkeypatch):
    """Gradients that fit without a turned copy still do."""
    from neuronx_distributed_amd import ops

    def full(*a, **k):
        raise torch.OutOfMemoryError("full")

    x = torch.randn(16, 8)
    monkeypatch.setattr(torch, "empty", full)
    assert ops._turned(x) is x
    monkeypatch.setattr(ops, "input_weight", lambda dy, w: ops._turned(w))
    w = torch.randn(8, 4)
    torch.testing.assert_close(ops.input_grad(x, w), x @ w)
