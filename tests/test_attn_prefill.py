"""Prefill attention with the keys split over a workgroup's waves (csrc/attention.hip
k_attn_pre) against the softmax in 64 bits, at the edges of its tiles: query sub-tiles of 32
(1, 2 and 4 per workgroup), key blocks of 32, partly and wholly masked blocks and rows.

Tolerance: scores, weights and sums are fp32 (products of exact fp16 pairs), so an output is
off by a few fp32 roundings of sums of n_kv terms of the same size: 2e-6 of the largest
output. Fewer than 64 query rows round the query to fp16, as the reference rows here do."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from ggmlc_amd import ops
from test_gemm_q8_model import bench_lib

DEV = "cuda"


def run(Hq, Hkv, D, S, n_kv, mask, strided=False):
    g = torch.Generator(device=DEV)
    g.manual_seed(Hq * 1000 + S + n_kv + D)
    q = torch.randn((S, Hq, D), generator=g, device=DEV)
    ctx = n_kv + (40 if strided else 0)
    k = torch.randn((Hkv, ctx, D), generator=g, device=DEV).to(torch.float16)
    v = torch.randn((Hkv, ctx, D), generator=g, device=DEV).to(torch.float16)
    k[:, n_kv:], v[:, n_kv:] = float("nan"), float("nan")  # rows past the view are never used
    scale = 1.0 / math.sqrt(D)
    got = ops.flash_attn_ext(q.permute(1, 0, 2), k[:, :n_kv], v[:, :n_kv], mask, scale)
    torch.cuda.synchronize()
    qd = (q.to(torch.float16) if S < 64 else q).double()
    kd, vd = (t[:, :n_kv].double().repeat_interleave(Hq // Hkv, 0) for t in (k, v))
    s = torch.matmul(qd.permute(1, 0, 2), kd.transpose(1, 2).contiguous()) * scale
    if mask is not None:
        s = s + mask.double()[None]
    w = torch.softmax(s, -1)
    w = torch.where(torch.isnan(w), torch.zeros_like(w), w)  # a row masked with -inf throughout: 0
    want = torch.matmul(w, vd).permute(1, 0, 2)
    assert torch.isfinite(got).all()
    err = (got.double() - want).abs().amax((1, 2)) / want.abs().max()
    # a row with only -32768 entries: fp32 holds s - 32768 to 2^-8 (its last place there), which
    # is the relative error of each weight
    tol = torch.full_like(err, 2e-6)
    if mask is not None:
        tol[mask.amax(-1) == -32768.0] = 2.0**-8
    assert (err < tol).all(), err.max().item()


def causal(S, n_kv, pos, fill=-32768.0):
    ok = torch.arange(n_kv, device=DEV)[None] <= pos + torch.arange(S, device=DEV)[:, None]
    return torch.where(ok, 0.0, fill).to(torch.float16)


CAUSAL = [
    (2, 1, 5, 256, 3),        # the smallest: 10 query vectors of a sub-tile of 32
    (1, 1, 31, 32, 1),        # one key block, one query short of a sub-tile
    (1, 1, 33, 36, 3),        # one query and one group of 4 keys past a tile
    (12, 2, 201, 2048, 1700),  # 6 query heads per kv head, a ragged chunk on a long past
    (32, 32, 257, 512, 250),  # more workgroups than CUs, one query past a sub-tile
    (40, 40, 512, 768, 131),  # two sub-tiles per workgroup, rows past the queries in none
    (32, 32, 545, 772, 227),  # two, the last sub-tile with one query
    (64, 32, 516, 516, 0),    # four sub-tiles per workgroup, the last with 8 query vectors
    (15, 5, 100, 100, 0),
    (4, 1, 65, 4096, 4000),   # the keys split over workgroups
]
# one workgroup per tile; one of several rounds; the keys split over workgroups; two and four sub-tiles
MASKS = [(4, 2, 70, 300), (32, 32, 300, 260), (32, 16, 70, 1044), (12, 2, 66, 3000), (32, 32, 545, 580), (64, 32, 530, 580)]


def launch(Hq, Hkv, S, n_kv, D=128):
    """plan_attn_pre: (32-query sub-tiles per workgroup, key splits over workgroups)"""
    nq, out = Hq // Hkv * S, (ctypes.c_int * 2)()
    need = ops.flash_attn_workspace_size(D, S, Hq, Hkv, n_kv)  # n_split * Hkv * NQ * (D + 2) floats
    lib = bench_lib()
    lib.gqbench_attn_pre_plan.argtypes = [ctypes.c_int64] * 4 + [ctypes.POINTER(ctypes.c_int)]
    lib.gqbench_attn_pre_plan.restype = None
    lib.gqbench_attn_pre_plan(nq, Hkv, n_kv, max(1, need // (Hkv * nq * (D + 2) * 4)), out)
    return tuple(out)


def test_shapes_cover_every_launch():
    for D in (64, 128):
        got = [launch(*c[:4], D=D) for c in CAUSAL]
        assert [n for n, _ in got] == [1, 1, 1, 1, 1, 2, 2, 4, 1, 1] and got[3][1] > 1 and got[9][1] > 1
        assert [launch(*c, D=D) for c in MASKS] == [(1, 1), (1, 1), (1, 2), (1, 5), (2, 1), (4, 1)]
    for Hq, Hkv, S, _ in MASKS[4:]:
        assert Hq // Hkv * S % 64 and Hq // Hkv * S % 128 > 32  # a remainder, and some sub-tile cut


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,S,n_kv,pos", CAUSAL)
def test_causal(D, Hq, Hkv, S, n_kv, pos):
    run(Hq, Hkv, D, S, n_kv, causal(S, n_kv, pos), strided=True)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,S,n_kv", MASKS)
def test_masks(Hq, Hkv, S, n_kv, D):
    """no mask; a sliding window (leading blocks left out); -inf holes; finite biases; rows
    masked throughout, which make the tile run again with every block"""
    run(Hq, Hkv, D, S, n_kv, None)
    i, j = torch.arange(S, device=DEV)[:, None], torch.arange(n_kv, device=DEV)[None]
    run(Hq, Hkv, D, S, n_kv, torch.where((j - i).abs() < 20, 0.0, -32768.0).to(torch.float16))
    holes = torch.where((i * 7 + j * 13) % 5 == 0, 0.0, float("-inf")).to(torch.float16)
    run(Hq, Hkv, D, S, n_kv, holes)
    run(Hq, Hkv, D, S, n_kv, (-0.01 * (i - j).abs()).to(torch.float16))
    run(Hq, Hkv, D, S, n_kv, causal(S, n_kv, n_kv - S))
    late = torch.where((j > n_kv - 40) & (j <= n_kv - 40 + i), 0.0, -32768.0)  # row 0 sees nothing,
    late[0, n_kv - 1] = 0.0  # the others one split's keys only
    run(Hq, Hkv, D, S, n_kv, late.to(torch.float16))
    one = torch.where((j - 37 * i) % n_kv == 0, 0.0, -32768.0)  # one key per row, all over the blocks
    run(Hq, Hkv, D, S, n_kv, one.to(torch.float16))
    m = causal(S, n_kv, 5)
    m[S // 3] = -32768.0  # one row without an unmasked key: uniform weights plus the scores
    run(Hq, Hkv, D, S, n_kv, m)
    m[S // 2] = float("-inf")  # and one with nothing at all: zeros
    run(Hq, Hkv, D, S, n_kv, m)


def masks(S, n_kv):
    """causal, banded, -inf holes, finite biases, one key no wave's first lane sees, a row without an
    unmasked key, one without any"""
    i, j = torch.arange(S, device=DEV)[:, None], torch.arange(n_kv, device=DEV)[None]
    yield causal(S, n_kv, n_kv - S)
    yield torch.where((j - i).abs() < 20, 0.0, -32768.0).to(torch.float16)
    yield torch.where((i * 7 + j * 13) % 5 == 0, 0.0, float("-inf")).to(torch.float16)
    yield (-0.01 * (i - j).abs()).to(torch.float16)
    m = causal(S, n_kv, 3)
    m[S // 2 + 1, n_kv - 2] = 0.0
    yield m
    m = causal(S, n_kv, 5)
    m[S // 3] = -32768.0
    m[S // 2] = float("-inf")
    yield m


def shifted(m):
    """the mask at an address that is not 8-byte aligned"""
    b = torch.empty(m.numel() + 1, dtype=m.dtype, device=DEV)[1:].view(m.shape)
    return b.copy_(m)


def odd_rows(m):
    """the mask's rows an odd number of values apart"""
    return torch.empty((m.shape[0], m.shape[1] + 1 + m.shape[1] % 2), dtype=m.dtype, device=DEV)[:, :-1][
        :, :m.shape[1]].copy_(m)


def past_2gib(m):
    """the mask's rows spread over more than 2 GiB"""
    step = 3 * 2**29 // m.shape[0] // 8 * 8  # values from row to row: a third of the rows behind 2 GiB
    b = torch.empty(step * (m.shape[0] - 1) + m.shape[1], dtype=m.dtype, device=DEV)
    assert 2 * (b.numel() - m.shape[1]) > 2**31 + 2**29
    return b.as_strided(m.shape, (step, 1)).copy_(m)


# tiles of 32 and of 64 query vectors
@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,S,n_kv", [(4, 2, 70, 300), (32, 32, 300, 304)])
def test_masks_the_split_kernel_does_not_read(Hq, Hkv, S, n_kv, D):
    """k_attn_mma: masks not 8-byte aligned, n_kv % 4 != 0, 2 GiB and more"""
    for m in masks(S, n_kv):
        run(Hq, Hkv, D, S, n_kv, shifted(m))
        run(Hq, Hkv, D, S, n_kv, odd_rows(m))
    for n in (n_kv + 1, n_kv + 3):
        for m in masks(S, n):
            run(Hq, Hkv, D, S, n, m)
    run(Hq, Hkv, D, S, n_kv, past_2gib(causal(S, n_kv, n_kv - S)))


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,S,n_kv", [(4, 2, 70, 300), (32, 32, 300, 304), (12, 2, 70, 2048)])
def test_mask_rows_that_overlap(Hq, Hkv, S, n_kv):
    """one mask row for every query, and rows that start one 8-byte step after another"""
    j = torch.arange(n_kv, device=DEV)
    run(Hq, Hkv, 128, S, n_kv, torch.where(j % 3 == 1, 0.0, -32768.0).to(torch.float16)[None].expand(S, n_kv))
    b = torch.where(torch.arange(n_kv + 4 * S, device=DEV) % 7 < 3, 0.0, -32768.0).to(torch.float16)
    run(Hq, Hkv, 128, S, n_kv, b.as_strided((S, n_kv), (4, 1)))
