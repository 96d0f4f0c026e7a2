"""The prefill GEMM's tiles, K splits and segments (csrc/plans.h plan_gemm_q8, k_reduce_q8) on the
GPU: every tile height, with and without splits and segments, outputs of odd width and spaced rows,
against the block formula in 64 bits.

Tolerance: block sums and scale products are exact, the sum over the nb blocks is fp32: nb
roundings of 2^-24 of partial sums no larger than a few times the largest output."""

from __future__ import annotations

import pytest
import torch

from ggmlc_amd import ops
from test_gemm_q8_model import bench_lib, chain_bound, plan

SHAPES = [
    (130, 512, 17), (131, 4096, 40),  # one 32-row tile; splits, rows not 16-byte aligned
    (12288, 1024, 300), (4096, 4096, 300), (22016, 512, 180), (4096, 4096, 333), (16384, 576, 512), (4096, 11008, 512),
    (32000, 960, 64), (12288, 4096, 512), (1600, 960, 37),  # sums in segments,
    (960, 2560, 64), (1536, 8960, 160), (22016, 4096, 200),  # also of K splits
]


def test_shapes_cover_every_launch():
    """every tile height, with and without K splits and segments, for each weight type"""
    for qt in (ops.Q8_0, ops.Q4_0):
        plans = [plan(qt, *s) for s in SHAPES]
        assert {(p[0], p[3] < p[2]) for p in plans} == {(1, False), (1, True), (2, False), (2, True), (3, False), (4, False)}
        assert {(p[1] > 1, p[3] < p[2]) for p in plans} == {(a, b) for a in (False, True) for b in (False, True)}


def _dequant(b, qt):
    d = b[..., :2].contiguous().view(torch.float16).double()
    qs = b[..., 2:].contiguous()
    q = qs.view(torch.int8).double() if qt == ops.Q8_0 else torch.cat([qs & 15, qs >> 4], -1).double() - 8
    return (q * d).flatten(1)


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [ops.Q8_0, ops.Q4_0])
@pytest.mark.parametrize("N,K,M", SHAPES)
def test_against_block_formula(qt, N, K, M):
    g = torch.Generator(device="cuda")
    g.manual_seed(N + K + M + qt)
    b = torch.randint(0, 256, (N, K // 32, ops.BLOCK_BYTES[qt]), generator=g, device="cuda", dtype=torch.uint8)
    d = (torch.rand((N, K // 32, 1), generator=g, device="cuda") * 0.01).to(torch.float16)
    b[..., :2] = d.view(torch.uint8)
    w = ops.QWeight(b.flatten(1).contiguous(), qt, K)
    x = torch.randn((M, K), generator=g, device="cuda")
    xq = ops.quantize_row_q8_0(x).view(M, K // 32, 34)
    want = _dequant(xq, ops.Q8_0) @ _dequant(b, qt).t()
    tol = 2.0**-24 * (K // 32) * want.abs().max().item()
    err = ops.mul_mat(w, x).double() - want
    assert err.abs().max().item() <= tol
    # c roundings of partial sums that grow like a random walk: each of variance ulp^2 / 12, ulp^2
    # on average 0.57 (2^-23)^2 of the square, c / 2 of the final sum's square in all; 1.1 for c's
    # own spread over the shapes
    c = chain_bound(qt, bench_lib().gqbench_fp16_pair_chain(N, K, M, 256))
    assert (err.norm() / want.norm()).item() <= 1.1 * 2.0**-23 * (c / 2 * 0.57 / 12) ** 0.5
    # rows of a wider buffer: split 0's slab keeps to its columns
    wide = torch.full((M, N + 5), 7.0, device="cuda")
    ops.mul_mat(w, x, out=wide[:, :N])
    assert (wide[:, :N].double() - want).abs().max().item() <= tol
    assert (wide[:, N:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [ops.Q8_0, ops.Q4_0])
def test_subnormal_scales(qt):
    """weight and activation scales below 2^-14, where fp16 keeps fewer bits: their products stay exact"""
    N, K, M = 200, 1088, 40
    g = torch.Generator(device="cuda")
    g.manual_seed(qt)
    b = torch.randint(0, 256, (N, K // 32, ops.BLOCK_BYTES[qt]), generator=g, device="cuda", dtype=torch.uint8)
    d = (torch.rand((N, K // 32, 1), generator=g, device="cuda") * 5e-5).to(torch.float16)
    b[..., :2] = d.view(torch.uint8)
    x = torch.randn((M, K), generator=g, device="cuda") * 1e-3
    xq = ops.quantize_row_q8_0(x).view(M, K // 32, 34)
    assert xq[..., :2].contiguous().view(torch.float16).max() < 2.0**-14 and d.max() < 2.0**-14
    want = _dequant(xq, ops.Q8_0) @ _dequant(b, qt).t()
    err = ops.mul_mat(ops.QWeight(b.flatten(1).contiguous(), qt, K), x).double() - want
    assert err.abs().max().item() <= 2.0**-24 * (K // 32) * want.abs().max().item()
