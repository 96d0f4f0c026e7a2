"""Products of weights with an odd number of blocks per row (csrc/gemm.hip: fp16 pairs, whose rows are
only 2-byte aligned) for more than 4 rows: 64- and 128-token tiles with and without K splits, the
last round of tiles as a launch of its own, row scales and the fused prologues, against the block
formula in 64 bits.

Tolerance: products of the fp16 pairs are exact; a block's sum and the sum over the nb blocks are
fp32, nb roundings of 2^-24 of partial sums no larger than a few times the largest output (those
inside a block are of its own, smaller, sum)."""

from __future__ import annotations

import pytest
import torch

import oracle as O
from ggmlc_amd import ops
from test_gemm_addressing import launches
from test_gemm_q8_plan import _dequant
from test_gpu_kernels import _big_rows, mar

SHAPES = [
    (300, 96, 17),        # 64-token tiles in one part, rows not 16-byte aligned
    (96, 11040, 17),      # in K splits
    (1024, 4128, 128),    # two tiles of tokens, splits
    (16500, 96, 130),     # 128-token tiles in one part
    (2048, 2080, 100),    # in K splits
    (16500, 1056, 130),   # the last round of tiles with K split as its own launch
    (96, 17440, 17),      # K past the one-launch prologue: blocks, then row scales in a pass of their own
]


def _weight(N, K, qt, g):
    b = torch.randint(0, 256, (N, K // 32, ops.BLOCK_BYTES[qt]), generator=g, device="cuda", dtype=torch.uint8)
    b[..., :2] = (torch.rand((N, K // 32, 1), generator=g, device="cuda") * 0.01).to(torch.float16).view(torch.uint8)
    return ops.QWeight(b.flatten(1).contiguous(), qt, K), b


def _want(x, b, qt):
    M, K = x.shape
    return _dequant(ops.quantize_row_q8_0(x).view(M, K // 32, 34), ops.Q8_0) @ _dequant(b, qt).t()


def test_shapes_cover_every_launch():
    got = [[(bm, ks > 1) for _, bm, ks, _ in launches(*s)] for s in SHAPES]
    assert got == [[(64, False)], [(64, True)], [(64, True)], [(128, False)], [(128, True)],
                   [(128, False), (128, True)], [(64, True)]]
    assert all(k // 32 % 2 for _, k, _ in SHAPES)


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [ops.Q8_0, ops.Q4_0])
@pytest.mark.parametrize("N,K,M", SHAPES)
def test_against_block_formula(qt, N, K, M):
    g = torch.Generator(device="cuda")
    g.manual_seed(N + K + M + qt)
    w, b = _weight(N, K, qt, g)
    x = torch.randn((M, K), generator=g, device="cuda")
    want = _want(x, b, qt)
    tol = 2.0**-24 * (K // 32) * want.abs().max().item()
    assert (ops.mul_mat(w, x).double() - want).abs().max().item() <= tol
    wide = torch.full((M, N + 5), 7.0, device="cuda")
    ops.mul_mat(w, x, out=wide[:, :N])
    assert (wide[:, :N].double() - want).abs().max().item() <= tol
    assert (wide[:, N:] == 7.0).all()
    if K <= 16384:  # the bias in the epilogue or the reduce
        bias = torch.randn((N,), generator=g, device="cuda")
        assert torch.equal(ops.mul_mat_fused(w, x, bias=bias), ops.mul_mat(w, x) + bias)


@pytest.mark.gpu
@pytest.mark.parametrize("qt", [ops.Q8_0, ops.Q4_0])
@pytest.mark.parametrize("N,K,M", [(1024, 4128, 17), (2048, 2080, 100), (96, 17440, 17)])
def test_large_activations(qt, N, K, M):
    """blocks with amax up to 8e6, where d * q leaves the fp16 range: the row scales"""
    g = torch.Generator(device="cuda")
    g.manual_seed(K + N + M)
    w = ops.quantize_weights(torch.randn((N, K), generator=g, device="cuda") * 0.02, qt)
    x = _big_rows(M, K, K + M)
    y = ops.mul_mat(w, torch.from_numpy(x).cuda()).cpu().numpy()
    want = O.mul_mat(w.data.cpu().numpy(), qt, K, x)
    for m in range(min(M, 6)):  # each large row at the bar on its own
        assert mar(y[m], want[m]) < 1e-5, m
    assert mar(y, want) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("K,N,M", [(4128, 300, 17), (2080, 2048, 100)])
def test_fused_prologues(K, N, M):
    """ADD, RMS_NORM and SWIGLU in front give the bits of the ops run one by one"""
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    w, _ = _weight(N, K, ops.Q8_0, g)
    x, d = (torch.randn((M, K), generator=g, device="cuda") for _ in range(2))
    xs = torch.empty_like(x)
    got = ops.mul_mat_fused(w, x, rms_eps=1e-5, x_add=d, x_sum=xs)
    s = ops.add(x, d)
    assert torch.equal(xs, s) and torch.equal(got, ops.mul_mat(w, ops.rms_norm(s, 1e-5)))
    gu = torch.randn((M, 2 * K), generator=g, device="cuda")
    assert torch.equal(ops.mul_mat_fused(w, gu, x_swiglu=True), ops.mul_mat(w, ops.swiglu(gu)))
