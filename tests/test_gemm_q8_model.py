"""Host model of the int8 prefill GEMM (csrc/gemm_q8.hip k_gemm_q8): every global load, LDS
address and store of a launch checked against the buffers, and its data path (prologue
layout, LDS staging, MFMA operands, accumulator layout) emulated lane by lane against the
block formula."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from test_gemm_addressing import launches

QK, BN, SBLK, ROW = 32, 128, 4, 128
Q8, Q4 = 8, 2
BB = {Q8: 34, Q4: 18}


def cdiv(a, b):
    return -(-a // b)


def part_room(N, K, M):
    """workspace left for the partials behind the activation (api.hip plan_mul_mat)"""
    from ggmlc_amd import _lib

    w = _lib.make_tensor(0x1000, _lib.Q8_0, [K, N], [34, K // QK * 34])
    x = _lib.make_tensor(0x1000, _lib.F32, [K, M], [4, 4 * K])
    return _lib.load().gq_mul_mat_workspace_size(w, x) - cdiv(cdiv(K, ROW) * M * (ROW + 8), 256) * 256


def bench_lib():
    """libgqbench.so, which answers the library's own plans without a device"""
    from ggmlc_amd import build

    lib = ctypes.CDLL(str(build.BENCH_LIB))
    lib.gqbench_gemm_q8_plan.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_size_t, ctypes.c_int64,
                                                                                 ctypes.POINTER(ctypes.c_int)]
    lib.gqbench_gemm_q8_plan.restype = None
    lib.gqbench_fp16_pair_chain.argtypes = [ctypes.c_int64] * 4
    lib.gqbench_fp16_pair_chain.restype = ctypes.c_double
    return lib


def plan(qt, N, K, M, ncu=256):
    """plan_gemm_q8: (32-token tiles per workgroup, K splits, stages per split, stages per segment)"""
    room, out = part_room(N, K, M), (ctypes.c_int * 4)()
    assert room >= 0
    bench_lib().gqbench_gemm_q8_plan(qt, N, K, M, room, ncu, out)
    assert (out[1] - 1) * 4 * M * N <= room  # split 0 stands in dst
    return tuple(out)


def act_layout(q, d, qt):
    """act_prep_q8's bytes of quants q [M, nb, 32] and fp16 scales d [M, nb]"""
    M, nb, _ = q.shape
    ns = cdiv(nb, SBLK)
    y = np.zeros(ns * M * (ROW + 8), np.uint8)
    for m in range(M):
        for b in range(ns * SBLK):
            row = (b >> 2) * M + m
            for part in range(4):
                at = ((part & 1) << 1) | (part >> 1) if qt == Q4 else part
                o = row * ROW + (b & 3) * 32 + at * 8
                y[o:o + 8] = q[m, b, 8 * part:8 * part + 8].view(np.uint8) if b < nb else 0
            o = ns * M * ROW + row * 8 + (b & 3) * 2
            y[o:o + 2] = (d[m, b:b + 1] if b < nb else np.zeros(1, np.float16)).view(np.uint8)
    return y


def buf_load(mem, base, nbytes, voff, soff, size):
    """raw buffer load: dwords whose vector offset is past the resource read 0, the others must
    lie in mem. The scalar offset moves the address and is no part of the check."""
    out = np.zeros(size, np.uint8)
    n = max(0, min(size, (nbytes - voff) & ~3))
    if n:
        at = base + voff + soff
        assert 0 <= at and at + n <= mem.size
        out[:n] = mem[at:at + n]
    return out


def weight_operand(lds, wr, h, j, qt):
    """the lane's 16 int8 and its scale dword pair; wr: dword index of the row in lds"""
    w = lambda i: int(lds[wr + i])  # noqa: E731
    if qt == Q8:
        w0 = (34 * j + 2) // 4 + 4 * h
        if j & 1:
            q = [w(w0 + i) for i in range(4)]
        else:
            x = [w(w0 + i) for i in range(5)]
            q = [((x[i] >> 16) | (x[i + 1] << 16)) & 0xffffffff for i in range(4)]
        dd = w(34 * j // 4)
    else:
        w0 = (18 * j + 2) // 4 + 2 * h
        if j & 1:
            u = [w(w0), w(w0 + 1)]
        else:
            x = [w(w0 + i) for i in range(3)]
            u = [((x[i] >> 16) | (x[i + 1] << 16)) & 0xffffffff for i in range(2)]
        q = [((v << 4) & 0xf0f0f0f0) ^ 0x80808080 for v in u] + [(v & 0xf0f0f0f0) ^ 0x80808080 for v in u]
        dd = w(18 * j // 4)
    m = dd & 0xffff0000 if j & 1 else dd & 0xffff
    pr = [m, 0] if j < 2 else [0, m]
    return np.array(q, np.uint32).view(np.int8), np.array(pr, np.uint32).view(np.float16)


def run_workgroup(qt, N, K, M, W, A, mt, s0, s1, seg, n0, m0):
    """sums [BN, 32 mt] of one workgroup (before the epilogue's power of two): segments of seg
    stages, each from zero, one after the other"""
    nb, ns = K // QK, cdiv(K, ROW)
    rb, sd = nb * BB[qt], BB[qt]
    pitch = sd + 1
    rows, toks = min(N - n0, BN), min(M - m0, 32 * mt)
    acc, total = np.zeros((BN, 32 * mt), np.float32), None
    for s in range(s0, s1 + 2):  # the pipeline requests two stages past its last: nothing is read
        lw = np.zeros(BN * pitch, np.uint32)
        la = np.zeros(32 * mt * ROW, np.uint8)
        ld = np.zeros(256 * 8, np.uint8)
        wrote = np.zeros(BN * pitch, bool)
        for tid in range(256):
            npc = sd // 2
            for u in range(cdiv(BN * npc, 256)):
                r, w = divmod(tid + 256 * u, npc)
                if r >= BN:
                    continue  # writes behind the rows
                off = r * rb + 8 * w if r < rows else 0x80000000
                wpos = pitch * r + 2 * w
                assert not wrote[wpos:wpos + 2].any()  # no dword has two writers
                wrote[wpos:wpos + 2] = True
                lw[wpos:wpos + 2] = buf_load(W, n0 * rb + s * sd * 4, rows * rb - s * sd * 4 if s < s1 else 0, off,
                                             0, 8).view(np.uint32)
            apos = (tid >> 3) * ROW + (((tid & 7) ^ ((tid >> 3) & 7)) << 4)
            for i in range(mt):
                la[apos + 4096 * i:apos + 4096 * i + 16] = buf_load(A, (s * M + m0) * ROW, toks * ROW * (s < s1),
                                                                    16 * tid + 4096 * i, 0, 16)
            v = buf_load(A, ns * M * ROW + (s * M + m0) * 8, toks * 8 * (s < s1), 8 * tid, 0, 8)
            ld[8 * tid:8 * tid + 8] = v
        if s >= s1:
            assert not lw.any() and not la.any() and not ld.any()
            continue
        if s > s0 and (s - s0) % seg == 0:
            total, acc = acc if total is None else acc + total, np.zeros_like(acc)
        for wave in range(4):
            q, d = {}, {}
            for lane in range(64):
                c, h = lane & 31, lane >> 5
                for j in range(SBLK):
                    q[lane, j], d[lane, j] = weight_operand(lw, (wave * 32 + c) * pitch, h, j, qt)
                    if s * SBLK + j >= nb:
                        d[lane, j] = np.zeros(4, np.float16)
            for j in range(SBLK):
                for i in range(mt):
                    S, P = np.zeros((32, 32), np.int64), np.zeros((32, 32), np.float64)
                    for h in range(2):
                        a = np.stack([q[32 * h + r, j] for r in range(32)]).astype(np.int64)
                        da = np.stack([d[32 * h + r, j] for r in range(32)]).astype(np.float64)
                        ps = [c * ROW + 4096 * i + (((2 * j + h) ^ (c & 7)) << 4) for c in range(32)]
                        x = np.stack([la[p:p + 16].view(np.int8) for p in ps]).astype(np.int64)
                        dx = np.stack([ld[8 * c + 256 * i:8 * c + 256 * i + 8].view(np.float16)
                                       for c in range(32)]).astype(np.float64)
                        S += a @ x.T
                        P += da @ dx.T
                    assert abs(S).max() < 2**24  # exact as fp32
                    sl = (slice(32 * wave, 32 * wave + 32), slice(32 * i, 32 * i + 32))
                    acc[sl] = (S * P + acc[sl]).astype(np.float32)
    return acc if total is None else acc + total


SHAPES = [(130, 64, 17), (100, 192, 33), (129, 960, 70), (33, 576, 100), (256, 128, 130), (5, 1152, 21),
          (40, 2048, 20)]


@pytest.mark.parametrize("qt", [Q8, Q4])
@pytest.mark.parametrize("N,K,M", SHAPES)
def test_data_path(qt, N, K, M):
    rng = np.random.default_rng(N + K + M + qt)
    nb = K // QK
    dw = rng.uniform(-0.01, 0.01, (N, nb)).astype(np.float16)
    dx = rng.uniform(0.001, 0.1, (M, nb)).astype(np.float16)
    qx = rng.integers(-127, 128, (M, nb, QK)).astype(np.int8)
    if qt == Q8:
        qw = rng.integers(-128, 128, (N, nb, QK)).astype(np.int8)
        body = qw.view(np.uint8)
    else:
        qw = rng.integers(-8, 8, (N, nb, QK)).astype(np.int8)
        u = (qw + 8).astype(np.uint8)
        body = u[..., :16] | (u[..., 16:] << 4)
    W = np.concatenate([dw[..., None].view(np.uint8), body], -1).reshape(-1)
    A = act_layout(qx, dx, qt)
    assert A.size == cdiv(K, ROW) * M * (ROW + 8)  # gemm_q8_act_bytes
    want = np.einsum("nbj,mbj,nb,mb->mn", qw.astype(np.float64), qx.astype(np.float64), dw.astype(np.float64),
                     dx.astype(np.float64))
    mt, ks, sps, seg = plan(qt, N, K, M)
    ns = cdiv(K, ROW)
    n_tiles, m_tiles = cdiv(N, BN), cdiv(M, 32 * mt)
    out = np.full((ks, M, N), np.nan, np.float32)
    seen = set()
    for blk in range(cdiv(n_tiles * ks, 8) * 8 * m_tiles):
        xcd, slot = blk & 7, blk >> 3
        col = slot // m_tiles * 8 + xcd
        if col >= n_tiles * ks:
            continue
        z = col // n_tiles
        n0, m0 = (col - z * n_tiles) * BN, (slot % m_tiles) * 32 * mt
        assert (z, n0, m0) not in seen
        seen.add((z, n0, m0))
        s0, s1 = z * sps, min(ns, z * sps + sps)
        assert s0 < s1
        acc = run_workgroup(qt, N, K, M, W, A, mt, s0, s1, seg, n0, m0)
        for wave in range(4):
            for lane in range(64):
                c, h = lane & 31, lane >> 5
                for g in range(4):
                    n = n0 + wave * 32 + 8 * g + 4 * h
                    for i in range(mt):
                        m = m0 + 32 * i + c
                        for e in range(4):
                            if m < M and n + e < N:
                                assert np.isnan(out[z, m, n + e])  # every output has one writer
                                out[z, m, n + e] = acc[wave * 32 + 8 * g + 4 * h + e, 32 * i + c] * (
                                    0.5 if qt == Q8 else 1 / 32)
    assert len(seen) == n_tiles * ks * m_tiles
    got = out[0]
    for z in range(1, ks):
        got = got + out[z]
    assert np.abs(got - want).max() <= 4e-7 * nb**0.5 * np.abs(want).max()


@pytest.mark.parametrize("N,K,M", [(4096, 4096, 512), (22016, 4096, 100), (4096, 11008, 17), (49152, 960, 333),
                                   (1536, 8960, 300), (2048, 1536, 40), (151936, 1536, 512), (32, 64, 1000)])
def test_plan_covers_k_once(N, K, M):
    for qt in (Q8, Q4):
        mt, ks, sps, seg = plan(qt, N, K, M)
        ns = cdiv(K, ROW)
        assert 1 <= mt <= 4 and ks >= 1 and (ks - 1) * sps < ns <= ks * sps and 1 <= seg <= sps
        # two workgroups' double-buffered stages fit a CU's LDS
        assert 2 * 2 * (BN * (BB[qt] + 1) * 4 + 16 + mt * 32 * ROW + 256 * 8) <= 160 * 1024


def chain(K, ks, sps, seg):
    """blocks per fp32 chain + chains a sum goes through, which its squared error grows with"""
    return min(4 * seg, K // QK) + cdiv(sps, seg) + ks - 1


def chain_bound(qt, old):
    """of the fp16 pairs' figure; their block sums round in Q8_0, which counts as 6 blocks, up to 20"""
    return max(old, min(old + 6, 20)) if qt == Q8 else old


@pytest.mark.parametrize("K", [64, 256, 320, 576, 832, 960, 1536, 2560, 4096, 8960, 11008, 16384])
def test_plan_rounds_no_more_than_the_fp16_pairs(K):
    """the sums are no longer than in the order of gemm.hip's plan (a last partial round of tiles
    counts by its share of the rows)"""
    lib = bench_lib()
    for N in (96, 960, 1536, 1600, 2048, 4096, 5120, 12288, 17920, 22016, 32000):
        for M in (5, 17, 40, 64, 65, 100, 160, 256, 300, 400, 512, 1000):
            old = 0.0
            for n, _, ks, spk in launches(N, K, M):
                old += n / N * (min(2 * spk, K // QK) + ks)
            assert abs(lib.gqbench_fp16_pair_chain(N, K, M, 256) - old) < 1e-9, (N, M)
            for qt in (Q8, Q4):
                _, ks, sps, seg = plan(qt, N, K, M)
                assert chain(K, ks, sps, seg) <= chain_bound(qt, old), (qt, N, M)
