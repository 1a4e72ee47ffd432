"""The GEMMs' row epilogues (16 lanes a row): destinations, gains and RoPE rows
of any alignment and stride, and SwiGLU arguments on both sides of its fast
reciprocal's range, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import bits_equal, describe_diff
from test_gpu_ops import dev, host, nrq_ref, rand_gemm

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from q3ops import ops  # noqa: E402

F = np.float32


@pytest.mark.parametrize("M", [66, 130, 512])
@pytest.mark.parametrize("off", [0, 1, 2])
@pytest.mark.parametrize("tile", [False, True])
def test_head_rows_any_alignment(cuda, monkeypatch, M, off, tile):
    if tile:
        monkeypatch.setenv("Q3_PREFILL_GEMM", "tile")
    rng = np.random.default_rng(M + off)
    K, N, H = 1024, 256, 2
    a, as_, b, bs = rand_gemm(rng, M, K, N, 256)
    nw = (1 + 0.1 * rng.normal(size=128)).astype(F)
    ang = rng.uniform(0, 6, (M, 64))
    cos, sin = np.cos(ang).astype(F), np.sin(ang).astype(F)
    q8 = torch.zeros((M, N + 5), dtype=torch.int8, device=cuda)[:, off:off + N]
    qs = torch.zeros((M, H + 1), dtype=torch.float32, device=cuda)[:, :H]
    tnw = torch.zeros((128, 3), dtype=torch.float32, device=cuda)[:, :1]
    tnw.copy_(dev(nw[:, None]))
    tc, ts = (torch.zeros((M, 64 + off), dtype=torch.float32, device=cuda)[:, off:] for _ in range(2))
    tc.copy_(dev(cos))
    ts.copy_(dev(sin))
    inv = F(1 / 128)
    ref = oracle.gemm_nt_group(a, as_, b, bs, 256)
    ops.gemm_nt_group_store(dev(a), dev(as_), dev(b), dev(bs), None, 256, q8=q8, qs=qs, nw=tnw, cos=tc, sin=ts,
                            inv_hd=float(inv))
    rq, rs = nrq_ref(ref, nw, cos, sin, H)
    assert bits_equal(host(q8), rq), describe_diff(host(q8), rq)
    assert bits_equal(host(qs), rs), describe_diff(host(qs), rs)
    ops.gemm_nt_group_store(dev(a), dev(as_), dev(b), dev(bs), None, 256, q8=q8, qs=qs)
    rq, rs = oracle.quant_rows_heads(ref, 128)
    assert bits_equal(host(q8), rq) and bits_equal(host(qs), rs)


@pytest.mark.parametrize("M", [66, 300])
@pytest.mark.parametrize("off", [0, 3])
@pytest.mark.parametrize("scale", [1e-4, 3e-3, 0.3])
def test_gate_up_rows_and_range(cuda, M, off, scale):
    """scale 0.3 gives gates of a few hundred: exp(-g) + 1 reaches 2^126 and
    +inf, and 0 + 1."""
    rng = np.random.default_rng(M)
    a, as_, wg, wgs = rand_gemm(rng, M, 1024, 512, 256)
    _, _, wu, wus = rand_gemm(rng, M, 1024, 512, 256)
    as_ = (as_ * F(scale)).astype(F)
    s8 = torch.zeros((M, 512 + 7), dtype=torch.int8, device=cuda)[:, off:off + 512]
    ss = torch.zeros((M, 2), dtype=torch.float32, device=cuda)
    ops.gemm_gate_up_swiglu_quant(dev(a), dev(as_), dev(wg), dev(wgs), dev(wu), dev(wus), s8, ss, 256)
    g = oracle.gemm_nt_group(a, as_, wg, wgs, 256)
    if scale == 0.3:
        assert g.min() < -90 and g.max() > 90
    r8, rs = oracle.quant_rows_heads(oracle.swiglu(g, oracle.gemm_nt_group(a, as_, wu, wus, 256)), 256)
    assert bits_equal(host(s8), r8), describe_diff(host(s8), r8)
    assert bits_equal(host(ss), rs), describe_diff(host(ss), rs)


@pytest.mark.parametrize("M", [2, 9, 16, 17, 32, 33, 64, 65, 256])
@pytest.mark.parametrize("N,group", [(128, 256), (1152, 256), (2176, 128)])
@pytest.mark.parametrize("padded", [False, True])
def test_argmax_rows_and_ties(cuda, M, N, group, padded):
    """One key per row and 128-column tile of the tile kernel (row tiles of 32
    and 64; padded weight rows, which the GEMV does not take, or more than 64
    rows), tile counts that are not a multiple of 8, and equal maxima in one
    tile and across tiles: the first column wins.  Up to 64 rows of dense
    weights the GEMV's keys."""
    rng = np.random.default_rng(M + N)
    a, as_, b, bs = rand_gemm(rng, M, 1024, N, group)
    for src in range(0, N, 37):  # copies of rows, later in the tile and in other tiles
        for dst in (src + 1, src + 65, src + 500):
            if dst < N:
                b[dst], bs[dst] = b[src], bs[src]
    best = torch.full((M, 1), -3.0e38, dtype=torch.float32, device=cuda)
    bidx = torch.zeros((M, 1), dtype=torch.int32, device=cuda)
    tb = torch.zeros((N, 1024 + 16 * padded), dtype=torch.int8, device=cuda)[:, :1024]
    tb.copy_(dev(b))
    ops.gemm_nt_group_argmax(dev(a), dev(as_), tb, dev(bs), best, bidx, group)
    ref = oracle.gemm_nt_group(a, as_, b, bs, group)
    assert host(bidx)[:, 0].tolist() == [int(i) for i in np.argmax(ref, axis=1)]
    assert bits_equal(host(best)[:, 0], ref.max(axis=1))


@pytest.mark.parametrize("N,group,M", [(65536, 128, 8), (65536, 128, 9), (98176, 128, 9), (98304, 128, 9),
                                       (98304, 128, 16), (98304, 128, 17), (98304, 256, 9)])
def test_argmax_wide_routes(cuda, N, group, M):
    """Both sides of the rules that share a wide argmax out between the GEMV
    and the tile kernel (rows, columns, group), with equal maxima."""
    rng = np.random.default_rng(M + N)
    a, as_, b, bs = rand_gemm(rng, M, 1024, N, group)
    for src in range(0, N, 997):
        for dst in (src + 1, src + 65, src + 50000):
            if dst < N:
                b[dst], bs[dst] = b[src], bs[src]
    best = torch.full((M, 1), -3.0e38, dtype=torch.float32, device=cuda)
    bidx = torch.zeros((M, 1), dtype=torch.int32, device=cuda)
    ops.gemm_nt_group_argmax(dev(a), dev(as_), dev(b), dev(bs), best, bidx, group)
    ref = oracle.gemm_nt_group(a, as_, b, bs, group)
    assert host(bidx)[:, 0].tolist() == [int(i) for i in np.argmax(ref, axis=1)]
    assert bits_equal(host(best)[:, 0], ref.max(axis=1))


def test_argmax_key_limit(cuda):
    """16 rows over more columns than the GEMV has keys for (one per 64
    columns), but the tile kernel (one per 128): as two calls over halves."""
    M, N, K, group = 16, (1 << 21) + 256, 1024, 128
    gen = torch.Generator(device=cuda)
    gen.manual_seed(21)
    b = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=cuda, generator=gen)
    bs = torch.rand((N, 1), device=cuda, generator=gen)
    a = torch.randint(-127, 128, (M, K), dtype=torch.int8, device=cuda, generator=gen)
    as_ = torch.rand((M, K // group), device=cuda, generator=gen)

    def argmax(lo, hi):
        best = torch.full((M, 1), -3.0e38, dtype=torch.float32, device=cuda)
        bidx = torch.zeros((M, 1), dtype=torch.int32, device=cuda)
        ops.gemm_nt_group_argmax(a, as_, b[lo:hi], bs[lo:hi], best, bidx, group)
        return host(best)[:, 0], host(bidx)[:, 0] + lo

    best, bidx = argmax(0, N)
    half = N // 2
    (b0, i0), (b1, i1) = argmax(0, half), argmax(half, N)
    assert bits_equal(best, np.maximum(b0, b1))
    assert np.array_equal(bidx, np.where(b1 > b0, i1, i0))
