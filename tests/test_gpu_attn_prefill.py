"""The prefill attention's P8 quantisation through the approximate reciprocal
and its exact path: quotients on and beside half-integers, and pmax outside the
reciprocal's range, against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import bits_equal, describe_diff
from test_gpu_ops import QK, dev, host, make_pages

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from q3ops import ops  # noqa: E402

F = np.float32


# (the largest unit keeps P8.V * pmax <= 32 * 127^2 units below 2^128)
@pytest.mark.parametrize("unit", [2.0**-6, 2.0**-120, 2.0**104, 3.0e-39])
@pytest.mark.parametrize("nudge", [0, 1, -1])
@pytest.mark.parametrize("rows,kv_len", [(7, 40), (33, 300)])
def test_prefill_p8_half_integers(cuda, unit, nudge, rows, kv_len):
    """All scores 0, so P = 1 and P * vs = vs: blocks whose scales are (k + 1/2)
    units (or one float beside) with a maximum of 127 units."""
    rng = np.random.default_rng(rows + nudge)
    heads, kvh = 16, 8
    n_pages = (kv_len + 31) // 32 + 1
    (k8, v8, ks, vs), (kp, vp, ksp, vsp, table) = make_pages(rng, kv_len, kvh * 128, kvh, n_pages)
    u = F(unit)
    vs[:] = ((rng.integers(0, 127, vs.shape) + F(0.5)) * u).astype(F)
    vs[:] = (vs.view(np.int32) + nudge).view(F)
    vs[::32] = F(127) * u
    t = np.arange(kv_len)
    vsp[table[t // 32], t % 32] = vs
    q8 = np.zeros((rows, heads * 128), np.int8)
    qs = rng.uniform(1e-3, 5e-2, (rows, heads)).astype(F)
    tk, tv, tks, tvs, tt = dev(kp), dev(vp), dev(ksp), dev(vsp), dev(table.view(np.int16))
    kv = ops.paged_kv(tk, tv, tks, tvs, tt)
    o8 = torch.zeros((rows, heads * 128), dtype=torch.int8, device=cuda)
    os_ = torch.zeros((rows, heads), dtype=torch.float32, device=cuda)
    ops.attention_heads_gqa_tokscale_paged(dev(q8), dev(qs), kv, kv_len, o8, os_, heads, kvh, 128, True, QK)
    attn = oracle.attention_heads_gqa_tokscale(q8, qs, k8, ks, v8, vs, heads, kvh, 128, True, QK)
    ro8, ros = oracle.quant_rows_heads(attn, 128)
    assert bits_equal(host(o8), ro8), describe_diff(host(o8), ro8)
    assert bits_equal(host(os_), ros), describe_diff(host(os_), ros)


@pytest.mark.parametrize("variant", ["", "pair"])
@pytest.mark.parametrize("nan", [0x7FC00000, 0x7FC00055, 0xFFC00001])
def test_prefill_nan_v_scale(cuda, monkeypatch, variant, nan):
    """A key whose V scale is a NaN quantises to P8 = 0 whatever the NaN's
    payload, in waves that otherwise take the approximate reciprocal."""
    monkeypatch.setenv("Q3_PREFILL_ATTN", variant)
    rng = np.random.default_rng(3)
    rows, kv_len, heads, kvh = 33, 300, 16, 8
    (k8, v8, ks, vs), (kp, vp, ksp, vsp, table) = make_pages(rng, kv_len, kvh * 128, kvh, 11)
    q8 = rng.integers(-127, 128, (rows, heads * 128)).astype(np.int8)
    qs = rng.uniform(1e-3, 5e-2, (rows, heads)).astype(F)
    t = np.arange(5, kv_len, 41)
    got = []
    for special in (False, True):
        # a NaN key's P * V is left out of the sum, as for a zero scale
        vsp[table[t // 32], t % 32] = np.array([nan if special else 0], np.uint32).view(F)[0]
        kv = ops.paged_kv(dev(kp), dev(vp), dev(ksp), dev(vsp), dev(table.view(np.int16)))
        o8 = torch.zeros((rows, heads * 128), dtype=torch.int8, device=cuda)
        os_ = torch.zeros((rows, heads), dtype=torch.float32, device=cuda)
        ops.attention_heads_gqa_tokscale_paged(dev(q8), dev(qs), kv, kv_len, o8, os_, heads, kvh, 128, True, QK)
        got.append((host(o8), host(os_)))
    vs[t] = 0
    attn = oracle.attention_heads_gqa_tokscale(q8, qs, k8, ks, v8, vs, heads, kvh, 128, True, QK)
    ro8, ros = oracle.quant_rows_heads(attn, 128)
    for o8, os_ in got:
        assert bits_equal(o8, ro8), describe_diff(o8, ro8)
        assert bits_equal(os_, ros), describe_diff(os_, ros)


@pytest.mark.parametrize("variant", ["", "pair", "walk"])
@pytest.mark.parametrize("page_tokens", [32, 128])
@pytest.mark.parametrize("rows,kv_len", [(2, 45), (33, 300), (301, 700)])
@pytest.mark.parametrize("row_bytes,scale_cols", [(1040, 8), (1088, 9), (1152, 11)])
def test_prefill_padded_rows(cuda, monkeypatch, variant, page_tokens, rows, kv_len, row_bytes, scale_cols):
    """K/V rows at any multiple of 16 bytes, not of 128 (row_bytes wider than
    the heads), and padded scale rows; the last head of the pool's last page
    is read."""
    monkeypatch.setenv("Q3_PREFILL_ATTN", variant)
    rng = np.random.default_rng(row_bytes + rows + page_tokens)
    heads, kvh, kw = 16, 8, 1024
    n_pages = (kv_len + page_tokens - 1) // page_tokens
    (k8, v8, ks, vs), (kp, vp, ksp, vsp, table) = make_pages(rng, kv_len, row_bytes, scale_cols, n_pages,
                                                             page_tokens=page_tokens)
    assert n_pages - 1 in table
    q8 = rng.integers(-127, 128, (rows, heads * 128)).astype(np.int8)
    qs = rng.uniform(1e-3, 5e-2, (rows, heads)).astype(F)
    kv = ops.paged_kv(dev(kp), dev(vp), dev(ksp), dev(vsp), dev(table.view(np.int16)), page_tokens)
    o8 = torch.zeros((rows, heads * 128), dtype=torch.int8, device=cuda)
    os_ = torch.zeros((rows, heads), dtype=torch.float32, device=cuda)
    ops.attention_heads_gqa_tokscale_paged(dev(q8), dev(qs), kv, kv_len, o8, os_, heads, kvh, 128, True, QK)
    cols = lambda t, n: np.ascontiguousarray(t[:, :n])  # noqa: E731
    attn = oracle.attention_heads_gqa_tokscale(q8, qs, cols(k8, kw), cols(ks, kvh), cols(v8, kw), cols(vs, kvh),
                                               heads, kvh, 128, True, QK)
    ro8, ros = oracle.quant_rows_heads(attn, 128)
    assert bits_equal(host(o8), ro8), describe_diff(host(o8), ro8)
    assert bits_equal(host(os_), ros), describe_diff(host(os_), ros)
