"""The split attention (k_attn_split.hip: a sequence's key blocks over
many workgroups) at the edges of its blocks (32 keys), workgroups (4 blocks)
and chain stages (16 blocks, 128 per pass), against the oracle in batches and
against the single-launch attention for one row; and the one-row whole-row
GEMM that its O projection takes."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import bits_equal, describe_diff
from test_gpu_batch import LD_TABLE, make_case, run_batch_case
from test_gpu_ops import dev, host, rand_gemm

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from q3ops import LM_LOGITS, ops  # noqa: E402
from q3ops.layout import InitConfig, Layout, ModelShape, init_random_blob  # noqa: E402
from q3ops.model import Model  # noqa: E402


@pytest.mark.parametrize("edge,ld_table", [
    ([0, 30, 31, 32, 33, 126, 127, 128, 129, 253], LD_TABLE),
    ([0, 510, 512, 2047, 4095, 4096, 4140], 132),
])
def test_split_batch_matches_oracle(cuda, monkeypatch, edge, ld_table):
    monkeypatch.setenv("Q3_ATTN_SPLIT", "1")
    n = len(edge)
    run_batch_case(cuda, n, *make_case(n, seed=700 + n, edge=edge, ld_table=ld_table))


def test_split_batch_shared_write_page(cuda, monkeypatch):
    """Rows that write into a page another row reads take the single launch,
    whose K/V rows are all written first: same ids with the split asked for."""
    lay, blob, ctx, tables, _, ids0 = make_case(5, seed=105)
    tables, ctx = tables.copy(), ctx.copy()
    tables[1], ctx[1] = tables[4], ctx[4] + 1  # row 1 reads row 4's new token
    tables[1, (ctx[1] // 32):] = tables[4, (ctx[1] // 32):]
    got = []
    for split in ("0", "1"):
        monkeypatch.setenv("Q3_ATTN_SPLIT", split)
        m = Model(lay, blob)
        out = torch.zeros(5, dtype=torch.int32, device=cuda)
        m.decode_batch(torch.from_numpy(ids0.copy()).to(cuda), ctx, tables, out)
        got.append((host(out), m.stage("x", 5)))
        m.close()
    assert np.array_equal(got[0][0], got[1][0]) and bits_equal(got[0][1], got[1][1])


def test_split_one_row_matches_fused(cuda, monkeypatch):
    """One decoding row at every edge: logits, residual row and the page rows
    equal the fused launch's, over a shuffled page table."""
    shape = ModelShape(layers=2, vocab=1024, seq=32, max_seq=4352)
    lay = Layout(shape)
    blob = init_random_blob(lay, InitConfig(n_prompt=1, n_gen=0, mode=0))
    rng = np.random.default_rng(9)
    o, ms = lay.offsets, lay.max_seq
    for li in range(shape.layers):
        base = o["kKV_BASE"] + li * o["kKV_STRIDE"]
        for off in (0, o["kKV_VOFF"]):
            n = ms * lay.kv_width
            blob[base + off:base + off + n] = rng.integers(-127, 128, n, dtype=np.int8).view(np.uint8)
            so = base + off + o["kKV_SOFF"]
            sc = rng.uniform(0.002, 0.03, ms * lay.kv_heads).astype(np.float32)
            blob[so:so + 4 * sc.size] = sc.view(np.uint8)
    table = rng.permutation(ms // 32).astype(np.uint16)
    ids = rng.integers(0, 1024, ms).astype(np.int32)
    res = {}
    for split in ("0", "1"):
        monkeypatch.setenv("Q3_ATTN_SPLIT", split)
        m = Model(lay, blob)
        m.set_page_table(table)
        m.set_ids(ids)
        for pos in (0, 30, 31, 32, 127, 128, 511, 512, 1567, 1568, 2047, 4095, 4096, 4351):
            m.forward_chunk(pos, 1, LM_LOGITS, True)
            res[split, pos] = [m.stage(nm, 1) for nm in ("logits", "x", "q8", "qs", "o8", "os")]
        res[split, "kv"] = [m.kv_cache(li, ms)[nm] for li in range(2) for nm in ("kc", "ks", "vc", "vs")]
        m.close()
    for (split, what), v in res.items():
        if split == "1":
            for a, b in zip(v, res["0", what]):
                assert bits_equal(a, b), (what, describe_diff(a, b))


def test_split_generate_graph_replays(cuda, monkeypatch):
    """The split decode steps captured in q3_generate's graph and replayed
    equal the fused ones."""
    shape = ModelShape(layers=2, vocab=1024, seq=64, max_seq=256)
    lay = Layout(shape)
    blob = init_random_blob(lay, InitConfig(n_prompt=100, n_gen=40, mode=0))
    got = []
    for split in ("0", "1"):
        monkeypatch.setenv("Q3_ATTN_SPLIT", split)
        s = torch.cuda.Stream()
        m = Model(lay, blob, stream=s)
        m.set_ctrl(100, 40, 0)
        for _ in range(3):
            m.generate()
            got.append(m.ids()[:140])
        m.close()
    assert all(np.array_equal(g, got[0]) for g in got[1:])


@pytest.mark.parametrize("K,group", [(1024, 128), (1024, 256), (2048, 128), (2048, 256), (3072, 256)])
@pytest.mark.parametrize("N", [128, 2048, 2176])
@pytest.mark.parametrize("per_group", [False, True])
def test_one_row_whole_row_gemm(cuda, K, group, N, per_group):
    rng = np.random.default_rng(K + N + group)
    a, as_, b, bs = rand_gemm(rng, 1, K, N, group)
    if per_group:
        bs = rng.uniform(1e-3, 1e-1, (N, K // group)).astype(np.float32)
    ref = (oracle.gemm_nt_group_bg if per_group else oracle.gemm_nt_group)(a, as_, b, bs, group)
    out = torch.zeros((1, N), dtype=torch.float32, device=cuda)
    ops.gemm_nt_group_store(dev(a), dev(as_), dev(b), dev(bs), out, group)
    assert bits_equal(host(out), ref), describe_diff(host(out), ref)
    x = rng.normal(size=(1, N)).astype(np.float32)
    xt = dev(x)
    ops.gemm_nt_group_store(dev(a), dev(as_), dev(b), dev(bs), None, group, add=xt)
    assert bits_equal(host(xt), (ref + x).astype(np.float32))


@pytest.mark.parametrize("M", [2, 4, 5, 8])
@pytest.mark.parametrize("K,group", [(1024, 128), (1024, 256), (2048, 128), (2048, 256), (3072, 256)])
@pytest.mark.parametrize("per_group", [False, True])
def test_few_rows_whole_row_gemm(cuda, M, K, group, per_group):
    """2 to 8 rows over the same weight registers, strided operands."""
    rng = np.random.default_rng(K + M + group)
    N = 384
    a, as_, b, bs = rand_gemm(rng, M, K, N, group)
    if per_group:
        bs = rng.uniform(1e-3, 1e-1, (N, K // group)).astype(np.float32)
    ta = torch.zeros((M, K + 16), dtype=torch.int8, device=cuda)[:, :K]
    ta.copy_(dev(a))
    tas = torch.zeros((M, K // group + 1), device=cuda)[:, :K // group]
    tas.copy_(dev(as_))
    ref = (oracle.gemm_nt_group_bg if per_group else oracle.gemm_nt_group)(a, as_, b, bs, group)
    out = torch.zeros((M + 1, N + 3), dtype=torch.float32, device=cuda)
    ops.gemm_nt_group_store(ta, tas, dev(b), dev(bs), out[:M, :N], group)
    assert bits_equal(host(out[:M, :N]), ref), describe_diff(host(out[:M, :N]), ref)
    assert not out[M].any() and not out[:, N:].any()
    x = rng.normal(size=(M, N)).astype(np.float32)
    xt = dev(x)
    ops.gemm_nt_group_store(ta, tas, dev(b), dev(bs), None, group, add=xt)
    assert bits_equal(host(xt), (ref + x).astype(np.float32))


def test_split_chunk_matches_tile_walk(cuda, monkeypatch):
    """Short chunks at the edges of 16-row tiles, 32-row blocks, key blocks,
    4-block workgroups and chain passes: logits of the last row and every
    stage row equal the prefill kernel's, over a shuffled page table, with the
    last layer on all rows and on the last one."""
    shape = ModelShape(layers=2, vocab=1024, seq=64, max_seq=4352)
    lay = Layout(shape)
    blob = init_random_blob(lay, InitConfig(n_prompt=1, n_gen=0, mode=0))
    rng = np.random.default_rng(11)
    o, ms = lay.offsets, lay.max_seq
    for li in range(shape.layers):
        base = o["kKV_BASE"] + li * o["kKV_STRIDE"]
        for off in (0, o["kKV_VOFF"]):
            n = ms * lay.kv_width
            blob[base + off:base + off + n] = rng.integers(-127, 128, n, dtype=np.int8).view(np.uint8)
            so = base + off + o["kKV_SOFF"]
            sc = rng.uniform(0.002, 0.03, ms * lay.kv_heads).astype(np.float32)
            blob[so:so + 4 * sc.size] = sc.view(np.uint8)
    table = rng.permutation(ms // 32).astype(np.uint16)
    ids = rng.integers(0, 1024, ms).astype(np.int32)
    chunks = [(0, 2), (30, 3), (127, 8), (4095, 2), (0, 9), (0, 64), (31, 16), (111, 17), (112, 16), (500, 33),
              (1003, 37), (4032, 64), (4063, 33), (4351 - 32, 32)]
    res = {}
    for split in ("0", "1"):
        monkeypatch.setenv("Q3_ATTN_SPLIT", split)
        m = Model(lay, blob)
        m.set_page_table(table)
        m.set_ids(ids)
        for pos, rows in chunks:
            for tail in (False, True):
                m.forward_chunk(pos, rows, LM_LOGITS, tail)
                res[split, pos, rows, tail] = ([m.stage("logits", 1)] +
                                               [m.stage(nm, rows) for nm in ("x", "q8", "qs", "o8", "os")])
        res[split, "kv"] = [m.kv_cache(li, ms)[nm] for li in range(2) for nm in ("kc", "ks", "vc", "vs")]
        m.close()
    for (split, *what), v in res.items():
        if split == "1":
            for a, b in zip(v, res[("0", *what)]):
                assert bits_equal(a, b), (what, describe_diff(a, b))


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, -0.02, 1e-44])
def test_split_special_scales(cuda, monkeypatch, which, value):
    """Rows over infinite, NaN, negative or subnormal scales in the pool come
    out as from the kernels that take the same rows without the split; with
    infinite or NaN scores a chunk's row has scale 0, a decoding row's NaN."""
    lay = Layout(ModelShape(layers=1, vocab=1024, seq=64, max_seq=1024))
    blob = init_random_blob(lay, InitConfig(n_prompt=1, n_gen=0, mode=0))
    rng = np.random.default_rng(17)
    o, ms = lay.offsets, lay.max_seq
    for off in (0, o["kKV_VOFF"]):
        at = o["kKV_BASE"] + off
        n = ms * lay.kv_width
        blob[at:at + n] = rng.integers(-127, 128, n, dtype=np.int8).view(np.uint8)
        sc = rng.uniform(0.002, 0.03, ms * lay.kv_heads).astype(np.float32)
        if (off == 0) == (which == "k"):
            sc.reshape(-1, lay.kv_heads)[40::300, ::2] = value
        blob[at + o["kKV_SOFF"]:at + o["kKV_SOFF"] + 4 * sc.size] = sc.view(np.uint8)
    ids = rng.integers(0, 1024, ms).astype(np.int32)
    tables = np.tile(np.arange(ms // 32, dtype=np.uint16), (3, 1))
    pos = np.array([20, 500, 1000], np.int32)
    got = {}
    for split in ("0", "1"):
        monkeypatch.setenv("Q3_ATTN_SPLIT", split)
        m = Model(lay, blob)
        m.set_ids(ids)
        pool = m.blob.clone()
        for at, rows in ((20, 2), (100, 16), (500, 37), (960, 64), (1000, 1)):
            m.blob.copy_(pool)
            m.forward_chunk(at, rows, LM_LOGITS, False)
            got[split, at, rows] = m.stage("o8", rows), m.stage("os", rows)
        m.blob.copy_(pool)
        out = torch.zeros(3, dtype=torch.int32, device=cuda)
        m.decode_batch(torch.from_numpy(ids[:3].copy()).to(cuda), pos, tables, out)
        got[split, "batch"] = m.stage("o8", 3), m.stage("os", 3)
        m.close()
    for (split, *what), (o8, os_) in got.items():
        if split == "1":
            w8, ws = got[("0", *what)]
            assert np.array_equal(o8, w8) and np.array_equal(os_, ws, equal_nan=True), what
    if which == "k" and not np.isfinite(value):
        assert np.isnan(got["1", 1000, 1][1]).any() and not np.isnan(got["1", 960, 64][1]).any()


@pytest.mark.parametrize("split", ["0", "1"])
def test_split_kernel_timing(cuda, monkeypatch, split):
    """Every route of the decode classes is timed, one launch per layer: the
    split attention, projections of several rows with their norm or quant
    kernel, chunks on both sides of the prologue GEMVs' row limit."""
    monkeypatch.setenv("Q3_ATTN_SPLIT", split)
    lay = Layout(ModelShape(layers=3, vocab=1024, seq=32, max_seq=2048))
    m = Model(lay, init_random_blob(lay, InitConfig(n_prompt=1, n_gen=0, mode=0)))
    m.set_ids(np.zeros(2048, np.int32))

    def counts(call):
        m.set_kernel_timing(True)
        call()
        kt = m.kernel_times()
        m.set_kernel_timing(False)
        assert all((ms > 0) == (n > 0) for ms, n in kt.values()), kt
        return {k: n for k, (_, n) in kt.items()}

    n = counts(lambda: m.forward_chunk(1600, 1, LM_LOGITS, True))
    assert n["attn_decode"] == 3, n
    if split == "1":
        assert n["gemv_qkv"] == n["gemv_o"] == n["gemv_gate_up"] == n["gemv_down"] == 3, n
    for rows in (4, 8, 9, 16):
        for tail in (False, True):  # (the last layer's single row is a decode attention)
            n = counts(lambda: m.forward_chunk(1000, rows, LM_LOGITS, tail))
            assert n["attn_decode"] == int(tail), (rows, n)
            assert n["gemv_qkv"] == n["gemv_o"] == n["gemv_gate_up"] == n["gemv_down"] == 3, (rows, n)
    assert not any(counts(lambda: m.forward_chunk(1000, 17, LM_LOGITS, True)).values())
    tables = np.stack([np.arange(64), np.arange(64)[::-1]]).astype(np.uint16)  # (no page of both in use)
    out = torch.zeros(2, dtype=torch.int32, device=cuda)
    n = counts(lambda: m.decode_batch(out, np.array([40, 1500], np.int32), tables, out))
    assert n["attn_decode"] == 3, n
    m.close()


def test_split_chunk_matches_oracle(cuda, monkeypatch):
    """A prompt in short chunks, all of them on the split attention, against
    the oracle: the last layer's attention output and residual rows of every
    chunk, and the logits."""
    monkeypatch.setenv("Q3_ATTN_SPLIT", "1")
    shape = ModelShape(layers=2, vocab=1024, seq=64, max_seq=640)
    lay = Layout(shape)
    blob = init_random_blob(lay, InitConfig(n_prompt=600, n_gen=0, mode=0))
    om = oracle.OracleModel(blob, lay.offsets, dict(shape.__dict__))
    ids = lay.global_views(blob)["ids"][:600].copy()
    m = Model(lay, blob)
    pos = 0
    for rows in (64, 33, 2, 17, 9, 64, 16, 8, 3, 40, 64, 48, 5, 31, 64, 61, 24, 11):
        logits, rec = om.forward_chunk(ids[pos:pos + rows], pos, rows, True, record=True)
        m.forward_chunk(pos, rows, LM_LOGITS, False)
        assert bits_equal(m.stage("logits", 1)[0], logits), (pos, rows)
        for st in ("x", "o8", "os"):
            assert bits_equal(m.stage(st, rows), rec[st]), (pos, rows, st)
        pos += rows
    m.close()
