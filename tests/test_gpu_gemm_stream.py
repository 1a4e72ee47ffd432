"""The register-streamed GEMM's tile shapes by size (64, 128 and 256 columns;
32- and 64-row head tiles), ragged row counts, against the oracle and the
LDS-staged tile kernel."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from conftest import bits_equal, describe_diff
from test_gpu_ops import dev, host, rand_gemm

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from q3ops import LM_LOGITS, ops  # noqa: E402
from q3ops.layout import InitConfig, Layout, ModelShape, init_random_blob  # noqa: E402
from q3ops.model import Model  # noqa: E402


@pytest.mark.parametrize("M,N", [(512, 1024), (545, 1024), (1057, 1024), (993, 1152), (65, 256)])
@pytest.mark.parametrize("K,group", [(1024, 256), (1024, 128), (2048, 128), (3072, 256), (3072, 128)])
def test_plain_columns_by_size(cuda, M, N, K, group):
    rng = np.random.default_rng(M + K + group)
    a, as_, b, bs = rand_gemm(rng, M, K, N, group)
    ref = oracle.gemm_nt_group(a, as_, b, bs, group)
    args = dev(a), dev(as_), dev(b)
    out = torch.zeros((M + 1, N + 4), dtype=torch.float32, device=cuda)
    ops.gemm_nt_group_store(*args, dev(bs), out[:M, :N], group)
    assert bits_equal(host(out[:M, :N]), ref), describe_diff(host(out[:M, :N]), ref)
    assert not out[M].any() and not out[:, N:].any()
    x = rng.normal(size=(M, N)).astype(np.float32)
    xt = dev(x)
    ops.gemm_nt_group_store(*args, dev(bs), None, group, add=xt)
    assert bits_equal(host(xt), (ref + x).astype(np.float32))
    bsg = rng.uniform(1e-3, 1e-1, (N, K // group)).astype(np.float32)
    ref = oracle.gemm_nt_group_bg(a, as_, b, bsg, group)
    ops.gemm_nt_group_store(*args, dev(bsg), out[:M, :N], group)
    assert bits_equal(host(out[:M, :N]), ref), describe_diff(host(out[:M, :N]), ref)


@pytest.mark.parametrize("rows", [961, 1090])
def test_chunk_tiles_by_size(cuda, monkeypatch, rows):
    """A chunk on the packed weights (64-row Q|K|V tiles, 128- or 256-column
    O and down tiles) equals the one on the LDS-staged tile kernel."""
    lay = Layout(ModelShape(layers=2, vocab=1024, seq=1090, max_seq=1120))
    blob = init_random_blob(lay, InitConfig(n_prompt=1090, n_gen=2, mode=0))
    got = []
    for packed in ("0", "1"):
        monkeypatch.setenv("Q3_PACKED_WEIGHTS", packed)
        if packed == "0":
            monkeypatch.setenv("Q3_PREFILL_GEMM", "tile")
        else:
            monkeypatch.delenv("Q3_PREFILL_GEMM")
        m = Model(lay, blob)
        m.forward_chunk(0, rows, LM_LOGITS, optimize_tail=False)
        r = {"logits": m.stage("logits", 1)[0]}
        for st in ("h8", "q8", "qs", "o8", "s8", "ss", "x"):
            r[st] = m.stage(st, rows)[1:]
        for li in range(2):
            c = m.kv_cache(li, rows)
            r.update({(li, st): c[st] for st in ("kc", "ks", "vc", "vs")})
        m.close()
        got.append(r)
    for k in got[0]:
        assert bits_equal(got[1][k], got[0][k]), (k, describe_diff(got[1][k], got[0][k]))
