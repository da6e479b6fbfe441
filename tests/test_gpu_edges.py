"""Exact-mode kernels at the edges of their ranges (remainders of the vector widths, tiles and
register batches), bit for bit against the CPU oracle."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

import oracle
from conftest import ptr, rope_tables

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden"))

import quant_models as QM  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def jy():
    import jieyu_amd
    if jieyu_amd.device_count() < 1:
        pytest.fail("no HIP device visible")
    return jieyu_amd


def bits_equal(a, b):
    return a.shape == b.shape and np.array_equal(np.ascontiguousarray(a).view(np.uint8),
                                                 np.ascontiguousarray(b).view(np.uint8))


def check_forward(jy, olib, spec, seqs, seed=5):
    """one small model: every layer's states of consecutive chunks equal the oracle's bits"""
    QM.SPECS["edge"] = spec
    try:
        m = QM.build_model("edge", seed)
    finally:
        del QM.SPECS["edge"]
    d, keep = QM.desc_of(m)
    L, H, max_seq = d.num_layers, d.hidden, sum(seqs)
    cos, sin = rope_tables(olib, max_seq, d.head_dim, d.rope_theta)
    okv = oracle.JyoKV()
    assert olib.jyo_kv_init(C.byref(okv), L, max_seq, d.num_kv_heads, d.head_dim) == 0
    g = jy.GpuModel(d, max_seq)
    kv = g.kv(max_seq)
    rng = np.random.default_rng(seed)
    start = 0
    try:
        for seq in seqs:
            X = rng.standard_normal((seq, H)).astype(np.float32)
            want, lo = X.copy(), np.zeros((L, seq, H), np.float32)
            assert olib.jyo_forward_cached(C.byref(d), ptr(want), ptr(cos), ptr(sin), seq, start, C.byref(okv),
                                           ptr(lo)) == 0
            got, log = g.forward_cached(kv, X, start, layer_out=True)
            assert bits_equal(log, lo), f"layers, rows {seq} at {start}"
            assert bits_equal(got, want), f"final norm, rows {seq} at {start}"
            start += seq
    finally:
        olib.jyo_kv_free(C.byref(okv))
        kv.close()
        g.close()


# the RMSNorm's row widths: under one 16-wide step, 8-wide and scalar tails, under and over one
# batch of 16 steps (256), an odd and an even number of batches, the register forms' limits
# (1024, 4096, 8192) and the scalar form (not a multiple of 4, past 8192)
@pytest.mark.parametrize("hidden", [4, 12, 20, 28, 255, 256, 260, 512, 780, 1024, 1028, 4096, 4108, 8192, 8196])
def test_rmsnorm_widths(jy, oracle_lib, hidden):
    spec = dict(hidden=hidden, heads=1, kv=1, hd=16, inter=8, vocab=16, theta=10000.0, bias=False,
                layers=[{s: QM.JY_F32 for s in QM.SLOTS}], embed=QM.JY_F32, lm=QM.JY_F32, tied=False)
    check_forward(jy, oracle_lib, spec, (3, 1))
