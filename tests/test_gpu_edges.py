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


# k-quant decode: the launches with RMSNorm (q/k/v of different types, gate/up of one type) at
# input widths under, at and over one register buffer of super-blocks (an odd number of buffers
# per row: 256, 1280, 2304; the register norm's limits 4096 and 8192, and past it), row counts
# that leave partial row groups and workgroups, more row groups than one pass of waves covers
# (the lm_head), and groups whose types do not fuse
@pytest.mark.parametrize("hidden,inter,types,vocab,bias", [
    (256, 512, "445", 70, True), (1280, 256, "654", 1031, False), (2304, 768, "446", 66000, True),
    (4096, 1024, "446", 300, False), (4352, 512, "556", 90, True), (8192, 256, "444", 41, False),
    (8448, 256, "646", 41, False)])
def test_kquant_decode_widths(jy, oracle_lib, hidden, inter, types, vocab, bias):
    t = {"4": QM.JY_Q4_K, "5": QM.JY_Q5_K, "6": QM.JY_Q6_K}
    q, k, v = (t[c] for c in types)
    up = q if inter != 768 else k  # gate and up of different types once
    layer = dict(Wq=q, Wk=k, Wv=v, Wo=k, W1=q, W2=v, W3=up)
    spec = dict(hidden=hidden, heads=4, kv=2, hd=64, inter=inter, vocab=vocab, theta=10000.0, bias=bias,
                layers=[layer], embed=v, lm=q, tied=False)
    check_forward(jy, oracle_lib, spec, (2, 1, 1))
    # the head: norm + lm_head in one launch, greedy picks against the oracle's logits
    QM.SPECS["edge"] = spec
    try:
        m = QM.build_model("edge", 3)
    finally:
        del QM.SPECS["edge"]
    d, keep = QM.desc_of(m)
    cos, sin = rope_tables(oracle_lib, 16, 64, d.rope_theta)
    prompt = QM.prompt_of(m, 3)
    want, wl = np.zeros(17, np.int32), np.zeros(vocab, np.float32)
    n = oracle_lib.jyo_generate(C.byref(d), ptr(prompt), 3, None, 0, ptr(cos), ptr(sin), 16, 4, 0.0, 1.0, ptr(want),
                                None, ptr(wl))
    g = jy.GpuModel(d, 16)
    ids, _, logits = g.generate(prompt, 4, want_logits=True)
    g.close()
    assert ids.tolist() == want[:n].tolist()
    assert bits_equal(logits, wl)


# a q/k/v group with one matrix of another kind, and a gate/up pair of two types: one kernel each
@pytest.mark.parametrize("wv,w3", [(QM.JY_Q8_0, QM.JY_Q4_K), (QM.JY_Q6_K, QM.JY_F16)])
def test_kquant_groups_that_do_not_fuse(jy, oracle_lib, wv, w3):
    layer = dict(Wq=QM.JY_Q4_K, Wk=QM.JY_Q4_K, Wv=wv, Wo=QM.JY_Q4_K, W1=QM.JY_Q4_K, W2=QM.JY_Q6_K, W3=w3)
    spec = dict(hidden=512, heads=4, kv=2, hd=64, inter=768, vocab=64, theta=10000.0, bias=True, layers=[layer] * 2,
                embed=QM.JY_Q6_K, lm=QM.JY_Q4_K, tied=False)
    check_forward(jy, oracle_lib, spec, (1, 1, 2, 1))

def check_generate(jy, oracle_lib, spec):
    """greedy picks and the last logits against the oracle's"""
    QM.SPECS["edge"] = spec
    try:
        m = QM.build_model("edge", 3)
    finally:
        del QM.SPECS["edge"]
    d, keep = QM.desc_of(m)
    cos, sin = rope_tables(oracle_lib, 16, spec["hd"], d.rope_theta)
    prompt = QM.prompt_of(m, 3)
    want, wl = np.zeros(17, np.int32), np.zeros(spec["vocab"], np.float32)
    n = oracle_lib.jyo_generate(C.byref(d), ptr(prompt), 3, None, 0, ptr(cos), ptr(sin), 16, 4, 0.0, 1.0, ptr(want),
                                None, ptr(wl))
    g = jy.GpuModel(d, 16)
    ids, _, logits = g.generate(prompt, 4, want_logits=True)
    g.close()
    assert ids.tolist() == want[:n].tolist()
    assert bits_equal(logits, wl)


# the k-quant matvec alone: rows of one buffer (up to 1024 inputs), of a remainder of the two
# buffers' 8 or 16 chunks, either side of the longer buffers' 8192 inputs; row groups cut short, and
# more than a workgroup per CU
@pytest.mark.parametrize("t", [QM.JY_Q4_K, QM.JY_Q5_K, QM.JY_Q6_K])
@pytest.mark.parametrize("n,k", [(1, 256), (66, 768), (4103, 1024), (13, 1280), (130, 2048), (5, 2304), (67, 3328),
                                 (17000, 512), (4100, 4352), (9, 8192), (18, 8448), (4098, 8448), (1030, 14336)])
def test_kquant_matvec_widths(jy, oracle_lib, t, n, k):
    check_exact_gemm(jy, oracle_lib, t, n, k, 1)


# dense decode: the launches with RMSNorm (q/k/v, gate/up, the head) and with SiLU (down) at input
# widths under, at and over one block of the panel (256 f32, 512 f16 rows), not a multiple of a
# 16-byte piece, at and past the widest row the launch holds (6144), outputs that cut a panel,
# f32, f16, and groups of two dense types, which take one kernel per matrix
@pytest.mark.parametrize("hidden,inter,t,vocab,bias", [
    (20, 8, "ff", 70, False), (255, 131, "ff", 65, True), (256, 260, "hh", 130, True), (516, 1031, "ff", 66, False),
    (513, 512, "hh", 64, False), (1120, 3040, "hh", 1031, True), (6144, 72, "ff", 40, False), (6148, 72, "ff", 40, True),
    (6144, 40, "hh", 41, False), (6160, 40, "hh", 41, False), (260, 136, "hf", 70, True), (260, 136, "fh", 70, False)])
def test_dense_decode_widths(jy, oracle_lib, hidden, inter, t, vocab, bias):
    a, b = [QM.JY_F32 if c == "f" else QM.JY_F16 for c in t]
    layer = dict(Wq=a, Wk=a, Wv=b, Wo=a, W1=a, W2=b, W3=b)
    spec = dict(hidden=hidden, heads=2, kv=1, hd=16, inter=inter, vocab=vocab, theta=10000.0, bias=bias,
                layers=[layer] * 2, embed=a, lm=b, tied=False)
    check_forward(jy, oracle_lib, spec, (2, 1, 1))
    check_generate(jy, oracle_lib, spec)


# the prompt GEMMs' tokens per wave (1, 2, 4, 8, 16: by rows and columns), rows that leave a partial
# wave and workgroup, 64-column tiles cut short, chunks of 256 cut to 32, 64, 96 and 224 (Q8_0),
# dense widths under one piece, under one register buffer and with a tail
@pytest.mark.parametrize("t,n,k", [
    (QM.JY_Q8_0, 130, 32), (QM.JY_Q8_0, 65, 96), (QM.JY_Q8_0, 1, 320), (QM.JY_Q8_0, 4099, 480),
    (QM.JY_Q4_K, 67, 256), (QM.JY_Q5_K, 4100, 512), (QM.JY_Q6_K, 129, 768),
    (QM.JY_F32, 63, 3), (QM.JY_F32, 65, 66), (QM.JY_F32, 130, 513), (QM.JY_F32, 4099, 300),
    (QM.JY_F16, 64, 7), (QM.JY_F16, 70, 130), (QM.JY_F16, 4098, 515)])
@pytest.mark.parametrize("m", [2, 5, 17, 33, 70])
def test_exact_gemm_tiles(jy, oracle_lib, t, n, k, m):
    check_exact_gemm(jy, oracle_lib, t, n, k, m)


# the widest form (16 tokens per wave): a partial last tile and wave, dense K under 16 and with a tail
@pytest.mark.parametrize("t,n,k,m", [
    (QM.JY_Q8_0, 24003, 96, 61), (QM.JY_Q6_K, 24003, 256, 50), (QM.JY_F32, 3100, 83, 200), (QM.JY_F32, 3100, 9, 200),
    (QM.JY_F16, 24003, 83, 61), (QM.JY_F16, 3100, 150, 211)])
def test_exact_gemm_wide_tiles(jy, oracle_lib, t, n, k, m):
    check_exact_gemm(jy, oracle_lib, t, n, k, m)


def check_exact_gemm(jy, oracle_lib, t, n, k, m):
    rng = np.random.default_rng(m + n + k + t)
    w = QM.rand_matrix(rng, t, n, k)
    wm = QM.WMat(w.ctypes.data_as(C.c_void_p), t)
    a = rng.standard_normal((m, k)).astype(np.float32)
    want = np.zeros((m, n), np.float32)
    oracle_lib.jyo_matmul_w(C.byref(wm), m, n, k, ptr(a), ptr(want))
    W = jy.WeightMatrix(w, t, n, k)
    got = W.matmul(a)
    W.close()
    assert bits_equal(got, want)
