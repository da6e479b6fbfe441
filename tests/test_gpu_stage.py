"""The rows of a forward call through the pinned ring: any row count and hidden size that ends
inside a copy piece (64 KiB), a slot (512 KiB) or past the whole ring (4 MiB), in place and to
another array, the same values as the rows one by one."""
import numpy as np
import pytest

from conftest import ptr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def jy():
    import jieyu_amd
    if jieyu_amd.device_count() < 1:
        pytest.fail("no HIP device visible")
    return jieyu_amd


# bytes: one slot less a row, exactly, and a row more; under and over 1 MiB (helpers); the ring
# and a row more; twice the ring and an odd rest; rows wider than a piece
@pytest.mark.parametrize("hidden,rows", [(256, 511), (256, 512), (256, 513), (256, 1023), (256, 1025), (1120, 937),
                                         (1024, 1024), (1024, 1025), (1024, 2307), (20480, 53)])
def test_rows_round_trip(jy, oracle_lib, hidden, rows):
    from jieyu_amd.model import Synth, synth_config
    print(f"[gpu-case] stage {hidden} x {rows}", flush=True)
    s = Synth(oracle_lib, synth_config("tiny-f32", num_layers=1, hidden=hidden, num_heads=1, num_kv_heads=1, head_dim=16,
                                       intermediate=16, vocab_size=16))
    g = jy.GpuModel(s.desc, rows)
    kv = g.kv()
    X = np.random.default_rng(hidden + rows).standard_normal((rows, hidden)).astype(np.float32)
    keep = X.copy()
    for _ in range(2):  # the second call finds the ring used
        out = g.forward_cached(kv, X, 0)
        assert np.array_equal(X, keep)
    inplace = X.copy()
    assert jy.lib().jyhip_forward_cached(g.h, kv.h, ptr(inplace), rows, 0, None) == 0
    assert np.array_equal(inplace.view(np.uint32), out.view(np.uint32))
    for r in (0, 1, rows // 2, rows - 2):
        assert np.array_equal(g.forward_cached(kv, X[r:r + 1], r).view(np.uint32), out[r:r + 1].view(np.uint32))
    # (the reference's SiLU takes the last elements of an array one by one, with another exp)
    assert np.max(np.abs(g.forward_cached(kv, X[-1:], rows - 1) - out[-1:])) < 5e-3
    kv.close()
    g.close()
    s.close()


# under and over a slot, and over the helpers' 1 MiB: the entry point that allocates nothing copies
# on the calling thread alone
@pytest.mark.parametrize("rows", [3, 513, 1025])
def test_noalloc_rows(jy, oracle_lib, rows):
    from jieyu_amd.model import Synth, synth_config
    hidden = 256
    print(f"[gpu-case] noalloc stage {hidden} x {rows}", flush=True)
    s = Synth(oracle_lib, synth_config("tiny-f32", num_layers=1, hidden=hidden, num_heads=1, num_kv_heads=1, head_dim=16,
                                       intermediate=16, vocab_size=16))
    g = jy.GpuModel(s.desc, rows)
    kv = g.kv()
    X = np.random.default_rng(rows).standard_normal((rows, hidden)).astype(np.float32)
    first = g.forward_cached_noalloc(kv, X, 0)
    want = g.forward_cached(kv, X, 0)
    again = g.forward_cached_noalloc(kv, X, 0)
    for got in (first, again):
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    kv.close()
    g.close()
    s.close()
