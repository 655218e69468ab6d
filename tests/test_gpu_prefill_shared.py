"""Prefill at the edges of its launch shapes, against the oracle's
token-by-token loop: append and attention in one launch (one, two and four
key tiles a workgroup; several workgroups to a query tile), the planes'
kernel with 1 to 8 workgroups to a query tile, head groups of 1, 2 and
4; and buffers that overlap.

Tolerance: as test_gpu_prefill.py (1e-4 on outputs; cache bit-exact).  The
states of a query tile are merged in a fixed order, so a second call gives
the same bits."""
import ctypes as C

import numpy as np
import pytest

from helpers import PREFILL_TOL, bits, device_arrays, log, max_err
from test_gpu_prefill import gpu_prefill, oracle_prefill

pytestmark = pytest.mark.gpu

SHAPES = [
    # one launch: 1, 2, 3, 4 key tiles, whole and with a remainder
    (1, 32, 4, 0, 2), (22, 32, 4, 0, 32), (1, 32, 4, 0, 33), (2, 32, 4, 31, 33), (1, 32, 4, 0, 65),
    (1, 32, 4, 0, 128), (1, 12, 4, 70, 50),
    # and several workgroups to a query tile (its first query tiles have one)
    (1, 32, 4, 0, 129), (1, 32, 4, 477, 3), (1, 32, 4, 900, 120), (1, 12, 1, 200, 40), (2, 32, 4, 0, 256),
    # head groups of one and two
    (1, 8, 8, 0, 20), (1, 8, 8, 130, 5), (1, 4, 2, 40, 100), (1, 8, 4, 300, 70),
    # planes: 8, 4, 6, 5, 3, 2 and 1 workgroups to a query tile
    (1, 32, 4, 1500, 100), (1, 32, 4, 1000, 256), (1, 32, 4, 700, 300), (1, 32, 4, 700, 330), (1, 8, 8, 0, 500), (2, 32, 4, 0, 300), (2, 32, 4, 100, 200), (22, 32, 4, 300, 40),
    (22, 32, 4, 477, 3), (22, 16, 2, 200, 220),
]


@pytest.mark.parametrize("layers,n_head,n_head_kv,pos0,n_tok", SHAPES)
def test_prefill_launch_shapes(O, W, engines, layers, n_head, n_head_kv, pos0, n_tok):
    n_ctx = pos0 + n_tok + 3
    case = W.make_prefill(n_layers=layers, n_tok=n_tok, pos0=pos0, n_head=n_head, n_head_kv=n_head_kv,
                          salt=pos0 + n_tok)
    g = np.random.default_rng(7)
    kv = [g.standard_normal((1, layers, n_ctx, n_head_kv * 64)).astype(np.float32) for _ in range(2)]
    eng = engines(layers, n_ctx, n_head=n_head, n_head_kv=n_head_kv)
    out, kc, vc = gpu_prefill(eng, case, kc_init=kv[0], vc_init=kv[1])
    again, _, _ = gpu_prefill(eng, case, kc_init=kv[0], vc_init=kv[1])
    ref, rkc, rvc = oracle_prefill(O, case, layers, n_ctx, kc=kv[0].ravel().copy(), vc=kv[1].ravel().copy())
    err = max_err(out, ref)
    log(f"    max-abs {err:.3e}")
    assert err <= PREFILL_TOL
    assert np.array_equal(bits(kc.ravel()), bits(rkc)) and np.array_equal(bits(vc.ravel()), bits(rvc))
    assert np.array_equal(bits(out), bits(again))


@pytest.mark.parametrize("pos0,n_tok", [(0, 20), (37, 60), (100, 9)])
def test_prefill_rows_already_in_the_cache(W, engines, pos0, n_tok):
    """k and v rows that lie in their own place in the cache, and an output in
    place of q, give what separate buffers give."""
    n_ctx = 192
    case = W.make_prefill(n_layers=1, n_tok=n_tok, pos0=pos0, salt=3)
    g = np.random.default_rng(8)
    kv = [g.standard_normal((1, 1, n_ctx, 256)).astype(np.float32) for _ in range(2)]
    eng = engines(1, n_ctx)
    out, kc, vc = gpu_prefill(eng, case, kc_init=kv[0], vc_init=kv[1])
    with device_arrays() as track:
        dkc, dvc = eng.kv_cache(1)
        track(dkc), track(dvc)
        for d, init, rows in ((dkc, kv[0], case.k), (dvc, kv[1], case.v)):
            init = init.copy()
            init[0, 0, pos0:pos0 + n_tok] = rows.reshape(n_tok, 256)
            d.upload(init)
        q = track(eng.array(case.q))
        off = pos0 * 256 * 4
        eng.prefill(pos0, n_tok, 0, 1, q.ptr, q.ptr, dkc.ptr + off, dvc.ptr + off, dkc.ptr, dvc.ptr)
        assert max_err(q.download(), out) <= PREFILL_TOL
        assert np.array_equal(bits(dkc.download()), bits(kc)) and np.array_equal(bits(dvc.download()), bits(vc))


def free_bytes(tla):
    free, total = C.c_size_t(), C.c_size_t()
    assert tla.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("layers,pos0,n_tok,shared", [(1, 0, 20, False), (22, 0, 200, False), (1, 300, 1, True)])
def test_prefill_allocates_what_it_uses(tla, W, layers, pos0, n_tok, shared):
    """The workspace of shared query tiles (51 MiB) comes with the first launch
    that shares one, not with a launch that does not; the planes with a launch
    that reads them."""
    n_ctx = pos0 + n_tok
    case = W.make_prefill(n_layers=layers, n_tok=n_tok, pos0=pos0, salt=1)
    eng = tla.Engine(tla.Config(layers, 2048, 32, 4, n_ctx, 10000.0))
    try:
        with device_arrays() as track:
            q, k, v = (track(eng.array(a)) for a in (case.q, case.k, case.v))
            out = track(eng.array(case.q.shape))
            kc, vc = eng.kv_cache(1)
            track(kc), track(vc)
            eng.synchronize()
            before = free_bytes(tla)
            for _ in range(2):
                eng.prefill(pos0, n_tok, 0, layers, out.ptr, q.ptr, k.ptr, v.ptr, kc.ptr, vc.ptr)
            eng.synchronize()
            used = before - free_bytes(tla)
    finally:
        eng.close()
    planes = layers * 4 * ((n_ctx + 31) // 32) * 24576 if layers > 1 else 0
    log(f"    {used >> 20} MiB")
    assert used - planes < 8 << 20 if not shared else 51 << 20 <= used < 60 << 20
