"""GPU parity of the backward kernels (backward.hip) against the oracle's fp64
restatement, which is itself pinned by finite differences (test_oracle.py).

Per row (dQ: (row, head); dK/dV: (token, kv head)): max|a - ref| / max|ref| <=
1e-5 (f32) or 2e-3 (f16), the path's tolerances.  The gradient pools are
accumulated into, as the reference's atomic adds do; keys before the window
start stay untouched.
"""
import numpy as np
import pytest

import oracle
from helpers import TOL, row_rel_err, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,T,H,hkv,d,bs,W", [
    (0, 40, 8, 2, 64, 16, 0),
    (0, 33, 4, 4, 128, 8, 20),     # window: keys 0..12 get no gradient
    (1, 64, 16, 4, 128, 16, 0),
    (1, 50, 8, 8, 64, 16, 0),
    (0, 17, 2, 1, 256, 16, 0),     # d = 256, MQA
    # f16, d = 128: the MFMA kernels (ragged row and key tiles, windows, G = 1..8)
    (1, 300, 32, 4, 128, 16, 0),
    (1, 257, 8, 8, 128, 32, 100),
    (1, 131, 16, 2, 128, 16, 0),
    (1, 96, 64, 8, 128, 16, 45),
    (1, 2100, 4, 4, 128, 1, 0),    # 2100 one-token blocks: the dQ kernel's large block-table form
])
def test_backward_parity(dtype, T, H, hkv, d, bs, W):
    import torch
    from pagedattentionmetal_amd import PagedAttentionEngine, PagedLayerSpec
    eng = PagedAttentionEngine()
    eng.set_graceful_degradation(False)
    rng = np.random.default_rng(300 + T + d)
    io = np.float32 if dtype == 0 else np.float16
    nbl = (T + bs - 1) // bs
    nb = nbl + 3
    bt = rng.permutation(nb)[:nbl].astype(np.int32)
    kp = rng.standard_normal((nb, bs, hkv, d)).astype(io)
    vp = rng.standard_normal((nb, bs, hkv, d)).astype(io)
    q = rng.standard_normal((T, H, d)).astype(io)
    go = rng.standard_normal((T, H, d)).astype(io)
    m, l, _ = oracle.forward_stats(q, kp, vp, bt, window=W)
    dq_r, dk_r, dv_r = oracle.backward(q, kp, vp, bt, go, m, l, window=W)
    init = np.zeros((nb, bs, hkv, d), io) if dtype == 1 else (0.1 * rng.standard_normal((nb, bs, hkv, d))).astype(io)
    dkp, dvp = to_dev(init.copy()), to_dev(init.copy())
    dq = torch.zeros((T, H, d), dtype=torch.float32 if dtype == 0 else torch.float16, device="cuda")
    lay = PagedLayerSpec(d, H, hkv, bs, dtype, W)
    eng.backward(to_dev(q), to_dev(kp), to_dev(vp), to_dev(bt), to_dev(go), to_dev(m.astype(np.float32)),
                 to_dev(l.astype(np.float32)), dq, dkp, dvp, T, lay)
    assert eng.last_stats["operation"] == 7
    assert row_rel_err(to_host(dq), dq_r) <= TOL[dtype]
    j = np.arange(T)
    slots = (bt[j // bs], j % bs)
    base = init[slots].astype(np.float64)
    got_k = to_host(dkp)[slots].astype(np.float64)
    got_v = to_host(dvp)[slots].astype(np.float64)
    ws = max(0, T - W) if W else 0
    assert row_rel_err(got_k[ws:], base[ws:] + dk_r[ws:]) <= TOL[dtype]
    assert row_rel_err(got_v[ws:], base[ws:] + dv_r[ws:]) <= TOL[dtype]
    assert np.array_equal(got_k[:ws], base[:ws]) and np.array_equal(got_v[:ws], base[:ws])
    # blocks the sequence does not use are untouched
    unused = np.setdiff1d(np.arange(nb), bt)
    assert np.array_equal(to_host(dkp)[unused], init[unused])


def test_backward_refuses_fp8(torch_mod=None):
    from pagedattentionmetal_amd import PagedAttentionEngine, PagedAttentionError, PagedLayerSpec
    import torch
    eng = PagedAttentionEngine()
    eng.set_graceful_degradation(False)
    x = torch.zeros(64, device="cuda")
    with pytest.raises(PagedAttentionError, match="f32 or f16"):
        eng.backward(x, x, x, x, x, x, x, x, x, x, 4, PagedLayerSpec(16, 2, 2, 16, 2))


@pytest.mark.parametrize("H,hkv,d,T", [(32, 32, 256, 19), (12, 4, 96, 26), (8, 1, 64, 33), (16, 4, 128, 70)])
def test_backward_f32_error_against_the_valu_kernels(H, hkv, d, T):
    """The f32 matrix kernels' gradients are no further from 64 bits than those of the
    VALU kernels, which take buffers that are not 16-byte aligned (5% for what the
    ratio of the error norms moves with the inputs)."""
    import torch
    from pagedattentionmetal_amd import PagedAttentionEngine, PagedLayerSpec
    bs, err = 16, np.zeros((2, 3))
    shifted = lambda a: torch.cat([torch.zeros(1, device="cuda"), to_dev(a).reshape(-1)])[1:].view(a.shape)
    for seed in range(3):
        rng = np.random.default_rng(700 + seed)
        nbl = (T + bs - 1) // bs
        bt = rng.permutation(nbl).astype(np.int32)
        kp, vp = (0.5 * rng.standard_normal((nbl, bs, hkv, d)).astype(np.float32) for _ in range(2))
        q, go = (rng.standard_normal((T, H, d)).astype(np.float32) for _ in range(2))
        m, l, _ = oracle.forward_stats(q, kp, vp, bt, window=0)
        m, l = m.astype(np.float32), l.astype(np.float32)
        ref = oracle.backward(q, kp, vp, bt, go, m, l, window=0)
        slots = (bt[np.arange(T) // bs], np.arange(T) % bs)
        for i, put in enumerate((to_dev, shifted)):
            eng = PagedAttentionEngine()
            eng.set_graceful_degradation(False)
            dq, dkp, dvp = torch.zeros((T, H, d), device="cuda"), to_dev(np.zeros_like(kp)), to_dev(np.zeros_like(vp))
            eng.backward(put(q), to_dev(kp), to_dev(vp), to_dev(bt), to_dev(go), to_dev(m), to_dev(l), dq, dkp, dvp, T,
                         PagedLayerSpec(d, H, hkv, bs, 0, 0))
            for x, (a, b) in enumerate(zip((to_host(dq), to_host(dkp)[slots], to_host(dvp)[slots]), ref)):
                err[i, x] += np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)
    assert (err[0] <= 1.05 * err[1]).all(), err
