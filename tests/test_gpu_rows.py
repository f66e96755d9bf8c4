"""The row-block kernels (rows.hip): prefill of f32 caches and of the f16 / e4m3
head and block sizes the dense kernel does not take; decode of f32 caches, small
head groups and those sizes.  Parity with the oracle at the edges of their blocks
(32 rows, 16 heads), tiles (16 keys), partitions and head-size tiles; keys that
hold Inf or NaN reach exactly the rows that see them, as on the VALU kernel; the
code object runs them bit for bit."""
import numpy as np
import pytest

import oracle
from helpers import TOL, make_case, row_rel_err, to_dev, to_host
from test_gpu_kernels import build_fp8, layer

pytestmark = pytest.mark.gpu

IO = {0: np.float32, 1: np.float16, 2: np.float16}


def _engine():
    from pagedattentionmetal_amd import PagedAttentionEngine
    e = PagedAttentionEngine()
    e.set_graceful_degradation(False)
    return e


def _prefill(eng, q, kd, vd, bt, T, lay, causal, off, ks=None, vs=None):
    import torch
    out = torch.full(q.shape, 7.0, dtype=torch.float32 if q.dtype == np.float32 else torch.float16, device="cuda")
    eng.prefill(to_dev(q), kd, vd, to_dev(bt), out, T, lay, causal=causal, q_offset=off, k_scale=ks, v_scale=vs)
    return to_host(out)


@pytest.mark.parametrize("dtype,T,off,H,hkv,d,bs,causal,window,part", [
    (0, 32, 0, 8, 8, 128, 16, True, 0, 0),
    (0, 33, 31, 8, 8, 128, 16, True, 0, 0),      # a second block of one row, a second tile of one key
    (0, 31, 1000, 8, 2, 64, 16, True, 0, 0),     # several partitions and the reduce
    (0, 70, 45, 6, 2, 80, 12, True, 0, 48),      # G = 3, head size between tiles, short partitions
    (0, 70, 245, 6, 2, 80, 12, True, 0, 48),     # past 256 keys, where the VALU kernel no longer takes it
    (0, 5, 300, 4, 4, 256, 8, True, 0, 0),
    (0, 90, 10, 4, 1, 32, 1, False, 0, 0),       # one-token blocks, not causal
    (0, 200, 0, 4, 4, 36, 16, True, 77, 0),      # rows before the window see no key
    (0, 1, 0, 2, 2, 4, 16, True, 0, 0),          # one row, one key, one slice
    (1, 130, 77, 12, 4, 96, 16, True, 0, 0),
    (1, 65, 0, 40, 2, 64, 16, True, 0, 0),       # more than 16 heads a kv head
    (1, 47, 500, 8, 8, 128, 24, True, 100, 0),   # a block size that is not a power of two
    (2, 64, 33, 8, 2, 96, 16, True, 0, 0),
    (2, 40, 0, 4, 4, 160, 4, False, 0, 0),
])
def test_rows_parity(dtype, T, off, H, hkv, d, bs, causal, window, part):
    rng = np.random.default_rng(900 + T + d)
    eng = _engine()
    _, k, v, bt, lens = make_case(rng, 1, H, hkv, d, bs, dtype, [off + T])
    q = rng.standard_normal((T, H, d)).astype(IO[dtype])
    if dtype == 2:
        kd, vd, ksd, vsd, k, v, ks, vs = build_fp8(eng, rng, k, v, bt, lens, hkv, d, bs)
        ks, vs = ks.view(np.uint16), vs.view(np.uint16)
    else:
        kd, vd, ksd, vsd, ks, vs = to_dev(k), to_dev(v), None, None, None, None
    eng.set_partition_tokens(part)
    o = _prefill(eng, q, kd, vd, bt[0], T, layer(H, hkv, d, bs, dtype, window), causal, off, ksd, vsd).astype(np.float64)
    ref = oracle.prefill(dtype, q, k, v, bt[0], off, causal=causal, window=window, k_scale=ks, v_scale=vs, n_threads=8)
    fin = np.isfinite(ref).all(axis=-1)
    assert np.isnan(o[~fin]).all(), "rows with no key in range are 0/0"
    assert row_rel_err(o[fin], ref[fin]) <= TOL[dtype]


@pytest.mark.parametrize("dtype,d", [(0, 128), (0, 40), (1, 96)])
def test_rows_inf_and_nan_stay_with_the_rows_that_see_them(dtype, d):
    """Against the VALU kernel (set_decode_kernel(1)) with single Inf and NaN elements
    of K and V at keys that some rows of a block mask."""
    T, off, H, hkv, bs = 70, 20, 4, 2, 16
    rng = np.random.default_rng(77)
    _, k, v, bt, _ = make_case(rng, 1, H, hkv, d, bs, dtype, [off + T])
    q = rng.standard_normal((T, H, d)).astype(IO[dtype])
    at = lambda j: (bt[0][j // bs], j % bs)
    v[at(50)][0, 3], v[at(61)][1, d - 1], k[at(75)][0, 1], v[at(89)][1, 0] = np.inf, np.nan, np.nan, -np.inf
    got = {}
    for choice in (0, 1):
        eng = _engine()
        eng.set_decode_kernel(choice)
        got[choice] = _prefill(eng, q, to_dev(k), to_dev(v), bt[0], T, layer(H, hkv, d, bs, dtype), True, off)
    a, b = got[0].astype(np.float64), got[1].astype(np.float64)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
    assert np.array_equal(a[np.isinf(a)], b[np.isinf(b)])
    assert np.isfinite(a[:30]).all() and not np.isfinite(a[30:, :, 3]).all()
    fin = np.isfinite(b).all(axis=-1)
    assert row_rel_err(a[fin], b[fin]) <= 2 * TOL[dtype]


@pytest.mark.parametrize("dtype,d", [(0, 128), (0, 64), (1, 96), (0, 32), (0, 200)])
def test_rows_code_object_bit_identical(dtype, d):
    T, off, H, hkv, bs = 45, 700, 8, 4, 16
    rng = np.random.default_rng(78)
    _, k, v, bt, _ = make_case(rng, 1, H, hkv, d, bs, dtype, [off + T])
    q = rng.standard_normal((T, H, d)).astype(IO[dtype])
    got = []
    for module in (False, True):
        eng = _engine()
        if module:
            eng.load_module()
            eng.set_module_strict(True)
        got.append(_prefill(eng, q, to_dev(k), to_dev(v), bt[0], T, layer(H, hkv, d, bs, dtype), True, off))
    assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))


@pytest.mark.parametrize("dtype,H,hkv,d,bs,lens,window,part", [
    (0, 8, 2, 128, 16, [0, 1, 15, 16, 17, 255, 256, 257], 0, 0),
    (0, 32, 8, 64, 16, [5000, 33, 1290], 0, 0),         # several partitions and the reduce
    (0, 6, 2, 80, 12, [700, 1, 64], 0, 48),             # G = 3, head size between tiles
    (0, 20, 1, 36, 16, [100, 17], 0, 0),                # 20 heads a kv head: two slots, the second of 4
    (0, 4, 4, 256, 8, [1500, 0, 300], 0, 0),
    (0, 2, 2, 4, 1, [3, 40], 0, 0),
    (0, 4, 2, 16, 16, [3, 17] * 33000, 0, 0),           # more rows than a grid's z takes: the VALU kernel
    (0, 4, 4, 16, 16, [2100, 130], 0, 16),              # 132 partitions: more than the reduce loads ahead
    (1, 16, 16, 64, 16, [3000, 100, 17, 0], 0, 0),
    (1, 8, 4, 128, 16, [2000, 500], 333, 0),
    (1, 34, 2, 96, 32, [900, 31], 0, 0),                # 17 heads a kv head
    (1, 8, 8, 256, 16, [260, 4], 0, 0),
    (2, 8, 8, 128, 16, [1000, 1, 77], 0, 0),
    (2, 12, 4, 64, 16, [2000, 48], 100, 32),
    (2, 8, 4, 96, 4, [513, 2], 0, 0),
])
def test_decode_rows_parity(dtype, H, hkv, d, bs, lens, window, part):
    import torch
    rng = np.random.default_rng(1300 + d + len(lens))
    eng = _engine()
    q, k, v, bt, lens = make_case(rng, len(lens), H, hkv, d, bs, dtype, lens)
    if dtype == 2:
        kd, vd, ksd, vsd, k, v, ks, vs = build_fp8(eng, rng, k, v, bt, lens, hkv, d, bs)
        ks, vs = ks.view(np.uint16), vs.view(np.uint16)
    else:
        kd, vd, ksd, vsd, ks, vs = to_dev(k), to_dev(v), None, None, None, None
    eng.set_partition_tokens(part)
    out = torch.full(q.shape, 7.0, dtype=torch.float32 if dtype == 0 else torch.float16, device="cuda")
    eng.decode(to_dev(q), kd, vd, to_dev(bt), to_dev(lens), out, len(lens), bt.shape[1],
               layer(H, hkv, d, bs, dtype, window), k_scale=ksd, v_scale=vsd)
    ref = oracle.decode(dtype, q, k, v, bt, lens, H, window=window, k_scale=ks, v_scale=vs, n_threads=8)
    o = to_host(out).astype(np.float64)
    assert np.isnan(o[lens == 0]).all(), "a row without keys is 0/0"
    assert row_rel_err(o[lens > 0], ref[lens > 0]) <= TOL[dtype]


@pytest.mark.parametrize("dtype,d", [(0, 128), (1, 64), (1, 96)])
def test_decode_rows_read_nothing_past_a_row(dtype, d):
    """NaN and Inf in the tail of a row's last block, and in its last visible key."""
    import torch
    H, hkv, bs = 8, 4, 16
    rng = np.random.default_rng(79)
    q, k, v, bt, lens = make_case(rng, 3, H, hkv, d, bs, dtype, [37, 300, 5])
    for i, L in enumerate(lens):
        b = bt[i][(L - 1) // bs]
        k[b, L % bs:], v[b, L % bs:] = np.nan, np.inf
    v[bt[1][299 // bs], 299 % bs, 0, 2] = np.inf
    got = {}
    for choice in (0, 1):
        eng = _engine()
        eng.set_decode_kernel(choice)
        out = torch.empty(q.shape, dtype=torch.float32 if dtype == 0 else torch.float16, device="cuda")
        eng.decode(to_dev(q), to_dev(k), to_dev(v), to_dev(bt), to_dev(lens), out, 3, bt.shape[1],
                   layer(H, hkv, d, bs, dtype))
        got[choice] = to_host(out).astype(np.float64)
    a, b = got[0], got[1]
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
    assert np.isinf(a).sum() == H // hkv
    fin = np.isfinite(b).all(axis=-1)
    assert row_rel_err(a[fin], b[fin]) <= 2 * TOL[dtype]


@pytest.mark.parametrize("dtype,d,lens", [(0, 128, [700, 40]), (1, 64, [1000, 3]), (2, 96, [90, 300])])
def test_decode_rows_code_object_bit_identical(dtype, d, lens):
    import torch
    H, hkv, bs = 8, 4, 16
    rng = np.random.default_rng(80)
    q, k, v, bt, lens = make_case(rng, len(lens), H, hkv, d, bs, dtype, lens)
    ksd = vsd = None
    if dtype == 2:
        kd, vd, ksd, vsd, *_ = build_fp8(_engine(), rng, k, v, bt, lens, hkv, d, bs)
    else:
        kd, vd = to_dev(k), to_dev(v)
    got = []
    for module in (False, True):
        eng = _engine()
        if module:
            eng.load_module()
            eng.set_module_strict(True)
        out = torch.empty(q.shape, dtype=torch.float32 if dtype == 0 else torch.float16, device="cuda")
        eng.decode(to_dev(q), kd, vd, to_dev(bt), to_dev(lens), out, len(lens), bt.shape[1], layer(H, hkv, d, bs, dtype),
                   k_scale=ksd, v_scale=vsd)
        got.append(to_host(out))
    assert np.array_equal(got[0].view(np.uint8), got[1].view(np.uint8))


@pytest.mark.parametrize("dtype,T,H,hkv,d,bs,W", [
    (0, 17, 3, 1, 32, 16, 0),        # G = 3, one row tile and one key past a tile
    (0, 70, 6, 2, 80, 12, 33),       # head size between tiles, window inside a tile, odd blocks
    (0, 260, 8, 1, 64, 16, 0),       # several shares per key block
    (0, 100, 4, 2, 128, 16, 48),     # window at a tile boundary
    (0, 40, 2, 2, 36, 1, 0),
    (1, 33, 5, 1, 96, 16, 0),
    (1, 300, 12, 4, 128, 16, 0),     # f16 d = 128 with a group that is no power of two
    (1, 129, 32, 2, 64, 8, 100),
    (1, 50, 4, 4, 256, 16, 0),
    (1, 20, 2, 1, 40, 4, 0),
])
def test_backward_rows_parity(dtype, T, H, hkv, d, bs, W):
    import test_gpu_backward
    test_gpu_backward.test_backward_parity(dtype, T, H, hkv, d, bs, W)


# MFMA decode as partitions (mfma_part_tiles): one partition, and the shortest and
# longest partition lengths the rule picks, on both sides of its lines
@pytest.mark.parametrize("dtype,H,hkv,d,bs,lens,window", [
    (1, 32, 8, 128, 16, [512, 1, 0, 300], 0),        # 32 tiles: one partition
    (1, 32, 8, 128, 16, [513, 17], 0),               # 33 tiles: 128-token partitions
    (1, 8, 1, 128, 16, [8200], 0),                   # 512-token partitions, the last of 8 tokens
    (1, 32, 8, 64, 8, [2000] + [5] * 20, 0),         # 8-token blocks, most rows in the first partition
    (1, 64, 8, 256, 16, [256, 2, 40], 0),
    (1, 64, 8, 256, 16, [257, 100], 0),
    (2, 32, 8, 128, 16, [1500, 100, 16, 0], 0),
    (2, 16, 4, 64, 32, [3000, 7], 900),
    (1, 16, 4, 128, 16, [5000] * 3, 700),
])
def test_decode_partitions_parity(dtype, H, hkv, d, bs, lens, window):
    test_decode_rows_parity(dtype, H, hkv, d, bs, lens, window, 0)


@pytest.mark.parametrize("dtype,d,lens", [(1, 128, [700, 0, 40]), (2, 128, [90, 300]), (1, 64, [2000, 1])])
def test_decode_layers_partitions_bit_identical(dtype, d, lens):
    """Layers fused over partitions (and their reduce) against single-layer decodes,
    from the library and (d = 128) from the code object."""
    import torch
    H, hkv, bs, n = 32, 8, 16, 3
    rng = np.random.default_rng(81)
    q, k, v, bt, lens = make_case(rng, len(lens), H, hkv, d, bs, dtype, lens)
    ksd = vsd = None
    if dtype == 2:
        kd, vd, ksd, vsd, *_ = build_fp8(_engine(), rng, k, v, bt, lens, hkv, d, bs)
    else:
        kd, vd = to_dev(k), to_dev(v)
    qs = [to_dev(rng.standard_normal(q.shape).astype(np.float16)) for _ in range(n)]
    btd, lnd, lay = to_dev(bt), to_dev(lens), layer(H, hkv, d, bs, dtype)
    single = []
    eng = _engine()
    for x in qs:
        o = torch.empty(q.shape, dtype=torch.float16, device="cuda")
        eng.decode(x, kd, vd, btd, lnd, o, len(lens), bt.shape[1], lay, k_scale=ksd, v_scale=vsd)
        single.append(to_host(o))
    for module in (False, True) if d == 128 else (False,):
        eng = _engine()
        if module:
            eng.load_module()
            eng.set_module_strict(True)
        outs = [torch.empty(q.shape, dtype=torch.float16, device="cuda") for _ in range(n)]
        eng.decode_layers(qs, kd, vd, btd, lnd, outs, len(lens), bt.shape[1], [lay] * n, k_scale=ksd, v_scale=vsd)
        for a, b in zip(single, outs):
            assert np.array_equal(a.view(np.uint16), to_host(b).view(np.uint16))


@pytest.mark.parametrize("H,hkv,d", [(32, 8, 128), (16, 4, 64), (32, 4, 256)])
@pytest.mark.parametrize("lens", [[900, 5, 17, 24, 8], [1, 33, 7, 40, 16], [2003, 130]])
def test_decode_e4m3_small_blocks_beside_other_entries(H, hkv, d, lens):
    """e4m3 rows of 8-token blocks whose tables go on past the rows (in a wider table)
    with a block of the pool that has scales and codes of its own: a row with an odd
    number of blocks ends inside a 16-token tile.  Single layer and fused layers."""
    import torch
    bs = 8
    rng = np.random.default_rng(82 + d + len(lens))
    eng = _engine()
    q, k, v, bt, lens = make_case(rng, len(lens), H, hkv, d, bs, 2, lens)
    kd, vd, ksd, vsd, kp, vp, ks, vs = build_fp8(eng, rng, k, v, bt, lens, hkv, d, bs)
    other = sorted(set(range(k.shape[0])) - {int(bt[b, i]) for b, L in enumerate(lens) for i in range(-(-int(L) // bs))})[0]
    kp[other], vp[other], ks[other], vs[other] = 0x7E, 0x7E, np.inf, np.nan
    kd, vd, ksd, vsd = to_dev(kp), to_dev(vp), to_dev(ks), to_dev(vs)
    wide = np.full((len(lens), bt.shape[1] + 9), other, np.int32)
    for b, L in enumerate(lens):
        wide[b, :-(-int(L) // bs)] = bt[b, :-(-int(L) // bs)]
    lay = layer(H, hkv, d, bs, 2)
    ref = oracle.decode(2, q, kp, vp, wide, lens, H, k_scale=ks.view(np.uint16), v_scale=vs.view(np.uint16), n_threads=8)
    out = torch.full(q.shape, 7.0, dtype=torch.float16, device="cuda")
    eng.decode(to_dev(q), kd, vd, to_dev(wide), to_dev(lens), out, len(lens), wide.shape[1], lay, k_scale=ksd, v_scale=vsd)
    assert row_rel_err(to_host(out).astype(np.float64), ref) <= TOL[2]
    outs = [torch.full(q.shape, 7.0, dtype=torch.float16, device="cuda") for _ in range(2)]
    eng.decode_layers([to_dev(q)] * 2, kd, vd, to_dev(wide), to_dev(lens), outs, len(lens), wide.shape[1], [lay] * 2,
                      k_scale=ksd, v_scale=vsd)
    for o in outs:
        assert np.array_equal(to_host(o).view(np.uint16), to_host(out).view(np.uint16))


def _attend64(q, k, v, lens):
    """float64 attention of rows q [n, H, d], row i over the first lens[i] of its keys k[i], v[i] [L, hkv, d]."""
    out = np.empty(q.shape)
    G = q.shape[1] // k[0].shape[1]
    for i, L in enumerate(lens):
        kk, vv = (np.repeat(x[i][:L].astype(np.float64), G, axis=1) for x in (k, v))
        s = np.einsum("hd,jhd->hj", q[i].astype(np.float64), kk) / np.sqrt(q.shape[2])
        p = np.exp(s - s.max(1, keepdims=True))
        out[i] = np.einsum("hj,jhd->hd", p / p.sum(1, keepdims=True), vv)
    return out


def _norm_err(a, ref):
    return np.linalg.norm(a.astype(np.float64) - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("H,hkv,d,T,off", [(64, 8, 128, 101, 0), (16, 4, 128, 143, 0), (32, 2, 96, 40, 300),
                                           (8, 4, 256, 90, 20)])
def test_rows_f32_prefill_error_against_the_valu_kernel(H, hkv, d, T, off):
    """The matrix units' f32 sums are no further from 64 bits than the VALU kernel's
    (a ratio of error norms over tens of thousands of outputs moves by 1% with the
    inputs; 3% allowed)."""
    bs, err = 16, {0: 0.0, 1: 0.0}
    for seed in range(3):
        rng = np.random.default_rng(500 + seed)
        _, k, v, bt, _ = make_case(rng, 1, H, hkv, d, bs, 0, [off + T])
        k, v = 0.5 * k, 0.5 * v
        q = rng.standard_normal((T, H, d)).astype(np.float32)
        kr, vr = (x[bt[0]].reshape(-1, hkv, d) for x in (k, v))
        ref = _attend64(q, [kr] * T, [vr] * T, [off + i + 1 for i in range(T)])
        for choice in err:
            eng = _engine()
            eng.set_decode_kernel(choice)
            err[choice] += _norm_err(_prefill(eng, q, to_dev(k), to_dev(v), bt[0], T, layer(H, hkv, d, bs, 0), True, off), ref)
    assert err[0] <= 1.03 * err[1], err


@pytest.mark.parametrize("H,hkv,d,B,hi", [(8, 1, 256, 49, 244), (8, 1, 128, 40, 69), (32, 8, 64, 64, 36), (32, 8, 256, 29, 191)])
def test_rows_f32_decode_error_against_the_valu_kernel(H, hkv, d, B, hi):
    """As above, short decodes (fewer outputs: 5%)."""
    import torch
    bs, err = 16, {0: 0.0, 1: 0.0}
    for seed in range(3):
        rng = np.random.default_rng(600 + seed)
        lens = rng.integers(hi // 4, hi + 1, B)
        lens[0] = hi
        q, k, v, bt, lens = make_case(rng, B, H, hkv, d, bs, 0, lens)
        k, v = 0.5 * k, 0.5 * v
        rows = lambda x: [x[bt[i]].reshape(-1, hkv, d) for i in range(B)]
        ref = _attend64(q, rows(k), rows(v), [int(L) for L in lens])
        for choice in err:
            eng = _engine()
            eng.set_decode_kernel(choice)
            out = torch.full(q.shape, 7.0, dtype=torch.float32, device="cuda")
            eng.decode(to_dev(q), to_dev(k), to_dev(v), to_dev(bt), to_dev(lens), out, B, bt.shape[1], layer(H, hkv, d, bs, 0))
            err[choice] += _norm_err(to_host(out), ref)
    assert err[0] <= 1.05 * err[1], err


def _wide(bt, pool, width):
    """Tables widened to `width` blocks, and a pool that may hold them (a call checks that)."""
    w = np.zeros((bt.shape[0], width), np.int32)
    w[:, :bt.shape[1]] = bt
    need = max(0, w.size - pool.shape[0])
    return w, np.concatenate([pool, np.zeros((need,) + pool.shape[1:], pool.dtype)])


@pytest.mark.parametrize("H,hkv,d,lens,width,valu", [
    (4, 4, 256, [250, 3, 64], 32, True),      # one head a kv head, d > 128: up to 512 tokens
    (4, 4, 256, [250, 3, 64], 33, False),
    (4, 4, 256, [300] * 33, 24, True),        # more heads: up to 384
    (4, 4, 256, [300] * 33, 25, False),
    (8, 8, 128, [190, 40], 24, True),         # few heads: up to 384
    (8, 8, 128, [190, 40], 25, False),
    (8, 8, 128, [190] * 3, 24, False),
    (4, 4, 256, [300] * 17, 32, False),
    (12, 4, 256, [177, 20], 24, True),        # an odd group
    (12, 4, 256, [177, 20] * 3, 24, False),
    (12, 4, 96, [177], 24, True),
    (12, 4, 96, [177, 20], 24, False),
    (8, 4, 256, [177, 20], 16, False),        # an even group
])
def test_f32_decode_rows_of_few_keys_stay_on_the_valu_kernel(H, hkv, d, lens, width, valu):
    """By the table's width, in blocks of 16: the same bits as with set_decode_kernel(1)."""
    import torch
    rng = np.random.default_rng(85)
    q, k, v, bt, lens = make_case(rng, len(lens), H, hkv, d, 16, 0, lens)
    bw, k = _wide(bt, k, width)
    _, v = _wide(bt, v, width)
    got = []
    for choice in (0, 1):
        eng = _engine()
        eng.set_decode_kernel(choice)
        out = torch.full(q.shape, 7.0, dtype=torch.float32, device="cuda")
        eng.decode(to_dev(q), to_dev(k), to_dev(v), to_dev(bw), to_dev(lens), out, len(lens), width, layer(H, hkv, d, 16, 0))
        got.append(to_host(out))
    assert row_rel_err(got[0].astype(np.float64), oracle.decode(0, q, k, v, bw, lens, H, n_threads=8)) <= TOL[0]
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)) == valu


@pytest.mark.parametrize("H,hkv,d,T,off,valu", [
    (8, 4, 128, 95, 0, True), (8, 8, 128, 101, 0, True), (8, 8, 96, 112, 0, False), (8, 8, 256, 95, 0, False),
    (8, 8, 64, 94, 0, False), (24, 8, 128, 72, 0, True), (24, 8, 128, 75, 0, False), (24, 4, 128, 39, 0, True),
    (24, 4, 96, 9, 122, True), (24, 4, 128, 44, 0, False), (24, 4, 256, 30, 0, False),
])
def test_f32_prefills_of_few_keys_stay_on_the_valu_kernel(H, hkv, d, T, off, valu):
    """By (row, head, key) triples: the same bits as with set_decode_kernel(1)."""
    rng = np.random.default_rng(87)
    _, k, v, bt, _ = make_case(rng, 1, H, hkv, d, 16, 0, [off + T])
    q = rng.standard_normal((T, H, d)).astype(np.float32)
    got = []
    for choice in (0, 1):
        eng = _engine()
        eng.set_decode_kernel(choice)
        got.append(_prefill(eng, q, to_dev(k), to_dev(v), bt[0], T, layer(H, hkv, d, 16, 0), True, off))
    assert row_rel_err(got[0].astype(np.float64), oracle.prefill(0, q, k, v, bt[0], off, causal=True, window=0, n_threads=8)) <= TOL[0]
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)) == valu


@pytest.mark.parametrize("dtype,H,hkv,d,B,width,most", [
    (1, 8, 1, 256, 9, 1456, 512),    # 9 to 16 pairs: 512 tokens
    (2, 16, 4, 64, 3, 1500, 512),
    (1, 32, 2, 128, 3, 1984, 256),   # up to 8 pairs: 256 while a CU has no three partitions
    (2, 8, 1, 256, 4, 772, 256),
])
def test_mfma_decode_of_few_pairs_keeps_short_partitions(dtype, H, hkv, d, B, width, most):
    """Tables much wider than their rows (blocks of 16)."""
    import torch
    rng = np.random.default_rng(86)
    eng = _engine()
    q, k, v, bt, lens = make_case(rng, B, H, hkv, d, 16, dtype, rng.integers(100, 700, B))
    if dtype == 2:
        kd, vd, ksd, vsd, k, v, ks, vs = build_fp8(eng, rng, k, v, bt, lens, hkv, d, 16)
        ks, vs = ks.view(np.uint16), vs.view(np.uint16)
    else:
        ks = vs = None
    bw, kp = _wide(bt, k, width)
    kd, vd = to_dev(kp), to_dev(_wide(bt, v, width)[1])
    ksd, vsd = (None, None) if ks is None else (to_dev(np.resize(x, kp.shape[0]).view(np.float16)) for x in (ks, vs))
    out = torch.full(q.shape, 7.0, dtype=torch.float16, device="cuda")
    eng.decode(to_dev(q), kd, vd, to_dev(bw), to_dev(lens), out, B, width, layer(H, hkv, d, 16, dtype), k_scale=ksd, v_scale=vsd)
    parts = eng.last_stats["temporary_bytes"] // (B * H * (d + 2) * 4)
    assert parts >= -(-width * 16 // most)
    ref = oracle.decode(dtype, q, k, v, bw, lens, H, k_scale=ks, v_scale=vs, n_threads=8)
    assert row_rel_err(to_host(out).astype(np.float64), ref) <= TOL[dtype]


@pytest.mark.parametrize("H,hkv,d,ctx,new,valu", [
    (4, 4, 256, [491, 60, 0], [5, 1, 17], True),      # d > 128: up to 31 tiles of 16 tokens
    (4, 4, 256, [492, 60, 0], [5, 1, 17], False),
    (8, 8, 128, [300, 60, 0], [5, 1, 17], False),
    (32, 32, 64, [40, 623], [255, 1], True),          # 8192 pairs: up to 39
    (32, 32, 64, [40, 624], [255, 1], False),
    (32, 32, 64, [40, 300], [254, 1], False),
    (32, 32, 64, [40, 1007], [511, 1], True),         # 16384: up to 63
    (32, 32, 64, [40, 1008], [511, 1], False),
    (32, 32, 64, [40, 1007], [510, 1], False),
    (32, 16, 64, [40, 1007], [511, 1], False),        # an even group
])
def test_f32_mixed_steps_of_few_keys_stay_on_the_valu_kernel(H, hkv, d, ctx, new, valu):
    """By the longest row and the (row, head) pairs: the same bits as with set_decode_kernel(1)."""
    import torch
    rng = np.random.default_rng(88)
    lens = [c + n for c, n in zip(ctx, new)]
    _, k, v, bt, _ = make_case(rng, len(lens), H, hkv, d, 16, 0, lens)
    q = rng.standard_normal((sum(new), H, d)).astype(np.float32)
    got = []
    for choice in (0, 1):
        eng = _engine()
        eng.set_decode_kernel(choice)
        out = torch.full(q.shape, 7.0, dtype=torch.float32, device="cuda")
        eng.mixed_step(to_dev(q), out, to_dev(k), to_dev(v), to_dev(bt), ctx, new, layer(H, hkv, d, 16, 0))
        got.append(to_host(out))
    at = 0
    for i, n in enumerate(new):
        ref = oracle.prefill(0, q[at:at + n], k, v, bt[i], ctx[i], causal=True, window=0, n_threads=8)
        assert row_rel_err(got[0][at:at + n].astype(np.float64), ref) <= TOL[0]
        at += n
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)) == valu
