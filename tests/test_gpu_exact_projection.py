"""The batched prefill's exact projections on the matrix cores (k_bgemm)
against the CPU restatement, bit for bit, where the kernel's tiling can go
wrong: token counts around its 16- and 48-token tiles and the count at which
it takes over, widths that leave a partial visit pair, a partial line group or
a single visit, and row counts that end inside a tile.

Then the products alone (cq35_device_exact_gemm), in every epilogue and both
tile shapes, for the values that the route is chosen by: sums that show the
order and the rounding of every step, products that are exact while their sums
are subnormal (the matrix cores keep them), and what a fused multiply-add
would round differently, recomputed by k_bgemm_fix: products whose lowest bits
lie below the F32 subnormals, products beyond the largest F32, infinities and
NaN. Against the batched order in numpy F32, which is the restatement's (first
test); where the fix matters, the fused sums are shown to differ first."""
import ctypes
import time

import numpy as np
import pytest
import torch

import cq35
import cq35.config as cc
from cq35 import _lib

pytestmark = pytest.mark.gpu


def config(hidden, intermediate, value_heads=4):
    cfg = cc.preset("mini")
    cfg.update(vocab=512, hidden=hidden, intermediate=intermediate, value_heads=value_heads)
    return cfg


def compare(oracle, cfg, weights, prompt):
    gm, om = cq35.Model.from_arrays(cfg, weights), oracle.Model(cfg, weights)
    gs, os_ = gm.session(len(prompt)), om.session(len(prompt))
    gl, gt = gs.step_raw(prompt)
    ot, ol = os_.step(prompt, 0)
    assert gt == ot
    assert np.array_equal(gl, ol), "logits"
    assert np.array_equal(gs.export_state(0), os_.cache()), "state"
    gm.close()


# hidden 576: nine lines (visits of one and two); 1024: one visit pair; 320:
# less than one visit. intermediate 1344: 21 lines, 84 tiles; 1416: 22.125
# lines (not whole ones: the vector kernel) with gate rows ending inside a
# tile; 200: rows ending inside a tile.
@pytest.mark.parametrize("hidden, intermediate, tokens", [
    (576, 1344, 7), (576, 1344, 8), (576, 1344, 17), (1024, 3584, 48), (576, 1416, 49), (320, 200, 257), (576, 1344, 289),
])
def test_tiles_match_restatement(oracle, hidden, intermediate, tokens):
    cfg = config(hidden, intermediate)
    print("exact projection", hidden, intermediate, tokens, flush=True)
    prompt = np.random.default_rng(tokens).integers(0, cfg["vocab"], tokens).tolist()
    compare(oracle, cfg, oracle.synthetic_weights(cfg, 29), prompt)


@pytest.mark.parametrize("tokens", [20, 300])
def test_products_below_the_exact_range(oracle, tokens):
    cfg = config(512, 1408)
    weights = oracle.synthetic_weights(cfg, 30)
    full = cfg["full_interval"] - 1
    base = 1 + 14 * full  # first attention layer: its input norm, and three tensors on attn_v
    specs = oracle.weight_specs(cfg)
    assert specs[base + 3][1] == cfg["kv_heads"] * cfg["head_dim"] and specs[base + 3][2] == cfg["hidden"]
    # inputs of about 2^-16 and weights of about 2^-120: products of 16 bits
    # around 2^-136, the lowest below 2^-149
    weights[base] = weights[base] * np.float32(2.0 ** -16)
    w = weights[base + 3]
    exponent = (w.astype(np.int32) >> 7) & 0xff
    assert exponent.max() < 127
    scaled = np.where(exponent > 114, (w & 0x807f) | ((exponent - 114) << 7).astype(np.uint16), 0)
    assert (scaled != 0).mean() > 0.8
    weights[base + 3] = scaled.astype(np.uint16)
    print("exact projection, tiny weights", tokens, flush=True)
    prompt = np.random.default_rng(tokens).integers(0, cfg["vocab"], tokens).tolist()
    compare(oracle, cfg, weights, prompt)


# ------------------------------------------------------- the products alone


def widen(bits):
    return (np.asarray(bits, np.uint16).astype(np.uint32) << 16).view(np.float32)


def narrow(f):  # nearest even, NaN quieted
    u = np.ascontiguousarray(f, np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return np.where(np.isnan(f), ((u >> 16) | 0x40).astype(np.uint16), r)


def b256(x, w, fused=False):
    """F32 totals [n][rows] of the batched order: lane l of 256 adds the low
    and the high product of its pairs l, l + 256, ... to one accumulator, then
    the lanes' halving tree. `fused`: each product and its sum rounded once
    (through F64: off at most where F64 rounds the sum itself)."""
    (n, cols), rows = x.shape, w.shape[0]
    visits = -(-cols // 512)
    pad = lambda a: np.pad(widen(a), ((0, 0), (0, 512 * visits - cols))).reshape(len(a), visits, 256, 2)
    xs, ws = pad(x), pad(w)
    acc = np.zeros((n, rows, 256), np.float32)
    with np.errstate(all="ignore"):
        for v in range(visits):
            for half in range(2):
                a, b = xs[:, None, v, :, half], ws[None, :, v, :, half]
                if fused:
                    acc = (acc.astype(np.float64) + a.astype(np.float64) * b.astype(np.float64)).astype(np.float32)
                else:
                    acc = acc + a * b
        while acc.shape[-1] > 1:
            h = acc.shape[-1] // 2
            acc = acc[..., :h] + acc[..., h:]
    return acc[..., 0]


def silu(x):
    x = np.ascontiguousarray(x, np.float32)
    y = np.empty_like(x)
    fp = ctypes.POINTER(ctypes.c_float)
    assert _lib.load().cq35_device_numeric(1, x.ctypes.data_as(fp), y.ctypes.data_as(fp), x.size) == 0
    return y


def epilogue(mode, total, up, res):
    with np.errstate(all="ignore"):
        if mode == 0:
            return narrow(total)
        if mode == 1:
            return narrow(widen(narrow(total)) + widen(res))
        return narrow(widen(narrow(silu(widen(narrow(total))))) * widen(narrow(up)))


def exact_gemm(x, w, w2, res, mode, kernel):
    (n, cols), rows = x.shape, w.shape[0]
    out = np.empty((n, rows), np.uint16)
    ptr = lambda a: a.ctypes.data if a is not None else None
    rc = _lib.load().cq35_device_exact_gemm(ptr(x), ptr(w), ptr(w2), ptr(res), n, rows, cols, mode, kernel, ptr(out))
    assert rc == 0, _lib.load().cq35_last_error()
    return out


def odd(rng, shape, exponent):
    """+-(an odd whole number of eight bits) * 2^exponent."""
    m = rng.integers(64, 128, shape) * 2 + 1
    return narrow((np.where(rng.random(shape) < 0.5, -m, m) * 2.0 ** exponent).astype(np.float32))


def operands(kind, mode, n, rows, cols, rng):
    """x, w, w2, res and whether the fused sums have to differ."""
    x = narrow(rng.standard_normal((n, cols)).astype(np.float32))
    w = narrow((rng.standard_normal((rows, cols)) * 0.05).astype(np.float32))
    w2 = narrow((rng.standard_normal((rows, cols)) * 0.05).astype(np.float32)) if mode == 2 else None
    res = narrow(rng.standard_normal((n, rows)).astype(np.float32)) if mode == 1 else None
    differs = False
    if kind == "cancelling":
        # four lanes: products of +-2^18 that cancel within the lane, small
        # ones between them whose low bits go where the order says
        w[:] = 0
        for lane in (0, 5, 130, 255):
            c = np.array([512 * v + 2 * lane + h for v in range(-(-cols // 512)) for h in (0, 1)])
            c = c[c < cols]
            big = rng.permutation(len(c))[:len(c) // 4 * 2]
            big.sort()
            x[:, c] = narrow(rng.uniform(1, 2, (n, len(c))).astype(np.float32))
            w[:, c] = narrow(rng.uniform(-2, 2, (rows, len(c))).astype(np.float32))
            x[:, c[big]] = narrow(np.float32([512.0]))
            w[:, c[big]] = narrow(np.where(np.arange(len(big)) % 2, -512.0, 512.0).astype(np.float32))
    elif kind == "subnormal sums":
        # products odd * 2^-149: exact, their sums below 2^-126
        x, w = odd(rng, (n, cols), -70), odd(rng, (rows, cols), -79)
        w = np.where(rng.random((rows, cols)) < 0.25, w, 0).astype(np.uint16)
        if mode == 1:
            res = narrow((rng.integers(-64, 64, (n, rows)) * 2.0 ** -132).astype(np.float32))
        if mode == 2:
            w2 = narrow(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(2.0 ** 60))
    elif kind == "tiny":
        # in one row tile, in turn an odd multiple of 2^-149 and an odd one of
        # 2^-150: the halves are ties, to even before the sum or with it. The
        # second's residues of 4 make the sums apart by a unit a pair; signs
        # keep them below 2^-126, where BF16 has 2^16 units.
        tile = 8 if mode == 2 else 16
        m = rng.integers(32, 64, (n, cols)) * 4 + 1
        x = narrow((m * np.where(np.arange(cols) % 2, 2.0 ** -71, 2.0 ** -70)).astype(np.float32))
        m = rng.integers(32, 64, (tile, cols)) * 4
        small = narrow((np.where(rng.random(m.shape) < 0.5, m + 1, -(m + 3)) * 2.0 ** -79).astype(np.float32))
        w = narrow(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(2.0 ** 60))
        if mode == 2:  # ordinary gates over such up sums, and the other way round
            w2 = w.copy()
            w2[tile:2 * tile] = small
            w[2 * tile:3 * tile] = small
        else:
            w[tile:2 * tile] = small
        if mode == 1:
            res = narrow((rng.integers(-64, 64, (n, rows)) * 2.0 ** -132).astype(np.float32))
        differs = True
    elif kind == "huge":
        # -1.5 * 2^127 + 2^128 in one lane: beyond the largest F32 in between
        for t in (1, n - 1):
            x[t, 10:12] = narrow(np.float32([2.0 ** 64, 2.0 ** 64]))
        beyond = narrow(np.float32([-1.5 * 2.0 ** 63, 2.0 ** 64]))
        w[:, 10:12] = 0
        w[rows - 1, 10:12] = beyond
        if mode == 2:
            w2[:, 10:12] = 0
            w2[0, 10:12] = beyond
        differs = True
    elif kind == "not finite":
        x[n // 2, 3] = narrow(np.float32([np.inf]))[0]
        x[n - 1, 4] = narrow(np.float32([np.nan]))[0]
        w[1, 7] = narrow(np.float32([-np.inf]))[0]
        w[rows - 1, 0] = narrow(np.float32([np.nan]))[0]
        if mode == 2:
            w2[2, 9] = narrow(np.float32([np.inf]))[0]
    elif kind == "zeros":
        x[:], w[:2 * 16] = 0x8000, 0
    return x, w, w2, res, differs


# 17 tokens: 16 x 16 tiles in every mode; 49 tokens: 48 x 16 in gate mode; 300
# tokens: 48 x 16 in all. 36 rows (plain, residual: three row tiles, gate:
# five) end inside a tile.
@pytest.mark.parametrize("mode, n", [(0, 17), (0, 300), (1, 17), (1, 300), (2, 17), (2, 49)])
@pytest.mark.parametrize("kind", ["ordinary", "cancelling", "subnormal sums", "tiny", "huge", "not finite", "zeros"])
def test_products_alone(kind, mode, n):
    rows, cols = 36, {"tiny": 4096, "cancelling": 2112}.get(kind, 1088)
    print("exact products", kind, "mode", mode, "tokens", n, flush=True)
    rng = np.random.default_rng(100 * mode + n)
    x, w, w2, res, differs = operands(kind, mode, n, rows, cols, rng)
    up = b256(x, w2) if mode == 2 else None
    want = epilogue(mode, b256(x, w), up, res)
    nan = np.isnan(widen(want))
    if differs:
        fused = epilogue(mode, b256(x, w, True), b256(x, w2, True) if mode == 2 else None, res)
        assert ((fused != want) & ~(nan & np.isnan(widen(fused)))).sum() >= 2, "the values do not tell the routes apart"
    if kind == "cancelling":
        assert (b256(x[:, ::-1], w[:, ::-1]) != b256(x, w)).mean() > 0.9, "the order does not show"
    if kind == "subnormal sums":
        total = np.abs(b256(x, w))
        assert (total < 2.0 ** -126).mean() > 0.5 and (widen(narrow(total)) > 0).mean() > 0.8
    for kernel in (0, 1):
        got = exact_gemm(x, w, w2, res, mode, kernel)
        assert np.array_equal(nan, np.isnan(widen(got))), (kernel, "NaN")
        assert np.array_equal(got[~nan], want[~nan]), (kernel, int((got[~nan] != want[~nan]).sum()))


@pytest.mark.parametrize("mode, n, rows", [(0, 777, 5001), (1, 300, 2050), (2, 777, 3100), (2, 20, 1100)])
def test_every_region_recomputed(mode, n, rows):
    """Whole matrices of products that the matrix cores round differently: more
    row groups than the recomputation has groups of waves, more than one batch
    of 64 regions each, ragged ends. Against the vector kernel, bit for bit."""
    cols = 512
    print("every region, mode", mode, "tokens", n, "rows", rows, flush=True)
    rng = np.random.default_rng(rows)
    x = operands("tiny", 0, n, 32, cols, rng)[0]
    m = rng.integers(32, 64, (rows, cols)) * 4
    small = narrow((np.where(rng.random(m.shape) < 0.5, m + 1, -(m + 3)) * 2.0 ** -79).astype(np.float32))
    plain = narrow(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(2.0 ** 60))
    res = narrow((rng.integers(-64, 64, (n, rows)) * 2.0 ** -132).astype(np.float32)) if mode == 1 else None
    w, w2 = (plain, small) if mode == 2 else (small, None)
    few = slice(0, 64)
    assert (narrow(b256(x[:20], small[few], True)) != narrow(b256(x[:20], small[few]))).mean() > 0.001
    want, got = exact_gemm(x, w, w2, res, mode, 0), exact_gemm(x, w, w2, res, mode, 1)
    assert np.array_equal(want, got), int((want != got).sum())


def test_numpy_order_is_the_restatement(oracle):
    rng = np.random.default_rng(9)
    for kind in ("ordinary", "cancelling", "subnormal sums", "tiny", "huge"):
        x, w, _, _, _ = operands(kind, 0, 3, 32, 2112, rng)
        total = b256(x, w)
        for t in range(3):
            for r in range(32):
                assert np.float32(oracle.dot_b256(x[t], w[r])).view(np.uint32) == total[t, r].view(np.uint32) or \
                    np.isnan(total[t, r])


def test_inexact_tiles_cost_no_cliff(oracle):
    """A prompt whose weight tiles are all recomputed (one subnormal weight in
    every eight rows), and one with a single such row tile per matrix: within
    six times the ordinary prompt's time (the vector kernel's rate is a third
    of the matrix cores'; measured 3.4 and 1.1)."""
    cfg = config(1024, 3584, value_heads=16)
    tokens = 768
    rng = np.random.default_rng(12)
    prompt = rng.integers(0, cfg["vocab"], tokens).tolist()
    specs = oracle.weight_specs(cfg)
    plain = oracle.synthetic_weights(cfg, 31)

    def with_tiny(rows):
        out = []
        for i, ((dtype, r, c, _), w) in enumerate(zip(specs, plain)):
            if dtype == "bf16" and c % 64 == 0 and 0 < i < len(specs) - 1:
                w = w.reshape(r, c).copy()
                w[rows, 5] = 1
            out.append(w)
        return out

    def seconds(weights, what):
        m = cq35.Model.from_arrays(cfg, weights)
        best = np.inf
        for _ in range(4):
            s = m.session(tokens)
            print("inexact tiles:", what, flush=True)
            t = time.perf_counter()
            s.step_raw(prompt)
            best = min(best, time.perf_counter() - t)
        m.close()
        print(f"  {1e3 * best:.2f} ms", flush=True)
        return best

    ordinary = seconds(plain, "none")
    assert seconds(with_tiny(slice(3, 4)), "one row tile per matrix") < 6 * ordinary
    assert seconds(with_tiny(slice(0, None, 8)), "all") < 6 * ordinary


def test_borrowed_weights_off_the_lds_alignment(oracle):
    """Weights that a caller placed at addresses of 8 modulo 16: the same
    prompt as with the library's own, bit for bit (the vector kernel's loads
    take any address; the loads into LDS ask for 16 bytes)."""
    cfg = config(576, 1344)
    weights = oracle.synthetic_weights(cfg, 33)
    tensors = []
    for w in weights:
        t = torch.empty(w.nbytes + 64, dtype=torch.uint8, device="cuda")
        at = 8 - t.data_ptr() % 16 + 16
        t[at:at + w.nbytes] = torch.from_numpy(np.ascontiguousarray(w).view(np.uint8)).cuda()
        tensors.append((t, at))
    torch.cuda.synchronize()
    pointers = (ctypes.c_void_p * len(weights))(*[t.data_ptr() + at for t, at in tensors])
    c, handle = cc.to_c(cfg), ctypes.c_void_p()
    _lib.check(_lib.load().cq35_model_create(ctypes.byref(c), pointers, 1, ctypes.byref(handle)))
    borrowed, own = cq35.Model(handle.value, cfg), cq35.Model.from_arrays(cfg, weights)
    prompt = np.random.default_rng(2).integers(0, cfg["vocab"], 70).tolist()
    print("borrowed weights", flush=True)
    a, b = borrowed.session(70), own.session(70)
    (la, ta), (lb, tb) = a.step_raw(prompt), b.step_raw(prompt)
    assert ta == tb and np.array_equal(la, lb) and np.array_equal(a.export_state(0), b.export_state(0))
