"""GPU: the head's matrix-core forms at the edges of their tiles and of the rule that picks them (split-K
tiles of 16 x 16 up to 32 x 96, tiled 32 x 64 and 64 x 128; partial last tiles in rows, outputs and k,
padded leading dimensions, unaligned output rows), bf16 and int8, within gamma_K sum |x w| of the
exact product, the bound of any fp32 order; and infinities and NaN in hidden rows and weights as IEEE
products and sums give them."""
import numpy as np
import pytest

from oracle.head_np import head_bound, head_exact, head_int8_bound, head_int8_exact, pack_int8
from test_gpu_head import _bf16, _run, _run_int8
from voxwerk_amd.hip import DeviceArray, Event

pytestmark = pytest.mark.gpu

# rows, k, n, pad: the form the rule takes
SHAPES = [(4, 8, 7, 0), (3, 1032, 40, 8), (16, 1024, 4096, 0), (15, 72, 1001, 8),   # split-K 16 x 16
          (17, 1024, 4095, 8), (33, 520, 2048, 0),                                  # 16 x 32
          (64, 1024, 3072, 0), (49, 136, 2993, 16),                                 # 16 x 48
          (128, 1024, 3072, 0), (65, 448, 4033, 8),                                 # 32 x 48
          (250, 1016, 2047, 0), (256, 512, 3072, 8),                                # 32 x 64, 32 x 96
          (255, 504, 3071, 0), (700, 136, 2049, 8), (513, 2048, 700, 0),            # tiled 32 x 64
          (1100, 264, 3001, 8), (2048, 64, 1601, 0)]                                # tiled 64 x 128


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("rows,k,n,pad", SHAPES)
def test_head_tiles_within_bound(ctx, rows, k, n, pad, int8):
    rng = np.random.default_rng(rows * 7919 + k * 31 + n)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    w = _bf16(rng.standard_normal((n, k)) * 0.05)
    if int8:
        q, scale = pack_int8(w)
        got = _run_int8(ctx, x, q, scale, ldx=k + pad, ldq=k + pad, ldo=n + pad // 8)
        exact, bound = head_int8_exact(x, q, scale), head_int8_bound(x, q, scale)
    else:
        got = _run(ctx, x, w, ldx=k + pad, ldw=k + pad, ldo=n + pad // 8)
        exact, bound = head_exact(x, w), head_bound(x, w)
    err = np.abs(got - exact)
    assert np.all(err <= bound), f"max err/bound {np.max(err / bound):.3f}"


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("rows,k,n", [(5, 1024, 600), (256, 512, 3072), (400, 72, 2050), (1100, 264, 3001)])
def test_head_tiles_nonfinite(ctx, rows, k, n, int8):
    """A hidden row with +inf, one with NaN, one with both infinities; a weight row with -inf, one with
    NaN (bf16), one with zeros where the infinities meet it (0 * inf = NaN)."""
    rng = np.random.default_rng(rows + k)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    wf = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    x[0, 3], x[rows - 1, k - 1], x[2, 5], x[2, 6] = np.inf, np.nan, np.inf, -np.inf
    wf[4, 3] = 0.0
    if int8:
        q, scale = pack_int8(_bf16(wf))
        got, wd = _run_int8(ctx, x, q, scale), q * scale[:, None]
    else:
        wf[1, 9], wf[n - 1, k - 2] = -np.inf, np.nan
        got, wd = _run(ctx, x, _bf16(wf)), (_bf16(wf).astype(np.uint32) << 16).view(np.float32)
    with np.errstate(invalid="ignore"):  # elementwise products and a plain sum, no library shortcuts
        for r in (0, 1, 2, rows - 1):
            want = (x[r].astype(np.float64) * wd.astype(np.float64)).sum(axis=1)
            for cls in (np.isnan, np.isposinf, np.isneginf):
                assert np.array_equal(cls(got[r]), cls(want)), (r, cls)
        for c in (1, 4, n - 1):
            want = (x.astype(np.float64) * wd[c].astype(np.float64)).sum(axis=1)
            for cls in (np.isnan, np.isposinf, np.isneginf):
                assert np.array_equal(cls(got[:, c]), cls(want)), (c, cls)


def head_us(ctx, x, n):
    rows, k = x.shape
    w = _bf16(np.random.default_rng(n).standard_normal((n, k)) * 0.05)
    d_x, d_w, d_o = DeviceArray.from_numpy(x), DeviceArray.from_numpy(w), DeviceArray((rows, n), np.float32)
    best = np.inf
    for _ in range(8):
        a, b = Event(), Event()
        a.record(ctx.stream())
        for _ in range(4):
            ctx.head_device(rows, k, n, d_x, k, d_w, k, d_o, n)
        b.record(ctx.stream())
        b.synchronize()
        best = min(best, 250 * a.elapsed_ms(b))
    return best


@pytest.mark.parametrize("rows,k,n", [(24, 1024, 2048), (256, 1024, 3072), (4096, 1024, 3072)])
def test_head_nonfinite_rows_cost_little(ctx, rows, k, n):
    """One hidden row of NaN (a finished sequence's slot, say) or with an infinity, and NaN in every row,
    against the finite call."""
    x = np.random.default_rng(rows).standard_normal((rows, k)).astype(np.float32)
    us = {"finite": head_us(ctx, x, n)}
    for name, r, c, v in (("NaN row", rows // 2, slice(None), np.nan), ("one NaN", rows // 2, k - 1, np.nan),
                          ("one inf", rows // 2, 7, np.inf), ("all rows", slice(None), k - 1, np.nan)):
        bad = x.copy()
        bad[r, c] = v
        us[name] = head_us(ctx, bad, n)
    print(us, flush=True)
    assert max(us.values()) < 2 * us["finite"] + 10
