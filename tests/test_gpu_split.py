"""GPU: wide rows of small batches, sampled by several workgroups each (ids only), against the kernel with
one workgroup per row (the same call asking for the write-back logits): the two use the same exact sums,
so every id is the same; and against the oracle. Sizes at the edges of the segments (4096 and 10240
entries), all option mixes, ties across segments, special rows, resident stores with generators, a
captured call (which keeps one workgroup per row) and streams of the caller's."""
import numpy as np
import pytest

from oracle import ref
from parity import compare_ids
from voxwerk_amd._lib import PARAMS_DTYPE
from voxwerk_amd.hip import DeviceArray, Event

pytestmark = pytest.mark.gpu


def options(rng, rows, vocab, **fixed):
    p = np.zeros(rows, dtype=PARAMS_DTYPE)
    p["do_sample"] = 1
    p["top_k"] = rng.choice([0, 0, 1, 50, 200, 256, 257, 1000, vocab], size=rows)
    p["top_p"] = rng.choice([1.0, 0.95, 0.8, 0.3, 1e-6], size=rows).astype(np.float32)
    p["temperature"] = rng.choice([0.7, 1.0, 1.3], size=rows).astype(np.float32)
    p["rep_penalty"] = rng.choice([1.0, 1.05, 1.1, 0.9], size=rows).astype(np.float32)
    supp = rng.random(rows) < 0.4
    p["supp_begin"], p["supp_end"] = np.where(supp, vocab - 1024, 0), np.where(supp, vocab, 0)
    p["keep_id"], p["ban_id"] = np.where(supp, vocab - 1024 + 102, -1), -1
    for k, v in fixed.items():
        p[k] = v
    return p


def check(ctx, x, p, u, off=None, hist=None, label=""):
    print(f"{label}: {x.shape}", flush=True)
    ids = ctx.sample(x, p, u, off, hist, raise_on_error=False)
    one, _, _ = ctx.sample(x, p, u, off, hist, want_logits=True, raise_on_error=False)
    bad = np.nonzero(ids != one)[0]
    assert not len(bad), f"{label}: rows {bad[:8]}: {ids[bad[:8]]} / {one[bad[:8]]} params {p[bad[:4]]}"
    rep = compare_ids(ids, ref.sample(x, p, u, off, hist, threads=8))
    assert not rep.unexplained, f"{label}: {rep}"
    return ids


@pytest.mark.parametrize("rows,vocab", [(24, 8193), (7, 12288), (24, 20481), (190, 9001), (24, 40960), (70, 61441),
                                        (13, 151936), (64, 151936), (136, 151935), (3, 524288)])
def test_split_option_mixes(ctx, rows, vocab):
    rng = np.random.default_rng(rows * 31 + vocab)
    x = (rng.standard_normal((rows, vocab), dtype=np.float32) * rng.choice([0.5, 2.0, 4.0], size=(rows, 1))).astype(np.float32)
    if rows >= 6:
        x[3] = np.round(x[3])            # many ties
        x[4] = np.round(x[4] * 16) / 16
        x[5, ::2] = -np.inf
    hl = rng.integers(0, 600, size=rows)
    off = np.concatenate([[0], np.cumsum(hl)]).astype(np.int32)
    hist = rng.integers(0, vocab, size=off[-1]).astype(np.int32)
    p = options(rng, rows, vocab)
    p["do_sample"][::6] = 0
    check(ctx, x, p, rng.random(rows), off, hist, label=f"mix {rows} x {vocab}")


@pytest.mark.parametrize("vocab", [10240, 33000, 151936])
def test_split_nucleus_ties_and_cuts(ctx, vocab):
    """Nucleus rows whose top-p cut falls among equal values (one value, two values, quantised logits),
    sorted rows either way, a row with one finite entry per segment, far outliers."""
    rng = np.random.default_rng(vocab)
    rows = 16
    x = rng.standard_normal((rows, vocab)).astype(np.float32)
    x[0] = 0.5
    x[1] = np.where(rng.random(vocab) < 0.5, 0.5, 0.25)
    x[2] = np.round(x[2] * 8) / 8
    x[3] = np.round(x[3] * 64) / 64
    x[4] = np.sort(x[4])
    x[5] = -np.sort(-x[5])
    x[6] = -np.inf
    x[6, ::4096] = 1.0
    x[7, 77] = 40.0
    x[8] *= 20
    x[9] = np.linspace(0, -1e-3, vocab)
    x[10, : vocab // 2] = -np.inf
    for top_p in (0.95, 0.5, 0.05, 1.0):
        for k in (0, 50, 256, 300, vocab // 3):
            p = options(rng, rows, vocab, top_p=np.float32(top_p), top_k=k, rep_penalty=np.float32(1.0), temperature=np.float32(1.0))
            for u in (rng.random(rows), np.full(rows, 0.0), np.full(rows, 1.0 - 2.0**-53)):
                check(ctx, x, p, u, label=f"ties V={vocab} p={top_p} k={k}")


def topk_us(ctx, x, k):
    """Device time of a call with this top-k, the best of several."""
    rows, vocab = x.shape
    p = np.zeros(rows, dtype=PARAMS_DTYPE)
    p["do_sample"], p["top_k"], p["top_p"], p["temperature"], p["rep_penalty"] = 1, k, np.float32(0.95), 1.0, 1.0
    p["keep_id"] = p["ban_id"] = -1
    d_x, d_p, d_u = DeviceArray.from_numpy(x), DeviceArray.from_numpy(p), DeviceArray.from_numpy(np.full(rows, 0.4))
    d_out, best = DeviceArray((rows,), np.int32), np.inf
    for _ in range(8):
        a, b = Event(), Event()
        a.record(ctx.stream())
        for _ in range(4):
            ctx.sample_device(rows, vocab, d_x, vocab, d_p, 1, d_u, d_out)
        b.record(ctx.stream())
        b.synchronize()
        best = min(best, 250 * a.elapsed_ms(b))
    return best


@pytest.mark.parametrize("rows,vocab", [(2, 20000), (16, 151936)])
def test_split_topk_near_256_stays_split(ctx, rows, vocab):
    """As k nears 256, the bound a segment gets from its 256 thread maxima lets more entries through than its
    list holds. It is raised then: a row sampled again by one workgroup takes ten times as long and more."""
    x = np.random.default_rng(vocab).standard_normal((rows, vocab)).astype(np.float32)
    us = {k: topk_us(ctx, x, k) for k in (128, 245, 250, 254, 256)}
    print(us, flush=True)
    assert max(us.values()) < 4 * us[128]


@pytest.mark.parametrize("vocab", [20000, 151936])
@pytest.mark.parametrize("k", [60, 250, 256])
def test_split_topk_bound_raised(ctx, vocab, k):
    """Rows whose segments get more entries than the list from the first bound: over every magnitude, of both
    signs, subnormal, with outliers, finite at few threads, large at few threads, tied."""
    rng = np.random.default_rng(vocab + k)
    x = rng.standard_normal((10, vocab))
    i = np.arange(vocab)
    x[1] = np.copysign(10.0 ** rng.uniform(-38, 38, vocab), x[1])
    x[2] *= 1e-40
    x[3, [5, vocab - 9]] = 2e38, -2e38
    x[4, i % 1024 >= 20] = -np.inf
    x[5, i % 1024 < 4 * k] += 30
    x[6] = np.round(x[6] * 16) / 16
    x[7] = np.where(rng.random(vocab) < 0.5, -1.0, -0.0)
    x[8] = -np.abs(x[8])
    x = x.astype(np.float32)
    p = options(rng, 10, vocab, top_k=k, top_p=np.float32(0.95), rep_penalty=np.float32(1.0), supp_begin=0, supp_end=0)
    for u in (rng.random(10), rng.random(10)):
        check(ctx, x, p, u, label=f"raised V={vocab} k={k}")


def test_split_special_rows(ctx):
    vocab, rows = 40000, 10
    x = np.full((rows, vocab), -1.0, np.float32)
    x[0] = -np.inf                      # all masked: V-1
    x[1] = 0.5
    x[2, 123] = np.nan                  # rejected
    x[3, [7, 39999]] = 3.0              # tied maxima
    x[4] = np.linspace(-5, 5, vocab)
    x[6, 30000] = np.inf                # rejected
    x[7, 39000] = np.nan                # greedy: rejected
    p = np.zeros(rows, dtype=PARAMS_DTYPE)
    p["do_sample"] = [1, 1, 1, 1, 1, 0, 1, 0, 1, 1]
    p["top_k"] = [0, 100, 0, 0, 0, 0, 50, 0, 0, 20]
    p["top_p"] = [0.9, 0.5, 1.0, 1e-7, 0.9, 0.9, 1.0, 1.0, -1.0, 0.9]
    p["temperature"], p["rep_penalty"], p["keep_id"], p["ban_id"] = 1.0, 1.1, -1, -1
    off = np.array([0, 2, 4, 6, 8, 10, 12, 14, 16, 18, 20], np.int32)
    hist = np.full(20, 5, np.int32)
    hist[17] = vocab                    # row 8: an id outside the vocabulary
    hist[19] = -1                       # row 9, top-k
    ids = check(ctx, x, p, np.linspace(0.05, 0.95, rows), off, hist, label="special")
    assert ids[0] == vocab - 1 and ids[2] == -3 and ids[3] == 39999 and ids[6] == -3 and ids[7] == -3
    assert ids[8] == -2 and ids[9] == -2


@pytest.mark.parametrize("top_k,top_p,do_sample", [(50, 1.0, 1), (0, 0.9, 1), (300, 0.9, 1), (0, 1.0, 0)])
def test_split_reads_no_history_without_a_penalty(ctx, top_k, top_p, do_sample):
    """Device calls whose rows have the penalty off and whose offsets were never filled (they point far past
    the ids): nothing of the history is read, the ids are those of the call without one."""
    rng = np.random.default_rng(top_k)
    rows, vocab = 5, 30000
    x = rng.standard_normal((rows, vocab)).astype(np.float32)
    p = options(rng, rows, vocab, top_k=top_k, top_p=np.float32(top_p), do_sample=do_sample, rep_penalty=np.float32(1.0))
    d_x, d_p, d_u = DeviceArray.from_numpy(x), DeviceArray.from_numpy(p), DeviceArray.from_numpy(rng.random(rows))
    off = (np.arange(rows + 1) * 4096 + (1 << 30)).astype(np.int32)
    d_off, d_ids, d_out = DeviceArray.from_numpy(off), DeviceArray.from_numpy(np.zeros(4, np.int32)), DeviceArray((rows,), np.int32)
    ctx.sample_device(rows, vocab, d_x, vocab, d_p, 1, d_u, d_out)
    ctx.synchronize()
    want = d_out.numpy().copy()
    ctx.sample_device(rows, vocab, d_x, vocab, d_p, 1, d_u, d_out, d_off, d_ids)
    ctx.synchronize()
    assert np.array_equal(d_out.numpy(), want)


def test_split_resident_store_with_generators(ctx):
    """Stages over a resident store: ids, appended histories and device generators as the calls with one
    row at a time's worth of host state give them."""
    from voxwerk_amd.sampler import DotNetRandom

    rng = np.random.default_rng(8)
    rows, vocab, steps = 6, 30000, 4
    store = ctx.history(rows, 64)
    gens, hists = [DotNetRandom(100 + r) for r in range(rows)], [list(rng.integers(0, vocab, 5)) for _ in range(rows)]
    for r in range(rows):
        store.set(r, np.array(hists[r], np.int32))
        store.seed(r, 100 + r)
    p = options(rng, rows, vocab, rep_penalty=np.float32(1.2), temperature=np.float32(1.0))
    p["top_k"], p["top_p"] = [0, 0, 50, 300, 0, 0], np.float32([0.9, 1.0, 0.9, 0.9, 0.9, 0.9])
    p["do_sample"] = [1, 1, 1, 1, 0, 1]
    for _ in range(steps):
        x = (rng.standard_normal((rows, vocab)) * 2).astype(np.float32)
        ids = ctx.sample_batch(store, x, np.arange(rows), p, None, append=True, rng="talker")
        u = np.array([gens[r].NextDouble() if p["do_sample"][r] else 0.0 for r in range(rows)])
        off = np.concatenate([[0], np.cumsum([len(h) for h in hists])]).astype(np.int32)
        one, _, _ = ctx.sample(x, p, u, off, np.concatenate(hists).astype(np.int32), want_logits=True)
        assert np.array_equal(ids, one)
        for r in range(rows):
            hists[r].append(int(ids[r]))
            assert list(store.get(r)) == hists[r]
    store.close()


@pytest.mark.parametrize("ticks", [0, 30, 100, 300, 1000])
def test_split_meetings_given_up(ticks):
    """Workgroups that wait for each other for too short a time (10 ns a tick; none at all at 0) give the row
    up at one meeting or another, and one samples it alone: the same ids, histories and generators; and the
    workspace, with normal waits again, serves the next call."""
    from voxwerk_amd.sampler import Context

    rng = np.random.default_rng(ticks)
    rows, vocab = 24, 70000
    p = options(rng, rows, vocab, temperature=np.float32(1.0))
    p["top_k"], p["top_p"] = [0, 0, 300, 40000, 0, 50] * 4, np.float32([0.9, 1.0, 0.9, 1.0, 0.3, 0.9] * 4)
    hists = [rng.integers(0, vocab, 5).astype(np.int32) for _ in range(rows)]
    logits = [(rng.standard_normal((rows, vocab)) * 2).astype(np.float32) for _ in range(3)]
    out = []
    for wait in (ticks, 50000):
        with Context(0) as c:
            store = c.history(rows, 64)
            for r in range(rows):
                store.set(r, hists[r])
                store.seed(r, 100 + r)
            ids = []
            for x in logits:
                for w in (wait, 50000):
                    assert c._lib.vxs_set_split_wait(c.handle, w) == 0
                    ids.append(c.sample_batch(store, x, np.arange(rows), p, None, append=True, rng="talker"))
            if wait == 0:  # the path is taken: one workgroup per row takes many times as long
                d = [DeviceArray.from_numpy(v) for v in (logits[0], p)] + [DeviceArray((rows,), np.int32)]
                us = []
                for w in (0, 50000):
                    c._lib.vxs_set_split_wait(c.handle, w)
                    a, b = Event(), Event()
                    a.record(c.stream())
                    for _ in range(4):
                        c.sample_device(rows, vocab, d[0], vocab, d[1], 1, None, d[2])
                    b.record(c.stream())
                    b.synchronize()
                    us.append(250 * a.elapsed_ms(b))
                print(us, flush=True)
                assert us[0] > 3 * us[1]
            out.append((np.array(ids), [list(store.get(r)) for r in range(rows)], [list(store.draw(r, "talker", 3)) for r in range(rows)]))
            store.close()
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]


def test_split_on_callers_streams_and_in_a_graph():
    import os
    import subprocess
    import sys

    script = os.path.join(os.path.dirname(__file__), "split_streams.py")
    p = subprocess.run([sys.executable, "-u", script], timeout=100, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    print(p.stdout, flush=True)
    assert p.returncode == 0, p.stdout[-2000:]
