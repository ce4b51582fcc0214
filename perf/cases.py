"""The work a user of the sampler has it do, as cases that can be timed and checked.

A case is a dict of plain values. Its ``kind`` says which public calls one pass makes:

``host``    ``Context.sample`` on host arrays, ``calls`` times in a row (a single talker step, the
            fifteen dependent code-predictor steps of a frame); synchronous, ids back on the host.
``sample``  ``Context.sample_device`` on rows already on the GPU: one sampling stage of a batch.
``head``    ``Context.head_device`` / ``head_int8_device``, ``heads`` weights in a row: logits from
            hidden rows, for one sequence up to a large batch.
``step``    one batched generation step on the device: talker head, sampler over resident histories
            with the slots' own generators, fifteen code-predictor heads and samplers, embedding.
``embed``   ``Context.frame_embed_device``: the next talker input of every sequence of a batch.

Shapes come from the workloads of ``voxwerk_amd/workloads.py`` and ``bench.py``: the talker's 3072
codes, the code predictor's 2048, hidden size 1024, a wide vocabulary of 151936.
"""
from __future__ import annotations

import math

import numpy as np
import torch  # before the library, which then binds to the same HIP runtime

from voxwerk_amd._lib import PARAMS_DTYPE
from voxwerk_amd.sampler import Context

TALKER_VOCAB, CP_VOCAB, EOS_ID, WIDE_VOCAB = 3072, 2048, 2150, 151936
GROUPS, HIDDEN = 16, 1024
MAX_ENTRIES = 1024 * WIDE_VOCAB      # logits of the largest sampling stage
MAX_PRODUCTS = 4096 * 1024 * 3072    # multiply-adds of the largest drawn head
STEP_SLOT_SETS, STEP_CAP = 8, 65536


def listed():
    talker = {"top_k": 50, "top_p": 1.0, "temperature": 0.9, "penalty": 1.05}
    return [
        # one sequence: a talker step called from host code, where latency is all
        {"name": "talker_step_host", "kind": "host", "calls": 1, "rows": 1, "vocab": 3072, "hist": 256,
         "suppress": False, "logits": "normal", "write_back": False, **talker},
        # the fifteen dependent code-predictor steps of one frame of a small batch, from host code
        {"name": "code_predictor_frame_host", "kind": "host", "calls": 15, "rows": 16, "vocab": 2048, "hist": 0,
         "suppress": False, "logits": "normal", "write_back": False, **dict(talker, penalty=1.0)},
        # a batched talker stage late in long sequences
        {"name": "batched_talker", "kind": "sample", "rows": 256, "vocab": 3072, "hist": 2048, "ragged": False,
         "per_row": True, "suppress": True, "logits": "normal", "write_back": False, **dict(talker, top_p=0.9)},
        # serving scale, full-vocabulary nucleus sampling
        {"name": "full_vocab_nucleus", "kind": "sample", "rows": 4096, "vocab": 3072, "hist": 512, "ragged": False,
         "per_row": False, "suppress": False, "logits": "mixture", "write_back": False, "top_k": 0, "top_p": 0.95,
         "temperature": 1.0, "penalty": 1.1},
        # serving scale, the talker's own options
        {"name": "talker_topk", "kind": "sample", "rows": 4096, "vocab": 3072, "hist": 256, "ragged": False,
         "per_row": False, "suppress": True, "logits": "normal", "write_back": False, **dict(talker, top_p=0.95)},
        # a wide (text model) vocabulary at serving scale
        {"name": "wide_vocab", "kind": "sample", "rows": 1024, "vocab": WIDE_VOCAB, "hist": 4096, "ragged": False,
         "per_row": False, "suppress": True, "logits": "zipf", "write_back": False, "top_k": 200, "top_p": 0.8,
         "temperature": 0.7, "penalty": 1.05},
        # the same vocabulary for the few sequences of an ordinary decode step
        {"name": "wide_few_rows", "kind": "sample", "rows": 16, "vocab": WIDE_VOCAB, "hist": 1024, "ragged": True,
         "per_row": True, "suppress": False, "logits": "zipf", "write_back": False, "top_k": 50, "top_p": 0.95,
         "temperature": 0.7, "penalty": 1.05},
        # nucleus sampling without a top-k over the wide vocabulary, a medium batch
        {"name": "wide_nucleus", "kind": "sample", "rows": 64, "vocab": WIDE_VOCAB, "hist": 1024, "ragged": True,
         "per_row": True, "suppress": False, "logits": "zipf", "write_back": False, "top_k": 0, "top_p": 0.95,
         "temperature": 1.0, "penalty": 1.05},
        # the sixteen int8 heads of one frame of a single sequence
        {"name": "int8_heads_frame", "kind": "head", "format": "int8", "heads": 16, "rows": 1, "k": 1024, "n": 2048},
        # the talker head that feeds the batched talker stage
        {"name": "codec_head_batch", "kind": "head", "format": "bf16", "heads": 1, "rows": 256, "k": 1024, "n": 3072},
        # a whole generation step of a medium batch, everything on the device
        {"name": "device_step", "kind": "step", "rows": 24},
        # the next talker inputs of a large batch
        {"name": "frame_embedding", "kind": "embed", "rows": 4096, "groups": GROUPS, "hidden": HIDDEN},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_options(rng, vocab):
    return {
        "top_k": rng.choice([0, 1, 20, 50, 64, 100, 200, min(400, vocab - 1)]),
        "top_p": rng.choice([1.0, 0.95, 0.9, 0.8]),
        "temperature": rng.choice([0.7, 0.9, 1.0, 1.2]),
        "penalty": rng.choice([1.0, 1.05, 1.1]),
    }


def draw(rng):
    kind = rng.choice(["host", "sample", "sample", "sample", "head", "head", "step", "embed"])
    if kind == "host":
        vocab = rng.choice([CP_VOCAB, TALKER_VOCAB, _log_int(rng, 500, 8192)])
        return {"kind": kind, "calls": rng.choice([1, 1, 4]), "rows": _log_int(rng, 1, 64), "vocab": vocab,
                "hist": _log_int(rng, 1, 2048), "suppress": rng.random() < 0.5, "logits": "normal",
                "write_back": rng.random() < 0.3, **_draw_options(rng, vocab)}
    if kind == "sample":
        vocab = rng.choice([CP_VOCAB, TALKER_VOCAB, WIDE_VOCAB, _log_int(rng, 1000, WIDE_VOCAB)])
        return {"kind": kind, "rows": _log_int(rng, 1, min(4096, MAX_ENTRIES // vocab)), "vocab": vocab,
                "hist": _log_int(rng, 1, 4096), "ragged": rng.random() < 0.5, "per_row": rng.random() < 0.5,
                "suppress": rng.random() < 0.3, "logits": "zipf" if vocab > 8192 else rng.choice(["normal", "mixture"]),
                "write_back": rng.random() < 0.15, **_draw_options(rng, vocab)}
    if kind == "head":
        k, n = 8 * _log_int(rng, 32, 256), rng.choice([CP_VOCAB, TALKER_VOCAB, _log_int(rng, 500, 4096)])
        return {"kind": kind, "format": rng.choice(["bf16", "bf16", "int8"]), "heads": 1,
                "rows": _log_int(rng, 1, min(4096, MAX_PRODUCTS // (k * n))), "k": k, "n": n}
    if kind == "step":
        return {"kind": kind, "rows": _log_int(rng, 1, 128)}
    return {"kind": kind, "rows": _log_int(rng, 16, 4096), "groups": GROUPS, "hidden": rng.choice([1024, 1024, 2048])}


# ---- inputs -----------------------------------------------------------------------------------

_context = None


def _ctx():
    """The one context a program keeps (its stream and staging)."""
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def _params(case, n):
    p = np.zeros(n, dtype=PARAMS_DTYPE)
    p["do_sample"], p["top_k"], p["top_p"] = 1, case["top_k"], np.float32(case["top_p"])
    p["temperature"], p["rep_penalty"] = np.float32(case["temperature"]), np.float32(case["penalty"])
    p["keep_id"] = p["ban_id"] = -1
    if case["suppress"]:  # special tokens: the last 1024 ids, but for EOS
        p["supp_begin"], p["supp_end"], p["keep_id"] = _special(case), case["vocab"], _eos(case)
    return p


def _special(case):
    return case["vocab"] - min(1024, case["vocab"] // 3)


def _eos(case):
    return min(_special(case) + EOS_ID - 2048, case["vocab"] - 1)


def _logits(case, rows, g):
    """Normal logits (talker and code predictor), a 90/10 mixture of two levels, or Zipf-distributed
    ranks with noise (a text vocabulary)."""
    shape, dev = (rows, case["vocab"]), g.device
    if case["logits"] == "normal":
        return torch.randn(shape, generator=g, device=dev) * 3.0
    if case["logits"] == "mixture":
        high = torch.rand(shape, generator=g, device=dev) < 0.1
        return torch.randn(shape, generator=g, device=dev).add_(high, alpha=4.0)
    rank = torch.rand(shape, generator=g, device=dev).mul_(case["vocab"]).add_(1.0).floor_()
    return torch.randn(shape, generator=g, device=dev).mul_(0.5).sub_(rank.log_(), alpha=1.1)


def _histories(case, rows, g):
    top = _special(case) if case["suppress"] else case["vocab"]
    lens = torch.full((rows,), case["hist"], dtype=torch.int64)
    if case.get("ragged"):
        lens = torch.randint(case["hist"] // 2, case["hist"] + 1, (rows,), generator=g, device=g.device).cpu()
    off = torch.zeros(rows + 1, dtype=torch.int32)
    off[1:] = torch.cumsum(lens, 0)
    ids = torch.randint(0, top, (int(off[-1]),), generator=g, device=g.device, dtype=torch.int32)
    return off, ids


def _bf16_weight(n, k, scale, g):
    return (torch.randn((n, k), generator=g, device=g.device) * scale).to(torch.bfloat16)


def _sampling_inputs(case, seed, device):
    g = torch.Generator(device=device).manual_seed(seed)
    calls = [_logits(case, case["rows"], g) for _ in range(case.get("calls", 1))]
    off, ids = _histories(case, case["rows"], g)
    u = torch.rand(case["rows"], generator=g, device=device, dtype=torch.float64)
    return calls, off, ids, u


def _head_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn((case["rows"], case["k"]), generator=g, device="cuda")
    return x, [_bf16_weight(case["n"], case["k"], 0.05, g) for _ in range(case["heads"])]


def prepare(case, seed):
    kind, rows = case["kind"], case["rows"]
    s = {"case": case, "ctx": _ctx()}
    if kind == "host":
        calls, off, ids, u = _sampling_inputs(case, seed, "cpu")
        s.update(logits=[c.numpy() for c in calls], u=u.numpy(), params=_params(case, rows), off=None, ids=None, out=None)
        if case["hist"]:
            s.update(off=off.numpy(), ids=ids.numpy())
        if case["write_back"]:
            s["out"] = [np.empty((rows, case["vocab"]), np.float32) for _ in calls]
    elif kind == "sample":
        (x,), off, ids, u = _sampling_inputs(case, seed, "cuda")
        params = _params(case, rows if case["per_row"] else 1)
        s.update(logits=x, off=off.cuda(), ids=ids, u=u, params=torch.from_numpy(params.view(np.uint8).copy()).cuda(),
                 out=torch.empty(rows, dtype=torch.int32, device="cuda"),
                 wb=torch.empty_like(x) if case["write_back"] else None)
    elif kind == "head":
        x, w = _head_inputs(case, seed)
        s.update(x=x, w=w, out=torch.empty((case["heads"], rows, case["n"]), device="cuda"))
        if case["format"] == "int8":
            s["q"] = [torch.empty((case["n"], case["k"]), dtype=torch.int8, device="cuda") for _ in w]
            s["scale"] = [torch.empty(case["n"], device="cuda") for _ in w]
            torch.cuda.synchronize()
            for a, q, sc in zip(w, s["q"], s["scale"]):
                s["ctx"].head_pack_int8_device(case["k"], case["n"], a, case["k"], q, case["k"], sc)
            s["ctx"].synchronize()
            s["w"] = None
    elif kind == "step":
        s.update(_step_state(rows, seed))
    else:
        g = torch.Generator(device="cuda").manual_seed(seed)
        s.update(_tables(case["hidden"], g))
        codes = [torch.randint(0, TALKER_VOCAB if i == 0 else CP_VOCAB, (rows, 1), generator=g, device="cuda")
                 for i in range(case["groups"])]
        s.update(codes=torch.cat(codes, 1).to(torch.int32), text=torch.randn((rows, case["hidden"]), generator=g, device="cuda"),
                 out=torch.empty((rows, case["hidden"]), device="cuda"),
                 status=torch.empty(rows, dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    return s


def _tables(hidden, g):
    return {"codec": _bf16_weight(TALKER_VOCAB, hidden, 1.0, g),
            "cp": _bf16_weight((GROUPS - 1) * CP_VOCAB, hidden, 1.0, g)}


def _step_state(rows, seed):
    """The state of a serving loop: the weights, the batch's resident histories (256 ids each) and
    generators. Successive passes advance successive sets of sequences of the one store."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    talker = {"vocab": TALKER_VOCAB, "top_k": 50, "top_p": 1.0, "temperature": 0.9, "penalty": 1.05, "suppress": True}
    sub = dict(talker, vocab=CP_VOCAB, penalty=1.0, suppress=False)
    n = STEP_SLOT_SETS * rows
    store = _ctx().history(n, STEP_CAP)
    r = np.random.default_rng(seed)
    for slot in range(n):
        store.set(slot, r.integers(0, 2048, 256))
        store.seed(slot, int(r.integers(0, 2**31)))
    sets = torch.arange(n, dtype=torch.int32, device="cuda").reshape(STEP_SLOT_SETS, rows)
    return {
        "x": torch.randn((rows, HIDDEN), generator=g, device="cuda"),
        "wt": _bf16_weight(TALKER_VOCAB, HIDDEN, 0.1, g),
        "wc": [_bf16_weight(CP_VOCAB, HIDDEN, 0.1, g) for _ in range(GROUPS - 1)],
        **_tables(HIDDEN, g),
        "store": store, "sets": [sets[i] for i in range(STEP_SLOT_SETS)], "turn": 0,
        "pt": torch.from_numpy(_params(talker, rows).view(np.uint8).copy()).cuda(),
        "pc": torch.from_numpy(_params(sub, rows).view(np.uint8).copy()).cuda(),
        "text": torch.randn((rows, HIDDEN), generator=g, device="cuda"),
        "lt": torch.empty((rows, TALKER_VOCAB), device="cuda"),
        "lc": torch.empty((GROUPS - 1, rows, CP_VOCAB), device="cuda"),
        "codes": torch.empty((GROUPS, rows), dtype=torch.int32, device="cuda"),
        "out": torch.empty((rows, HIDDEN), device="cuda"),
        "status": torch.empty(rows, dtype=torch.int32, device="cuda"),
    }


# ---- one pass ---------------------------------------------------------------------------------


def run(s):
    case, ctx, kind = s["case"], s["ctx"], s["case"]["kind"]
    rows = case["rows"]
    if kind == "host":
        if not case["write_back"]:
            return [ctx.sample(x, s["params"], s["u"], s["off"], s["ids"]) for x in s["logits"]]
        return [ctx.sample(x, s["params"], s["u"], s["off"], s["ids"], logits_out=o)[:2] for x, o in zip(s["logits"], s["out"])]
    if kind == "sample":
        ctx.sample_device(rows, case["vocab"], s["logits"], case["vocab"], s["params"], 1 if case["per_row"] else 0,
                          s["u"], s["out"], s["off"], s["ids"], out_logits=s["wb"])
        return {"ids": s["out"], "logits": s["wb"]}
    if kind == "head":
        k, n = case["k"], case["n"]
        for i in range(case["heads"]):
            if case["format"] == "int8":
                ctx.head_int8_device(rows, k, n, s["x"], k, s["q"][i], k, s["scale"][i], s["out"][i], n)
            else:
                ctx.head_device(rows, k, n, s["x"], k, s["w"][i], k, s["out"][i], n)
        return s["out"]
    if kind == "step":
        slots = s["sets"][s["turn"]]
        s["turn"] = (s["turn"] + 1) % STEP_SLOT_SETS
        ctx.head_device(rows, HIDDEN, TALKER_VOCAB, s["x"], HIDDEN, s["wt"], HIDDEN, s["lt"], TALKER_VOCAB)
        ctx.sample_batch_device(s["store"], rows, TALKER_VOCAB, s["lt"], TALKER_VOCAB, slots, s["pt"], 1, None,
                                s["codes"][0], append=True, rng="talker")
        for g in range(1, GROUPS):
            ctx.head_device(rows, HIDDEN, CP_VOCAB, s["x"], HIDDEN, s["wc"][g - 1], HIDDEN, s["lc"][g - 1], CP_VOCAB)
            ctx.sample_batch_device(s["store"], rows, CP_VOCAB, s["lc"][g - 1], CP_VOCAB, slots, s["pc"], 1, None,
                                    s["codes"][g], append=False, rng="sub")
        ctx.frame_embed_device(rows, GROUPS, HIDDEN, s["codes"], 1, s["codec"], TALKER_VOCAB, s["cp"], CP_VOCAB,
                               s["out"], HIDDEN, s["status"], addend=s["text"], ld_addend=HIDDEN, group_stride=rows)
        return {"talker_logits": s["lt"], "cp_logits": s["lc"], "codes": s["codes"], "embedding": s["out"]}
    ctx.frame_embed_device(rows, case["groups"], case["hidden"], s["codes"], case["groups"], s["codec"], TALKER_VOCAB,
                           s["cp"], CP_VOCAB, s["out"], case["hidden"], s["status"], addend=s["text"],
                           ld_addend=case["hidden"])
    return {"embedding": s["out"], "status": s["status"]}


# ---- what a pass cannot do without, and how exact it is ------------------------------------------


def _head_work(rows, k, n, int8):
    return {"bytes": n * k * (1 if int8 else 2) + (4 * n if int8 else 0) + 4 * rows * (k + n), "flops": 2 * rows * k * n}


def _embed_work(rows, groups, hidden):
    return {"bytes": rows * (2 * groups * hidden + 8 * hidden + 4 * groups + 4), "flops": rows * groups * hidden}


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind in ("host", "sample"):
        hist = case["hist"] * (0.75 if case.get("ragged") else 1.0)
        params = 36.0 if case.get("per_row", True) else 0.0
        per_row = 4 * case["vocab"] * (2 if case["write_back"] else 1) + 4 * hist + 4 + 8 + 4 + params
        return {"bytes": case.get("calls", 1) * rows * per_row, "flops": 0}
    if kind == "head":
        w = _head_work(rows, case["k"], case["n"], case["format"] == "int8")
        return {name: case["heads"] * v for name, v in w.items()}
    if kind == "embed":
        return _embed_work(rows, case["groups"], case["hidden"])
    parts = [_head_work(rows, HIDDEN, TALKER_VOCAB, False), _embed_work(rows, GROUPS, HIDDEN)]
    parts += [_head_work(rows, HIDDEN, CP_VOCAB, False)] * (GROUPS - 1)
    ids = rows * (4 * TALKER_VOCAB + 4 * 256 + (GROUPS - 1) * 4 * CP_VOCAB)
    return {"bytes": sum(p["bytes"] for p in parts) + ids, "flops": sum(p["flops"] for p in parts)}


def tolerance(case):
    """Ids: the rule of the sampler decides them, so another correct implementation gives the same but
    where a uniform or the top-p cut lies within the rounding of a 32-bit exponential (1e-6 of the
    mass): about one row in a million. Write-back logits and embeddings: the same operations in the
    same order. Heads: 32-bit products and sums in another order (measured 1.0e-7 to 1.2e-7 against
    64 bits; the worst of some million entries lies about five times further out)."""
    if case["kind"] == "embed":
        return "exact"
    if case["kind"] in ("host", "sample"):
        return {"rel": 0.0, "max": 0.0, "differ": 1e-3}
    return {"rel": 5e-7, "max": 4e-6, "differ": 1e-3}


# ---- the same in 64 bits, in plain torch ---------------------------------------------------------


def _exact_sample(case, x, off, ids, u):
    """The sampling rule row by row: penalty, suppression, temperature and top-k as 32-bit values (they
    are defined so), probabilities and running sums in 64 bits."""
    rows, vocab = x.shape
    p = _params(case, 1)[0]
    x = x.clone()
    seen = torch.zeros((rows, vocab), dtype=torch.bool, device=x.device)
    row_of = torch.repeat_interleave(torch.arange(rows, device=x.device), (off[1:] - off[:-1]).to(x.device))
    seen[row_of, ids.long()] = True
    rho = float(p["rep_penalty"])
    if rho != 1.0:
        pen = torch.where(x < 0, x.double() * rho, x.double() / rho).float()
        x = torch.where(seen, pen, x)
    if case["suppress"]:
        keep = x[:, _eos(case)].clone()
        x[:, int(p["supp_begin"]):int(p["supp_end"])] = -math.inf
        x[:, _eos(case)] = keep
    x = x * float(np.float32(1.0) / p["temperature"])
    k = int(p["top_k"])
    if 0 < k < vocab:
        kth = torch.topk(x, k, dim=1).values[:, -1:]
        x = torch.where(x < kth, torch.full_like(x, -math.inf), x)
    prob = torch.exp((x - x.max(1, keepdim=True).values).double())
    prob /= prob.sum(1, keepdim=True)
    if p["top_p"] < 1.0:
        thr = float(np.float32(1.0) - p["top_p"])
        order = torch.sort(prob, dim=1, stable=True)
        cut = torch.cumsum(order.values, 1) <= thr
        cut[:, -1] = False
        prob.scatter_(1, order.indices, torch.where(cut, torch.zeros_like(prob), order.values))
        prob /= prob.sum(1, keepdim=True)
    hit = (torch.cumsum(prob, 1) > u[:, None]) & (prob > 0)
    last = vocab - 1 - (prob > 0).to(torch.int8).flip(1).argmax(1)
    out = torch.where(hit.any(1), hit.to(torch.int8).argmax(1), last).to(torch.int32)
    return out, x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "sample"):
        calls, off, ids, u = _sampling_inputs(case, seed, "cpu" if kind == "host" else "cuda")
        got = []
        for x in calls:
            if not case["hist"]:
                off, ids = off * 0, ids[:0]
            step = max(1, (1 << 24) // case["vocab"])  # rows at a time
            parts = [_exact_sample(case, x[r:r + step], off[r:r + step + 1], ids[int(off[r]):int(off[min(r + step, len(x))])],
                                   u[r:r + step]) for r in range(0, len(x), step)]
            o = torch.cat([a for a, _ in parts])
            got.append([o, torch.cat([b for _, b in parts])] if case["write_back"] else o)
        if kind == "host":
            return got
        return {"ids": got[0][0], "logits": got[0][1]} if case["write_back"] else {"ids": got[0], "logits": None}
    if kind == "head":
        x, w = _head_inputs(case, seed)
        out = []
        for a in w:
            a = a.double()
            if case["format"] == "int8":
                # symmetric per-output scales as the packing defines them: each step rounded to 32 bits
                top = a.abs().amax(1)
                scale = torch.where(top > 0, (top / 127.0).float().double(), torch.ones_like(top))
                inv = (1.0 / scale).float().double()
                a = torch.round((a * inv[:, None]).float()).clamp_(-127, 127).double() * scale[:, None]
            out.append(x.double() @ a.t().contiguous())
        return torch.stack(out)
    if kind == "step":
        s = _step_state(case["rows"], seed)
        x = s["x"].double()
        s["store"].close()
        return {"talker_logits": x @ s["wt"].double().t().contiguous(),
                "cp_logits": torch.stack([x @ w.double().t().contiguous() for w in s["wc"]]), "codes": None, "embedding": None}
    s = prepare(case, seed)
    out, codes = s["text"].double(), s["codes"].long()
    for i in range(case["groups"]):
        table = s["codec"] if i == 0 else s["cp"][(i - 1) * CP_VOCAB:i * CP_VOCAB]
        out = out + table[codes[:, i]].double()
    return {"embedding": out, "status": torch.zeros_like(s["status"])}
