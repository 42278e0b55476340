"""The work that a program has the hot path do, as cases to measure.

Five kinds of call, each through the public entry points of kvmem_amd.api:

  step      a decode step of every layer: scoring, selection, stage plan and
            attention over the window (steady state: the plan is empty)
  attend    decode / verify attention over a window, without retrieval
  prefill   attention of a prompt chunk over the window and its own cells
  ingest    what comes with a chunk's or a step's new tokens: query sums,
            mean-K upkeep, K / V rows quantised and written into the window
  retrieve  a retrieval whose selection changes: scoring, selection and the
            stage-in of the blocks that moved or are new

Sizes are the framework's own (24 query heads on 4 kv heads of 256 dims, 8 on 2
of 128, 128-token blocks, 32,768-cell windows, histories to 262,144 tokens)
and generic ones between them.  Values are N(0, 1) before quantisation, as the
benchmark's; a query is close to the blocks it should retrieve.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kvmem-llama.cpp_amd"))
from kvmem_amd import _lib as L, api  # noqa: E402

BT = 128                                  # tokens per block
N_ROT, FREQ_BASE = 64, 1e7
TYPES = {"q8_0": (L.T_Q8_0, L.T_Q4_0), "q4_0": (L.T_Q4_0, L.T_Q4_0), "f16": (L.T_F16, L.T_F16)}
BLOCK = {"q8_0": (34, 18), "q4_0": (18, 18), "f16": (64, 64)}     # bytes of 32 K / V values

_state = None


def _st():
    """The program's execution state: one for the process."""
    global _state
    if _state is None:
        _state = api.State(0)
    return _state


# ---- the cases -----------------------------------------------------------------
def _case(name, kind, **kw):
    c = {"kind": kind, "head_dim": 256, "kv_heads": 4, "group": 6, "cache": "q8_0", "query": "bf16"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the benchmark's decode step (4 verified tokens), four layers of a model after each other
        _case("step_256k_32k_mtp4", "step", layers=4, lanes=1, history=262144, window=32768, gen=16384, tokens=4),
        # a short conversation on a small model, one token: the smallest step
        _case("step_8k_4k_1tok", "step", head_dim=128, kv_heads=2, group=4, layers=1, lanes=1, history=8192,
              window=4096, gen=300, tokens=1),
        # four conversations decoded together, one token each
        _case("step_4lanes_64k_256k", "step", layers=2, lanes=4, history=262144, window=32768, gen=16384, tokens=1),
        # the fp16 16K-token configuration: 32 retrieved blocks and a 512-cell reserve
        _case("attend_f16_4608_1tok", "attend", head_dim=128, kv_heads=2, group=4, cache="f16", query="f32",
              window=4608, filled=4608, tokens=1),
        # draft verification over a part-filled q4_0 window, an odd number of tiles
        _case("attend_q4_20608_5tok", "attend", cache="q4_0", query="f32", window=20608, filled=19111, tokens=5),
        # the benchmark's prompt chunk: the largest call
        _case("prefill_2048_34816", "prefill", window=34816, filled=34816, tokens=2048),
        # the ragged end of a prompt
        _case("prefill_37_32768", "prefill", window=34816, filled=32805, tokens=37),
        # a mid-sized chunk on an fp16 cache
        _case("prefill_f16_700_8192", "prefill", head_dim=128, kv_heads=2, group=4, cache="f16", query="f32",
              window=9216, filled=8892, tokens=700),
        # a prompt chunk's new tokens into the sums, the index and the window
        _case("ingest_2048", "ingest", window=34816, history=262144, pos0=98304, cell0=32768, tokens=2048, turn="all"),
        # the new tokens of one verified decode step
        _case("ingest_4", "ingest", query="f32", window=32768, history=262144, pos0=98301, cell0=17003, tokens=4,
              turn="decode"),
        # the topic drifts: the oldest retrieved block leaves and a new one joins, the others move one slot
        _case("retrieve_drift_32k", "retrieve", window=32768, history=262144, fresh=1, shadow=True),
        # a new topic: every retrieved block but the sink comes from the host
        _case("retrieve_new_32k", "retrieve", window=32768, history=262144, fresh=127, shadow=False),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step", "attend", "prefill", "prefill", "ingest", "retrieve"])
    dim, kv, grp = rng.choice([(256, 4, 6), (256, 4, 6), (128, 2, 4), (128, 8, 4), (256, 2, 8), (128, 1, 8)])
    c = _case(None, kind, head_dim=dim, kv_heads=kv, group=grp, query=rng.choice(["bf16", "f32"]))
    if kind in ("attend", "prefill"):
        c["cache"] = rng.choice(["q8_0", "q8_0", "q4_0", "f16"])
        c["window"] = 128 * _log(rng, 8, 256)
        c["filled"] = max(64, int(c["window"] * rng.uniform(0.5, 1.0)))
        most = 32 // grp
        c["tokens"] = rng.randint(1, most) if kind == "attend" else min(c["filled"], _log(rng, most + 1, 1500))
    elif kind == "step":
        c["cache"] = rng.choice(["q8_0", "q8_0", "q4_0"])
        c["layers"], c["lanes"] = rng.randint(1, 3), rng.choice([1, 1, 2, 3])
        c["window"] = 256 * _log(rng, 8, 128)
        c["history"] = max(_log(rng, 4096, 262144) // BT * BT, c["lanes"] * c["window"])
        c["gen"] = rng.randint(32, c["window"] // 2)
        c["tokens"] = rng.randint(1, 32 // grp)
    elif kind == "ingest":
        c["cache"] = rng.choice(["q8_0", "q8_0", "q4_0", "f16"])
        c["tokens"] = _log(rng, 1, 2048)
        c["window"] = 128 * _log(rng, 32, 256)
        c["cell0"] = rng.randint(0, c["window"] - c["tokens"])
        c["history"] = 262144
        c["pos0"] = rng.randint(0, c["history"] - c["tokens"])
        c["turn"] = "decode" if c["tokens"] <= 8 else rng.choice(["all", "tail"])
    else:
        c["cache"] = rng.choice(["q8_0", "q8_0", "q4_0"])
        c["window"] = 256 * _log(rng, 16, 128)
        n_sel = c["window"] // 2 // BT
        c["history"] = max(_log(rng, 16384, 262144) // BT * BT, 2 * c["window"])
        c["fresh"] = _log(rng, 1, n_sel - 1)
        c["shadow"] = rng.random() < 0.7
    return c


# ---- inputs ------------------------------------------------------------------
def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _blocks(kind, x):
    """(codes, scales) of 32-value blocks, as ggml's quantisers form them in fp32."""
    x = x.reshape(-1, 32)
    if kind == "q8_0":
        d = x.abs().amax(1) / 127.0
        i = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
        y = x * i[:, None]
        return torch.trunc(y + torch.copysign(torch.full_like(y, 0.5), y)).to(torch.int8), d.to(torch.float16)
    top = x.gather(1, x.abs().argmax(1, keepdim=True))[:, 0]
    d = top * -0.125
    i = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    return (x * i[:, None] + 8.5).to(torch.int32).clamp(0, 15).to(torch.uint8), d.to(torch.float16)


def _rows(kind, x):
    """Cache rows (uint8 [tokens][bytes]) of fp32 values [tokens][values]."""
    n = x.shape[0]
    if kind == "f16":
        return x.to(torch.float16).view(torch.uint8).reshape(n, -1)
    q, d = _blocks(kind, x)
    if kind == "q4_0":
        q = q[:, :16] | (q[:, 16:] << 4)
    return torch.cat([d[:, None].view(torch.uint8), q.view(torch.uint8)], 1).reshape(n, -1)


def _values(kind, x):
    """The 64-bit values that the cache rows of `x` hold."""
    if kind == "f16":
        return x.to(torch.float16).double()
    q, d = _blocks(kind, x)
    v = (q.double() - (8.0 if kind == "q4_0" else 0.0)) * d.double()[:, None]
    return v.reshape(x.shape)


def _kv_kinds(case):
    return ("f16", "f16") if case["cache"] == "f16" else (case["cache"], "q4_0")


def _window_values(case, seed, lane, n):
    """fp32 K and V of n window cells."""
    e = case["kv_heads"] * case["head_dim"]
    g = _gen(seed, 11 + lane)
    return _randn(g, n, e), _randn(g, n, e)


def _queries(case, seed, lane, n):
    q = _randn(_gen(seed, 101 + lane), n, case["kv_heads"] * case["group"], case["head_dim"])
    return q.to(torch.bfloat16) if case["query"] == "bf16" else q


def _history(case, seed, lane, n, keep=None):
    """Pinned history rows of n tokens; keep: the token blocks whose fp32 K and V are returned."""
    e = case["kv_heads"] * case["head_dim"]
    kk, vk = _kv_kinds(case)
    kb, vb = (e // 32 * b for b in BLOCK[case["cache"]])
    bufs = None if keep is not None else (api.HostBuffer(n * kb), api.HostBuffer(n * vb))
    kept = {}
    for c0 in range(0, n, 32768):
        m = min(32768, n - c0)
        g = _gen(seed, 1000 + 64 * lane + c0 // 32768)
        k, v = _randn(g, m, e), _randn(g, m, e)
        if keep is None:
            torch.from_numpy(bufs[0].u8[c0 * kb:(c0 + m) * kb]).copy_(_rows(kk, k).view(-1))
            torch.from_numpy(bufs[1].u8[c0 * vb:(c0 + m) * vb]).copy_(_rows(vk, v).view(-1))
        else:
            for b in keep:
                if c0 <= b * BT < c0 + m:
                    kept[b] = (k[b * BT - c0:(b + 1) * BT - c0].clone(), v[b * BT - c0:(b + 1) * BT - c0].clone())
    if keep is not None:
        return kept
    h = api.History.__new__(api.History)
    h.kbuf, h.vbuf, h.n_tokens = bufs[0], bufs[1], n
    h.c = L.History(bufs[0].ptr, bufs[1].ptr, n)
    return h


def _topics(case, seed, lane, layer, n_blocks, sets):
    """Block sums [n_blocks][e] whose blocks of sets[i] lie near topic i, and each topic's query rows [4][heads * dim]."""
    H, D, G = case["kv_heads"], case["head_dim"], case["group"]
    g = _gen(seed, 100000 + 64 * lane + layer)
    sums = _randn(g, n_blocks, H, D) * BT ** 0.5
    queries = []
    for ids in sets:
        u = torch.nn.functional.normalize(_randn(g, H, D), dim=1)
        sums[torch.from_numpy(np.asarray(ids)).cuda()] += u * (2.0 * BT)
        rows = (u[:, None, :] + 0.02 * _randn(g, H, 4 * G, D))
        queries.append(rows.reshape(H, 4, G, D).permute(1, 0, 2, 3).reshape(4, H * G * D).contiguous())
    return sums.reshape(n_blocks, H * D), queries


def _pick(seed, salt, n, lo, hi):
    return np.sort(np.random.default_rng([int(seed), salt]).choice(np.arange(lo, hi), n, replace=False))


def _lane_blocks(case, lane):
    return case["history"] * (lane + 1) // case["lanes"] // BT


def _step_set(case, seed, lane, layer):
    n_sel = case["window"] // 2 // BT
    return np.concatenate([[0], _pick(seed, 200 + 64 * lane + layer, n_sel - 1, 1, _lane_blocks(case, lane))])


def _drift_sets(case):
    """Two selections: `fresh` of the oldest blocks after the sink leave, as many new ones join."""
    n_sel, n_blocks, f = case["window"] // 2 // BT, case["history"] // BT, case["fresh"]
    step = (n_blocks - f - 1) // (n_sel - 1)
    old = 1 + np.arange(n_sel - 1) * step
    return np.concatenate([[0], old]), np.concatenate([[0], old[f:], np.arange(n_blocks - f, n_blocks)])


def _index(case, n_blocks, sums):
    ix = api.MeanKIndex(_st(), 1, n_blocks, case["kv_heads"], case["head_dim"], BT, norms=True)
    if sums is not None:
        ix.set_block_sums(sums[None])
        ix.mean_tokens.fill_(BT)
        ix.present.fill_(1)
        ix.refresh()
    return ix


def _accumulator(case, rows=None):
    qa = api.QueryAcc(_st(), 1, case["kv_heads"] * case["group"], case["head_dim"], n_head_kv=case["kv_heads"])
    qa.reset()
    if rows is not None:
        qa.add(0, rows)
    return qa


def _window(case, shadow=False):
    kt, vt = TYPES[case["cache"]]
    return api.KVWindow(_st(), case["window"], case["kv_heads"], case["head_dim"], BT, kt, vt, shadow=shadow)


def _filled_window(case, seed):
    w = _window(case)
    n = case["filled"]
    k, v = _window_values(case, seed, 0, n)
    kk, vk = _kv_kinds(case)
    w.import_rows(0, _rows(kk, k), _rows(vk, v), torch.arange(n, dtype=torch.int32, device="cuda"))
    return w


def _prepare_step(case, seed):
    st, H, G, D = _st(), case["kv_heads"], case["group"], case["head_dim"]
    n_sel, base = case["window"] // 2 // BT, case["window"] // 2
    hist = [_history(case, seed, i, _lane_blocks(case, i) * BT) for i in range(case["lanes"])]
    kk, vk = _kv_kinds(case)
    calls, outs = [], []
    for layer in range(case["layers"]):
        lanes = []
        for i in range(case["lanes"]):
            nb = _lane_blocks(case, i)
            sums, (rows,) = _topics(case, seed, i, layer, nb, [_step_set(case, seed, i, layer)])
            salt = 16 * layer + i
            k, v = _window_values(case, seed, salt, case["gen"])
            w = _window(case)
            sel = api.SelectionBuffers(st, nb, n_sel)
            ln = dict(index=_index(case, nb, sums), query=_accumulator(case, rows), n_blocks=nb,
                      n_tokens=torch.full((nb,), BT, dtype=torch.int32, device="cuda"), budget_blocks=n_sel,
                      sink_blocks=1, window=w, sel=sel, history=hist[i], q=_queries(case, seed, salt, case["tokens"]),
                      q_pos=torch.arange(base + case["gen"] - case["tokens"], base + case["gen"], dtype=torch.int32,
                                         device="cuda"),
                      out=torch.empty((case["tokens"], H * G, D), device="cuda"))
            api.score_topk(st, ln["index"], ln["query"], nb, ln["n_tokens"], n_sel, 1, 0, None, w, sel)
            api.stagein_selection(st, hist[i], w, sel, N_ROT, FREQ_BASE)
            w.import_rows(base, _rows(kk, k), _rows(vk, v),
                          torch.arange(base, base + case["gen"], dtype=torch.int32, device="cuda"))
            lanes.append(ln)
            outs.append({"out": ln["out"], "scores": sel.scores, "ids": sel.ids, "to_base": sel.to_base})
        if case["lanes"] == 1:
            ln = lanes[0]
            calls.append(api.prepare_decode_step(st, ln["index"], ln["query"], ln["n_blocks"], ln["n_tokens"], n_sel,
                                                 1, 0, ln["window"], ln["sel"], ln["history"], ln["q"], ln["q_pos"],
                                                 H * G, D ** -0.5, ln["out"], N_ROT, FREQ_BASE))
        else:
            calls.append(api.prepare_decode_step_lanes(st, lanes, H * G, D ** -0.5, N_ROT, FREQ_BASE))
    return {"kind": "step", "calls": calls, "outs": outs}


def prepare(case, seed):
    kind, st = case["kind"], _st()
    H, G, D = case["kv_heads"], case["group"], case["head_dim"]
    if kind == "step":
        return _prepare_step(case, seed)
    if kind in ("attend", "prefill"):
        n, w = case["tokens"], _filled_window(case, seed)
        q = _queries(case, seed, 0, n)
        pos = torch.arange(case["filled"] - n, case["filled"], dtype=torch.int32, device="cuda")
        out = torch.empty((n, H * G, D), device="cuda")
        s = {"kind": kind, "w": w, "q": q, "pos": pos, "out": out, "heads": H * G, "scale": D ** -0.5}
        if kind == "attend":
            s["call"] = api.prepare_fa_decode(st, w, q, pos, H * G, D ** -0.5, out)
        return s
    if kind == "ingest":
        n = case["tokens"]
        q, k, kr, v = _ingest_values(case, seed)
        keep = None if case["turn"] != "tail" else np.arange(n) >= n - n // 4
        return {"kind": kind, "decode": case["turn"] == "decode", "q": q, "k": k, "kr": kr, "v": v, "keep": keep,
                "w": _window(case), "ix": _index(case, case["history"] // BT, None), "qa": _accumulator(case),
                "cell0": case["cell0"], "pos0": case["pos0"], "types": TYPES[case["cache"]],
                "pos": torch.arange(case["pos0"], case["pos0"] + n, dtype=torch.int32, device="cuda")}
    sets = _drift_sets(case)
    nb, n_sel = case["history"] // BT, len(sets[0])
    sums, rows = _topics(case, seed, 0, 0, nb, sets)
    ix, hist, w = _index(case, nb, sums), _history(case, seed, 0, nb * BT), _window(case, case["shadow"])
    sel = api.SelectionBuffers(st, nb, n_sel)
    n_tokens = torch.full((nb,), BT, dtype=torch.int32, device="cuda")
    calls = [api.prepare_score_topk_stagein(st, ix, _accumulator(case, r), nb, n_tokens, n_sel, 1, 0, w, sel, hist,
                                            N_ROT, FREQ_BASE) for r in rows]
    calls[0]()                                # the conversation so far; the passes go to the other topic and back
    return {"kind": kind, "calls": calls, "next": 1, "w": w, "sel": sel}


def _ingest_values(case, seed):
    n, e = case["tokens"], case["kv_heads"] * case["head_dim"]
    q = _queries(case, seed, 0, n)
    g = _gen(seed, 7)
    k = _randn(g, n, case["kv_heads"], case["head_dim"])
    return q, k.to(torch.bfloat16) if case["query"] == "bf16" else k, _randn(g, n, e), _randn(g, n, e)


# ---- one pass ------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "step":
        for call in s["calls"]:
            call()
        return s["outs"]
    if kind == "attend":
        s["call"]()
        return s["out"]
    if kind == "prefill":
        return api.fa_prefill(_st(), s["w"], s["q"], s["pos"], s["heads"], s["scale"], s["out"])
    if kind == "ingest":
        qa, ix, w = s["qa"], s["ix"], s["w"]
        if s["decode"]:
            qa.add_view(0, s["q"])
            ix.acc_add(0, s["k"], 0, s["k"].shape[0])
        else:
            qa.reset()
            qa.add_view(0, s["q"], s["keep"])
            ix.add_view(0, s["pos0"], s["k"])
        k_rows = api.quantize_rows(_st(), s["types"][0], s["kr"])
        v_rows = api.quantize_rows(_st(), s["types"][1], s["v"])
        w.import_rows(s["cell0"], k_rows, v_rows, s["pos"])
        return {"q_sum": qa.q_sum, "q_vec": qa.q_vec, "q_norm": qa.q_norm, "acc": ix.acc, "k_sum": ix.k_sum,
                "mean_tokens": ix.mean_tokens, "k_norm": ix.k_norm, "k": w.k, "v": w.v, "cell_pos": w.cell_pos}
    s["calls"][s["next"]]()
    s["next"] ^= 1
    w, sel = s["w"], s["sel"]
    return {"scores": sel.scores, "ids": sel.ids, "to_base": sel.to_base, "k": w.k, "v": w.v, "cell_pos": w.cell_pos}


# ---- what a pass cannot do without ---------------------------------------------
def _row_bytes(case):
    return sum(case["kv_heads"] * case["head_dim"] // 32 * b for b in BLOCK[case["cache"]])


def _attention(case, first, n):
    """(bytes, flops) of n queries at positions first .. over cells 0 .. first + n - 1."""
    H, G, D = case["kv_heads"], case["group"], case["head_dim"]
    pairs = n * first + n * (n + 1) // 2
    qb = 2 if case["query"] == "bf16" else 4
    return (first + n) * (_row_bytes(case) + 4) + n * H * G * D * (qb + 4), 4 * D * pairs * H * G


def work(case):
    kind = case["kind"]
    e, qe = case["kv_heads"] * case["head_dim"], case["kv_heads"] * case["group"] * case["head_dim"]
    if kind == "step":
        n, first = case["tokens"], case["window"] // 2 + case["gen"] - case["tokens"]
        b, f = _attention(case, first, n)
        nb = sum(_lane_blocks(case, i) for i in range(case["lanes"]))
        many = case["layers"] * case["lanes"]
        return {"bytes": many * b + case["layers"] * nb * (e * 4 + 16), "flops": many * f + case["layers"] * nb * e * 2}
    if kind in ("attend", "prefill"):
        b, f = _attention(case, case["filled"] - case["tokens"], case["tokens"])
        return {"bytes": b, "flops": f}
    if kind == "ingest":
        n, es = case["tokens"], 2 if case["query"] == "bf16" else 4
        kept = n // 4 if case["turn"] == "tail" else n
        return {"bytes": kept * qe * es + n * e * es + 2 * n * e * 4 + n * (_row_bytes(case) + 8) + qe * 4
                + (n // BT + 1) * e * 4, "flops": kept * qe + 3 * n * e}
    n_sel, nb = case["window"] // 2 // BT, case["history"] // BT
    staged = n_sel - 1
    return {"bytes": nb * (e * 4 + 16) + staged * BT * 2 * _row_bytes(case), "flops": nb * e * 2 + staged * BT * e * 12}


def tolerance(case):
    # sums, scores, selections and cache bytes have one right answer
    if case["kind"] in ("ingest", "retrieve"):
        return "exact"
    # attention: probabilities enter the P V product as 16-bit floats
    return {"rel": 2e-3, "max": 2e-2}


# ---- the same in 64 bits -------------------------------------------------------
def _attend64(case, q, q_pos, k, v, pos, round_q):
    """Softmax attention in 64 bits over cells with values k, v [cells][e] at positions pos."""
    H, G, D = case["kv_heads"], case["group"], case["head_dim"]
    n = q.shape[0]
    q = q.float()
    q = _values("q8_0", q.reshape(n, -1)) if round_q else q.double()
    q = q.reshape(n, H, G, D)
    out = torch.empty((n, H, G, D), dtype=torch.float64, device="cuda")
    for h in range(H):
        kh = k.reshape(-1, H, D)[:, h].t().contiguous()
        vh = v.reshape(-1, H, D)[:, h].contiguous()
        for t0 in range(0, n, 128):
            t1 = min(n, t0 + 128)
            s = (q[t0:t1, h].reshape(-1, D) @ kh) * D ** -0.5
            dead = pos[None, :] > q_pos[t0:t1, None]
            s.view(t1 - t0, G, -1).masked_fill_(dead[:, None, :], float("-inf"))
            out[t0:t1, h] = (torch.softmax(s, 1) @ vh).view(t1 - t0, G, D)
    return out.reshape(n, H * G, D)


def _scores64(case, sums, rows):
    """Mean over the kv heads of the cosine of the query mean and each block's key mean."""
    H, G, D = case["kv_heads"], case["group"], case["head_dim"]
    q = rows.double().sum(0).view(H, G, D).sum(1) / (rows.shape[0] * G)
    k = sums.double().view(-1, H, D) / BT
    dot = (k * q).sum(2)
    return (dot / (q.norm(dim=1) * k.norm(dim=2) + 1e-6)).mean(1)


def _staged64(case, kind, k, base):
    """A staged block's K: rotated to window positions base .., Hadamard transform, cache type again."""
    H, D = case["kv_heads"], case["head_dim"]
    x = _values(kind, k).reshape(BT, H, D)
    theta = np.power(np.float32(FREQ_BASE), np.arange(N_ROT // 2, dtype=np.float32) * np.float32(-2.0 / N_ROT))
    ang = np.arange(base, base + BT, dtype=np.float32)[:, None] * theta.astype(np.float32)
    c, s = (torch.from_numpy(f(ang.astype(np.float64))).cuda()[:, None, :] for f in (np.cos, np.sin))
    a, b = x[..., :N_ROT // 2].clone(), x[..., N_ROT // 2:N_ROT].clone()
    x[..., :N_ROT // 2], x[..., N_ROT // 2:N_ROT] = a * c - b * s, a * s + b * c
    had = torch.ones((1, 1), dtype=torch.float64, device="cuda")
    while had.shape[0] < D:
        had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)], 0)
    x = (x.reshape(-1, D) @ had.contiguous()) * D ** -0.5
    return _values(kind, x.float().reshape(BT, H * D))


def exact(case, seed):
    kind = case["kind"]
    kk, vk = _kv_kinds(case)
    if kind == "step":
        base, n, res = case["window"] // 2, case["tokens"], []
        sets = {(y, i): _step_set(case, seed, i, y) for y in range(case["layers"]) for i in range(case["lanes"])}
        hist = [_history(case, seed, i, _lane_blocks(case, i) * BT,
                         set(int(b) for y in range(case["layers"]) for b in sets[y, i])) for i in range(case["lanes"])]
        for layer in range(case["layers"]):
            for i in range(case["lanes"]):
                nb, salt = _lane_blocks(case, i), 16 * layer + i
                sums, (rows,) = _topics(case, seed, i, layer, nb, [sets[layer, i]])
                gk, gv = _window_values(case, seed, salt, case["gen"])
                ks = [_staged64(case, kk, hist[i][int(b)][0], j * BT) for j, b in enumerate(sets[layer, i])]
                vs = [_values(vk, hist[i][int(b)][1]) for b in sets[layer, i]]
                k, v = torch.cat(ks + [_values(kk, gk)]), torch.cat(vs + [_values(vk, gv)])
                pos = torch.arange(base + case["gen"], device="cuda")
                out = _attend64(case, _queries(case, seed, salt, n), pos[-n:], k, v, pos, True)
                res.append({"out": out, "scores": _scores64(case, sums, rows), "ids": None, "to_base": None})
        return res
    if kind in ("attend", "prefill"):
        n, m = case["tokens"], case["filled"]
        k, v = _window_values(case, seed, 0, m)
        pos = torch.arange(m, device="cuda")
        few = n * case["group"] <= 32            # few rows: q8_0 queries against a quantised cache
        return _attend64(case, _queries(case, seed, 0, n), pos[m - n:], _values(kk, k), _values(vk, v), pos,
                         few and case["cache"] != "f16")
    if kind == "ingest":
        H, G, D, n = case["kv_heads"], case["group"], case["head_dim"], case["tokens"]
        q, k, _, _ = _ingest_values(case, seed)
        q, k = q.double().reshape(n, -1), k.double().reshape(n, -1)
        kept = q[n - n // 4:] if case["turn"] == "tail" else q
        res = dict.fromkeys(("mean_tokens", "k", "v", "cell_pos"))
        res["q_sum"] = kept.sum(0)[None]
        res["q_vec"] = (res["q_sum"].view(1, H, G, D).sum(2) / max(1, kept.shape[0] * G))
        res["q_norm"] = (res["q_vec"] ** 2).sum(2)
        res["acc"] = (k.sum(0) if case["turn"] == "decode" else torch.zeros(H * D, device="cuda").double())[None]
        nb = case["history"] // BT
        sums = torch.zeros((nb, H * D), dtype=torch.float64, device="cuda")
        cnt = torch.zeros(nb, dtype=torch.float64, device="cuda")
        if case["turn"] != "decode":
            blk = torch.arange(case["pos0"], case["pos0"] + n, device="cuda") // BT
            sums.index_add_(0, blk, k)
            cnt.index_add_(0, blk, torch.ones(n, dtype=torch.float64, device="cuda"))
            cnt[blk[0]] += case["pos0"] % BT      # the block's earlier tokens count, their sums are zero here
        res["k_sum"] = torch.cat([sums, sums.new_zeros((-nb % 8, H * D))]).view(1, -1, 8, H * D).transpose(2, 3).contiguous()
        res["k_norm"] = ((sums / cnt.clamp(min=1)[:, None]).view(nb, H, D) ** 2).sum(2).t().contiguous()[None]
        return res
    sums, rows = _topics(case, seed, 0, 0, case["history"] // BT, _drift_sets(case))
    res = dict.fromkeys(("ids", "to_base", "k", "v", "cell_pos"))
    res["scores"] = _scores64(case, sums, rows[1])
    return res
