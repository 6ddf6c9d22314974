"""The work a user of the dedoppler search has it do, as a list of measurable cases.

Every case is one pass through public entry points of :mod:`seticore_amd`:

* ``search``   one coarse channel per call, ``Dedopplerer.search`` (the reference's call), with its
               default host-exact statistics or with device statistics;
* ``batch``    many coarse channels (beams) of one or several shapes planned once, ``batch.Batch``,
               plain or gated by the block-proposal network;
* ``tree``     the path sums of one drift block, ``Dedopplerer.taylor_tree`` (what the reference's own
               taylor_benchmark times);
* ``incoherent`` ``Dedopplerer.addIncoherentPower`` over the hits of the coherent beams;
* ``normalize`` float32 power to the half-width storage forms;
* ``forward`` / ``gradient`` the proposal network's scoring and training passes.

Inputs are synthetic power as the search meets it: exponential noise with a gain, a cosine taper over
the outer 5 % of a coarse channel, a DC spike at its centre, drifting tones and a few stationary
narrowband interferers. They are made by torch on the GPU from the seed alone. The telescope
parameters are those of the file-scale workload (2.79 Hz channels, 18.25 s time steps).
"""

import math

import numpy as np
import torch

import seticore_amd as sa
from seticore_amd import batch as sb

FOFF = -2.79e-6   # MHz
TSAMP = 18.25     # s
TYPES = {"f32": (sa.SC_F32, torch.float32), "f16": (sa.SC_F16, torch.float16),
         "bf16": (sa.SC_BF16, torch.bfloat16)}


def listed():
    return [
        # A few thousand channels and the default (reference-exact) statistics: a zoom around a
        # candidate, or the known-answer checks users run first. Latency and launches.
        {"name": "exact_small", "kind": "search", "stats": "exact", "T": 13, "N": 5003,
         "max_drift": 2.0, "snr": 25.0, "dtype": "f32"},
        # One file-scale coarse channel with the defaults a switching user has: host-exact statistics,
        # SNR 25, drifts up to 10 Hz/s.
        {"name": "exact_file", "kind": "search", "stats": "exact", "T": 16, "N": 1 << 20,
         "max_drift": 10.0, "snr": 25.0, "dtype": "f32"},
        # The single-coarse-channel workload (drifts up to 4 Hz/s, SNR 10) with device statistics, one
        # call per coarse channel as run_dedoppler makes them.
        {"name": "call_file", "kind": "search", "stats": "device", "T": 16, "N": 1 << 20,
         "max_drift": 4.0, "snr": 10.0, "dtype": "f32"},
        # A ragged middle size: 50 time steps (padded to 64), an odd width, half-width storage.
        {"name": "call_mid", "kind": "search", "stats": "device", "T": 50, "N": 300001,
         "max_drift": 5.0, "snr": 10.0, "dtype": "f16"},
        # The longest time axis: 256 steps of a file-scale coarse channel.
        {"name": "call_long", "kind": "search", "stats": "device", "T": 256, "N": 1 << 20,
         "max_drift": 5.0, "snr": 10.0, "dtype": "f32"},
        # A file: consecutive coarse channels of 16 x 2^20, one plan, one launch per pass.
        {"name": "batch_file", "kind": "batch", "shapes": "16x1048576", "copies": 16,
         "max_drift": 10.0, "snr": 10.0, "dtype": "f32", "gate": 0.0},
        # Beams with uneven time steps and channel widths, half-width storage.
        {"name": "batch_uneven", "kind": "batch",
         "shapes": "16x1048576 32x262144 64x131072 256x131072 200x262144 13x262144",
         "copies": 2, "max_drift": 5.0, "snr": 10.0, "dtype": "bf16", "gate": 0.0},
        # The learned gate over a file: the network scores every block, about 60 % are searched.
        {"name": "batch_gated", "kind": "batch", "shapes": "16x262144", "copies": 16,
         "max_drift": 10.0, "snr": 10.0, "dtype": "bf16", "gate": 0.6},
        # The reference's taylor_benchmark: one drift block of 256 x 2^20.
        {"name": "tree", "kind": "tree", "T": 256, "N": 1 << 20, "block": -2, "dtype": "f32"},
        # A few hundred hits of the coherent beams looked up in the incoherent one.
        {"name": "incoherent", "kind": "incoherent", "T": 16, "N": 1 << 19, "hits": 300,
         "max_drift": 10.0, "dtype": "f32"},
        # Half-width storage of a file-scale coarse channel.
        {"name": "normalize", "kind": "normalize", "T": 16, "N": 1 << 20, "dtype": "bf16"},
        # One training batch of the proposal network.
        {"name": "net_gradient", "kind": "gradient", "B": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "batch", "batch", "tree", "incoherent",
                       "normalize", "forward", "gradient"])
    if kind == "search":
        stats = rng.choice(["exact", "device", "device"])
        T = _log_int(rng, 4, 256)
        N = _log_int(rng, 1000 if stats == "exact" else 4096, min(1 << 20, (1 << 27) // max(T, 16)))
        return {"kind": kind, "stats": stats, "T": T, "N": N,
                "max_drift": round(rng.uniform(0.5, 10.0 if T <= 16 else 5.0), 2),
                "snr": 25.0 if stats == "exact" else round(rng.uniform(10.0, 30.0), 1),
                "dtype": rng.choice(["f32", "f32", "f16", "bf16"])}
    if kind == "batch":
        gate = rng.choice([0.0, 0.0, 0.6])
        if gate:
            shapes = ["16x%d" % (4096 * _log_int(rng, 2, 64))]
        else:
            shapes = ["%dx%d" % (rng.choice([13, 16, 16, 16, 30, 32, 64, 100, 200, 256]),
                                 _log_int(rng, 4096, 1 << 18)) for _ in range(rng.randint(1, 4))]
        return {"kind": kind, "shapes": " ".join(shapes), "copies": rng.randint(1, 16 // len(shapes)),
                "max_drift": round(rng.uniform(1.0, 10.0 if gate else 5.0), 2),
                "snr": round(rng.uniform(10.0, 30.0), 1),
                "dtype": rng.choice(["f32", "f32", "f16", "bf16"]), "gate": gate}
    if kind == "tree":
        T = _log_int(rng, 4, 512)
        return {"kind": kind, "T": T, "N": _log_int(rng, 20000, (1 << 26) // max(64, T)),
                "block": rng.randint(-2, 2), "dtype": rng.choice(["f32", "f16", "bf16"])}
    if kind == "incoherent":
        return {"kind": kind, "T": _log_int(rng, 8, 64), "N": _log_int(rng, 50000, 1 << 18),
                "hits": _log_int(rng, 1, 200), "max_drift": round(rng.uniform(1.0, 5.0), 2),
                "dtype": rng.choice(["f32", "f32", "f16", "bf16"])}
    if kind == "normalize":
        T = _log_int(rng, 4, 256)
        return {"kind": kind, "T": T, "N": _log_int(rng, 1000, (1 << 26) // max(T, 64)),
                "dtype": rng.choice(["bf16", "f16", "f32"])}
    return {"kind": kind, "B": _log_int(rng, 1, 2048 if kind == "forward" else 300)}


# ---------------------------------------------------------------------------
# Inputs.

def _rounded(T):
    r = 1
    while r < T:
        r *= 2
    return r


def _resolution(T):
    return 1e6 * FOFF / ((_rounded(T) - 1) * TSAMP)


def _drift_range(T, max_drift):
    steps = _rounded(T) - 1
    nmd = max_drift / abs(_resolution(T) * steps)
    return int(math.floor(-nmd)), int(math.floor(nmd)), int(2 * math.ceil(nmd * steps))


def _waterfall(T, N, max_drift, seed, gain=None):
    """float32 power [T_r][N]: noise, taper, DC spike, tones, interferers; rows from T on are zero."""
    T_r = _rounded(T)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = np.random.default_rng(seed)
    gain = float(r.uniform(0.5, 2.0)) if gain is None else gain
    x = torch.empty((T_r, N), dtype=torch.float32, device="cuda")
    x[:T].exponential_(1.0, generator=g)
    x[T:].zero_()
    x *= gain
    edge = N // 20
    if edge:
        taper = torch.ones(N, device="cuda")
        ramp = 0.5 - 0.5 * torch.cos(torch.linspace(0.0, math.pi, edge, device="cuda"))
        taper[:edge] = 0.25 + 0.75 * ramp
        taper[N - edge:] = taper[:edge].flip(0)
        x *= taper
    x[:T, N // 2] += 50.0 * gain
    steps = np.arange(T)
    rows, cols, vals = [], [], []
    for k in range(max(4, N // 65536)):
        drift = r.uniform(-max_drift, max_drift)
        amp = gain * (80.0 if k < 2 else 10 ** r.uniform(math.log10(9.0), math.log10(120.0))) / math.sqrt(T)
        # Mid-channel tones in the first two slots, so that every seed has hits.
        start = r.uniform(0.3, 0.7) * N if k < 2 else r.uniform(0.06, 0.94) * N
        if k < 2:
            drift = 0.3 * max_drift * (1 if k else -1)
        c = np.rint(start + steps * drift * TSAMP / (FOFF * 1e6)).astype(np.int64)
        ok = (c >= 0) & (c < N)
        rows.append(steps[ok]); cols.append(c[ok]); vals.append(np.full(ok.sum(), amp))
    for _ in range(N // 300000):
        c = int(r.integers(int(0.06 * N), int(0.94 * N)))
        rows.append(steps); cols.append(np.full(T, c)); vals.append(np.full(T, gain * 10 ** r.uniform(1.0, 4.0)))
    rows, cols, vals = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    x.index_put_((torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda()),
                 torch.from_numpy(vals).float().cuda(), accumulate=True)
    return x


def _stored(x, T, dtype):
    """The coarse channel as it is stored: float32 power, or normalised half-width power."""
    if dtype == "f32":
        return x
    y = x[:T].double()
    sd = y.std(unbiased=False)
    loc = y.sum(0).median() / T
    z = torch.zeros_like(x)
    z[:T] = ((y - loc) / sd).float().clamp(-65504.0, 65504.0)
    return z.to(TYPES[dtype][1])


def _channel(T, N, max_drift, seed, dtype):
    return _stored(_waterfall(T, N, max_drift, seed), T, dtype)


def _shapes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split()] * case["copies"]


def _tiles(B, seed):
    """Pooled, normalised tiles of noise with a drifting tone in about half of the blocks."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = torch.empty((B, 16, 1024, 4), device="cuda").exponential_(1.0, generator=g).sum(-1)
    r = np.random.default_rng(seed)
    t = np.arange(16)
    labels = (r.uniform(size=B) < 0.5).astype(np.float32)
    hot = np.nonzero(labels)[0]
    if len(hot):
        start, slope, amp = r.uniform(0, 1024, len(hot)), r.uniform(-8, 8, len(hot)), r.uniform(2, 40, len(hot))
        c = np.clip(np.rint(start[:, None] + t * slope[:, None]), 0, 1023).astype(np.int64)
        b = np.repeat(hot, 16)
        s[torch.from_numpy(b).cuda(), torch.from_numpy(np.tile(t, len(hot))).cuda(),
          torch.from_numpy(c.ravel()).cuda()] += torch.from_numpy(np.repeat(amp, 16)).float().cuda()
    z = (2.0 * (s - 4.0) / 3.2).clamp(-4.0, 32.0)
    return z.to(torch.bfloat16), torch.from_numpy(labels).cuda()


def _params(seed):
    """He-uniform float32 parameters in the network's layout."""
    r = np.random.default_rng(seed)

    def he(n, fan):
        return r.uniform(-1, 1, n) * math.sqrt(6.0 / fan)

    return np.concatenate([he(16 * 15, 15), np.zeros(16), he(32 * 15 * 16, 240), np.zeros(32),
                           he(32 * 15 * 32, 480), np.zeros(32), he(32, 32), np.zeros(1)]).astype(np.float32)


def _meta(N):
    return sa.FilterbankMetadata(fch1=8421.38671875, foff=FOFF, coarse_channel_size=N)


def _hit_list(case, seed):
    """Hits of coherent beams as a search reports them: start channel and drift inside the range."""
    T, N = case["T"], case["N"]
    bmin, bmax, _ = _drift_range(T, case["max_drift"])
    span = _rounded(T) - 1
    r = np.random.default_rng(seed + 1)
    drifts = np.arange(bmin * span, (bmax + 1) * span)
    out = []
    # Distinct drifts: hits of equal drift come back in no particular order.
    for d in r.choice(drifts, size=min(case["hits"], len(drifts)), replace=False):
        d = int(d)
        c = int(r.integers(max(0, -d), N - max(0, d)))
        out.append(sa.DedopplerHit(index=c, drift_steps=d, drift_rate=d * _resolution(T), snr=12.0,
                                   beam=0, num_timesteps=T, power=50.0))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        net = sa.ProposalNet(max_batch=case["B"])
        net.set_params(_params(seed))
        tiles, labels = _tiles(case["B"], seed)
        return {"kind": kind, "net": net, "tiles": tiles, "labels": labels}
    if kind == "batch":
        shapes = _shapes(case)
        data = [_channel(T, N, case["max_drift"], seed * 1009 + i, case["dtype"])
                for i, (T, N) in enumerate(shapes)]
        instances = [sb.instance(x, T, FOFF, TSAMP, case["max_drift"], 0.0, case["snr"], coarse_channel=i,
                                 dtype=TYPES[case["dtype"]][0], metadata=_meta(N))
                     for i, (x, (T, N)) in enumerate(zip(data, shapes))]
        slots = [_windows(T, N, case["max_drift"]) for T, N in shapes]
        if not case["gate"]:
            return {"kind": kind, "batch": sb.Batch(instances), "data": data, "slots": slots}
        net = sa.ProposalNet(max_batch=max(N for _, N in shapes) // sa.BLOCK_CHANNELS)
        net.set_params(_params(7))
        threshold = _gate_threshold(net, data, case["gate"])
        return {"kind": kind, "batch": sb.Batch(instances, proposal=net, logit_threshold=threshold),
                "data": data, "net": net, "slots": slots}
    T, N = case["T"], case["N"]
    if kind == "normalize":
        return {"kind": kind, "x": _waterfall(T, N, 5.0, seed)[:T], "dtype": TYPES[case["dtype"]][0]}
    x = _channel(T, N, case.get("max_drift", 5.0), seed, case["dtype"])
    buf = sa.FilterbankBuffer(_rounded(T), N, data=x, dtype=TYPES[case["dtype"]][0])
    dd = sa.Dedopplerer(T, N, FOFF, TSAMP)
    state = {"kind": kind, "buf": buf, "dd": dd, "meta": _meta(N), "case": case}
    if kind == "search":
        state["slots"] = _windows(T, N, case["max_drift"])
        if case["stats"] == "device":
            dd.set_stats_mode(sa.SC_STATS_DEVICE)
    if kind == "incoherent":
        state["hits"] = _hit_list(case, seed)
    if kind == "tree":
        state["columns"] = _valid_columns(case)
    return state


def _gate_threshold(net, data, share):
    """The logit threshold that flags about `share` of the blocks, in the middle of the widest gap
    between neighbouring logits around it."""
    logits = []
    for x in data:
        sums = x.float().sum(0)
        lo, hi = (int(f * sums.numel()) for f in (0.05, 0.95))
        ranked = sums.sort().values
        stats = torch.stack([ranked[sums.numel() // 2], ranked[lo:hi].std()])
        logits.append(net.forward(sa.ProposalNet.pool(x, stats)))
    z = torch.cat(logits).sort().values.cpu().numpy()
    a, b = int((0.85 - share) * len(z)), int((1.15 - share) * len(z))
    gaps = np.diff(z[a:b + 1])
    if not len(gaps):
        return float(z[0]) - 1.0
    k = a + int(np.argmax(gaps))
    return float(0.5 * (z[k] + z[k + 1]))


def _valid_columns(case):
    """Start channels all of whose paths in the drift block lie inside the coarse channel."""
    last = (_rounded(case["T"]) - 1) * case["block"]
    return max(0, -last), case["N"] - max(0, last + _rounded(case["T"]) - 1)


HIT = np.dtype(sa.DedopplerHit)


def _windows(T, N, max_drift):
    """Merge windows of a search: the most hits it can have."""
    return -(-N // _drift_range(T, max_drift)[2])


def _table(hits, slots):
    """The hits as columns, with zeros up to `slots` rows."""
    rows = np.zeros(slots, HIT)
    rows[:len(hits)] = np.frombuffer(b"".join(map(bytes, hits)), HIT)
    return rows


def _columns(rows):
    return {f: np.ascontiguousarray(rows[f])
            for f in ("index", "drift_steps", "drift_rate", "frequency", "snr", "power")}


def run(state):
    kind = state["kind"]
    if kind == "search":
        c, hits = state["case"], []
        state["dd"].search(state["buf"], state["meta"], -1, 0, c["max_drift"], 0.0, c["snr"], hits)
        return _columns(_table(hits, state["slots"]))
    if kind == "batch":
        b = state["batch"]
        b.run()
        return _columns(np.concatenate([_table(b.hits(i), n) for i, n in enumerate(state["slots"])]))
    if kind == "tree":
        lo, hi = state["columns"]
        return state["dd"].taylor_tree(state["buf"], state["case"]["block"])[:, lo:hi]
    if kind == "incoherent":
        hits = list(state["hits"])
        state["dd"].addIncoherentPower(state["buf"], hits)
        return {"drift_steps": np.array([h.drift_steps for h in hits], np.int64),
                "index": np.array([h.index for h in hits], np.int64),
                "incoherent_power": np.array([h.incoherent_power for h in hits], np.float32)}
    if kind == "normalize":
        y, loc, sd = sa.normalize(state["x"], state["dtype"])
        return {"y": y, "loc": loc, "std": sd}
    if kind == "forward":
        return state["net"].forward(state["tiles"])
    grad, loss = state["net"].gradient(state["tiles"], state["labels"])
    return {"grad": grad, "loss": loss}


# ---------------------------------------------------------------------------
# What a pass cannot do without.

_SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def _search_work(T, N, max_drift, dtype):
    bmin, bmax, _ = _drift_range(T, max_drift)
    T_r = _rounded(T)
    # One float per path sum and level (the pairwise tree), the running maximum aside.
    return T_r * N * _SIZE[dtype], (bmax - bmin + 1) * T_r * N * math.log2(T_r)


def work(case):
    kind = case["kind"]
    if kind == "search":
        b, f = _search_work(case["T"], case["N"], case["max_drift"], case["dtype"])
        return {"bytes": b, "flops": f}
    if kind == "batch":
        each = [_search_work(T, N, case["max_drift"], case["dtype"]) for T, N in _shapes(case)]
        share = case["gate"] or 1.0
        return {"bytes": sum(b for b, _ in each), "flops": share * sum(f for _, f in each)}
    if kind == "tree":
        T_r, N = _rounded(case["T"]), case["N"]
        return {"bytes": T_r * N * (_SIZE[case["dtype"]] + 4), "flops": T_r * N * math.log2(T_r)}
    if kind == "incoherent":
        T_r = _rounded(case["T"])
        return {"bytes": case["hits"] * T_r * _SIZE[case["dtype"]], "flops": case["hits"] * (T_r - 1)}
    if kind == "normalize":
        n = case["T"] * case["N"]
        return {"bytes": n * (4 + _SIZE[case["dtype"]]), "flops": 5 * n}
    macs = 16 * 512 * 16 * 15 + 8 * 256 * 32 * 240 + 4 * 128 * 32 * 480 + 512 * 32
    return {"bytes": case["B"] * 16 * 1024 * 2 + 4 * 23393, "flops": 2.0 * case["B"] * macs}


# ---------------------------------------------------------------------------
# The same results in 64 bits, with torch alone.

def _tree64(x, T_r, b):
    """Path sums [T_r][N] of drift block b for every start channel (samples outside are zero)."""
    N = x.shape[1]
    wide = N + T_r
    pad = (T_r - 1) * abs(b) + T_r
    xp = torch.nn.functional.pad(x, (pad, pad))
    v = torch.stack([xp[t, pad + t * b:pad + t * b + wide] for t in range(T_r)]).unsqueeze(1)
    L = 2
    while L <= T_r:
        # v [T_r/half][half offsets][wide]: combine neighbours, the second shifted by (p + 1) // 2.
        half = L // 2
        first, second = v[0::2], v[1::2]
        w = torch.zeros((T_r // L, L, wide), dtype=x.dtype, device=x.device)
        for p in range(L):
            s = (p + 1) // 2
            w[:, p, :wide - s] = first[:, p // 2, :wide - s] + second[:, p // 2, s:]
        v, L = w, 2 * L
    return v[0, :, :N]


def _search64(x, T, max_drift, snr):
    """(snr, power) of the hits, in ascending channel order, with zeros up to one per window."""
    T_r, N = x.shape
    x = x.double()
    sums = x.sum(0).sort().values
    median = float(sums[N // 2])
    kept = sums[math.ceil(0.05 * N):math.floor(0.95 * N) + 1]
    sd = float((kept - kept.mean()).square().mean().sqrt())
    threshold = snr * sd + median
    bmin, bmax, window = _drift_range(T, max_drift)
    top = torch.zeros(N, dtype=torch.float64, device=x.device)
    chan = torch.arange(N, device=x.device)
    offs = torch.arange(T_r, device=x.device)[:, None]
    for b in range(bmin, bmax + 1):
        last = chan + (T_r - 1) * b
        v = _tree64(x, T_r, b)
        v = torch.where((last >= 0) & (last + offs < N), v, 0.0)
        top = torch.maximum(top, v.amax(0))
    top = top.cpu().numpy()
    power = []
    for i in range(0, N, window):
        c = i + int(np.argmax(top[i:i + window]))
        if top[c] > threshold and not (top[max(0, c - window + 1):c + window] > top[c]).any():
            power.append(top[c])
    out = np.zeros((2, _windows(T, N, max_drift)))
    out[0, :len(power)] = (np.array(power) - median) / sd
    out[1, :len(power)] = power
    return out


def _network64(p, z):
    """Block logits; bfloat16 weights and activations as the network stores them."""
    def rounded(v):
        return v + (v.float().to(torch.bfloat16).double() - v).detach()

    def conv(x, w, b, sh, sw):
        B, C, H, W = x.shape
        cols = torch.nn.functional.unfold(x, (3, 5), padding=(1, 2), stride=(sh, sw))
        y = rounded(w) @ cols + b[:, None]
        return rounded(torch.relu(y)).reshape(B, len(b), H // sh, W // sw)

    at = np.cumsum([0, 240, 16, 7680, 32, 15360, 32, 32, 1])
    w1, b1, w2, b2, w3, b3, wh, bh = (p[a:b] for a, b in zip(at[:-1], at[1:]))
    h = conv(z[:, None], w1.reshape(16, 15), b1, 1, 2)
    h = conv(h, w2.reshape(32, 15, 16).transpose(1, 2).reshape(32, 240), b2, 2, 2)
    h = conv(h, w3.reshape(32, 15, 32).transpose(1, 2).reshape(32, 480), b3, 2, 2)
    s = (h.flatten(2) * wh[:, None]).sum(1) + bh
    return s.gather(1, s.argmax(1, keepdim=True)).squeeze(1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        tiles, labels = _tiles(case["B"], seed)
        p = torch.from_numpy(_params(seed)).cuda().double()
        if kind == "forward":
            with torch.no_grad():
                return torch.cat([_network64(p, t.double()) for t in tiles.split(64)])
        p.requires_grad_(True)
        loss = 0.0
        for t, y in zip(tiles.split(64), labels.double().split(64)):
            part = torch.nn.functional.binary_cross_entropy_with_logits(
                _network64(p, t.double()), y, reduction="sum") / case["B"]
            part.backward()
            loss += float(part)
        return {"grad": p.grad, "loss": torch.tensor([loss], dtype=torch.float64)}
    if kind == "batch":
        if case["gate"]:
            return None  # which blocks are searched is the network's decision
        pairs = [_search64(_channel(T, N, case["max_drift"], seed * 1009 + i, case["dtype"]), T,
                           case["max_drift"], case["snr"]) for i, (T, N) in enumerate(_shapes(case))]
        return {"index": None, "drift_steps": None, "drift_rate": None, "frequency": None,
                "snr": np.concatenate([a for a, _ in pairs]),
                "power": np.concatenate([b for _, b in pairs])}
    T, N = case["T"], case["N"]
    if kind == "normalize":
        x = _waterfall(T, N, 5.0, seed)[:T].double()
        loc = x.sum(0).sort().values[N // 2] / T
        sd = (x - x.mean()).square().mean().sqrt()
        return {"y": ((x - loc) / sd).clamp(-65504.0, 65504.0), "loc": float(loc), "std": float(sd)}
    x = _channel(T, N, case.get("max_drift", 5.0), seed, case["dtype"])
    if kind == "search":
        snr, power = _search64(x, T, case["max_drift"], case["snr"])
        return {"index": None, "drift_steps": None, "drift_rate": None, "frequency": None,
                "snr": snr, "power": power}
    if kind == "tree":
        lo, hi = _valid_columns(case)
        return _tree64(x.double(), _rounded(T), case["block"])[:, lo:hi]
    # The hits in the order addIncoherentPower leaves them (by drift), each with its path's sum.
    hits = _hit_list(case, seed)
    T_r = _rounded(T)
    order = sorted(range(len(hits)), key=lambda k: hits[k].drift_steps)
    y, out = x.double().cpu().numpy(), []
    for k in order:
        block, p = divmod(hits[k].drift_steps, T_r - 1)
        out.append(sum(y[t, hits[k].index + t * block + _shift(t, p, T_r)] for t in range(T_r)))
    return {"drift_steps": None, "index": None, "incoherent_power": np.array(out)}


def _shift(t, p, T_r):
    """Channels that path offset p has moved by at time step t (drift block 0)."""
    s, L = 0, T_r
    while L > 1:
        half = L // 2
        if t >= half:
            s += (p + 1) // 2
            t -= half
        p, L = p // 2, half
    return s
