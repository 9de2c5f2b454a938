"""Workloads of the correction engine that are timed.

Every case is work that a program built on `care_amd` has the engine do:
correcting reads of a resident read set (one pair, a batch, the whole set),
running a read set from host memory to corrected reads, listing the
candidates of reads, training the learned gate and evaluating it.  Read sets
are paired-end, drawn from a random genome with repeat families like the
simulator's repeat-pe and large-pe profiles: 2-bit packed, with the quality
widths the read store knows (none, 1, 2 or 8 bits per base), of one length or
ragged.

listed() holds the cases, draw(rng) gives further ones of the same ranges,
prepare() what a program holds before the call (the resident read set and its
tables, host arrays for the results, the gate's parameters), run() the call.
"""

import math

import numpy as np
import torch

import care_amd
from care_amd import gate

DEVICE = "cuda:0"

# Modes of correction: the plain method (every candidate, refinement), the
# plain method that also corrects the candidates of good anchors, and the
# gated one (the 20 candidates that most maps hit, no refinement, a learned
# gate on every doubtful column).
MODES = {
    "plain": {},
    "candidates": {"correct_candidates": 1},
    "gated": {"correction_type": 3, "candidate_limit": 20, "threshold_anchor": 0.99},
}


def _reads(name, kind, mode, reads, anchors, length, shortest, bits, maps, coverage, kmer=20):
    return {"name": name, "kind": kind, "mode": mode, "reads": reads, "anchors": anchors, "length": length,
            "shortest": shortest, "bits": bits, "maps": maps, "coverage": coverage, "kmer": kmer}


def listed():
    return [
        # one pair corrected against a small resident set: what an interactive caller waits for
        _reads("one-pair", "correct", "plain", 6000, 2, 150, 150, 2, 32, 30),
        # a small batch of trimmed (ragged) reads through the gate, a service's request
        _reads("small-gated-ragged", "correct", "gated", 20000, 250, 150, 75, 2, 32, 30),
        # a batch of reads of 100 to 250 bases with 1-bit qualities and other table options
        _reads("batch-plain-ragged", "correct", "plain", 60000, 10002, 250, 100, 1, 24, 50, 18),
        # long reads (2x300) without qualities, the whole of a small set
        _reads("long-plain-noqual", "correct", "plain", 40006, 40006, 300, 300, 0, 16, 30),
        # candidate correction with 8-bit qualities and 48 maps, a batch of a larger set
        _reads("batch-candidates", "correct", "candidates", 300000, 30000, 150, 150, 8, 48, 40),
        # the headline set, 1M reads of 150 bases at 30x, by the plain method
        _reads("set-plain", "correct", "plain", 1000000, 1000000, 150, 150, 2, 32, 30),
        # the headline set through the gate
        _reads("set-gated", "correct", "gated", 1000000, 1000000, 150, 150, 2, 32, 30),
        # a whole small program: context, upload, tables, gated correction
        _reads("program-small-gated", "program", "gated", 9998, 9998, 150, 150, 2, 32, 30),
        # a whole program over a bacterial-sized set, plain method
        _reads("program-plain", "program", "plain", 400002, 400002, 150, 150, 2, 32, 30),
        # candidate lists of a batch of reads, for overlap analyses
        _reads("candidate-lists", "query", "plain", 300000, 50001, 150, 150, 2, 32, 30),
        # one epoch of training the gate on its decision columns
        {"name": "gate-training", "kind": "train", "columns": 262147, "batch": 4096},
        # the gate's outputs on a validation set's columns
        {"name": "gate-evaluation", "kind": "infer", "columns": 500001},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["correct", "correct", "correct", "program", "query", "train", "infer"])
    if kind == "train":
        return {"kind": kind, "columns": _size(rng, 4096, 262147), "batch": rng.choice([1024, 4096, 4099])}
    if kind == "infer":
        return {"kind": kind, "columns": _size(rng, 100, 500001)}
    mode = rng.choice(["plain", "gated", "candidates"]) if kind != "query" else "plain"
    length = rng.choice([100, 101, 150, 151, 250, 300])
    shortest = length if rng.random() < 0.6 else max(40, int(length * rng.uniform(0.4, 0.9)))
    # at most the work of the largest listed set
    most = {"correct": 600000, "program": 200000, "query": 50000}[kind]
    if mode == "candidates":
        most = 30000
    most = int(most * min(1.0, (150.0 / length) ** 2))
    anchors = 2 * max(1, _size(rng, 2, most) // 2)
    reads = anchors if kind == "program" else min(600000, max(anchors, 2 * (_size(rng, 6000, 300000) // 2)))
    reads = max(reads, 2000)
    if kind == "program":
        anchors = reads
    maps, coverage, kmer = rng.choice([(32, 30, 20), (32, 30, 20), (16, 30, 20), (48, 40, 20), (24, 50, 18)])
    return {"kind": kind, "mode": mode, "reads": reads, "anchors": anchors, "length": length, "shortest": shortest,
            "bits": rng.choice([0, 1, 2, 2, 8]), "maps": maps, "coverage": coverage, "kmer": kmer}


# ---- inputs ----------------------------------------------------------------


def _genome(g, size):
    """Uniform bases with repeat families: about 7 % of the genome in copies of 1 to 5 kbp (shorter on small
    genomes), 5 to 20 copies a family, 1 % divergence."""
    seq = torch.randint(0, 4, (size,), generator=g, device=DEVICE, dtype=torch.int16)
    rng = np.random.default_rng(int(torch.randint(0, 2**31, (1,), generator=g, device=DEVICE).item()))
    for _ in range(max(1, round(size / 500000))):
        n = min(int(rng.integers(1000, 5001)), size // 20)
        template = torch.randint(0, 4, (n,), generator=g, device=DEVICE, dtype=torch.int16)
        for at in rng.integers(0, size - n, int(rng.integers(5, 21))):
            other = torch.randint(1, 4, (n,), generator=g, device=DEVICE, dtype=torch.int16)
            hit = torch.rand((n,), generator=g, device=DEVICE) < 0.01
            seq[at:at + n] = torch.where(hit, (template + other) & 3, template)
    return seq


def _pack(codes, bits, width):
    """Rows of `bits`-bit codes, first code in the top bits of 32-bit words."""
    per = 32 // bits
    words = (width + per - 1) // per
    rows = torch.zeros((codes.shape[0], words * per), device=DEVICE, dtype=torch.int32)
    rows[:, :width] = codes
    rows = rows.view(-1, words, per)
    out = torch.zeros(rows.shape[:2], device=DEVICE, dtype=torch.int32)
    for i in range(per):
        out |= rows[:, :, i] << (32 - bits * (i + 1))
    return out


def _read_set(case, seed):
    """Packed rows, lengths and quality rows of a paired-end read set, in host memory."""
    n, length, bits = case["reads"], case["length"], case["bits"]
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    lens = torch.randint(case["shortest"], length + 1, (n,), generator=g, device=DEVICE)
    size = max(4 * length + 2000, int(n * 0.5 * (length + case["shortest"]) / case["coverage"]))
    genome = _genome(g, size)
    ins = 2.0 * length + 0.2 * length * torch.randn((n // 2,), generator=g, device=DEVICE)
    ins = ins.round().long().clamp(length, 4 * length)
    start = (torch.rand((n // 2,), generator=g, device=DEVICE, dtype=torch.float64) * (size - ins + 1)).long()
    flip = torch.randint(0, 2, (n // 2,), generator=g, device=DEVICE)
    rev = torch.stack([flip, 1 - flip], 1).view(-1, 1)
    first = torch.stack([start, start], 1).view(-1, 1) + rev * (ins.repeat_interleave(2).view(-1, 1) - 1)
    i = torch.arange(length, device=DEVICE)
    base = genome[first + (1 - 2 * rev) * i].int()
    base = torch.where(rev == 1, 3 - base, base)
    # substitutions rise from 0.1 % to 2 % along a read
    p = 0.001 + 0.019 * i / max(1, length - 1)
    err = torch.rand((n, length), generator=g, device=DEVICE) < p
    other = torch.randint(1, 4, (n, length), generator=g, device=DEVICE, dtype=torch.int32)
    base = torch.where(err, (base + other) & 3, base)
    live = i < lens.view(-1, 1)
    seqs = _pack(torch.where(live, base, 0), 2, length)
    quals = None
    if bits == 8:
        # phred 35 on correct bases and 12 on substituted ones, as characters
        q = torch.where(err, 33 + 12, 33 + 35)
        rows = torch.zeros((n, (length + 3) // 4 * 4), device=DEVICE, dtype=torch.uint8)
        rows[:, :length] = torch.where(live, q, 0).to(torch.uint8)
        quals = rows.cpu().numpy().view(np.uint32)
    elif bits:
        # phred scores around the substitution rate, binned
        q = (-10 * torch.log10(p) + 2 * torch.randn((n, length), generator=g, device=DEVICE)).round().clamp(2, 41)
        bins = (q > 13).int() if bits == 1 else (q > 4).int() + (q > 13).int() + (q > 20).int()
        quals = _pack(torch.where(live, bins, 0), bits, length).cpu().numpy().view(np.uint32)
    return seqs.cpu().numpy().view(np.uint32), lens.int().cpu().numpy(), quals


def _columns(case, seed):
    """Decision columns as the gate sees them: shares, supports and flags of MSA columns, mostly in 0..1, and
    labels that depend on them."""
    rng = np.random.default_rng(int(seed))
    x = rng.random((case["columns"], 32), dtype=np.float32)
    x[:, 21:25] = x[:, 21:25] < 0.1
    x[:, [6, 7, 14, 15, 16, 26, 27, 30]] *= 1.5
    z = 6.0 * (x[:, 2] + x[:, 3] - x[:, 0] - x[:, 8]) + rng.standard_normal(len(x), dtype=np.float32)
    return x, (z > 0).astype(np.uint8)


def _parameters(seed):
    """A fresh 32-64-32-16-1 network."""
    rng = np.random.default_rng(int(seed) + 77)
    parts = []
    for outputs, inputs in ((64, 32), (32, 64), (16, 32), (1, 16)):
        limit = math.sqrt(6.0 / inputs)
        parts += [rng.uniform(-limit, limit, outputs * inputs), rng.uniform(-0.1, 0.1, outputs)]
    return np.concatenate(parts).astype(np.float32)


class State:
    """What a program holds: the engine, its inputs and its result arrays."""

    def __init__(self):
        self.engine = None

    def close(self):
        if self.engine is not None:
            self.engine.close()
            self.engine = None

    def __del__(self):
        self.close()


def _options(case):
    return care_amd.default_options(
        kmer_length=case["kmer"], num_hash_maps=case["maps"], coverage=float(case["coverage"]), paired_end=1,
        use_quality=int(case["bits"] > 0), **MODES[case["mode"]])


def _load(engine, s):
    if s.case["mode"] == "gated":
        engine.mlp_load(s.gate)
    engine.upload(s.seqs, s.lens, None, s.quals, s.case["bits"] or 8, s.case["length"])
    engine.build()


def prepare(case, seed):
    s = State()
    s.case = case
    if case["kind"] in ("train", "infer"):
        s.x, s.y = _columns(case, seed)
        s.params = _parameters(seed)
        s.engine = care_amd.Engine(care_amd.default_options(correction_type=3))
        return s
    s.seqs, s.lens, s.quals = _read_set(case, seed)
    s.gate = gate.load(gate.DEFAULT_GATE)
    n = case["anchors"]
    pitch = (case["length"] + 15) // 16 * 16
    # a batch starts inside the set where it is not the whole of it
    s.first = (case["reads"] - n) // 2 & ~1
    if case["kind"] == "query":
        s.ids = care_amd.pinned_empty((n * 8 * case["coverage"] + 4096,), np.uint32)
        s.ids[:] = 0
        s.offsets = np.zeros(n + 1, dtype=np.int32)
    else:
        s.out = (care_amd.pinned_empty((n,), np.uint8), care_amd.pinned_empty((n, pitch), np.uint8))
        if case["mode"] == "candidates":
            cap = 24 * n + 4096
            s.out += (care_amd.pinned_empty((cap,), np.uint32), care_amd.pinned_empty((cap, pitch), np.uint8))
            s.device_lens = torch.from_numpy(s.lens).to(DEVICE)
            s.merged = (torch.zeros((cap,), device=DEVICE, dtype=torch.int64),
                        torch.zeros((cap, pitch), device=DEVICE, dtype=torch.uint8))
        # ragged rows are read up to each read's length
        s.live = None
        if case["shortest"] < case["length"]:
            lens = s.lens[s.first:s.first + n]
            s.live = np.where(np.arange(pitch) < lens[:, None], np.uint8(255), np.uint8(0))
    if case["kind"] != "program":
        s.engine = care_amd.Engine(_options(case))
        _load(s.engine, s)
    return s


# ---- the work --------------------------------------------------------------


def _in_order(s, ids, rows):
    """Corrected candidates by read id, as a program merges them (they come in no order): rows on the device,
    sorted by id and, within a read, by content, at the front of the program's arrays."""
    ids = torch.from_numpy(ids.view(np.int32)).to(DEVICE).long()
    rows = torch.from_numpy(rows).to(DEVICE)
    live = torch.arange(rows.shape[1], device=DEVICE) < s.device_lens[ids].view(-1, 1)
    rows = torch.where(live, rows, 0)
    key = torch.zeros_like(ids)
    for word in rows.view(torch.int64).unbind(1):
        key = key * 6364136223846793005 + word
    order = torch.argsort(key)
    order = order[torch.argsort(ids[order], stable=True)]
    torch.index_select(ids, 0, order, out=s.merged[0][:len(order)])
    torch.index_select(rows, 0, order, out=s.merged[1][:len(order)])
    return s.merged


def _correct(s, engine):
    n = s.case["anchors"]
    status, seqs, ids, rows = engine.correct(s.first, n, candidate_capacity=len(s.out[2]) if len(s.out) > 2 else None,
                                             out=s.out)
    # rows of reads that stay as they are hold nothing
    seqs[np.flatnonzero((status & 1) == 0)] = 0
    if s.live is not None:
        np.bitwise_and(seqs, s.live, out=seqs)
    got = [status, seqs[:, :s.case["length"]]]
    if s.case["mode"] == "candidates":
        got += _in_order(s, ids, rows)
    return got


def run(s):
    kind = s.case["kind"]
    if kind == "train":
        return s.engine.mlp_train(s.x, s.y, s.params, epochs=1, batch=s.case["batch"], lr=1e-3, seed=1)
    if kind == "infer":
        return s.engine.mlp_infer(s.x, s.params)
    if kind == "query":
        # into the program's own buffers, by the C interface (include/care_amd.h)
        e = s.engine
        code = e.lib.care_minhash_query(e.ctx, s.first, s.case["anchors"], s.ids.ctypes.data, s.offsets.ctypes.data,
                                        s.ids.size)
        if code != care_amd.CARE_OK:
            raise care_amd.CareError(e.lib.care_last_error().decode())
        return s.ids, s.offsets
    if kind == "program":
        with care_amd.Engine(_options(s.case)) as engine:
            _load(engine, s)
            return _correct(s, engine)
    return _correct(s, s.engine)


def work(case):
    if case["kind"] == "train":
        # features and labels in; forward, input and weight gradients
        return {"bytes": case["columns"] * 129, "flops": case["columns"] * 3 * 2 * 4624}
    if case["kind"] == "infer":
        return {"bytes": case["columns"] * 132, "flops": case["columns"] * 2 * 4624}
    mean = 0.5 * (case["length"] + case["shortest"])
    row = 4 * ((case["length"] + 15) // 16) + 4 * ((case["length"] * case["bits"] + 31) // 32) + 4
    # reads that overlap an anchor enough to be candidates, and the table entries that name them
    cands = min(20.0, case["coverage"] * 1.4) if case["mode"] == "gated" else case["coverage"] * 1.4
    probes = case["maps"] * 24 + 4 * case["maps"] * 0.4 * case["coverage"]
    n = case["anchors"]
    if case["kind"] == "query":
        return {"bytes": n * (probes + 4 * cands + 4), "flops": 0}
    moved = n * (row + probes + cands * row + mean + 1)
    # one comparison of the overlap and one weighted vote per base of every candidate
    flops = n * cands * mean * 4
    if case["kind"] == "program":
        # rows up, every read's k-mer hashes in every map, tables written once
        moved += case["reads"] * (row + 24 * case["maps"])
        flops += case["reads"] * case["maps"] * mean
    return {"bytes": moved, "flops": flops}


# ---- 64-bit values ---------------------------------------------------------


def _layers(params):
    p = params.astype(np.float64)
    out, at = [], 0
    for outputs, inputs in ((64, 32), (32, 64), (16, 32), (1, 16)):
        w = p[at:at + outputs * inputs].reshape(outputs, inputs)
        at += outputs * inputs
        out.append((w, p[at:at + outputs]))
        at += outputs
    return out


def _forward(layers, x):
    acts = [x]
    for k, (w, b) in enumerate(layers):
        z = acts[-1] @ w.T + b
        acts.append(np.maximum(z, 0.0) if k < 3 else z)
    return acts


def _order(n, seed):
    """Shuffled row order of an epoch (Fisher-Yates over splitmix64)."""
    mask = (1 << 64) - 1
    state = (seed * 0x9E3779B97F4A7C15 + 0x632BE59BD9B4E019) & mask
    perm = list(range(n))
    for i in range(n - 1, 0, -1):
        state = (state + 0x9E3779B97F4A7C15) & mask
        z = ((state ^ (state >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % (i + 1)
        perm[i], perm[j] = perm[j], perm[i]
    return np.array(perm)


def exact(case, seed):
    if case["kind"] not in ("train", "infer"):
        return None  # bytes and read ids
    x, y = _columns(case, seed)
    x = x.astype(np.float64)
    params = _parameters(seed).astype(np.float64)
    if case["kind"] == "infer":
        return _forward(_layers(params), x)[-1][:, 0]
    m, v, losses = np.zeros_like(params), np.zeros_like(params), []
    perm = _order(len(x), 1)
    for step, at in enumerate(range(0, len(x), case["batch"]), 1):
        rows = perm[at:at + case["batch"]]
        layers = _layers(params)
        acts = _forward(layers, x[rows])
        z, t = acts[-1][:, 0], y[rows].astype(np.float64)
        losses.append(np.mean(np.logaddexp(0.0, z) - t * z))
        d = ((1.0 / (1.0 + np.exp(-z)) - t) / len(rows))[:, None]
        parts = []
        for k in range(3, -1, -1):
            parts.append((d.T @ acts[k], d.sum(0)))
            if k:
                d = (d @ layers[k][0]) * (acts[k] > 0)
        grad = np.concatenate([a.ravel() for pair in reversed(parts) for a in pair])
        m = 0.9 * m + 0.1 * grad
        v = 0.999 * v + 0.001 * grad * grad
        params = params - 1e-3 * (m / (1 - 0.9**step)) / (np.sqrt(v / (1 - 0.999**step)) + 1e-8)
    return params, np.array([np.mean(losses)])
