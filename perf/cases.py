"""Performance cases of the k-mer counting framework, through its public entry points.

Reads are drawn on the GPU from a seeded genome (GC content, interspersed and tandem repeats,
substitution errors, both strands), as the benchmark's read sets are, and handed over as the host
CSR arrays that every entry point takes. Six kinds of work, over read sets of a loader batch to
tens of millions of reads:

  resident  a batch already uploaded goes through phase 1 and the count and the table stays in
            HBM, as in a benchmark step: what both calls return comes back, every partition's
            bytes, superkmers, k-mers and rows and the distinct total (a copy of the whole table
            to the host would take many times the pass);
  table     the whole call of a program that wants its table: host reads in, the rows of every
            partition in ascending key order out;
  store     the counting call of the drop-in: reference-format partitions from the host, the
            ordered table out;
  stream    a loader's uneven batches appended into capacity-sized regions, then counted;
  sized     phase 1 and count with predicted region sizes (learned sizing);
  gradient  one loss and gradient of the sizing network on a training batch.
"""
import math

import numpy as np
import torch

from rapidgkc_amd import native

ALL = 0xFFFFFFFF
HIST_BINS, STATS = 4 ** 5, 3  # the sizing network's minimizer histogram and batch statistics


def _case(name, kind, reads, read_len, genome, k, p, parts, cmin=1, err=0.01, gc=0.41, repeats=0.10, tandem=0.0,
          long_bases=0, ragged=False, batches=0):
    c = {"kind": kind, "reads": reads, "read_len": read_len, "genome": genome, "k": k, "p": p, "parts": parts,
         "cmin": cmin, "err": err, "gc": gc, "repeats": repeats, "tandem": tandem, "long_bases": long_bases,
         "ragged": ragged, "batches": batches}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one loader batch of the reference (2000 reads) counted by itself: launches and latency
        _case("loader_batch", "table", 2_000, 150, 100_000, 31, 11, 512),
        # a small sequencing run, error k-mers dropped (min-count 2): the 1 Mbp benchmark workload, reads in, table out
        _case("uniform_1m_table", "table", 200_000, 150, 1_000_000, 31, 11, 512, cmin=2, err=0.005, gc=0.5, repeats=0.0),
        # a bacterial-size set at 30x, quality-trimmed reads of mixed lengths, min-count 2: reads in, table out
        _case("trimmed_30x_table", "table", 1_000_000, 151, 5_000_000, 31, 11, 512, cmin=2, ragged=True),
        # the headline workload's reads (30x, 1% errors, 10% repeats) at half its genome: one benchmark step
        _case("genome_30x", "resident", 10_000_000, 150, 50_000_000, 31, 11, 512),
        # short and long reads together, k=25, p=9: the mixed benchmark workload, a fifth of it
        _case("mixed_k25", "resident", 1_333_333, 150, 10_000_000, 25, 9, 512, err=0.005, gc=0.5, repeats=0.0,
              long_bases=20_000_000),
        # 128-bit keys: the k=55 tandem-repeat benchmark workload, a quarter of it
        _case("tandem_k55", "resident", 2_000_000, 250, 50_000_000, 55, 13, 512, gc=0.40, repeats=0.0, tandem=0.25),
        # 128-bit keys with the table as the product, few partitions
        _case("k55_table", "table", 60_000, 250, 1_000_000, 55, 13, 64, cmin=2, gc=0.40, repeats=0.0, tandem=0.05),
        # stores made elsewhere (the host phase 1, .skm files) counted through the drop-in's call
        _case("host_store", "store", 700_000, 150, 7_000_000, 31, 11, 512, cmin=2),
        # a loader handing over uneven batches of short and long reads
        _case("stream_k25", "stream", 666_667, 150, 5_000_000, 25, 9, 512, err=0.005, gc=0.5, repeats=0.0,
              long_bases=10_000_000, batches=32),
        # learned sizing: regions from predicted counts instead of a sizing pass
        _case("sized_30x", "sized", 4_000_000, 150, 20_000_000, 31, 11, 512),
        # the sizing network's training batch (16 genomes, 512 partitions, two heads)
        {"name": "sizer_gradient", "kind": "gradient", "batch": 16, "parts": 512, "hidden": 128},
    ]


def draw(rng):
    kind = rng.choice(["table", "table", "resident", "resident", "resident", "store", "stream", "sized", "gradient"])
    if kind == "gradient":
        return {"kind": kind, "batch": rng.randint(1, 64), "parts": rng.choice([64, 127, 256, 512, 1000]),
                "hidden": rng.choice([64, 100, 128])}
    k, p = rng.choice([(21, 7), (25, 9), (31, 11), (31, 11), (32, 11), (33, 11), (47, 13), (55, 13)])
    read_len = rng.choice([100, 125, 150, 151, 250, rng.randint(76, 300)])
    cov = rng.uniform(8, 40)
    most = {"table": 1.5e8, "store": 1e8, "stream": 1.2e8, "sized": 6e8, "resident": 1.5e9}[kind] / (3 if k > 32 else 1)
    bases = math.exp(rng.uniform(math.log(3e5 if kind != "stream" else 3e6), math.log(most)))
    longs = kind in ("resident", "stream") and rng.random() < 0.4
    reads = max(100, int(bases * (0.9 if longs else 1.0) / read_len)) | 1
    # a minimizer of 7 bases has few values: such sets are small ones
    if p == 7:
        reads = min(reads, 400_001)
    return _case(None, kind, reads, read_len, max(20_000, int(reads * read_len / cov)), k, p,
                 rng.choice([31, 64, 128, 300, 512, 512, 1000]), cmin=2 if kind in ("table", "store") else rng.choice([1, 1, 2]),
                 err=round(rng.uniform(0.002, 0.015), 4), gc=round(rng.uniform(0.35, 0.6), 3),
                 repeats=round(rng.uniform(0.0, 0.3), 3), tandem=rng.choice([0.0, 0.0, 0.1]),
                 long_bases=int(bases * 0.1) if longs else 0, ragged=rng.random() < 0.4,
                 batches=rng.randint(4, 48) if kind == "stream" else 0)


# ---- inputs ----------------------------------------------------------------------------------
def _genome(c, gen):
    """Bases 0..3 (A C G T) of the genome."""
    n, dev = c["genome"], "cuda"
    u = torch.rand(n, generator=gen, device=dev)
    at = (1.0 - c["gc"]) / 2.0
    g = (u >= at).to(torch.uint8) + (u >= 0.5).to(torch.uint8) + (u >= 1.0 - at).to(torch.uint8)
    blk = min(3000, n // 8)
    m = int(c["repeats"] * n / blk)
    slots = torch.randperm(n // blk, generator=gen, device=dev)
    if m:  # copies of other parts at 2% divergence
        span = torch.arange(blk, device=dev)
        src = torch.randint(0, n - blk, (m, 1), generator=gen, device=dev) + span
        cp = g[src]
        sub = torch.rand(m, blk, generator=gen, device=dev) < 0.02
        cp = torch.where(sub, (cp + 1) & 3, cp)
        g[slots[:m, None] * blk + span] = cp
    t = min(int(c["tandem"] * n / blk), n // blk - m)
    if t:  # blocks filled with a unit of 2 to 200 bases
        span = torch.arange(blk, device=dev)
        unit = torch.randint(2, min(201, blk), (t, 1), generator=gen, device=dev)
        base = slots[m:m + t, None] * blk
        g[base + span] = g[base + span % unit]
    return g


def _cut(g, lens, err, gen):
    """Reads of the given lengths at random places and strands with substitutions, as one array."""
    dev, n = g.device, len(g)
    lens = lens.to(dev)
    start = (torch.rand(len(lens), generator=gen, device=dev, dtype=torch.float64) * (n - lens + 1)).long()
    rev = torch.rand(len(lens), generator=gen, device=dev) < 0.5
    ends = torch.cumsum(lens, 0)
    place = torch.arange(int(ends[-1]), device=dev) - torch.repeat_interleave(ends - lens, lens)
    r = torch.repeat_interleave(rev, lens)
    at = torch.repeat_interleave(start, lens) + torch.where(r, torch.repeat_interleave(lens, lens) - 1 - place, place)
    b = g[at]
    b = torch.where(r, 3 - b, b)
    wrong = torch.rand(len(b), generator=gen, device=dev) < err
    shift = torch.randint(1, 4, (len(b),), generator=gen, device=dev, dtype=torch.uint8)
    return torch.where(wrong, (b + shift) & 3, b)


def _reads(c, seed):
    """(chars, offs) of the case's reads: host arrays, long reads spread among the short ones."""
    gen = torch.Generator(device="cuda").manual_seed(1 + int(seed))
    host = torch.Generator().manual_seed(1 + int(seed))
    g = _genome(c, gen)
    ascii_ = torch.tensor(list(b"ACGT"), dtype=torch.uint8, device="cuda")
    n = c["reads"]
    lens = torch.full((n,), c["read_len"], dtype=torch.int64)
    if c["ragged"]:  # trimmed: half the reads keep their length, the others lose up to half of it
        cut = torch.rand(n, generator=host) * 0.5 * (torch.rand(n, generator=host) < 0.5)
        lens = (lens * (1.0 - cut)).long()
    if c["long_bases"]:  # log-normal, mean 10 kbp, sd 6 kbp, 5% errors
        sigma = math.sqrt(math.log(1.36))
        m = max(1, c["long_bases"] // 10_000)
        ll = torch.exp(torch.randn(m, generator=host) * sigma + math.log(10_000) - sigma * sigma / 2)
        ll = ll.long().clamp(100, min(100_000, c["genome"] // 2))
        pos = torch.sort(torch.randint(0, n, (m,), generator=host)).values
    else:
        ll, pos = torch.zeros(0, dtype=torch.int64), torch.zeros(0, dtype=torch.int64)
    # pieces of at most ~64 M bases keep the index arrays small
    step = max(1, 64_000_000 // c["read_len"])
    all_lens, total = [], int(lens.sum()) + int(ll.sum())
    chars = torch.empty(total, dtype=torch.uint8, pin_memory=True)
    at = done = 0
    for lo in range(0, n, step):
        hi = min(n, lo + step)
        last = hi == n
        here = len(ll) if last else int((pos < hi).sum())
        pieces = [(lens[lo:hi], c["err"])]
        if here > done:
            pieces.append((ll[done:here], 0.05))
            done = here
        for ls, err in pieces:
            b = ascii_[_cut(g, ls, err, gen).long()]
            chars[at:at + len(b)].copy_(b)
            at += len(b)
            all_lens.append(ls)
    offs = np.zeros(len(lens) + len(ll) + 1, dtype=np.uint64)
    np.cumsum(torch.cat(all_lens).numpy(), out=offs[1:])
    del g
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return chars.numpy(), offs


def _net_inputs(c, seed):
    """Features, targets and weights of the sizing network, as its training loop makes them:
    standardised clipped features, targets around the training mean, He-initialised weights."""
    rng = np.random.default_rng(int(seed))
    n_in, h, n_out = HIST_BINS + 3 * c["parts"] + STATS, c["hidden"], 2 * c["parts"]
    x = np.clip(rng.standard_normal((c["batch"], n_in)), -8, 8).astype(np.float32)
    t = (0.3 * rng.standard_normal((c["batch"], n_out))).astype(np.float32)
    w = []
    for a, b in ((n_in, h), (h, h), (h, n_out)):
        w += [(rng.standard_normal(a * b) * math.sqrt(2.0 / a)).astype(np.float32), (0.01 * rng.standard_normal(b)).astype(np.float32)]
    return (n_in, h, h, n_out), x, t, np.concatenate(w)


def _most_rows(c):
    """Rows a program makes room for: every k-mer, or with a min-count what the genome can repeat."""
    n = c["reads"] * max(1, c["read_len"] - c["k"] + 1) + c["long_bases"]
    return n if c["cmin"] == 1 else min(n // c["cmin"], 3 * c["genome"]) + 4096


def prepare(case, seed):
    c = dict(case, counter=native.Counter(0))
    cnt = c["counter"]
    if c["kind"] == "gradient":
        dims, c["x"], c["t"], w = _net_inputs(case, seed)
        c["net"] = native.Mlp(cnt, *dims)
        c["net"].set_params(w)
        return c
    chars, offs = _reads(case, seed)
    k, p, parts = c["k"], c["p"], c["parts"]
    if c["kind"] in ("table", "store"):  # the program's buffers for the table
        cap = _most_rows(case)
        c["keys"] = np.zeros(cap * (1 if k <= 32 else 2), dtype=np.int64)
        c["counts"] = np.zeros(cap, dtype=np.int32)
    if c["kind"] == "resident":
        cnt.set_reads(chars, offs)
    elif c["kind"] == "table":
        c["chars"], c["offs"] = chars.copy(), offs  # a program's ordinary arrays
    elif c["kind"] == "store":
        maker = native.Counter(0)
        maker.set_reads(chars, offs)
        c["part_offs"], _, _ = maker.superkmers(k, p, parts)
        c["store"] = maker.copy_store(int(c["part_offs"][-1]))
        maker.close()
    else:
        # region sizes as a prediction gives them: 15% over the true counts
        cnt.set_reads(chars, offs)
        po, skm, _ = cnt.superkmers(k, p, parts)
        c["cap_bytes"] = (np.diff(po).astype(np.float64) * 1.15).astype(np.uint64) + np.uint64(512)
        c["cap_recs"] = (skm.astype(np.float64) * 1.15).astype(np.uint64) + np.uint64(64)
        if c["kind"] == "sized":
            rows, _ = cnt.count(1, ALL)
            c["distinct"] = rows.astype(np.float64)
        else:
            rng = np.random.default_rng(int(seed))
            n = len(offs) - 1
            b = [0] + sorted(int(v) for v in rng.choice(np.arange(1, n), c["batches"] - 1, replace=False)) + [n]
            c["loaded"] = [(chars[int(offs[i]):int(offs[j])].copy(), (offs[i:j + 1] - offs[i]).astype(np.uint64))
                           for i, j in zip(b[:-1], b[1:])]
            c["max_reads"] = max(len(o) - 1 for _, o in c["loaded"])
            c["max_bases"] = max(len(s) for s, _ in c["loaded"])
    return c


# ---- one pass --------------------------------------------------------------------------------
def _ordered_table(s, rows):
    """Each partition's rows ascending by key, partition after partition, in the program's buffers
    (128-bit keys as pairs of 64-bit words)."""
    cnt = s["counter"]
    cnt.sort_rows()
    if int(rows.sum()) > len(s["counts"]):
        raise RuntimeError("more rows than the program's buffers hold")
    if native.lib().rgkc_copy_table(cnt._h, s["keys"].ctypes.data, s["counts"].ctypes.data):
        raise RuntimeError("the table could not be copied")
    return s["keys"], s["counts"]


def run(s):
    cnt = s["counter"]
    if s["kind"] == "gradient":
        return s["net"].grad(s["x"], s["t"])
    k, p, parts, cmin = s["k"], s["p"], s["parts"], s["cmin"]
    if s["kind"] == "store":
        rows, distinct = cnt.count_host_store(s["store"], s["part_offs"], parts, k, p, cmin, ALL)
        return rows.view(np.int64), distinct, _ordered_table(s, rows)
    if s["kind"] == "stream":
        cnt.stream_begin(k, p, parts, s["max_reads"], s["max_bases"], s["cap_bytes"], s["cap_recs"])
        for chars, offs in s["loaded"]:
            cnt.stream_add(chars, offs)
        made = cnt.stream_end()
    elif s["kind"] == "sized":
        made = cnt.superkmers_sized(k, p, parts, s["cap_bytes"], s["cap_recs"])
        cnt.set_sizing(s["distinct"], margin=0.1)
    else:
        if s["kind"] == "table":
            cnt.set_reads(s["chars"], s["offs"])
        made = cnt.superkmers(k, p, parts)
    rows, distinct = cnt.count(cmin, ALL)
    counters = [v.view(np.int64) for v in (*made, rows)]
    if s["kind"] == "table":
        return counters, distinct, _ordered_table(s, rows)
    return counters, distinct


# ---- what a pass cannot do without ---------------------------------------------------------------
def work(case):
    c = case
    if c["kind"] == "gradient":
        n_in, h, n_out = HIST_BINS + 3 * c["parts"] + STATS, c["hidden"], 2 * c["parts"]
        params = n_in * h + h + h * h + h + h * n_out + n_out
        # features and targets in, weights read (16 bits) and gradients written (32 bits)
        return {"bytes": 4 * c["batch"] * (n_in + n_out) + 6 * params,
                "flops": 2 * c["batch"] * (3 * (params - n_in * h) + 2 * n_in * h)}
    mean_len = c["read_len"] * (0.875 if c["ragged"] else 1.0)
    bases = c["reads"] * mean_len + c["long_bases"]
    short = c["reads"] * max(0.0, mean_len - c["k"] + 1)
    n = short + c["long_bases"]
    true = c["genome"] * (1.0 - math.exp(-n / c["genome"]))
    false = short * (1.0 - (1.0 - c["err"]) ** c["k"]) + c["long_bases"] * (1.0 - 0.95 ** c["k"])
    rows = true + (false if c["cmin"] == 1 else 0.0)
    row_bytes = 12 if c["k"] <= 32 else 20
    # reads (or their packed records, about 1.4 bytes a k-mer) in, table rows out
    return {"bytes": (1.4 * n if c["kind"] == "store" else bases + 8.0 * c["reads"]) + rows * row_bytes, "flops": 0}


def exact(case, seed):
    """The gradient in 64 bits; the counts are whole numbers."""
    if case["kind"] != "gradient":
        return None
    dims, x, t, w = _net_inputs(case, seed)
    wt = torch.from_numpy(w)
    x, t = torch.from_numpy(x).double(), torch.from_numpy(t).double()
    ws, bs, o = [], [], 0
    for a, b in zip(dims[:-1], dims[1:]):
        ws.append(wt[o:o + a * b].bfloat16().double().reshape(a, b).requires_grad_())  # weights are read in bf16
        bs.append(wt[o + a * b:o + a * b + b].double().requires_grad_())
        o += a * b + b
    h = x
    for i in range(3):
        h = h @ ws[i] + bs[i]
        h = torch.relu(h) if i < 2 else h
    loss = ((h - t) ** 2).mean()
    loss.backward()
    return np.concatenate([v.grad.numpy().reshape(-1) for i in range(3) for v in (ws[i], bs[i])]), float(loss.detach())
