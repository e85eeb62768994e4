"""Workloads by which the speed of this package is followed from change to change.

Each case is one thing that a program using the package has it do: count the
k-mers of a read set, mostly with the histogram cutoff and the macro nodes
after it, through the Python entry points of pakman_plus_amd.api (the C ABI
of include/pakhip.h underneath).  The listed cases go from a read set of a
megabyte, where launches and waits decide, to 1.2e9 two-word k-mers, where
memory does; draw() gives further cases of the same ranges.

Read sets are made on the GPU: a random genome (with repeat families where
the case says so), reads from uniform positions on either strand, independent
substitution errors.  The bases come from the seed; where the reads lie and
where their errors are comes from the case, so that read sets of one case
differ in every base and have tables of one size.  The input is resident on
the device before the pass, as a program that keeps its read sets in HBM has
it, except where a case says "host".  A context (or server) is created once
per state and kept, as every caller does.

Outputs are the tables themselves, read where they lie on the device.  Where
their size depends on the bases (short k, N bytes, one rank's share) the pass
ends as a program's does that keeps a table beyond the context's next count:
with a copy into arrays of its own.  All values are whole numbers (keys as
64-bit words, counts, node records as 32-bit words).
"""
import ctypes
import json
import math
import zlib

import numpy as np
import torch

from pakman_plus_amd import api

# ---------------------------------------------------------------------------
# The cases.
#
# kind   count    count + cutoff(t = 21) + macro nodes, input on the device
#        host     the same from host memory, the node records back on the host
#        noalloc  count into the caller's arrays without device allocation
#        thresh   count + the PaK-graph builder's threshold cutoff + nodes
#        fastq    count of four-line FASTQ with "\r\n" line ends
#        builder  the builder API's count (fixed read length, whole-word keys)
#        share    one rank's share at 8 ranks (minimum-L-mer owner)
#        batch    a batch of uneven read sets on a server with four slots
# g      genome length; cov, len, err: coverage, read length, error rate
# ragged read lengths are log-uniform in [len, len_max], and "n" per base is
#        the rate of N bytes


def listed():
    return [
        # A drop-in call on one small read set (a plasmid, an amplicon pool):
        # host bytes in, node records out.
        dict(name="host_plasmid", kind="host", g=20_000, cov=60.0, len=100, err=0.005, k=32),
        # A serving loop that counts small read sets into its own arrays.
        dict(name="noalloc_small", kind="noalloc", g=40_000, cov=40.0, len=100, err=0.005, k=32),
        # The small end-to-end workload of the benchmark: 1 Mbp, 30x.
        dict(name="small_k32", kind="count", g=1_000_000, cov=30.0, len=100, err=0.005, k=32),
        # The bacterial workload of the benchmark: 4.6 Mbp, 80x, 1 % errors.
        dict(name="bacterial_k32", kind="count", g=4_600_000, cov=80.0, len=100, err=0.01, k=32),
        # A bacterial set with two-word keys and an odd k.
        dict(name="bacterial_k63", kind="count", g=5_000_000, cov=50.0, len=150, err=0.005, k=63),
        # The large workload of the benchmark (repeat families, k = 64) at
        # 40 Mbp, so that several read sets' working memory fits the card.
        dict(name="large_k64", kind="count", g=40_000_000, cov=50.0, len=150, err=0.005, k=64, rep=0.05),
        # Trimmed reads of uneven length with N bytes, short k, threshold cutoff.
        dict(name="ragged_k21", kind="thresh", g=3_000_000, cov=40.0, len=30, len_max=301, err=0.005, n=0.001, k=21),
        # Long reads: kilobases each, a few thousand of them.
        dict(name="long_reads_k31", kind="count", g=2_500_000, cov=30.0, len=2_000, len_max=20_000, err=0.003, k=31),
        # A sequencer's own file format.
        dict(name="fastq_k31", kind="fastq", g=2_000_000, cov=50.0, len=125, err=0.005, k=31),
        # The stand-alone table builder: every read's 100 bytes, 64-bit words.
        dict(name="builder_k32", kind="builder", g=2_000_000, cov=60.0, len=100, err=0.005, k=32, bits=64),
        # One rank's share of a bacterial set at its real shape.
        dict(name="share_k32", kind="share", g=4_600_000, cov=40.0, len=100, err=0.01, k=32),
        # Uneven read sets counted together, as the batched benchmark does.
        dict(name="batch_k32", kind="batch", g=600_000, cov=40.0, len=100, err=0.005, k=32, sets=16),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["count", "count", "count", "count", "host", "noalloc", "thresh", "ragged", "long", "fastq",
                       "builder", "share", "batch"])
    c = dict(kind=kind, g=int(_log_uniform(rng, 5e4, 6e6)), len=rng.choice([75, 100, 101, 125, 150, 250]),
             err=round(_log_uniform(rng, 0.002, 0.01), 5))
    c["k"] = rng.choice([15, 21, 27, 31, 31, 32, 32, 33] if c["len"] < 125 else [15, 21, 25, 31, 32, 32, 41, 55, 64])
    if kind == "count" and rng.random() < 0.3:
        c.update(rep=0.05, g=int(_log_uniform(rng, 4e6, 1.5e7)))
    elif kind == "host":
        c["g"] = int(_log_uniform(rng, 1e4, 3e5))
    elif kind == "noalloc":
        c.update(g=int(_log_uniform(rng, 1e4, 4e4)), len=100, k=rng.choice([21, 27, 31, 32]))
    elif kind in ("thresh", "ragged"):
        c.update(kind="thresh" if kind == "thresh" else "count", len=rng.randint(25, 60), len_max=rng.randint(150, 600),
                 n=round(rng.uniform(0.0, 0.003), 5), k=rng.choice([15, 19, 21, 25, 31]))
    elif kind == "long":
        c.update(kind="count", len=rng.randint(1_000, 3_000), len_max=rng.randint(8_000, 30_000),
                 err=round(rng.uniform(0.001, 0.004), 5), k=rng.choice([21, 31, 32, 51]))
    elif kind == "builder":
        c["bits"] = rng.choice([64, 128])
        c["k"] = 32 if c["bits"] == 64 else rng.choice([41, 55, 64])
        c["len"] = max(c["len"], 100)
    elif kind == "share":
        c["k"] = rng.choice([21, 31, 32])
    elif kind == "batch":
        c.update(g=int(_log_uniform(rng, 2e5, 1e6)), sets=rng.randint(6, 20), k=rng.choice([31, 32, 55]), len=150)
    # coverage: 12 to 26 error-free k-mers per position and strand, so that
    # the cutoff keeps some
    length = c["len"] if not c.get("len_max") else (c["len"] + c["len_max"]) // 3
    whole = max(1.0 - c["k"] / length, 0.1) * (1.0 - c["err"]) ** c["k"]
    c["cov"] = round(2.0 * rng.uniform(12.0, 26.0) / whole, 2)
    if kind == "noalloc":
        c["cov"] = min(c["cov"], 40.0)
    elif not c.get("rep"):
        c["g"] = int(min(c["g"], 4e8 / c["cov"]))
    return c


# ---------------------------------------------------------------------------
# Read sets.

_CHUNK = 1 << 20  # reads made at a time


def _rand(shape, gen, dtype=torch.float32):
    return torch.rand(shape, device="cuda", generator=gen, dtype=dtype)


def _genome(case, lay, gen, g):
    """Base codes A0 C1 T2 G3 of a random genome of g bases; with "rep", that
    share of it is copies of 50 repeat families at 2 % divergence.  `gen`
    gives the bases, `lay` where the copies and their differences are."""
    x = torch.randint(0, 4, (g,), dtype=torch.uint8, device="cuda", generator=gen)
    rep = case.get("rep", 0.0)
    if rep:
        # a copy and 64 bases on either side that are as good as random, in a
        # slot of its own
        rs = np.random.RandomState(int(torch.randint(0, 1 << 30, (1,), device="cuda", generator=lay)))
        fam = [torch.randint(0, 4, (int(n) + 128,), dtype=torch.uint8, device="cuda", generator=gen)
               for n in rs.randint(300, 5001, 50)]
        left = int(rep * g)
        for slot in rs.permutation(g // 5_200):
            if left <= 0:
                break
            f = fam[rs.randint(0, len(fam))]
            n = f.numel()
            rate = torch.full((n,), 0.75, device="cuda")
            rate[64:n - 64] = 0.02
            sub = torch.randint(1, 4, (n,), dtype=torch.uint8, device="cuda", generator=lay)
            at = int(slot) * 5_200
            x[at:at + n] = torch.where(_rand(n, lay) < rate, (f + sub) & 3, f)
            left -= n - 128
    return x


def _bases(case, lay, genome, start, flip, off, n):
    """The bases at `off` within reads of length n that start at `start` on
    the strand `flip` (all broadcast together), with errors, as bytes."""
    at = torch.where(flip, start + n - 1 - off, start + off)
    b = genome[at] ^ (flip.to(torch.uint8) << 1)  # the complement flips bit 1
    sub = torch.randint(1, 4, b.shape, dtype=torch.uint8, device="cuda", generator=lay)
    b = torch.where(_rand(b.shape, lay) < case["err"], (b + sub) & 3, b)
    letters = torch.tensor(list(b"ACTG"), dtype=torch.uint8, device="cuda")[b.long()]
    if case.get("n"):
        letters[_rand(b.shape, lay) < case["n"]] = ord("N")
    return letters


def _digits(first, count, mark):
    """(count, 10) bytes: the mark and the read's number in nine digits."""
    v = torch.arange(first, first + count, device="cuda")
    p = torch.tensor([10 ** i for i in range(8, -1, -1)], device="cuda")
    d = ((v[:, None] // p) % 10 + 48).to(torch.uint8)
    return torch.cat([torch.full((count, 1), ord(mark), dtype=torch.uint8, device="cuda"), d], 1)


def _read_set(case, seed, g=None, cov=None, length=None):
    """The read set's bytes on the device: strict single-line FASTA, or
    FASTQ with "\r\n" line ends for kind "fastq"."""
    gen, lay = torch.Generator(device="cuda"), torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1_000_003 + 17)
    g = int(g or case["g"])
    L = int(length or case["len"])
    cov = float(cov or case["cov"])
    shape = json.dumps([{k: v for k, v in case.items() if k != "name"}, g, L, cov], sort_keys=True)
    lay.manual_seed(zlib.crc32(shape.encode()))
    genome = _genome(case, lay, gen, max(g, case.get("len_max", L) + 1))
    g = genome.numel()
    if case.get("len_max"):
        lo, hi = math.log(L), math.log(case["len_max"])
        mean = (case["len_max"] - L) / (hi - lo)
        R = max(1, int(g * cov / mean))
        n = torch.exp(lo + (hi - lo) * _rand(R, lay, torch.float64)).long()
        start = (_rand(R, lay, torch.float64) * (g - n + 1)).long()
        flip = _rand(R, lay) < 0.5
        first = torch.cumsum(n + 12, 0) - (n + 12)  # header of 10, its '\n', the bases, '\n'
        out = torch.full((int((n + 12).sum()),), 10, dtype=torch.uint8, device="cuda")
        out[(first[:, None] + torch.arange(10, device="cuda")).reshape(-1)] = _digits(0, R, ">").reshape(-1)
        many = max(1, int(_CHUNK * 100 / mean))
        for r0 in range(0, R, many):
            r = slice(r0, min(R, r0 + many))
            row = torch.repeat_interleave(torch.arange(r.start, r.stop, device="cuda"), n[r])
            c = torch.cumsum(n[r], 0) - n[r]
            off = torch.arange(row.numel(), device="cuda") - c[row - r.start]
            out[first[row] + 11 + off] = _bases(case, lay, genome, start[row], flip[row], off, n[row])
        return out
    R = max(1, int(g * cov / L))
    fastq = case["kind"] == "fastq"
    # '@' header "\r\n" bases "\r\n" '+' "\r\n" qualities "\r\n", or '>' header '\n' bases '\n'
    width = 10 + 2 + L + 2 + 1 + 2 + L + 2 if fastq else 10 + 1 + L + 1
    out = torch.empty((R, width), dtype=torch.uint8, device="cuda")
    off = torch.arange(L, device="cuda")[None, :]
    for r0 in range(0, R, _CHUNK):
        m = min(R, r0 + _CHUNK) - r0
        o = out[r0:r0 + m]
        start = torch.randint(0, g - L + 1, (m, 1), device="cuda", generator=lay)
        flip = _rand((m, 1), lay) < 0.5
        b = _bases(case, lay, genome, start, flip, off, L)
        o[:, :10] = _digits(r0, m, "@" if fastq else ">")
        if fastq:
            crlf = torch.tensor([13, 10], dtype=torch.uint8, device="cuda")
            o[:, 10:12] = crlf
            o[:, 12:12 + L] = b
            o[:, 12 + L:14 + L] = crlf
            o[:, 14 + L] = ord("+")
            o[:, 15 + L:17 + L] = crlf
            o[:, 17 + L:17 + 2 * L] = torch.randint(35, 74, (m, L), dtype=torch.uint8, device="cuda", generator=gen)
            o[:, 17 + 2 * L:] = crlf
        else:
            o[:, 10] = 10
            o[:, 11:11 + L] = b
            o[:, 11 + L] = 10
    return out.reshape(-1)


def _batch_shapes(case):
    """(genome, coverage, read length) of the sets of a batch: genomes spread
    evenly over a factor of 30 in their logarithm, the largest of length g."""
    n = case["sets"]
    lens = [75, 100, 150, 250] if case["k"] <= 32 else [150, 250]
    return [(int(case["g"] * 30.0 ** (-i / max(n - 1, 1))), case["cov"] * (0.75 + 0.5 * ((i * 7) % n) / n),
             lens[i % len(lens)]) for i in range(n)]


# ---------------------------------------------------------------------------
# What a program holds before the call, and the call.


class _Device:
    """A device array of the library, for torch.as_tensor; the tensor holds
    it, and it holds the context or server that the memory belongs to."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


def _view(owner, ptr, shape, typestr):
    dtype = torch.int64 if typestr == "<i8" else torch.int32
    if 0 in shape:
        return torch.empty(shape, dtype=dtype, device="cuda")
    return torch.as_tensor(_Device(owner, int(ptr), shape, typestr), device="cuda")


def _table(owner, n, words, keys, counts):
    return {"keys": _view(owner, keys, (int(n), int(words)), "<i8"),
            "counts": _view(owner, counts, (int(n),), "<i4")}


def _keeps(case):
    """Whether the pass ends with copies into the program's own arrays: the
    number of distinct k-mers depends on the bases."""
    return case["kind"] == "share" or case["k"] < 31 or case.get("n", 0.0) > 0


def _kept(state, **views):
    """The tables copied into the state's own arrays, kept for the next pass."""
    for name, v in views.items():
        own = state["own"][name]
        if v.shape[0] > own.shape[0]:
            raise RuntimeError(f"{name}: {v.shape[0]} entries, room for {own.shape[0]}")
        own[:v.shape[0]].copy_(v)
    return {name: state["own"][name] for name in views}


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "batch":
        sets = [_read_set(case, seed * 1000 + i, g, cov, length) for i, (g, cov, length) in enumerate(_batch_shapes(case))]
        state.update(sets=sets, server=api.Server(0, n_slots=4), tickets=[],
                     jobs=[dict(device_ptr=s.data_ptr(), nbytes=s.numel(), k=case["k"], t=21) for s in sets])
        torch.cuda.synchronize()
        return state
    reads = _read_set(case, seed)
    state["ctx"] = api.Context(0)
    if kind == "host":
        state["host"] = reads.cpu().numpy()
    else:
        state["reads"] = reads
    words = 1 if case["k"] <= 32 and case.get("bits", 64) == 64 else 2
    if kind == "noalloc":
        cap = reads.numel()
        state["keys"] = torch.zeros((cap, words), dtype=torch.int64, device="cuda")
        state["counts"] = torch.zeros(cap, dtype=torch.int32, device="cuda")
    elif kind != "host" and _keeps(case):
        _, table, nodes = _expected(case, case["g"], case["cov"], case["len"])
        cap = 100_000 + int(table * (0.3 if kind == "share" else 1.2))
        state["own"] = {"keys": torch.zeros((cap, words), dtype=torch.int64, device="cuda"),
                        "counts": torch.zeros(cap, dtype=torch.int32, device="cuda")}
        if kind in ("count", "thresh"):
            state["own"]["nodes"] = torch.zeros((200_000 + int(nodes * 2.0), 12), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    kind, k = case["kind"], case["k"]
    if kind == "batch":
        return _run_batch(state)
    ctx = state["ctx"]
    if kind == "host":
        ctx.count(state["host"], k)
        hist, mb, _ = ctx.cutoff(21)
        ctx.macro_nodes()
        nodes = ctx.nodes_host().view(np.int32).reshape(-1, 12)
        if _keeps(case):  # into a record array of the program's own
            own = np.zeros((200_000 + 3 * case["g"], 12), dtype=np.int32)
            own[:nodes.shape[0]] = nodes
            nodes = own
        return {"hist": hist.view(np.int64), "min_bucket": mb, "nodes": nodes}
    reads = state["reads"]
    where = dict(device_ptr=reads.data_ptr(), nbytes=reads.numel())
    if kind == "noalloc":
        n = ctx.count_noalloc(reads.data_ptr(), reads.numel(), k, state["keys"].data_ptr(), state["counts"].data_ptr(),
                              state["counts"].numel())
        return {"n": n, "keys": state["keys"], "counts": state["counts"]}
    out = {}
    if kind == "fastq":
        t = ctx.count_format(None, k, "fastq", **where)
    elif kind == "builder":
        out["reads"] = ctx.builder_count(None, k, read_len=case["len"], kmer_bits=case["bits"], **where)
        t = ctx.table
    elif kind == "share":
        t = ctx.count_rank_share(None, k, 8, 3, **where)
    else:
        t = ctx.count(None, k, **where)
    out.update(_table(ctx, t.n, t.words, t.keys_ptr, t.counts_ptr))
    if kind in ("count", "thresh"):
        if kind == "count":
            hist, out["min_bucket"], out["kept"] = ctx.cutoff(21)
            out["hist"] = hist.view(np.int64)
        else:
            out["kept"] = ctx.cutoff_threshold(4)
        m = ctx.macro_nodes()
        out["nodes"] = _view(ctx, ctx.nodes_ptr, (m, 12), "<i4")
    if _keeps(case):
        out["n"] = t.n
        with torch.cuda.stream(torch.cuda.ExternalStream(ctx.stream)):  # after the context's last kernels
            out.update(_kept(state, **{name: out[name] for name in state["own"]}))
    return out


def _run_batch(state):
    """Submits the batch, waits for every job and returns the resident tables
    and nodes; the results of the batch before are given back first."""
    srv = state["server"]
    for t in state["tickets"]:
        srv.release(t)
    state["tickets"] = srv.submit_batch(state["jobs"])
    out = []
    for t in state["tickets"]:
        r = api._JobResult()
        srv._check(srv._lib.pk_server_wait(srv._h, t, ctypes.byref(r)))
        if r.status:
            raise RuntimeError(r.message.decode(errors="replace"))
        out.append({**_table(srv, r.table.n, r.table.words, r.table.keys, r.table.counts),
                    "nodes": _view(srv, r.nodes.nodes, (int(r.nodes.n), 12), "<i4")})
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without: the input read once, the table and the nodes
# written once.  The number of distinct k-mers is the expected one: the
# genome's, seen on either strand, and one of its own for every k-mer
# instance with an error.


def _expected(case, g, cov, length):
    k, mean, per = case["k"], float(length), max(length - case["k"] + 1, 0)
    if case.get("len_max"):
        lo, hi, mean = math.log(length), math.log(case["len_max"]), 0.0
        mean = (case["len_max"] - length) / (hi - lo)
        per = max(mean - k + 1, 0.0)
    reads = max(1.0, g * cov / mean)
    inst = reads * per
    bad = 1.0 - (1.0 - case["err"]) ** k * (1.0 - case.get("n", 0.0)) ** k
    genome = min(2.0 * g, 4.0 ** k)
    table = min(4.0 ** k, genome + inst * bad)
    size = reads * (mean + 12.0) if case["kind"] != "fastq" else reads * (2.0 * mean + 21.0)
    return size, table, genome


def work(case):
    words = 1 if case["k"] <= 32 and case.get("bits", 64) == 64 else 2
    shapes = _batch_shapes(case) if case["kind"] == "batch" else [(case["g"], case["cov"], case["len"])]
    total = 0.0
    for g, cov, length in shapes:
        size, table, nodes = _expected(case, g, cov, length)
        if case["kind"] == "share":
            table /= 8.0
        total += size + table * (8 * words + 4)
        if case["kind"] in ("count", "thresh", "batch", "host"):
            total += nodes * 48.0
    return {"bytes": total, "flops": 0.0}
