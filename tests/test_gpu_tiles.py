"""Tiled partition of the counting path (k_pack, k_valid, k_split_main,
k_split, the run maps and the retry of the bucket count) at the sizes where
it can go wrong, bit-exact against the oracle: inputs that end just before,
at and after a 16-byte word, a 64-byte group, a 16 KiB block and a tile;
lines, headers and reads across those borders; tiles without a k-mer; buckets
with far more runs than a map holds, with more distinct keys than a table,
and with nearly all keys of the input."""
from __future__ import annotations

import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _p(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def ctx():
    from pakman_plus_amd import api
    c = api.Context(0)
    yield c
    c.close()


def _bases(rng, n, alpha=b"ACGT"):
    return bytes(rng.choice(np.frombuffer(alpha, dtype=np.uint8), n))


def _check(ctx, oracle_mod, fa, k):
    ctx.count(fa, k)
    keys, counts = ctx.table_host()
    want_k, want_c = oracle_mod.count(fa, k)
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)


@pytest.mark.parametrize("size", [15, 16, 17, 63, 64, 65, 16383, 16384, 16385, 16384 + 63, 32767, 32768, 32769,
                                  3 * 16384 - 1, 3 * 16384])
@pytest.mark.parametrize("newline", [True, False])
def test_one_read_ends_at_a_border(ctx, oracle_mod, size, newline):
    """One record whose input is `size` bytes long, with and without the
    final line end, at the smallest, a middle and the largest k."""
    rng = np.random.default_rng(size)
    body = size - 3 - int(newline)
    fa = b">h\n" + _bases(rng, body, b"ACGTN") + (b"\n" if newline else b"")
    assert len(fa) == size
    for k in (8, 31, 32, 33, 64):
        _p(f"case: border size={size} newline={newline} k={k}")
        _check(ctx, oracle_mod, fa, k)


@pytest.mark.parametrize("shift", [0, 1, 31, 62, 63, 64])
def test_line_ends_around_a_block_border(ctx, oracle_mod, shift):
    """A read's start, a header and a short read on either side of byte 16384;
    then 40 KiB of header (whole tiles without a k-mer) and two reads."""
    rng = np.random.default_rng(100 + shift)
    first = b">a\n"
    fa = first + _bases(rng, 16384 - len(first) - shift) + b"\n>b\n" + _bases(rng, 40) + b"\n>c\n" + _bases(rng, 300)
    fa += b"\n>" + b"h" * 40960 + b"\n" + _bases(rng, 5000) + b"\n>d\n" + _bases(rng, 64) + b"\n"
    for k in (9, 32, 64):
        _p(f"case: block border shift={shift} k={k}")
        _check(ctx, oracle_mod, fa, k)


@pytest.mark.parametrize("k", [16, 32, 50])
@pytest.mark.parametrize("factor", [0.0, 0.02, 6.0])
def test_levels_and_retries(ctx, oracle_mod, k, factor):
    """All k-mers distinct (every table of the built-in size and of six times
    the load retries in several passes), at one, two and three levels."""
    rng = np.random.default_rng(7)
    fa = b"".join(b">r%d\n" % i + _bases(rng, 150) + b"\n" for i in range(6000))
    try:
        ctx.set_tuning(bucket_factor=factor)
        _p(f"case: levels k={k} bucket_factor={factor}")
        _check(ctx, oracle_mod, fa, k)
    finally:
        ctx.set_tuning()


@pytest.mark.parametrize("k", [21, 40])
def test_skewed_parent_with_many_short_runs(ctx, oracle_mod, k):
    """A-rich reads: one level-1 bucket holds most k-mers, so its rare second
    digits have a few keys in each of hundreds of tiles (more runs than a
    bucket's map), its common ones far more keys than a table."""
    rng = np.random.default_rng(11)
    reads = np.full((130_000, 100), ord("A"), dtype=np.uint8)
    hit = rng.random(reads.shape) < 0.02
    reads[hit] = rng.choice(np.frombuffer(b"CGT", dtype=np.uint8), int(hit.sum()))
    rows = np.concatenate([np.tile(np.frombuffer(b">r\n", dtype=np.uint8), (reads.shape[0], 1)), reads,
                           np.full((reads.shape[0], 1), 10, dtype=np.uint8)], axis=1)
    fa = rows.tobytes()
    try:
        ctx.set_tuning(l1_bits=6, bucket_factor=0.3)
        _p(f"case: skewed parent k={k}")
        _check(ctx, oracle_mod, fa, k)
    finally:
        ctx.set_tuning()


@pytest.mark.parametrize("klen,bits", [(11, 64), (32, 64), (40, 128), (64, 128)])
@pytest.mark.parametrize("reads", [1, 45, 700])
def test_builder_tiles(ctx, oracle_mod, klen, bits, reads):
    """Builder counts over one tile and several, with words that reach back
    to the read's start (klen below the word) and full ones."""
    rng = np.random.default_rng(klen + reads)
    fa = b"".join(b">r%d\n" % i + _bases(rng, 120, b"ACGTN") + b"\n" for i in range(reads))
    _p(f"case: builder tiles klen={klen} bits={bits} reads={reads}")
    n = ctx.builder_count(fa, klen, read_len=100, kmer_bits=bits)
    keys, counts = ctx.table_host()
    want_n, want_k, want_c = oracle_mod.builder_count(fa, klen, 100, bits)
    assert n == want_n
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)


@pytest.mark.parametrize("k", [12, 32, 33, 64])
@pytest.mark.parametrize("n", [1, 639, 640, 641, 20_000])
def test_macro_node_ranges(ctx, oracle_mod, k, n):
    """Node ranges of one element, of a full one and one more, and ranges
    with far more succ than pred elements (k-mers c + A...A + random: their
    succ keys crowd into a quarter of the pred keys' span), which are cut
    down, the records against the oracle's."""
    from pakman_plus_amd import api
    rng = np.random.default_rng(k * 1000 + n)
    same = min(10, k - 6)
    rows = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), (n, k))
    rows[:, 1:1 + same] = ord("A")
    fa = b"".join(b">r\n" + r.tobytes() + b"\n" for r in rows)
    _p(f"case: node ranges k={k} n={n}")
    ctx.count(fa, k)
    kept = ctx.cutoff_threshold(0)
    keys, counts = ctx.kept_host()
    assert kept == keys.shape[0]
    m = ctx.macro_nodes()
    got = api.nodes_as_arrays(ctx.nodes_host(), k)
    want = oracle_mod.macro_nodes(keys, counts, k)
    assert m == want["keys"].shape[0]
    for f in ("keys", "pre_cnt", "suf_cnt"):
        assert np.array_equal(got[f], want[f]), f


@pytest.mark.parametrize("k", [8, 9, 10, 11, 14, 15, 22, 23, 24, 32, 39, 40, 55, 56, 64])
def test_share_windows(ctx, k):
    """The share's window minima for every block size of the kernel and the
    edges between them, over reads shorter and longer than a tile, with clean
    stretches, isolated bytes whose third code bit is set, and runs of them;
    against the window-by-window restatement of the reference."""
    import rank_util as RU
    rng = np.random.default_rng(k)
    reads = []
    for n, p in ((k, 0.0), (k + 1, 0.3), (20_000, 0.0), (12_000, 0.002), (150, 0.0), (400, 0.05), (400, 1.0),
                 (k - 1, 0.0), (3_000, 0.2), (70, 0.02), (8_128 * 2, 0.0005)):
        r = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), n)
        bad = rng.random(n) < p
        r[bad] = rng.choice(np.frombuffer(b"NnHXYz", dtype=np.uint8), int(bad.sum()))
        reads.append(r.tobytes())
    reads.append(b"A" * 500 + b"N" + b"A" * 300)
    fa = b"".join(b">%d\n%s\n" % (i, r) for i, r in enumerate(reads))
    _p(f"case: share windows k={k}")
    freq = RU.lmer_freq(fa)
    assert np.array_equal(ctx.lmer_frequency(fa), freq)
    walk = RU.owner_walk(fa, k, 3, freq)
    for r in range(3):
        ctx.count_rank_share(fa, k, 3, r)
        keys, counts = ctx.table_host()
        assert RU.table_counter(keys, counts) == RU.share_counter(walk, r), r


def test_lmer_counts_past_16_bits(ctx):
    """L-mers of one kind filling a block's 16-bit counters several times over,
    between others, and frequencies that rank beyond the histogram's range."""
    rng = np.random.default_rng(5)
    acgt = np.frombuffer(b"ACGT", dtype=np.uint8)
    part = [b"A" * 3_000_000, rng.choice(acgt, 500_000).tobytes(), b"C" * 300_000, b"AC" * 100_000]
    reads = part * 8
    fa = b"".join(b">r\n" + r + b"\n" for r in reads)
    _p("case: L-mer counters past 16 bits")
    want = np.zeros(1 << 16, dtype=np.uint64)
    for r in part:
        c = (np.frombuffer(r, dtype=np.uint8) >> 1) & 3
        v = np.zeros(c.size - 7, dtype=np.int64)
        for j in range(8):
            v = (v << 2) | c[j:c.size - 7 + j]
        want += 8 * np.bincount(v, minlength=1 << 16).astype(np.uint64)
    assert np.array_equal(ctx.lmer_frequency(fa), want)
    ctx.count(fa, 31)
    keys, counts = ctx.table_host()
    full = dict(zip(keys[:, 0].tolist(), counts.tolist()))
    got = {}
    for r in range(2):
        ctx.count_rank_share(fa, 31, 2, r)
        keys, counts = ctx.table_host()
        one = dict(zip(keys[:, 0].tolist(), counts.tolist()))
        assert not set(one) & set(got)
        got.update(one)
    assert got == full


@pytest.mark.parametrize("u", [16_384 * 1024, 16_384 * 1024 + 1, 16_383, 16_385, 40])
@pytest.mark.parametrize("t", [2, 3])
def test_cutoff_plan(ctx, u, t):
    """Tables of one block of the cutoff, one entry less and more, and of as
    many blocks as one launch plans and one more entry: histogram, threshold
    and kept entries against the table's own counts."""
    rng = np.random.default_rng(u)
    k = 31
    r = rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), u + k - 1).tobytes()
    fa = b">a\n" + r + b"\n>b\n" + r[:min(u // 3 + k, 5000)] + b"\n"
    _p(f"case: cutoff u={u} t={t}")
    ctx.count(fa, k)
    keys, counts = ctx.table_host()
    assert keys.shape[0] == u
    hist, mb, nk = ctx.cutoff(t)
    want = np.bincount(counts, minlength=t)[:t].astype(np.uint64)
    assert np.array_equal(np.asarray(hist)[1:t], want[1:t])
    wmb = 1 + int(np.argmin(want[1:t]))
    keep = counts >= wmb
    assert mb == wmb and nk == int(keep.sum())
    kk, kc = ctx.kept_host()
    assert np.array_equal(kk, keys[keep]) and np.array_equal(kc, counts[keep])


@pytest.mark.parametrize("klen,bits", [(32, 64), (33, 64), (45, 64), (64, 128), (70, 128)])
@pytest.mark.parametrize("read_len", [70, 100, 120, 121, 122, 300])
def test_builder_window_ends(ctx, oracle_mod, klen, bits, read_len):
    """Words shorter than or equal to the window, counted from window ends:
    reads shorter than the line, equal to it, one and two bytes longer (the
    '\n', then the next record's '>'), and spanning records, whose windows
    overlap the next read's and need the read table."""
    rng = np.random.default_rng(klen + read_len)
    fa = b"".join(b">r%d\n" % i + _bases(rng, 120, b"ACGTN") + b"\n" for i in range(700))
    _p(f"case: builder window ends klen={klen} bits={bits} read_len={read_len}")
    n = ctx.builder_count(fa, klen, read_len=read_len, kmer_bits=bits)
    keys, counts = ctx.table_host()
    want_n, want_k, want_c = oracle_mod.builder_count(fa, klen, read_len, bits)
    assert n == want_n
    assert np.array_equal(keys.reshape(-1), np.asarray(want_k).reshape(-1))
    assert np.array_equal(counts, want_c)


@pytest.mark.parametrize("size", [1, 2, 13, 15, 16, 17, 31, 33, 100, 16_383, 16_384, 40_000])
@pytest.mark.parametrize("end", [b"\n", b"\r\n"])
def test_rewrite_by_output(ctx, oracle_mod, size, end):
    """Lines around a chunk, a block and more, and so short that a block holds
    more of them than its table, with and without a last line end."""
    rng = np.random.default_rng(size)
    n = max(3, min(9_000, 200_000 // size))
    _p(f"case: rewrite size={size} end={end!r}")
    seqs = [_bases(rng, int(rng.integers(max(size - 2, 0), size + 1)), b"ACGTN") for _ in range(n)]
    fq = b"".join(b"@%d" % (i % 10) + end + q + end + b"+" + end + b"I" * len(q) + end for i, q in enumerate(seqs))
    fa = b"".join((b">%d" % i + end if i % 5 == 0 else b"") + q + end for i, q in enumerate(seqs))
    for cut in (0, len(end)):
        for fmt, data in (("fastq", fq), ("fasta", fa)):
            data = data[:len(data) - cut]
            try:
                want = oracle_mod.normalize(data, fmt)
            except ValueError:  # an empty last line without its end is no line
                with pytest.raises(Exception, match="not a multiple of 4"):
                    ctx.normalize(data, fmt)
                continue
            assert ctx.normalize(data, fmt) == want, (fmt, cut)


def test_served_results_in_reused_blocks(ctx):
    """Result blocks of released jobs serve later jobs: sizes that fit a spare
    block, nearly fit and do not, two slots, results downloaded while others'
    blocks change hands."""
    from pakman_plus_amd import api
    rng = np.random.default_rng(11)
    sets = []
    for reads in (400, 430, 380, 2_000, 60, 405):
        one = b"".join(b">r\n" + _bases(rng, 90, b"ACGT") + b"\n" for _ in range(reads))
        sets.append(one * 3)
    want = []
    for fa in sets:
        ctx.count(fa, 31)
        want.append(ctx.table_host())
    srv = api.Server(0, n_slots=2)
    try:
        for rnd in range(4):
            order = rng.permutation(len(sets))
            _p(f"case: served round {rnd} order {order.tolist()}")
            tickets = [srv.submit(fasta=sets[int(i)], k=31, t=2) for i in order]
            for i, tk in zip(order, tickets):
                r = srv.wait(tk)
                got = srv.download(r)
                keys, counts = want[int(i)]
                assert np.array_equal(got["keys"], keys) and np.array_equal(got["counts"], counts)
                srv.release(tk)
    finally:
        srv.close()


@pytest.mark.parametrize("k", [21, 32, 55])
def test_budget_gives_idle_buffers_back(k):
    """Budgets below what a count holds without one: the same results, from
    buffers given back and asked for again, or PK_ENOMEM; two counts, cutoff
    and nodes per budget, and a count of the other kind between."""
    from pakman_plus_amd import api
    rng = np.random.default_rng(k)
    genome = _bases(rng, 30_000, b"ACGT")
    fa = b"".join(b">r\n" + genome[i:i + 100] + b"\n" for i in rng.integers(0, 29_900, 9_000))
    free = api.Context(0)
    free.count(fa, k)
    want = free.table_host()
    free.cutoff_threshold(2)
    free.macro_nodes()
    kept, nodes, held = free.kept_host(), free.nodes_host(), free.device_bytes
    free.close()
    done = 0
    for share in (1.0, 0.9, 0.8, 0.7, 0.6, 0.45):
        _p(f"case: budget k={k} share={share}")
        c = api.Context(0, int(held * share))
        try:
            for _ in range(2):
                c.count(fa, k)
                got = c.table_host()
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
                c.cutoff_threshold(2)
                c.macro_nodes()
                got = c.kept_host()
                assert np.array_equal(got[0], kept[0]) and np.array_equal(got[1], kept[1])
                assert np.array_equal(c.nodes_host(), nodes)
                assert c.device_bytes <= held * share
                try:  # needs more than the main path's count
                    c.builder_count(fa, k, read_len=90, kmer_bits=64 if k <= 32 else 128)
                except api.PakHipError as e:
                    assert e.code == api.PK_ENOMEM
            done += 1
        except api.PakHipError as e:
            assert e.code == api.PK_ENOMEM
        finally:
            c.close()
    assert done >= 2


def test_lmer_frequency_budgets():
    """L-mer frequencies with room for every block's table, for a few, and
    without room for the packed input (the read table's walk)."""
    from pakman_plus_amd import api
    import rank_util as RU
    rng = np.random.default_rng(2)
    fa = b"".join(b">r\n" + _bases(rng, 100, b"ACGTN") + b"\n" for _ in range(20_000))
    want = RU.lmer_freq(fa)
    done = 0
    for budget in (0, 40 << 20, 8 << 20, 4_200_000, 3_600_000, 3_300_000, 2_500_000):
        _p(f"case: L-mers budget={budget}")
        c = api.Context(0, budget)
        try:
            assert np.array_equal(c.lmer_frequency(fa), want)
            done += 1
        except api.PakHipError as e:
            assert e.code == api.PK_ENOMEM
        finally:
            c.close()
    assert done >= 4
