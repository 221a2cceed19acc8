"""KMatch with max_freq 1 (the device path that counts k-mers in buckets and chains on the device)
against KMatch's steps restated position by position (kmatch/KMatch.cc:21-318): records, their
order and the run's counts, at the sizes where that path can go wrong -- tiles of 1024 joined
positions, groups of 4096 positions, the look-back limit of 64, k-mers repeated more often than
one wave counts, table slots that no k-mer fills, many short records."""
from __future__ import annotations

import numpy as np
import pytest

from satsuma2_amd._lib import RESULT_DTYPE

pytestmark = pytest.mark.gpu

STRIDE = 10_000_000_000
CODE = {c: i for i, c in enumerate(b"ACGT")} | {c: i for i, c in enumerate(b"acgt")}
COMP = bytes.maketrans(b"ACGT", b"TGCA")


def table(records, K):
    """(entries that occur once, by k-mer, without the last; how many there were)."""
    seen, slots, filled = {}, 0, 0
    for index, s in enumerate(records, 1):
        if not s:
            continue
        slots += len(s) + 1 - K
        f = r = have = 0
        for p, c in enumerate(s):
            b = CODE.get(c)
            have = 0 if b is None else have + 1
            b = b or 0
            f = ((f << 2) | b) & ((1 << (2 * K)) - 1)
            r = (r >> 2) | ((3 - b) << (2 * (K - 1)))
            if have >= K:
                filled += 1
                pos = p - K + 2 + index * STRIDE
                k, v = (f, pos) if f <= r else (r, -pos)
                seen[k] = v if k not in seen else None
    for _ in range(min(2, slots - filled)):  # unfilled slots are entries {0, 0}
        seen[0] = 0 if 0 not in seen else None
    kept = sorted((k, v) for k, v in seen.items() if v is not None)
    return dict(kept[:-1]), len(kept)


def expected(query, target, K, min_length, jump):
    q, nq = table(query, K)
    t, nt = table(target, K)
    joined = sorted((abs(v), abs(t[k]), (not v > 0) != (not t[k] > 0)) for k, v in q.items() if k in t)
    lengths = [len(s) for s in query if s]
    out, active = [], []

    def close(b):
        q0, t0, rev, n = b
        if n + K >= min_length:
            qid = (q0 // STRIDE - 1) % 2**64
            tt = t0 - n if rev else t0
            out.append((qid, (t0 // STRIDE - 1) % 2**64, lengths[qid] if qid < len(lengths) else 0,
                        (q0 % STRIDE - 1) % 2**64, (tt % STRIDE - 1) % 2**64, n + K, rev, (0,) * 7, 1.0, 1.0))

    for qi, ti, rev in joined[1:]:  # the first joined position is skipped
        used, keep = False, []
        for b in active:
            d = qi - b[0]
            if d == (b[1] - ti if b[2] else ti - b[1]) and d - b[3] <= jump and b[2] == rev:
                b[3], used = d, True
            if d - b[3] > jump:
                close(b)
            else:
                keep.append(b)
        active = keep
        if not used:
            active.append([qi, ti, rev, 0])
    for b in active:
        close(b)
    return np.array(out, RESULT_DTYPE), nq, nt, len(joined)


@pytest.fixture(scope="module")
def ctx():
    from satsuma2_amd.api import Context

    c = Context(0)
    yield c
    c.close()


def rnd(rng, n):
    return np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, n)].tobytes()


def genomes(name):
    rng = np.random.default_rng(len(name))
    g = rnd(rng, 4200)
    if name.startswith("same "):  # a chain of that many joined positions (one is skipped, one dropped)
        s = rnd(rng, int(name[5:]))
        return [s], [s]
    if name == "reverse":
        return [g], [g.translate(COMP)[::-1]]
    if name == "records":
        return ([g[:1000], b"", g[1000:2500], rnd(rng, 31), g[2500:]],
                [rnd(rng, 40), g[500:3000], b"", g[3100:], rnd(rng, 32)])
    if name == "short records":
        q = [rnd(rng, int(n)) for n in rng.integers(31, 80, 200)]
        return q, [rnd(rng, int(n)) for n in rng.integers(31, 80, 150)] + [q[7] + q[90], g]
    if name == "changes":
        a = bytearray(g)
        for p in rng.integers(0, len(a), 90):
            a[p] = b"ACGTN"[int(rng.integers(0, 5))]
        return [g], [bytes(a[:1500]).lower() + bytes(a[1500:2600]).translate(COMP)[::-1] + bytes(a[2500:])]
    if name == "repeats":  # more copies of a k-mer than one wave counts, on both sides
        return [b"A" * 17000 + g + b"ACCTG" * 17000], [g[:3000] + b"CAGGT" * 17500 + b"T" * 40000]
    if name == "one unfilled":  # exactly one slot of either table is not filled
        return [b"N" + g[:300]], [b"N" + g[100:400]]
    assert name == "nothing"
    return [b"N" * 300], [g]


NAMES = ["same 62", "same 1035", "same 1046", "same 2069", "reverse", "records", "short records", "changes", "repeats",
         "one unfilled", "nothing"]


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("K,min_length,jump", [(3, 3, 2), (11, 11, 10), (21, 40, 20), (21, 21, 0), (31, 31, 64)])
def test_unique_kmers(ctx, name, K, min_length, jump):
    from satsuma2_amd.kmatch import kmatch

    query, target = genomes(name)
    print(f"[kmatch] {name} K={K} jump={jump}", flush=True)
    got, st = kmatch(ctx, query, target, K, min_length, jump, 1)
    want, nq, nt, joined = expected(query, target, K, min_length, jump)
    assert (st["query_kept"], st["target_kept"], st["joined"]) == (nq, nt, joined)
    assert got.tobytes() == want.tobytes()


def test_look_back_limit(ctx):
    """A gap of 64 is bridged on the device, 65 by the general path: the same step apart."""
    from satsuma2_amd.kmatch import kmatch

    rng = np.random.default_rng(5)
    a, b = rnd(rng, 400), rnd(rng, 400)
    for gap in (63, 64, 65, 66):
        query, target = [a + rnd(rng, gap - 11) + b], [a + rnd(rng, gap - 11) + b]
        for jump in (64, 65):
            got, _ = kmatch(ctx, query, target, 11, 11, jump, 1)
            assert got.tobytes() == expected(query, target, 11, 11, jump)[0].tobytes(), (gap, jump)


@pytest.mark.parametrize("jump", [20, 65])
@pytest.mark.parametrize("order", ["sls", "lsl", "ssl", "lss", "l", "s"])
def test_long_and_short_records(ctx, order, jump):
    """Neighbours cut from one sequence: a letter missing between two records gives k-mers across the cut."""
    from satsuma2_amd.kmatch import kmatch

    rng = np.random.default_rng(11)
    g = rnd(rng, 140000)
    query, at = [], 0
    for c in order:
        for n in (65536 + 3 * at % 7,) if c == "l" else (40, 31, 700):
            query.append(g[at:at + n])
            at += n
    target = [g[max(0, at - 900):at - 300], g[at - 300:at]] + query[::-1]
    for q, t in ((query, target), (query, [g[:at]])):
        got, st = kmatch(ctx, q, t, 15, 15, jump, 1)
        want, nq, nt, joined = expected(q, t, 15, 15, jump)
        assert (st["query_kept"], st["target_kept"], st["joined"]) == (nq, nt, joined)
        assert got.tobytes() == want.tobytes()


def one_bucket(n, bits, seed):
    """n records of 31 bases whose k-mers fall into bucket 0 of 2^bits (sxc_kmatch_unique.h: mix)."""
    rng = np.random.default_rng(seed)
    f = rng.integers(0, 1 << 62, n << (bits + 1), dtype=np.uint64)
    rc = np.zeros_like(f)
    for i in range(31):
        rc = (rc << np.uint64(2)) | (np.uint64(3) - ((f >> np.uint64(2 * i)) & np.uint64(3)))
    h = np.minimum(f, rc)
    for _ in range(2):
        h = h * np.uint64(0x9E3779B97F4A7C15)
        h ^= h >> np.uint64(32)
    f = f[(h & np.uint64((1 << bits) - 1)) == 0][:n]
    assert len(f) == n
    code = np.stack([(f >> np.uint64(2 * (30 - i))) & np.uint64(3) for i in range(31)], 1).astype(np.uint8)
    return [bytes(r) for r in np.frombuffer(b"ACGT", np.uint8)[code]]


@pytest.mark.parametrize("name", ["one wave", "several workgroups", "full", "just over"])
def test_more_kmers_than_a_bucket_holds(ctx, name):
    """More than 1024 different k-mers in one bucket: the general path decides, after the device path has
    run in part.  Records, order and counts as ever, and the next run on the context is its own."""
    from satsuma2_amd.kmatch import kmatch

    rng = np.random.default_rng(len(name))
    if name == "one wave":  # 1500 table slots: 4 buckets
        r = one_bucket(1250, 2, 1)
        query, target = r[:750], r[500:]
    elif name == "several workgroups":  # 20000 slots: 64 buckets, one of more than 16384 entries
        r = one_bucket(3000, 6, 2)
        query = r[:1800] + [r[int(i)] for i in rng.integers(0, 700, 8200)]
        target = r[1000:] + [r[int(i)] for i in rng.integers(1500, 2400, 8000)]
    else:  # 1024 k-mers fill the table, 1025 do not fit
        r = one_bucket(1024 if name == "full" else 1025, 2, 3)
        query, target = r[:700], r[300:]
    target = [t.translate(COMP)[::-1] if k % 3 == 0 else t for k, t in enumerate(target)]
    print(f"[kmatch] {name}: {len(query)} and {len(target)} records", flush=True)
    got, st = kmatch(ctx, query, target, 31, 31, 30, 1)
    want, nq, nt, joined = expected(query, target, 31, 31, 30)
    assert len(want) > 100
    assert (st["query_kept"], st["target_kept"], st["joined"], st["blocks"]) == (nq, nt, joined, len(want))
    assert got.tobytes() == want.tobytes()
    assert (st["sweep_ms"] > 0) == (name != "full")  # chained on the host: the general path
    q, t = genomes("records")
    got, st = kmatch(ctx, q, t, 21, 40, 20, 1)
    want, nq, nt, joined = expected(q, t, 21, 40, 20)
    assert (st["query_kept"], st["target_kept"], st["joined"]) == (nq, nt, joined)
    assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("tail", [b"A" * 26, b"AC" * 13, b"AGTACCATTGACATTTAGCAGGCATA"])
def test_kmers_that_differ_in_their_first_bases(ctx, tail):
    """All 1024 k-mers of five bases before one 26-mer, as before homopolymer runs, with a few hundred others:
    they spread over the buckets (the device path decides), from either strand."""
    from satsuma2_amd.kmatch import kmatch

    rng = np.random.default_rng(8)
    heads = [bytes(b"ACGT"[(k >> (2 * i)) & 3] for i in range(5)) for k in range(1024)]
    query = [h + tail for h in heads] + [rnd(rng, 31) for _ in range(200)]
    target = [h + tail for h in heads[::3]] + query[1000:] + [rnd(rng, 31) for _ in range(100)]
    target = [t.translate(COMP)[::-1] if k % 2 else t for k, t in enumerate(target)]
    got, st = kmatch(ctx, query, target, 31, 31, 30, 1)
    want, nq, nt, joined = expected(query, target, 31, 31, 30)
    assert len(want) > 100 and st["sweep_ms"] == 0
    assert (st["query_kept"], st["target_kept"], st["joined"]) == (nq, nt, joined)
    assert got.tobytes() == want.tobytes()
