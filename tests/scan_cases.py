"""Chunk pairs at the sizes where the scan's slices (29 blocks of 32 positions), its kinds of pair
and its queue change over."""
import numpy as np

# diagonals of 45 .. 47 positions (the window), 78 (block 1's flags), a slice's last block and the
# next one's first (32 * (29 t + 1) positions, t = 1, 2), whole and ragged words
LENGTHS = [1, 45, 46, 47, 63, 64, 65, 78, 959, 960, 961, 962, 992, 1007, 1024]
LETTERS = ["acgt", "n_gap", "few", "words", "dense", "zero"]


def other_letters(seq: bytes, letters: str, rng) -> bytes:
    s = bytearray(seq)
    n = len(s)
    if letters == "n_gap":
        s[n // 3: n // 3 + min(60, n // 3 + 1)] = b"N" * len(s[n // 3: n // 3 + min(60, n // 3 + 1)])
    elif letters == "few":  # a letter at the ends and one inside
        for at, c in ((0, b"R"), (n // 2, b"K"), (n - 1, b"Y")):
            s[at:at + 1] = c
    elif letters == "words":  # one word in 8 of both chunks, the most that is scanned in slices
        for w in range(0, n, 128):
            s[w] = ord("S")
    elif letters == "dense":
        for at in range(0, n, 9):
            s[at] = b"RYKMSWN"[int(rng.integers(7))]
    elif letters == "zero":  # a byte without a codec row
        s[n // 2] = ord("*")
    return bytes(s)


def related(lt: int, lq: int, letters: str, seed: int, reverse=False):
    """(target, query): random bases, the query's middle copied from the target with 12% changed."""
    rng = np.random.default_rng(seed)
    t = rng.choice(list(b"ACGT"), lt).astype(np.uint8)
    q = rng.choice(list(b"ACGT"), lq).astype(np.uint8)
    n = min(lt, lq) * 2 // 3
    if n:
        piece = t[(lt - n) // 2:(lt - n) // 2 + n].copy()
        change = rng.random(n) < 0.12
        piece[change] = rng.choice(list(b"ACGT"), int(change.sum()))
        if reverse:
            piece = np.frombuffer(piece.tobytes().translate(bytes.maketrans(b"ACGT", b"TGCA"))[::-1], np.uint8)
        at = (lq - n) // 3
        q[at:at + n] = piece
    return other_letters(t.tobytes(), letters, rng), bytes(q.tobytes())


# (target total, gate of pure pairs, gate of pairs with few other letters): the shortest stretch a kept run
# can have (keep_min_run) is looked for 1, 2, 4 or 8 positions at a time
GATES = [(1e3, 1, 1), (3e4, 2, 1), (5e4, 2, 1), (1e5, 4, 2), (2e5, 4, 2), (1e6, 4, 4), (4e6, 8, 4), (1e7, 8, 4), (1e9, 8, 8)]


def short_runs(n: int, letters: str, seed: int):
    """(target, query) whose kept runs are short: the target all G/C, the query all A/T but for stretches of
    24 to 40 positions where they agree, on as many A/T as G/C, so that little is expected by chance."""
    rng = np.random.default_rng(seed)
    t = rng.choice(list(b"GC"), n).astype(np.uint8)
    q = rng.choice(list(b"AT"), n).astype(np.uint8)
    shift, at = int(rng.integers(5, 40)), 60 + seed % 32
    while at + 110 < n - shift:
        m = int(rng.integers(24, 41))
        hit = at + rng.permutation(m)[:m - int(rng.integers(0, 4))]
        t[hit] = rng.permutation(np.resize(rng.permutation(list(b"ACGT")), len(hit)))
        q[hit + shift] = t[hit]
        at += m + int(rng.integers(50, 70))
    return other_letters(t.tobytes(), letters, rng), bytes(q.tobytes())


def composed(lt: int, lq: int, gc: float, other: float, seed: int):
    """(target, query) of a G/C content, related, with that share of other letters in both: pairs on either
    side of the limits up to which slices pay."""
    rng = np.random.default_rng(seed)
    p = [(1 - gc) / 2, gc / 2, gc / 2, (1 - gc) / 2]
    t, q = (rng.choice(list(b"ACGT"), n, p=p).astype(np.uint8) for n in (lt, lq))
    n = min(lt, lq) // 2
    q[lq - n:] = np.where(rng.random(n) < 0.15, q[lq - n:], t[:n])
    for s in (t, q):
        at = rng.random(len(s)) < other
        at[len(s) // 3] = True
        s[at] = rng.choice(list(b"RYKMSW"), int(at.sum()))
    return t.tobytes(), q.tobytes()
