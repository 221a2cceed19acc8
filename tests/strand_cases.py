"""Batches of chunk pairs with every form of chunk the pair and spectra kernels tell apart -- full and
odd lengths, a query of up to N bases, an empty one, letters of one, two and three bases, N runs,
signal tails -- and their oracle."""
import ctypes as C

import numpy as np

import oracle
from scan_cases import related
from satsuma2_amd import _lib


def batch(N: int, n: int, seed: int, tails: bool = True):
    """(pairs, target tails, query tails): n pairs of n distinct targets, the first ones long."""
    H = N // 2
    shapes = [(H, H), (H - 1, N - 5), (H - N // 8 + 3, H // 2 + 1), (H // 3, H), (H // 2 + 7, 0), (H, 60)]
    pairs, tt, qt = [], [], []
    rng = np.random.default_rng(seed)
    for k in range(n):
        lt, lq = shapes[k] if k < len(shapes) else (61 + (7 * k) % min(190, H - 61), 100 + (5 * k) % min(150, H - 100))
        t, q = related(lt, lq, ("acgt", "n_gap", "few")[k % 3], seed + k, reverse=k % 2 == 1)
        if k % 4 == 1:  # letters of three bases, whose channel sums are sequential
            t, q = (bytes(b"BDHV"[i % 4] if i % 37 == 5 else c for i, c in enumerate(s)) for s in (t, q))
        pairs.append(dict(tseq=t, qseq=q, t_record=k, q_record=k, q_record_len=len(q), fast=int(k % 7 == 3)))
        both = []
        for s in (t, q):
            tail = []
            if tails and k % 5 == 2 and len(s) + 300 <= N:
                a, b = (rng.choice(list(b"ACGTN"), len(s) + m).astype(np.uint8).tobytes() for m in (150, 300))
                tail = [(len(s) + 140, a, k % 2), (len(s) + 299, b, (k // 5) % 2)]
            both.append(tail)
        tt.append(both[0])
        qt.append(both[1])
    return pairs, tt, qt


def tail_table(tails):
    """sxc_signal_tail of every pair (and what it points to, to be kept)."""
    out, keep = (_lib.SignalTail * len(tails))(), []
    for k, segs in enumerate(tails):
        if segs:
            arr = (_lib.TailSeg * len(segs))(*[_lib.TailSeg(end, len(s), s, strand, 0) for end, s, strand in segs])
            keep.append((arr, segs))
            out[k] = _lib.SignalTail(arr, len(segs), 0)
    return out, keep


def reference(pairs, tt, qt, N, target_total=1e6):
    return np.concatenate(oracle.align_batch(pairs, oracle.make_params(N=N, target_total=target_total), threads=8,
                                             cap_per_pair=1024, t_tails=tt, q_tails=qt))


def pair_table(pairs):
    return (_lib.Pair * len(pairs))(*[_lib.Pair(p["tseq"], len(p["tseq"]), p["qseq"], len(p["qseq"]), 0, 0, p["t_record"],
                                                p["q_record"], p["q_record_len"], p["fast"]) for p in pairs])


def params(N, target_total=1e6):
    p = _lib.Params()
    C.memset(C.byref(p), 0, C.sizeof(p))
    p.N, p.q_chunk, p.strands, p.cutoff, p.cutoff_fast, p.min_prob, p.target_total = N, 4096, 2, 1.8, 2.9, 0.99, target_total
    return p
