"""The scan's slices on the CPU workgroup emulator against the oracle: lengths around a slice's and
a window's ends, every kind of pair, every gate (the keep threshold's shortest run), more blocks
than the queue holds.  Records and the count of runs equal the oracle's; probabilities come from
the same library functions."""
import ctypes as C

import numpy as np
import pytest

import hostbuild
import oracle
from conftest import dense_run_pair
from scan_cases import GATES, LENGTHS, LETTERS, composed, related, short_runs
from test_emu import COLS, emu_batch


@pytest.fixture(scope="module")
def emu():
    return C.CDLL(hostbuild.emu_library())


def check(emu, pairs, N, target_total):
    got, _, st = emu_batch(emu, pairs, N=N, target_total=target_total)
    ref = np.concatenate(oracle.align_batch([dict(p, q_record_len=len(p["qseq"])) for p in pairs],
                                            oracle.make_params(N=N, target_total=target_total)))
    for c in COLS:
        assert np.array_equal(got[c], ref[c]), c
    for ps in range(2 * len(pairs)):
        p = pairs[ps // 2]
        qs = p["qseq"] if ps % 2 == 0 else oracle.reverse_complement(p["qseq"])
        xc = oracle.xcorr(oracle.encode(p["tseq"], N), oracle.encode(qs, N))
        assert st[ps, 1] == len(oracle.matchup(qs, p["tseq"], xc, 1.8)), (ps, len(p["tseq"]), len(qs))
    return ref


@pytest.mark.parametrize("letters", LETTERS)
def test_lengths(emu, letters):
    pairs = []
    for k, n in enumerate(LENGTHS):
        t, q = related(n, 1024 if k % 2 else n, letters, 31 * k + 5, reverse=k % 3 == 0)
        pairs.append(dict(tseq=t, qseq=q, t_record=k, q_record=k))
    assert len(check(emu, pairs, 2048, 1024.0 * 1024)) > 0


@pytest.mark.parametrize("letters", ["acgt", "few", "dense"])
@pytest.mark.parametrize("target_total", [1.0, 30.0, 1e3, 1e9])
def test_gates(emu, letters, target_total):
    pairs = []
    for k, n in enumerate((200, 700, 1000)):
        t, q = related(n, 1000, letters, 7 * k + 3, reverse=k == 1)
        pairs.append(dict(tseq=t, qseq=q, t_record=k, q_record=k))
    assert len(check(emu, pairs, 2048, target_total)) > 0


@pytest.mark.parametrize("letter", [b"", b"R"])
def test_more_blocks_than_the_queue(emu, letter):
    t = dense_run_pair(length=2048)
    t = t[:700] + letter + t[700 + len(letter):]
    assert len(check(emu, [dict(tseq=t, qseq=t, t_record=0, q_record=0)], 4096, 10.0)) > 0


@pytest.mark.parametrize("letters", ["acgt", "few", "words"])
@pytest.mark.parametrize("target_total,pure,general", GATES)
def test_every_gate(emu, target_total, pure, general, letters):
    """Gates 1, 2, 4 and 8, each by a target size whose shortest kept run asks for it; the runs start at
    every position of a block."""
    least = (C.c_int32 * 3)()
    emu.emu_min_run(C.c_double(0.99), C.c_double(target_total), least)
    assert [max(g for g in (1, 2, 4, 8) if g <= n) for n in (least[0], least[2])] == [pure, general]
    pairs = []
    for k in range(35):
        t, q = short_runs(500, letters, k) if k < 32 else related(900, 1000, letters, k, reverse=k == 33)
        pairs.append(dict(tseq=t, qseq=q, t_record=k, q_record=k))
    assert len(check(emu, pairs, 2048, target_total)) >= (3 if target_total > 1e8 else 25)


@pytest.mark.parametrize("split", ["", "16"])
@pytest.mark.parametrize("target_total", [1e3, 1e5, 1e6, 1e9])
def test_slices_or_segments(emu, monkeypatch, target_total, split):
    """General pairs on both sides of slices_pay's limits: composition, other letters, gate, share of lags.
    Each pair alone and in one batch."""
    if split:
        monkeypatch.setenv("SXC_EMU_SPLIT", split)
    pairs = []
    for k, (gc, other) in enumerate((g, o) for g in (0.1, 0.25, 0.35, 0.41, 0.5) for o in (0.0, 0.002, 0.005)):
        t, q = composed(1000 - 7 * k, 1024 - 31 * k, gc, other, 90 + k)
        pairs.append(dict(tseq=t, qseq=q, t_record=k, q_record=k))
    assert len(check(emu, pairs, 2048, target_total)) > 0
