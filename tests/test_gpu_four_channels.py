"""The pair and spectra kernels that take a chunk's four channels in one workgroup, on the GPU against
the oracle.  Launches of at most 128 strands (or target chunks) take a workgroup per channel, in the
default geometry; the batches here have more of both, so every compiled geometry runs: full and odd
lengths, queries up to N, letters of three bases (whose window entropies and channel sums take their own
path), N runs, signal tails.
Bar: accepted lags, coordinates, lengths, strands, identities bit-exact; prob within 1e-11 relative."""
import ctypes as C

import numpy as np
import pytest

import oracle
from conftest import unpack2
from strand_cases import batch, pair_table, params, reference, tail_table
from test_gpu_parity import GEOMETRIES, assert_results_equal

pytestmark = pytest.mark.gpu

PAIRS = 133  # 266 strands and 133 target chunks
DEFAULT = {nb: (32 if nb == 15 else 16, 3, 0, 0) for nb in range(9, 16)}


@pytest.fixture(scope="module")
def ctx():
    from satsuma2_amd.api import Context

    c = Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def cases():
    made = {}

    def of(nb):
        if nb not in made:
            N = 1 << nb
            pairs, tt, qt = batch(N, PAIRS, 10 * nb)
            lags = []
            for p, t, q in zip(pairs[:6], tt, qt):
                for qs in (p["qseq"], oracle.reverse_complement(p["qseq"])):
                    xc = oracle.xcorr(oracle.encode(p["tseq"], N), oracle.encode(qs, N))
                    lags.append(None if t or q else oracle.findtop(xc, 2.9 if p["fast"] else 1.8))
            made[nb] = pairs, tt, qt, reference(pairs, tt, qt, N), lags
        return made[nb]

    return of


def run_and_check(ctx, nb, case):
    """The batch with its signal tails, run eagerly and replayed."""
    from satsuma2_amd._lib import Result, check

    pairs, tt, qt, ref, lags = case
    L, h, prm = ctx.L, C.c_void_p(), params(1 << nb)
    t, keep_t = tail_table(tt)
    q, keep_q = tail_table(qt)
    check(L.sxc_batch_create_tails(ctx.handle, pair_table(pairs), len(pairs), C.byref(prm), t, q, C.byref(h)))
    try:
        for k in range(2):
            check(L.sxc_batch_run(h))
            out = np.zeros(len(ref) + 64, oracle.RESULT_DTYPE)
            n = C.c_int64(0)
            check(L.sxc_batch_results(h, out.ctypes.data_as(C.POINTER(Result)), len(out), C.byref(n)))
            assert_results_equal(out[:n.value], ref, f"N = {1 << nb}, run {k}")
        for ps, want in enumerate(lags):
            got, m = np.zeros(1 << 15, np.int32), C.c_int32(0)
            check(L.sxc_batch_lags(h, ps // 2, ps % 2, got.ctypes.data_as(C.POINTER(C.c_int32)), len(got), C.byref(m)))
            assert want is None or np.array_equal(got[:m.value], want), ps
    finally:
        L.sxc_batch_destroy(h)


@pytest.mark.parametrize("nb,sa,km,occ,lean", [(nb, *g) for nb, g in DEFAULT.items()] + GEOMETRIES)
def test_every_geometry(ctx, cases, nb, sa, km, occ, lean):
    from satsuma2_amd.api import Geometry

    N = 1 << nb
    case = cases(nb)
    assert len(case[3]) > 30 and sum(map(bool, case[1])) > 20
    print(f"[geometry] N {N} stage A {sa} rounds {km} occ {occ} lean {lean}", flush=True)
    try:
        for kernel in ("pairs", "spectra"):
            ctx.set_geometry(N, kernel, Geometry(sa, km, occ, lean))
        run_and_check(ctx, nb, case)
    finally:
        for kernel in ("pairs", "spectra"):
            ctx.set_geometry(N, kernel, Geometry(*DEFAULT[nb]))


@pytest.mark.parametrize("n", [64, 65])
def test_both_sides_of_the_limit(ctx, n):
    """128 and 130 strands give the same pairs' records."""
    N = 2048
    pairs, tt, qt = batch(N, n, 3)
    run_and_check(ctx, 11, (pairs, tt, qt, reference(pairs, tt, qt, N), []))


def test_golden_pairs_after_autotune(ctx, golden):
    """The golden pairs three times over (192 targets), in the geometries the autotuner chose."""
    from satsuma2_amd.api import ChunkPair, Geometry, HomologyByXCorr, SlaveParams

    g = golden("uniform_pairs.npz")
    P = g["t"].shape[0]
    try:
        ctx.autotune(8192)
        pairs = [ChunkPair(bytes(bytearray(unpack2(g["t"][r], 4096))), unpack2(g["q"][r], 4096), t_record=r, q_record=r,
                           q_record_len=4096, fast=int(g["fast"][r])) for _ in range(3) for r in range(P)]
        assert len({id(p.tseq) for p in pairs}) > 128
        got = HomologyByXCorr(ctx, SlaveParams(target_total=float(4096 * P))).align_batch(pairs)
        assert_results_equal(got, np.concatenate([g["results"]] * 3), "after autotune")
    finally:
        for kernel in ("pairs", "spectra"):
            ctx.set_geometry(8192, kernel, Geometry(*DEFAULT[13]))
