"""The pair and spectra kernels with a workgroup per channel, and their sum, on the CPU workgroup
emulator against the oracle: every length, every form of chunk, signal tails, resident query spectra,
threads in any order, and under AddressSanitizer."""
import ctypes as C

import numpy as np
import pytest

import hostbuild
import oracle
from strand_cases import batch, pair_table, params, reference, tail_table
from test_emu import COLS, _run_check


@pytest.fixture(scope="module")
def emu():
    return C.CDLL(hostbuild.emu_library())


def run(emu, pairs, tt, qt, N):
    out = np.zeros(1 << 14, oracle.RESULT_DTYPE)
    n = C.c_int64(0)
    xc = np.zeros((2 * len(pairs), N), np.float32)
    st = np.zeros((2 * len(pairs), 2), np.int32)
    t, keep_t = tail_table(tt)
    q, keep_q = tail_table(qt)
    prm = params(N)
    assert emu.emu_align_batch_tails(pair_table(pairs), len(pairs), C.byref(prm), t, q, out.ctypes.data_as(C.c_void_p),
                                     C.c_int64(len(out)), C.byref(n), xc.ctypes.data_as(C.c_void_p),
                                     st.ctypes.data_as(C.c_void_p)) == 0
    return out[:n.value].copy(), xc, st


@pytest.mark.parametrize("nb", range(9, 16))
def test_a_workgroup_per_channel(emu, monkeypatch, nb):
    N = 1 << nb
    pairs, tt, qt = batch(N, 8 if nb < 14 else 6, nb)
    one, xc1, st1 = run(emu, pairs, tt, qt, N)
    monkeypatch.setenv("SXC_EMU_PARTS", "1")
    got, xc, st = run(emu, pairs, tt, qt, N)
    ref = reference(pairs, tt, qt, N)
    assert len(ref) > 0
    for c in COLS:
        assert np.array_equal(got[c], ref[c]), c
    assert got.tobytes() == one.tobytes() and xc.tobytes() == xc1.tobytes() and np.array_equal(st, st1)


@pytest.mark.parametrize("nb", [9, 11, 13, 15])
def test_a_workgroup_per_channel_with_query_spectra(emu, monkeypatch, nb):
    N = 1 << nb
    pairs, tt, qt = batch(N, 5, nb + 50, tails=False)
    monkeypatch.setenv("SXC_EMU_PARTS", "1")
    monkeypatch.setenv("SXC_EMU_QSPEC", "1")
    got, _, _ = run(emu, pairs, tt, qt, N)
    ref = reference(pairs, tt, qt, N)
    for c in COLS:
        assert np.array_equal(got[c], ref[c]), c


@pytest.mark.parametrize("order", ["", "reverse", "shuffle"])
@pytest.mark.parametrize("nb", [9, 12, 14, 15])
def test_asan_a_workgroup_per_channel(monkeypatch, tmp_path, nb, order):
    monkeypatch.setenv("SXC_EMU_PARTS", "1")
    monkeypatch.setenv("SXC_EMU_ORDER", order)
    pairs, _, _ = batch(1 << nb, 6, nb + 90)
    _run_check(hostbuild.emu_checker(), tmp_path, [(p["tseq"], p["qseq"], p["fast"]) for p in pairs], 1 << nb)
