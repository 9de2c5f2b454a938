"""Calls of different sizes on one context, the order of the correction's
work queue, and candidate results up to and beyond the caller's capacity.

CPU through the HIP emulation; the GPU tests run the device.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import care_amd
from tests import helpers

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    return care_amd._bind(ctypes.CDLL(os.path.join(EMU_DIR, "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)


def _readset(d, genome, length=60):
    path, _ = helpers.simulate({"profile": "repeat-pe", "seed": 430, "genome": genome,
                                "sim_args": ["--length", str(length)]}, d)
    return care_amd.ReadSet([path], paired_end=True, qual_bits=0)


def _engine(lib, rs, **options):
    opt = care_amd.default_options(**dict(dict(kmer_length=20, num_hash_maps=16, coverage=30.0, paired_end=1,
                                               min_overlap=20), **options))
    eng = care_amd.Engine(opt, device=0, lib=lib)
    eng.upload_readset(rs)
    eng.build()
    return eng


def _rows(eng, status, seqs):
    return status.tobytes(), seqs[(status & 1) != 0, :eng.max_length].tobytes()


def _sizes(lib, rs, large):
    """A graph is replayed around calls that make the buffers grow."""
    def pinned(eng, n):
        pitch = (rs.max_length + 15) // 16 * 16
        return (care_amd.pinned_empty((n,), np.uint8, lib=eng.lib),
                care_amd.pinned_empty((n, pitch), np.uint8, lib=eng.lib))

    want = {}
    for n in (2, 64, large):
        with _engine(lib, rs) as eng:
            want[n] = _rows(eng, *eng.correct(0, n)[:2])
    with _engine(lib, rs) as eng:
        outs = {n: pinned(eng, n) for n in want}
        for n, graph in ((64, True), (64, True), (2, False), (64, True), (large, False), (64, True), (64, True),
                         (large, True), (2, True), (large, True), (64, False), (large, False)):
            for a in outs[n]:
                a[:] = 0
            assert _rows(eng, *eng.correct(0, n, out=outs[n], graph=graph)[:2]) == want[n], (n, graph)


def test_emulated_sizes_and_graphs(emu, tmp_path):
    rs = _readset(str(tmp_path), 2400)
    _sizes(emu, rs, rs.n & ~1)
    rs.close()


@pytest.mark.gpu
def test_gpu_sizes_and_graphs(tmp_path):
    print("sizes and graphs", flush=True)
    rs = _readset(str(tmp_path), 60000)
    _sizes(None, rs, rs.n & ~1)
    rs.close()


def _queue(lib, rs, batch):
    """Anchors with long candidate lists are corrected first; the call without
    allocation takes all in read order."""
    with _engine(lib, rs) as eng:
        eng.set_tuning(batch_anchors=batch)
        ids, offs = eng.query(0, rs.n)
        long = np.diff(offs) > 96  # more than 96 or three times the coverage
        # of several batches some hold long lists; most reads have short ones
        per_batch = [long[i:i + batch].sum() for i in range(0, rs.n, batch)]
        assert len(per_batch) > 2 and sum(p > 0 for p in per_batch) > 1 and 0 < long.sum() < rs.n // 2
        n = rs.n & ~1
        assert _rows(eng, *eng.correct(0, n)[:2]) == _rows(eng, *eng.correct(0, n, noalloc=True)[:2])


def test_emulated_long_lists_first(emu, tmp_path):
    rs = _readset(str(tmp_path), 6000, 100)
    _queue(emu, rs, 512)
    rs.close()


@pytest.mark.gpu
def test_gpu_long_lists_first(tmp_path):
    print("long lists first", flush=True)
    rs = _readset(str(tmp_path), 300000, 100)
    _queue(None, rs, 16384)
    rs.close()


def _capacity(lib, rs):
    """Candidate results in as many rows as the caller gives; one row less is
    an error, however many of a group of rows are beyond."""
    with _engine(lib, rs, correct_candidates=1) as eng:
        n = rs.n & ~1
        status, seqs, cids, cseqs = eng.correct(0, n, candidate_capacity=64 * n)
        order = np.lexsort(cseqs[:, :rs.max_length].T[::-1].tolist() + [cids])
        total = len(cids)
        assert total > 64
        for short in (1, 15, 16, 17, total - 1, total):
            with pytest.raises(care_amd.CareError, match="candidate_capacity exceeded"):
                eng.correct(0, n, candidate_capacity=total - short)
            got = eng.correct(0, n, candidate_capacity=total)
            assert _rows(eng, *got[:2]) == _rows(eng, status, seqs) and len(got[2]) == total
            again = np.lexsort(got[3][:, :rs.max_length].T[::-1].tolist() + [got[2]])
            assert np.array_equal(got[2][again], cids[order])
            assert np.array_equal(got[3][again, :rs.max_length], cseqs[order, :rs.max_length])


def test_emulated_candidate_capacity(emu, tmp_path):
    rs = _readset(str(tmp_path), 1200)
    _capacity(emu, rs)
    rs.close()


@pytest.mark.gpu
def test_gpu_candidate_capacity(tmp_path):
    print("candidate capacity", flush=True)
    rs = _readset(str(tmp_path), 30000)
    _capacity(None, rs)
    rs.close()
