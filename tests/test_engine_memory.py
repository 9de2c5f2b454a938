"""Device memory of a context: what a call leaves after a failed allocation.

CPU through the HIP emulation, which can make the k-th allocation fail and
counts live bytes (tests/emu/hip/hip_runtime.h).
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import care_amd
from tests import helpers

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    return care_amd._bind(ctypes.CDLL(os.path.join(EMU_DIR, "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)


@pytest.fixture(scope="module")
def reads(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("reads"))
    path, _ = helpers.simulate({"profile": "repeat-pe", "seed": 401, "genome": 2200, "sim_args": ["--length", "60"]}, d)
    rs = care_amd.ReadSet([path], paired_end=True, qual_bits=0)
    yield rs
    rs.close()


def _engine(lib, rs, **options):
    opt = care_amd.default_options(kmer_length=20, num_hash_maps=2, coverage=30.0, paired_end=1, min_overlap=20, **options)
    eng = care_amd.Engine(opt, device=0, lib=lib)
    eng.upload_readset(rs)
    eng.build()
    return eng


def _results(eng, n):
    """Everything a call returns for the first n reads, candidates in a fixed order."""
    status, seqs, cids, cseqs = eng.correct(0, n, candidate_capacity=32 * n)
    ids, offs = eng.query(0, n)
    width = eng.max_length
    cands = sorted((int(i), bytes(r[:width])) for i, r in zip(cids, cseqs))
    return status.tobytes(), seqs[(status & 1) != 0, :width].tobytes(), cands, ids.tobytes(), offs.tobytes()


@pytest.mark.parametrize("call,most", [("correct", 99), ("query", 99), ("autotune", 8)])
def test_small_call_after_a_failed_growth(emu, reads, call, most):
    """A call needs larger buffers, one of their allocations fails (each in
    turn, at most `most`); a small call that the old buffers served still
    gives its results."""
    assert reads.n > 1024
    big = reads.n & ~1
    calls = {"correct": lambda e: e.correct(0, big, candidate_capacity=1 << 18),
             "query": lambda e: e.query(0, big), "autotune": lambda e: e.autotune(0, big)}
    with _engine(emu, reads, correct_candidates=1) as eng:
        want = _results(eng, 2)
    failures = 0
    while failures < most:
        with _engine(emu, reads, correct_candidates=1) as eng:
            assert _results(eng, 2) == want
            emu.care_emu_fail_alloc(failures + 1)
            try:
                calls[call](eng)
                assert emu.care_emu_fail_pending() > 0
                break
            except care_amd.CareError:
                failures += 1
            finally:
                emu.care_emu_fail_alloc(0)
            assert _results(eng, 2) == want, failures
    assert failures >= 3


def _live(lib):
    live, peak = ctypes.c_uint64(), ctypes.c_uint64()
    lib.care_emu_memory(ctypes.byref(live), ctypes.byref(peak))
    return live.value


def test_gate_buffers_are_given_back(emu):
    """The features of a large training set do not stay on the device after
    the call (here one that ends at a non-finite feature); what small calls
    use stays, bounded by 32 MiB of staged features and 32 MiB of converted
    ones."""
    with care_amd.Engine(care_amd.default_options(), device=0, lib=emu) as eng:
        before = _live(emu)
        p = np.zeros(care_amd.MLP_PARAMS, np.float32)
        x = np.zeros((1 << 20, 32), np.float32)
        y = np.zeros(len(x), np.uint8)
        eng.mlp_train(x[:100], y[:100], p, epochs=1, batch=16, lr=1e-3, seed=1)
        kept = _live(emu)
        assert kept > before
        eng.mlp_train(x[:100], y[:100], p, epochs=1, batch=16, lr=1e-3, seed=1)
        assert _live(emu) == kept
        x[-1, -1] = np.inf
        for call in (lambda: eng.mlp_train(x, y, p, epochs=1, batch=16, lr=1e-3, seed=1),
                     lambda: eng.mlp_gradient(x, y, p)):
            with pytest.raises(care_amd.CareError):
                call()
            assert _live(emu) - before <= 64 << 20


def test_growing_calls_allocate_seldom(emu, reads):
    """Calls that grow by a pair at a time find most of their buffers there:
    records per workgroup are not allocated again for each of them."""
    with _engine(emu, reads) as eng:
        eng.set_tuning(correct_blocks_per_cu=64)  # 128 workgroups
        allocations = 0
        for n in range(2, 131, 2):
            emu.care_emu_fail_alloc(1 << 30)
            eng.correct(0, n)
            allocations += (1 << 30) - emu.care_emu_fail_pending()
            emu.care_emu_fail_alloc(0)
        # two buffers of records for each power of two from 2 to 128, and at most a dozen others
        assert allocations <= 2 * 7 + 12


# A call with 64,000 candidate slots an anchor on a device of 256 compute units: peak memory above what was live
# before it, and the results.  argv: emulation folder, read file, anchors per batch (0 automatic), workgroups per CU.
WIDE = """
import ctypes, hashlib, os, sys
import care_amd
lib = care_amd._bind(ctypes.CDLL(os.path.join(sys.argv[1], "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)
rs = care_amd.ReadSet([sys.argv[2]], paired_end=True, qual_bits=0)
opt = care_amd.default_options(kmer_length=20, num_hash_maps=64, coverage=400.0, paired_end=1, min_overlap=20)
live, peak = ctypes.c_uint64(), ctypes.c_uint64()
with care_amd.Engine(opt, device=0, lib=lib) as eng:
    eng.upload_readset(rs)
    eng.build()
    eng.set_tuning(batch_anchors=int(sys.argv[3]), correct_blocks_per_cu=int(sys.argv[4]), query_lds_hits=16,
                   query_register_hits=64)
    lib.care_emu_memory(ctypes.byref(live), ctypes.byref(peak))
    before = live.value
    n = min(1024, rs.n)
    status, seqs, _, _ = eng.correct(0, n)
    lib.care_emu_memory(ctypes.byref(live), ctypes.byref(peak))
    print(n, peak.value - before)
    print(hashlib.md5(status.tobytes() + seqs[(status & 1) != 0, :eng.max_length].tobytes()).hexdigest())
"""


def test_batch_memory_is_bounded(tmp_path):
    """The scratch of a call stays within a quarter of the free memory (2 GiB
    of the emulated 8), and with a batch size set by the caller within 36
    bytes a candidate slot; with fewer rows than anchors the results are the
    same."""
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    path, _ = helpers.simulate({"profile": "repeat-pe", "seed": 402, "genome": 2200,
                                "sim_args": ["--length", "60"]}, str(tmp_path))
    got = []
    for batch, per_cu in ((0, 8), (64, 8)):
        p = subprocess.run([sys.executable, "-c", WIDE, EMU_DIR, path, str(batch), str(per_cu)],
                           env=dict(os.environ, EMU_CUS="256", PYTHONPATH=helpers.ROOT), stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, text=True, timeout=600)
        assert p.returncode == 0, p.stdout[-2000:]
        n, took, digest = p.stdout.split()
        outputs = int(n) * (64 + 64)  # rows of results, counters
        assert int(took) <= (36 * 64000 * batch if batch else 2 << 30) + outputs + (1 << 20), (batch, took)
        got.append(digest)
    assert got[0] == got[1]
