"""Scratch limits of table building and queries, met on small sets.

CPU through the HIP emulation, built with a scratch of three maps of 600
reads at a time, 2^16 slots of a scratch table and eight query wavefronts
(CARE_SMALL_SCRATCH in care_amd/csrc/engine.h), against the usual build and
the oracle.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import care_amd
from tests import helpers

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")


def _library(kind):
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh"), kind], check=True)
    return care_amd._bind(ctypes.CDLL(os.path.join(EMU_DIR, "_build", kind, "libcare_amd_emu.so")),
                          care_amd.ENGINE_SYMBOLS)


@pytest.fixture(scope="module")
def usual():
    return _library("")


@pytest.fixture(scope="module")
def small():
    return _library("small")


def _reads(n, length, genome, seed):
    """Reads of a random genome, 2-bit packed."""
    rng = np.random.default_rng(seed)
    g = rng.integers(0, 4, genome)
    at = rng.integers(0, genome - length, n)
    seqs = np.zeros((n, (length + 15) // 16), np.uint32)
    for i in range(length):
        seqs[:, i // 16] |= (g[at + i] << (30 - 2 * (i % 16))).astype(np.uint32)
    return seqs, np.full(n, length, np.int32)


def _tables(lib, seqs, lens, maps, coverage):
    opt = care_amd.default_options(kmer_length=16, num_hash_maps=maps, coverage=coverage)
    with care_amd.Engine(opt, device=0, lib=lib) as eng:
        eng.upload(seqs, lens)
        eng.build()
        return [eng.export_map(m) for m in range(maps)]


def test_every_slot_of_a_scratch_table(usual, small):
    """The scratch tables of 32,768 reads have as many slots as a slot index
    tells apart, and keys lie in the last one."""
    seqs, lens = _reads(32768, 20, 14000, 1)
    want, got = _tables(usual, seqs, lens, 6, 30.0), _tables(small, seqs, lens, 6, 30.0)
    for m in range(6):
        for a, b in zip(want[m], got[m]):
            assert np.array_equal(a, b), m


def _group(lib, reads, maps):
    """Maps that are built together (care_engine::build_group)."""
    f = lib._ZN11care_engine11build_groupEmi
    f.argtypes, f.restype = [ctypes.c_uint64, ctypes.c_int], ctypes.c_int
    return f(reads, maps)


def _lists_like_oracle(lib, rs, maps, coverage, anchors, **tuning):
    """Candidate lists of the given anchors against the oracle's."""
    orc = helpers.oracle()
    seqs, lens = np.ascontiguousarray(rs.seqs), np.ascontiguousarray(rs.lengths)
    t = orc.orc_tables_build(seqs.ctypes.data, rs.pitch, lens.ctypes.data, rs.n, 20, maps, coverage)
    buf = np.zeros(maps * 400, dtype=np.uint32)
    opt = care_amd.default_options(kmer_length=20, num_hash_maps=maps, coverage=coverage)
    longest = 0
    with care_amd.Engine(opt, device=0, lib=lib) as eng:
        eng.upload_readset(rs)
        eng.build()
        if tuning:
            eng.set_tuning(**tuning)
        ids, offs = eng.query(0, rs.n)
        for i in anchors:
            c = orc.orc_tables_query(t, seqs[i].ctypes.data, int(lens[i]), i, buf.ctypes.data, len(buf))
            assert np.array_equal(ids[offs[i]:offs[i + 1]], buf[:c]), i
            longest = max(longest, c)
    orc.orc_tables_free(t)
    return longest


@pytest.mark.parametrize("maps", [1, 2, 6, 7, 64])
def test_map_groups_and_spill_rows(small, maps, tmp_path):
    """Maps built in groups that do and do not divide them evenly, and queries
    whose wavefronts take one anchor after another through the same spill
    row."""
    path, _ = helpers.simulate({"profile": "repeat-pe", "seed": 421, "genome": 1500,
                                "sim_args": ["--length", "75"]}, str(tmp_path))
    rs = care_amd.ReadSet([path], paired_end=True, qual_bits=0)
    assert rs.n > 8 * 32 and _group(small, rs.n, maps) == min(maps, 3)
    longest = _lists_like_oracle(small, rs, maps, 30.0, range(rs.n), query_lds_hits=16, query_register_hits=64)
    assert longest > 16
    rs.close()


@pytest.mark.gpu
def test_gpu_several_map_groups(tmp_path):
    """64 maps of 60,000 reads take more scratch than a group may."""
    print("map groups", flush=True)
    path, _ = helpers.simulate({"profile": "repeat-pe", "seed": 422, "genome": 300000}, str(tmp_path))
    rs = care_amd.ReadSet([path], paired_end=True, qual_bits=0)
    assert 2 * _group(care_amd.engine(), rs.n, 64) >= 64 > _group(care_amd.engine(), rs.n, 64) >= 32
    _lists_like_oracle(None, rs, 64, 30.0, range(0, rs.n, 97))
    rs.close()
