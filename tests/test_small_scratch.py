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
