"""Launch shapes against the limits of a workgroup.

The host functions that size the correction kernel's LDS are called by name;
the emulation build of the engine has the same ones as the device build.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import care_amd
from tests import helpers

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")
MAX_LDS = 64 * 1024


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    return care_amd._bind(ctypes.CDLL(os.path.join(EMU_DIR, "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)


def _function(lib, name, ints, result=ctypes.c_size_t):
    """care_engine::name, taking `ints` int arguments."""
    f = getattr(lib, "_ZN11care_engine%d%sE%s" % (len(name), name, "i" * ints))
    f.argtypes, f.restype = [ctypes.c_int] * ints, result
    return f


# gate mode (bit 0 the anchor gate, bit 1 the candidate gate), candidate correction
MODES = [(0, 0), (0, 1), (1, 0), (1, 1), (3, 1)]


@pytest.mark.parametrize("gated,candidates", MODES)
def test_accepted_shapes_launch_within_the_lds_limit(emu, gated, candidates):
    """Every shape that the capacity rule accepts is launched with no more
    than the limit, whatever the columns that candidate correction may add."""
    lds = _function(emu, "correct_lds_bytes", 8)
    capacity = _function(emu, "correct_capacity_bytes", 6)
    accepted = 0
    for length in range(1, 1001):
        for bits in (0, 1, 2, 8):
            qpitch = (bits * length + 31) // 32
            # workgroup, and the one that the capacity is computed for (256 unless it was set)
            for threads, asked in ((128, 128), (192, 192), (256, 256), (128, 256)):
                for chunk in (0, 16, 17, 23, 32, 64, 101, 128, 256):
                    if capacity(length, int(bits > 0), qpitch, asked, gated, chunk) > MAX_LDS:
                        continue
                    accepted += 1
                    assert qpitch <= threads, (length, bits, threads)  # rows are staged a word a thread
                    for columns in (15, length // 2, length, 1 << 20) if candidates else (0,):
                        got = lds(length, int(bits > 0), qpitch, threads, gated, chunk, candidates, columns)
                        assert got <= MAX_LDS, (length, bits, threads, asked, chunk, columns)
    assert accepted > 10000


def _largest_chunk(lib, length, bits, threads, gated):
    capacity = _function(lib, "correct_capacity_bytes", 6)
    qpitch = (bits * length + 31) // 32
    return max(c for c in range(16, 257) if capacity(length, int(bits > 0), qpitch, threads, gated, c) <= MAX_LDS)


def _compact_like_default(lib, sizes, d, length, bits, threads, genome):
    """The largest accepted staging area with columns of a whole read on
    either side leaves no room for the usual LDS layout: the results are
    those of the smallest staging area, which has it."""
    chunk = _largest_chunk(sizes, length, bits, threads, 0)
    lds = _function(sizes, "correct_lds_bytes", 8)
    qpitch = (bits * length + 31) // 32
    # 8 bytes of keys and a staged row per candidate: the layouts differ if the sizes do not follow the chunk
    row = 16 + 4 * ((length + 15) // 16 + qpitch) + 16 * ((length + 31) // 32 + 3) + 8
    small = lds(length, int(bits > 0), qpitch, threads, 0, 16, 1, length)
    assert lds(length, int(bits > 0), qpitch, threads, 0, chunk, 1, length) < small + (chunk - 16) * row
    reads, _ = helpers.simulate({"profile": "repeat-pe", "seed": 410 + length, "genome": genome,
                                 "sim_args": ["--length", str(length)]}, d)
    rs = care_amd.ReadSet([reads], paired_end=True, qual_bits=bits)
    opt = care_amd.default_options(kmer_length=20, num_hash_maps=16, coverage=30.0, paired_end=1,
                                   use_quality=int(bits > 0), correct_candidates=1, new_columns_to_correct=length)
    results = []
    for c in (16, chunk):
        with care_amd.Engine(opt, device=0, lib=lib) as eng:
            eng.upload_readset(rs)
            eng.build()
            eng.set_tuning(correct_threads=threads, msa_chunk=c)
            status, seqs, cids, cseqs = eng.correct(0, rs.n, candidate_capacity=64 * rs.n)
            corrected = (status & 1) != 0
            assert corrected.sum() > rs.n // 4 and len(cids) > rs.n
            rows = sorted((int(i), bytes(r[:rs.lengths[i]])) for i, r in zip(cids, cseqs))
            results.append((status.tobytes(), seqs[corrected, :length].tobytes(), rows))
    assert results[0] == results[1]
    rs.close()


COMPACT = [(300, 0, 128), (270, 2, 256), (280, 8, 192)]


@pytest.mark.parametrize("length,bits,threads", COMPACT)
def test_emulated_compact_layout(emu, length, bits, threads, tmp_path):
    _compact_like_default(emu, emu, str(tmp_path), length, bits, threads, 2400)


@pytest.mark.gpu
@pytest.mark.parametrize("length,bits,threads", COMPACT)
def test_gpu_compact_layout(length, bits, threads, tmp_path):
    print("compact layout", length, bits, threads, flush=True)
    _compact_like_default(None, care_amd.engine(), str(tmp_path), length, bits, threads, 60000)


@pytest.mark.parametrize("columns", [1 << 20, 1 << 30, (1 << 31) - 1, -(1 << 31)])
def test_emulated_any_number_of_new_columns(emu, columns, tmp_path):
    """Beyond the longest read more (or fewer) new columns change nothing."""
    reads, _ = helpers.simulate({"profile": "repeat-pe", "seed": 405, "genome": 1500,
                                 "sim_args": ["--length", "100"]}, str(tmp_path))
    rs = care_amd.ReadSet([reads], paired_end=True, qual_bits=0)
    results = []
    for new in (1000 if columns > 0 else -1000, columns):
        opt = care_amd.default_options(kmer_length=20, num_hash_maps=8, coverage=30.0, paired_end=1,
                                       correct_candidates=1, new_columns_to_correct=new)
        with care_amd.Engine(opt, device=0, lib=emu) as eng:
            eng.upload_readset(rs)
            eng.build()
            status, seqs, cids, cseqs = eng.correct(0, rs.n, candidate_capacity=64 * rs.n)
            corrected = (status & 1) != 0
            assert corrected.any() and (len(cids) > 0) == (columns > 0)
            rows = sorted((int(i), bytes(r[:rs.lengths[i]])) for i, r in zip(cids, cseqs))
            results.append((status.tobytes(), seqs[corrected, :100].tobytes(), rows))
    assert results[0] == results[1]
    rs.close()


@pytest.mark.parametrize("gated,candidates", MODES)
@pytest.mark.parametrize("length,bits", [(100, 0), (150, 2), (250, 8)])
def test_reported_chunk_is_the_launched_one(emu, length, bits, gated, candidates):
    """The staging area that care_get_tuning reports, set by hand, takes the
    LDS of the automatic one."""
    opt = care_amd.default_options(kmer_length=20, num_hash_maps=4, coverage=30.0, use_quality=int(bits > 0),
                                   correct_candidates=candidates, correction_type=3 if gated else 0,
                                   correction_type_cands=3 if gated & 2 else 0)
    qpitch = (bits * length + 31) // 32
    with care_amd.Engine(opt, device=0, lib=emu) as eng:
        eng.upload(np.zeros((2, (length + 15) // 16), np.uint32), np.full(2, length, np.int32), None,
                   np.zeros((2, qpitch), np.uint32) if bits else None, bits or 8, length)
        t = eng.tuning()
    lds = _function(emu, "correct_lds_bytes", 8)
    args = (length, int(bits > 0), qpitch, t["correct_threads"], gated)
    assert lds(*args, t["msa_chunk"], candidates, 15) == lds(*args, 0, candidates, 15)


@pytest.mark.parametrize("length,bits,limit,threads",
                         [(150, 2, 0, 128), (225, 1, 0, 128), (250, 2, 0, 128), (250, 8, 0, 256), (300, 0, 0, 256),
                          (300, 8, 0, 256), (400, 0, 0, 256), (250, 8, 20, 128), (300, 2, 20, 128), (300, 8, 20, 256)])
def test_two_wavefronts_an_anchor_where_lds_has_room(emu, length, bits, limit, threads):
    """The workgroup of a large call; 256 where 128 threads were measured slower."""
    opt = care_amd.default_options(kmer_length=20, num_hash_maps=4, coverage=30.0, use_quality=int(bits > 0),
                                   candidate_limit=limit, correction_type=3 if limit else 0)
    qpitch = (bits * length + 31) // 32
    with care_amd.Engine(opt, device=0, lib=emu) as eng:
        eng.upload(np.zeros((2, (length + 15) // 16), np.uint32), np.full(2, length, np.int32), None,
                   np.zeros((2, qpitch), np.uint32) if bits else None, bits or 8, length)
        assert eng.tuning()["correct_threads"] == threads
