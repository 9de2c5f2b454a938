"""The kernels at the edges of their tiles, windows and dispatch rules.

Corrections of read sets whose lengths meet each alignment window (2 to 4
words of 32 bases), each quality width and equal or mixed lengths, packed
candidate lists around the tile of 1,024 anchors and with limits below and
above a list's length, tables built in one and in several groups of maps, and
gate batches around a block of 64 rows are compared with the oracle.  CPU
through the HIP emulation; the GPU tests run the device.
"""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import care_amd
from tests import helpers

sys.path.insert(0, os.path.join(helpers.ROOT, "oracle"))
import mlp_oracle  # noqa: E402

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")


@pytest.fixture(scope="module")
def emu():
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    return care_amd._bind(ctypes.CDLL(os.path.join(EMU_DIR, "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)


def _run(exe, reads, out, args):
    p = subprocess.run([exe, "-i", reads, "-o", "r.fastq", "-d", out, "-t", "4"] + args, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=600)
    assert p.returncode == 0, p.stdout[-2000:]
    return helpers.md5(os.path.join(out, "r.fastq"))


def _trim(reads, seed):
    """The reads cut to between 40 % and all of their bases."""
    rng = np.random.default_rng(seed)
    with open(reads) as f:
        lines = f.read().split("\n")
    for i in range(1, len(lines) - 2, 4):
        n = int(rng.integers(int(0.4 * len(lines[i])), len(lines[i]) + 1))
        lines[i], lines[i + 2] = lines[i][:n], lines[i + 2][:n]
    with open(reads, "w") as f:
        f.write("\n".join(lines))


SHAPES = [(100, 0, False), (101, 2, True), (151, 1, True), (250, 8, False), (300, 2, True)]


def _correct_like_oracle(exe, d, length, bits, ragged, genome, extra=()):
    case = {"profile": "repeat-pe", "seed": 300 + length + bits, "genome": genome,
            "sim_args": ["--length", str(length)]}
    reads, _ = helpers.simulate(case, d)
    if ragged:
        _trim(reads, length)
    args = ["-c", "30", "--pairmode", "PE", "-k", "20", "-h", "16", "--candidateCorrection"]
    if bits:
        args += ["-q", "--qualityScoreBits", str(bits)]
    want = _run(helpers.ORACLE_EXE, reads, os.path.join(d, "oracle"), args)
    assert _run(exe, reads, os.path.join(d, "out"), ["-g", "0"] + args) == want


@pytest.mark.parametrize("length,bits,ragged", SHAPES)
def test_emulated_corrections_by_length_and_quality(emu, length, bits, ragged, tmp_path):
    _correct_like_oracle(os.path.join(EMU_DIR, "_build", "care-gpu-emu"), str(tmp_path), length, bits, ragged, 2400)


@pytest.mark.gpu
@pytest.mark.parametrize("length,bits,ragged", SHAPES)
def test_gpu_corrections_by_length_and_quality(length, bits, ragged, tmp_path):
    print("corrections", length, bits, ragged, flush=True)
    _correct_like_oracle(os.path.join(helpers.ROOT, "care_amd", "_build", "care-gpu"), str(tmp_path), length, bits,
                         ragged, 60000)


def _lists_like_oracle(lib, d, genome, maps, limits, counts, check):
    reads, _ = helpers.simulate({"profile": "repeat-pe", "seed": 320, "genome": genome}, d)
    rs = care_amd.ReadSet([reads], paired_end=True, qual_bits=0)
    orc = helpers.oracle()
    seqs, lens = np.ascontiguousarray(rs.seqs), np.ascontiguousarray(rs.lengths)
    t = orc.orc_tables_build(seqs.ctypes.data, rs.pitch, lens.ctypes.data, rs.n, 20, maps, 30.0)
    buf = np.zeros(maps * 400, dtype=np.uint32)
    for limit in limits:
        opt = care_amd.default_options(kmer_length=20, num_hash_maps=maps, coverage=30.0, candidate_limit=limit)
        with care_amd.Engine(opt, device=0, lib=lib) as eng:
            eng.upload_readset(rs)
            eng.build()
            for n in counts:
                n = min(n, rs.n)
                ids, offs = eng.query(0, n)
                assert offs[0] == 0 and offs[n] == len(ids)
                for i in sorted({0, n - 1, n // 2, *range(0, n, max(1, n // check))}):
                    args = (t, seqs[i].ctypes.data, int(lens[i]), i)
                    c = (orc.orc_tables_query_limited(*args, limit, buf.ctypes.data, len(buf)) if limit
                         else orc.orc_tables_query(*args, buf.ctypes.data, len(buf)))
                    assert np.array_equal(ids[offs[i]:offs[i + 1]], buf[:c]), (limit, n, i)
    orc.orc_tables_free(t)


def test_emulated_packed_lists(emu, tmp_path):
    _lists_like_oracle(emu, str(tmp_path), 8000, 8, (0, 1, 20, 1000), (1, 1023, 1024, 1025, 1600), 200)


@pytest.mark.gpu
def test_gpu_packed_lists_and_map_groups(tmp_path):
    # 60,000 reads and 48 maps: more scratch than one group of maps may take
    print("packed lists", flush=True)
    _lists_like_oracle(None, str(tmp_path), 300000, 48, (0, 20), (1, 1023, 1024, 1025, 60000), 500)


def _gate(lib, rows):
    rng = np.random.default_rng(rows)
    x = rng.uniform(0.0, 1.5, size=(rows, 32)).astype(np.float32)
    y = (x[:, 0] + 0.5 * x[:, 3] > 0.9).astype(np.uint8)
    p = mlp_oracle.init_params(31)
    with care_amd.Engine(care_amd.default_options(), device=0, lib=lib) as eng:
        g, loss = eng.mlp_gradient(x, y, p)
        lo, go = mlp_oracle.loss_and_grad(x, y, p)
        assert abs(loss - lo) < 1e-4 * max(1.0, abs(lo))
        # the tolerance of the gradient test at 100 rows
        assert np.linalg.norm(np.asarray(g, np.float64) - go) < 2e-3 * np.linalg.norm(go)
        z = eng.mlp_infer(x, p)
        zo, _ = mlp_oracle.forward(x, p)
        assert np.max(np.abs(z - zo)) < 1e-3 * max(1.0, np.max(np.abs(zo)))
        # a feature that is not finite is refused, wherever it is
        for bad in (np.inf, -np.inf, np.nan):
            xb = x.copy()
            xb[rows - 1, 31] = bad
            for call in (lambda: eng.mlp_infer(xb, p), lambda: eng.mlp_gradient(xb, y, p),
                         lambda: eng.mlp_train(xb, y, p, epochs=1, batch=16, lr=1e-3, seed=1)):
                with pytest.raises(care_amd.CareError):
                    call()


@pytest.mark.parametrize("rows", [16, 63, 64, 65, 130])
def test_emulated_gate_rows(emu, rows):
    _gate(emu, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [16, 63, 64, 65, 4099])
def test_gpu_gate_rows(rows):
    print("gate rows", rows, flush=True)
    _gate(None, rows)


@pytest.mark.gpu
def test_gpu_gate_feature_chunks():
    """Features beyond one staged chunk of 2^18 rows: every row's logit has
    the bits that the row has in a call of its own chunk alone, and a
    non-finite feature in the last chunk is refused.  (Against the oracle a
    maximum over so many rows meets hidden activations that fall on either
    side of a bfloat16 rounding boundary; bits between calls have no such
    tail.)"""
    print("gate feature chunks", flush=True)
    n, chunk = (1 << 18) + 5, 1 << 18
    x = np.random.default_rng(41).uniform(0.0, 1.5, size=(n, 32)).astype(np.float32)
    p = mlp_oracle.init_params(31)
    with care_amd.Engine(care_amd.default_options(), device=0) as eng:
        z = eng.mlp_infer(x, p)
        assert np.array_equal(z[chunk:], eng.mlp_infer(x[chunk:], p))
        assert np.array_equal(z[:1000], eng.mlp_infer(x[:1000], p))
        assert np.array_equal(z[chunk - 1000:chunk], eng.mlp_infer(x[chunk - 1000:chunk], p))
        x[n - 1, 0] = np.nan
        with pytest.raises(care_amd.CareError):
            eng.mlp_infer(x, p)
