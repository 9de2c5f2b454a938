"""Setting the launch shapes that care_get_tuning reported changes nothing.

Automatic shapes depend on the size of a call; what is launched is seen in
the device memory that a call takes (records per workgroup).
CPU through the HIP emulation.
"""
import os
import subprocess
import sys

from tests import helpers

EMU_DIR = os.path.join(helpers.ROOT, "tests", "emu")

# Prints what the calls of an engine allocate, tuned by argv[1], and the shapes it reports.
SCRIPT = """
import ctypes, os, sys
import numpy as np
import care_amd
lib = care_amd._bind(ctypes.CDLL(os.path.join(sys.argv[2], "_build", "libcare_amd_emu.so")), care_amd.ENGINE_SYMBOLS)
rng = np.random.default_rng(1)
n, length = 600, 60
genome = rng.integers(0, 4, 2000)
at = rng.integers(0, len(genome) - length, n)
seqs = np.zeros((n, 4), np.uint32)
for i in range(length):
    seqs[:, i // 16] |= (genome[at + i] << (30 - 2 * (i % 16))).astype(np.uint32)
opt = care_amd.default_options(kmer_length=20, num_hash_maps=4, coverage=20.0, min_overlap=20)
with care_amd.Engine(opt, device=0, lib=lib) as eng:
    eng.upload(seqs, np.full(n, length, np.int32), None, None, 8, length)
    eng.build()
    how = sys.argv[1]
    if how in ("all", "one"):
        shape = eng.tuning()
        if how == "one":
            shape["query_lds_hits"] = 256
        eng.set_tuning(**shape)
    elif how == "autotuned":
        shape = eng.tuning()
        eng.set_tuning(correct_threads=192, msa_chunk=20, batch_anchors=64, correct_blocks_per_cu=5)
        eng.tuning()
        eng.set_tuning(**shape)
    elif how == "pinned":
        eng.set_launch_config(0, 128)
    live, peak = ctypes.c_uint64(), ctypes.c_uint64()
    for k in (2, 64, 600):
        eng.correct(0, k)
        lib.care_emu_memory(ctypes.byref(live), ctypes.byref(peak))
        print(k, live.value, eng.stats().launches)
    print(sorted((k, v) for k, v in eng.tuning().items() if k != "query_lds_hits"))
"""


def _run(how):
    env = dict(os.environ, EMU_CUS="256", PYTHONPATH=helpers.ROOT)
    p = subprocess.run([sys.executable, "-c", SCRIPT, how, EMU_DIR], env=env, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-2000:]
    return p.stdout


def test_reported_shapes_set_again(tmp_path):
    subprocess.run(["sh", os.path.join(EMU_DIR, "build_emu.sh")], check=True)
    default = _run("none")
    assert _run("all") == default
    assert _run("one") == default
    assert _run("autotuned") == default
    # another workgroup size is seen in what is launched
    assert _run("pinned") != default
