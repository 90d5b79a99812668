"""Writes the energies that test_gpu_fp32_bits.py holds the FP32 kernels to.

    python tests/golden/make_fp32_energies.py TREE OUT.npz

TREE is a built checkout whose FP32 transforms are the ones to keep; the
systems come from the test's own tables.
"""
import os
import sys

tree, out = os.path.abspath(sys.argv[1]), sys.argv[2]
tests = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path[:0] = [tree, tests]

import numpy as np  # noqa: E402

import test_gpu_fp32_bits as T  # noqa: E402

made = {}
for table in (T.REGISTER, T.OTHER):
    for i, (name, case) in enumerate(table.items()):
        print(name, case, flush=True)
        made[name] = T.energies(case, i)
np.savez_compressed(out, **made)
