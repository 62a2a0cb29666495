"""Writes tests/golden/stopped_iterates.npz: MINRES solutions after a fixed number of
steps (tests/test_gpu_stopped_iterates.py), from the library as it is built.  The
committed values are those of revision 89a5a5b on an MI355X, whose steps took the cell
product line by line before another kernel existed.

Run from the repository root on a GPU:  python tests/golden/make_stopped_iterates.py
"""
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

import invdft_amd  # noqa: E402
from tests import test_gpu_stopped_iterates as t  # noqa: E402


def main():
    lib = invdft_amd.load()
    np.savez_compressed(t.FIX, **{t.name(c): t.iterate(lib, *c) for c in t.CASES})


if __name__ == "__main__":
    main()
