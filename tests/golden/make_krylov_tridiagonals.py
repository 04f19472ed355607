"""Writes krylov_tridiagonals.npz: the Lanczos coefficients (a_i, b_i+1) of
tests/test_gpu_krylov_order.py's cases as the library in qpc-tdse-cpc_amd (or
in the directory given) computes them.  Needs an MI355X.

    python tests/golden/make_krylov_tridiagonals.py [library directory [output]]
"""
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, os.path.join(HERE, ".."))
sys.path.insert(0, sys.argv[1] if len(sys.argv) > 1 else os.path.join(ROOT, "qpc-tdse-cpc_amd"))

import qpc_gpu  # noqa: E402
from test_gpu_krylov_order import CASES, case_name, tridiagonal  # noqa: E402


def main():
    out = {}
    for c in CASES:
        out[case_name(c)] = tridiagonal(qpc_gpu, c)
        print(case_name(c), len(out[case_name(c)]), "vectors", flush=True)
    np.savez_compressed(sys.argv[2] if len(sys.argv) > 2 else os.path.join(HERE, "krylov_tridiagonals.npz"), **out)


if __name__ == "__main__":
    main()
