"""Writes flow_values.npz, the kept samples of tests/test_gpu_flow_values.py,
from the library that turbins_amd loads (run on a GPU)."""
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.dirname(HERE), os.path.dirname(os.path.dirname(HERE))]

import test_gpu_flow_values as T  # noqa: E402

out = sys.argv[1] if len(sys.argv) > 1 else T.GOLDEN
np.savez_compressed(out, **{f"{f}_{n}": a for f in T.FLOWS for n, a in T.flow_samples(f).items()})
