"""FP16-stored fields of the library itself (not the reference's, which has no
FP16), from the revision before any kernel made several steps per launch: its
collision in moments, one step per launch.  Needs the GPU and that revision's
package first in sys.path.

usage: PYTHONPATH=<that tree> python tests/golden/make_f16.py OUTPUT.npz
"""
import os
import sys

import numpy as np

sys.path.append(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import test_gpu_f16_bits as T  # noqa: E402

np.savez_compressed(sys.argv[1], **{name: T.run(name) for name in T.RUNS})
print("wrote", sys.argv[1])
