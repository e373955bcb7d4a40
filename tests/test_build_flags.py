"""Device build flags against what the sources rely on (CPU)."""
import glob
import os

from gonn_amd import build as gbuild


def test_files_that_look_for_nan_honour_it():
    # nonfinite() and SplitCheck (common.h) find an operand without a three-piece
    # split by the NaN that its pieces make; a build without NaNs may drop it.
    users = [f for f in glob.glob(os.path.join(gbuild.CSRC, "*.hip"))
             if any(x in open(f).read() for x in ("nonfinite(", "SplitCheck"))]
    assert len(users) >= 4, "fp32 forward, dK/dV, dQ and the cache attend"
    for f in users:
        for flag in gbuild.CFLAGS + gbuild.FILE_FLAGS.get(os.path.basename(f), []):
            assert flag not in ("-fno-honor-nans", "-ffinite-math-only", "-ffast-math", "-mno-amdgpu-ieee"), (f, flag)
