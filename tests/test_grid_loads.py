"""The class-grid kernels fetch scan points ahead of their use, past the end of
their chunk, and leave those loads to the buffer descriptor's range check.  A
raw buffer's check covers the vector offset and the instruction's constant; a
scalar offset is outside it (past the descriptor's end the check would let the
load through, up to 192 points behind the scan's allocation).  So every buffer
load of the compiled kernels has the scalar offset 0."""
import os
import re
import subprocess

from tsdf_localization_amd import build


def test_buffer_loads_have_no_scalar_offset(tmp_path):
    out = tmp_path / "grid_eval.s"
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S", "-o", str(out),
                    os.path.join(build.CSRC, "grid_eval.hip")], check=True, capture_output=True)
    loads = re.findall(r"^\s*(buffer_load_\S+)\s+(.*)$", out.read_text(), flags=re.M)
    points = [(op, args) for op, args in loads if "offen" in args]
    assert len(points) >= 12  # six kernels, at least the pipeline's two loads each
    for op, args in points:
        soffset = args.split("],")[-1].split()[0]
        assert soffset == "0", f"{op} {args}"
