"""The raster service's kernel reads its jobs' tables with vector loads only: they
change while it runs, and the scalar cache is invalidated only when a kernel
starts, so a scalar load could return an earlier job's record. Its scalar loads
are those of its own arguments."""
import os
import re
import subprocess

from rusterizer_amd import build


def test_service_kernel_reads_no_job_table_through_the_scalar_cache(tmp_path):
    out = tmp_path / "k.s"
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "-S", "--cuda-device-only",
                    os.path.join(build.CSRC, "rz_kernels.hip"), "-o", str(out)], check=True, capture_output=True)
    text = out.read_text()
    body = text[re.search(r"^_ZN3rzk16k_raster_service\w*:", text, re.M).start():]
    body = body[:body.index(".Lfunc_end")]
    loads = re.findall(r"^\s+(s_load_\w+ .*|s_buffer_load_\w+ .*)$", body, re.M)
    assert 1 <= len(loads) <= 4, loads
