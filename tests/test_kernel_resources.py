"""The hybrid linears keep their partial sums in registers: no instance of
k_q35_mv, whole or ragged K, uses scratch memory.  (Left free to sink the f64
adds past the loop's branch, the compiler held a whole chunk's widened products
at once: 512 registers and up to 2,740 bytes of scratch where K is not a
multiple of 64, twice the time at 48 rows.)"""
import importlib.util
import os
import re
import subprocess

from conftest import PKG


def test_hybrid_linears_use_no_scratch(tmp_path):
    spec = importlib.util.spec_from_file_location("cohx_build", os.path.join(PKG, "build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    out = tmp_path / "q35.s"
    subprocess.run([b._hipcc(), *b.FLAGS, "-x", "hip", "--cuda-device-only", "-S",
                    os.path.join(PKG, "csrc", "q35_kernels.hip"), "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", out.read_text(), re.S)
    scratch = {name: int(re.search(r"private_segment_fixed_size (\d+)", body)[1])
               for name, body in kernels if "k_q35_mvI" in name}
    assert len(scratch) == 32, len(scratch)  # 4 epilogues x 4 splits x 2 forms of K
    assert not any(scratch.values()), scratch
