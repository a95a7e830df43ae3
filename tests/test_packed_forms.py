"""The packed product of 2 to 16 rows, read in the assembly that is made here from its source: launches of one product carry nothing of the
form that takes several.  The kernel has no scalar registers to spare, and a decode step of a small model is a chain of such launches."""
import os
import re
import subprocess

import pytest


def test_one_product_pays_nothing_for_several_in_one_launch(tmp_path):
    """Nothing but the form for several products asks for the grid's third dimension, which numbers them."""
    from rust_inference_amd.errors import KernelError
    from rust_inference_amd.kernels import build
    try:
        hipcc = build._hipcc()
    except KernelError as e:
        pytest.skip(str(e))
    name, out = "gemm_skinny_bf16.hip", str(tmp_path / "kernels.s")
    subprocess.run([hipcc, *build.HIPCC_FLAGS, *build.FILE_FLAGS.get(name, []), "--cuda-device-only", "-S", os.path.join(build.CSRC, name), "-o", out],
                   check=True, env=dict(os.environ, HOME=os.environ.get("HOME", str(tmp_path))), capture_output=True)
    with open(out) as f:
        text = f.read()
    third = {kernel: int(re.search(r"\.amdhsa_system_sgpr_workgroup_id_z (\d)", body)[1])
             for kernel, body in re.findall(r"\.amdhsa_kernel (\S*gemm_skinny_packed_kernel\S*)\n(.*?)\.end_amdhsa_kernel", text, re.S)}
    # (the last template argument but for the closing ones: ...Lb<batch>EEv; the forms of one product are 4 and 8 wavefronts, with the
    # activation or not, both result types, two steps to a load or one)
    batch = {kernel for kernel in third if re.search(r"ELb1EEv", kernel.split("packed_kernel")[1])}
    assert len(third) == 24 and len(batch) == 8
    assert {kernel for kernel, z in third.items() if z} == batch
