"""Registers of the surrogate kernels (compiled here, no GPU): the network's fragments fill the register
file, and what does not fit is spilled inside the KMC step loop."""
import os
import re
import subprocess

from latticemontecarlo_amd import build as B


def test_surrogate_kernels_scratch(tmp_path):
    """At most 224 bytes of scratch per thread, what C = 3 needs for its bookkeeping; 364 bytes took 18 %
    longer per KMC step. The evaluation kernels (one step) need none."""
    name = "lmc_surrogate_kmc.hip"
    asm = str(tmp_path / "k.s")
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *B.FLAGS, *B.SOURCE_FLAGS.get(name, []),
                    "-I" + os.path.join(B.ROOT, "include"), "-I" + B.CSRC, "--cuda-device-only", "-S",
                    os.path.join(B.CSRC, name), "-o", asm], check=True, capture_output=True)
    text = open(asm).read()
    found = re.findall(r"\.name: +(\S*SurrogateKernel\S*)\n\s+\.private_segment_fixed_size: (\d+)", text)
    assert len(found) == 16
    for kernel, scratch in found:
        kmc = re.search(r"SurrogateKernelILi\dELi\dELi\d+ELb(\d)", kernel).group(1) == "1"
        assert int(scratch) <= (224 if kmc else 0), kernel
