"""The FP64 Roe flux of the stage kernels rounds as IEEE quotients and roots do: its rms error against extended precision,
with the hardware's reciprocals modelled on the host (tests/abi/roe_accuracy.cpp), is no larger than theirs."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_roe_flux_rounds_as_quotients_do(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    out = str(tmp_path / "roe_accuracy")
    subprocess.run([os.path.join(rocm, "llvm", "bin", "clang++"), "-std=c++17", "-O2", "-mfma", "-ffp-contract=fast", "-w",
                    "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "hopefoam_amd", "csrc"), "-isystem", os.path.join(rocm, "include"),
                    os.path.join(HERE, "abi", "roe_accuracy.cpp"), "-o", out], check=True)
    lines = subprocess.run([out], check=True, capture_output=True, text=True, timeout=120).stdout.split("\n")[:3]
    for line in lines:
        kernel, quotients = map(float, line.split())
        # two rms errors of 4e5 samples each, partly the same roundings: their ratio scatters by less than 0.3 %
        assert kernel <= 1.005 * quotients, line
