"""CPU: the resident decode step as hipcc made it: two waves a SIMD, one workgroup to a CU, nothing in scratch (a spilled register would wait for the weights in flight)."""
import os

import pytest

PATH = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-candle_amd", "kernel_resources_resident.txt")


def test_registers():
    if not os.path.exists(PATH):
        pytest.skip("not built here")
    kernels, name = {}, None
    for line in open(PATH):
        key, value = line.strip().rsplit(": ", 1)
        if key == "Function Name":
            name = value
        else:
            kernels.setdefault(name, {})[key] = int(value)
    steps = {n: r for n, r in kernels.items() if "resident_step_kernel" in n}
    assert len(steps) == 4, sorted(kernels)
    for n, r in steps.items():
        assert r["ScratchSize [bytes/lane]"] == 0 and r["Occupancy [waves/SIMD]"] == 2, (n, r)
