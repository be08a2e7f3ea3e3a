"""CPU: hand-offs between the waves of a launch and to the host, in the code objects as hipcc made them here.  Values rarely show a missing wait: what is late by a
microsecond is there when the test looks.  And what a loop hands to its next turn."""
import os
import re
import shutil
import subprocess

import pytest

from nano_vllm_candle_amd._lib import LIB_PATH

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def instructions(tmp_path_factory):
    """instructions(part): the instructions of the kernel whose name holds `part`"""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("objects")
    run = lambda *a: subprocess.run([OBJDUMP, *map(str, a)], cwd=d, check=True, capture_output=True, text=True).stdout.splitlines()
    shutil.copy(LIB_PATH, d / "lib.so")
    run("--offloading", d / "lib.so")
    found = [(obj, line.split()[-1]) for obj in sorted(d.glob("lib.so.*gfx950")) for line in run("--syms", obj) if " F " in line]

    def of(part):
        (obj, name), = [f for f in found if part in f[1]]
        return [re.sub(r"\s*//.*", "", line).strip() for line in run("-d", f"--disassemble-symbols={name}", obj) if line.startswith("\t")]

    return of


def test_a_copy_to_the_host_waits_for_the_stores_of_every_wave(instructions):
    # One thread counts for its workgroup.  On gfx950 neither a barrier nor another wave's fence waits for a wave's stores.
    ops = instructions("copy_out_kernel")
    barrier = ops.index("s_barrier")
    stores = [i for i, o in enumerate(ops[:barrier]) if o.startswith("global_store")]
    assert stores and any(re.match(r"s_waitcnt .*vmcnt\(0\)", o) for o in ops[stores[-1]:barrier]), ops[stores[-1]:barrier + 1]


def test_a_decode_records_position_is_read_by_the_lane_that_writes_it(instructions):
    # Sixteen lanes move a record on and all of them need the position that one of them overwrites: they have it from that lane, and no store comes before.
    ops = instructions("advance_decode_kernel")
    across = [i for i, o in enumerate(ops) if re.match(r"ds_bpermute|ds_swizzle|v_readlane|v_mov_b32_dpp", o)]
    assert across, ops
    stores = [i for i, o in enumerate(ops) if o.startswith("global_store")]
    record = [i for i in stores if i > across[0]]
    reads = [i for i, o in enumerate(ops) if o.startswith("global_load") and i > across[0]]
    assert record and reads and not any("offset:8" in ops[i] for i in reads), ops


@pytest.mark.parametrize("hd,sets,lo", [(128, 1, 0), (128, 1, 1), (128, 1, 2), (128, 2, 0), (128, 2, 1), (128, 2, 2), (64, 1, 0), (64, 2, 0)])
def test_the_sum_over_v_stays_in_its_registers_from_tile_to_tile(instructions, hd, sets, lo):
    # A K/V tile's last products write where the next tile's read: no pair of registers moves between the first product and the last.
    ops = instructions(f"attn_prefill_kernelILi{hd}ELi2ELi{sets}ELi{lo}E")
    products = [i for i, o in enumerate(ops) if "mfma" in o]
    moves = [o for o in ops[products[0]:products[-1]] if o.startswith("v_mov_b64")]
    assert products and not moves, moves
