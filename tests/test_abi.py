"""CPU: the C-ABI library loads and exports every symbol include/nvllm_amd.h declares; failures are loud."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "nvllm_amd.h")              # the boundary a maintainer binds
DEBUG_HEADER = os.path.join(ROOT, "include", "nvllm_amd_debug.h")  # profiling / parity-debug / tuning exports


def header_functions(paths=(HEADER, DEBUG_HEADER)):
    names = set()
    for path in paths:
        src = open(path).read()
        src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
        names.update(re.findall(r"\b(nvllm_[a-z0-9_]+)\s*\(", src))
    return sorted(names)


def test_boundary_header_holds_no_debug_or_tuning_exports():
    names = header_functions((HEADER,))
    assert not [n for n in names if "_debug_" in n or "_profile_" in n], names


def test_library_exports_every_header_symbol():
    import ctypes

    import nano_vllm_candle_amd as pkg

    lib = ctypes.CDLL(pkg._lib.LIB_PATH)
    names = header_functions()
    assert len(names) >= 40
    for n in names:
        assert hasattr(lib, n), f"{n} declared in include/nvllm_amd.h but not exported"


def test_python_binding_covers_the_header():
    import nano_vllm_candle_amd as pkg

    assert sorted(pkg._lib.EXPORTED_SYMBOLS) == header_functions()


def test_library_is_in_tree_and_no_cpu_fallback():
    import nano_vllm_candle_amd as pkg

    assert os.path.dirname(pkg._lib.LIB_PATH).endswith("nano-vllm-candle_amd")
    # the product never imports the oracle
    for root, _, files in os.walk(os.path.join(ROOT, "nano-vllm-candle_amd")):
        for f in files:
            if f.endswith((".py", ".cpp", ".hip", ".h")):
                txt = open(os.path.join(root, f)).read()
                assert "import oracle" not in txt and "from oracle" not in txt and "qwen3_oracle" not in txt, f


@pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="a GPU is present")
def test_context_creation_fails_loudly_without_a_gpu():
    import nano_vllm_candle_amd as pkg

    with pytest.raises(pkg._lib.NvllmError):
        pkg.Context(0)


def test_missing_library_raises(monkeypatch, tmp_path):
    import nano_vllm_candle_amd as pkg

    monkeypatch.setattr(pkg._lib, "_lib", None)
    monkeypatch.setattr(pkg._lib, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(pkg._lib.NvllmLibraryMissing):
        pkg._lib.lib()


def _kernel_resources():
    out = {}
    for name in ("kernel_resources.txt", "kernel_resources_tile.txt", "kernel_resources_stream.txt", "kernel_resources_latent_ops.txt", "kernel_resources_latent.txt", "kernel_resources_latent_prefill.txt", "kernel_resources_bias_attn.txt",
                 "kernel_resources_recurrent.txt", "kernel_resources_recurrent_chunk.txt", "kernel_resources_scan.txt", "kernel_resources_moe.txt",
                 "kernel_resources_conv_attn.txt"):
        path = os.path.join(ROOT, "nano-vllm-candle_amd", name)
        if not os.path.exists(path):
            pytest.skip(name + " missing: rebuild the library (make -C nano-vllm-candle_amd/csrc)")
        for blk in open(path).read().split("Function Name: ")[1:]:
            lines = blk.strip().splitlines()
            out[lines[0].strip()] = {k.strip(): int(v) for k, v in (l.split(":", 1) for l in lines[1:])}
    return out


def test_hot_kernels_keep_their_register_budget():
    # hipcc's own per-kernel report, written beside the library by the build.  The decode path is tuned to exact wave
    # counts per SIMD: the decode attention kernel at 2 waves (<= 256 registers; at 269 it silently ran at 1 wave per
    # SIMD and the whole step lost 12 %), the register-direct GEMMs of the 0.6B layer at >= 4 (16-wave workgroups),
    # none of them with scratch in its inner loop.
    res = _kernel_resources()
    want = {  # mangled-name prefix -> minimum waves per SIMD
        "_ZN5nvllm17attn_paged_kernelILi128ELi4ELb1ELi0EEE": 2,   # fused decode attention, head_dim 128
        "_ZN5nvllm17attn_paged_kernelILi128ELi4ELb0ELi0EEE": 2,
        "_ZN5nvllm17attn_paged_kernelILi128ELi4ELb1ELi1EEE": 2,   # ... with the 24-bit V cache (one tile set per wave)
        "_ZN5nvllm17attn_paged_kernelILi128ELi4ELb1ELi2EEE": 2,   # ... with 24-bit K and V
        "_ZN5nvllm18gemm_rowdir_kernelILi4ELi16ELi2ELi2EEE": 4,   # QKV        (0.6B: N 4096, K 1024)
        "_ZN5nvllm18gemm_rowdir_kernelILi1ELi16ELi4ELi0EEE": 4,   # o_proj     (N 1024, K 2048)
        "_ZN5nvllm18gemm_rowdir_kernelILi6ELi16ELi2ELi1EEE": 4,   # gate/up    (N 6144, K 1024)
        "_ZN5nvllm18gemm_rowdir_kernelILi1ELi16ELi6ELi0EEE": 4,   # down_proj  (N 1024, K 3072)
        "_ZN5nvllm23gemm_rowdir_loop_kernelILi4ELi16ELi2ELi2EEE": 4,  # the same four where a workgroup walks several row blocks
        "_ZN5nvllm23gemm_rowdir_loop_kernelILi1ELi16ELi4ELi0EEE": 4,
        "_ZN5nvllm23gemm_rowdir_loop_kernelILi6ELi16ELi2ELi1EEE": 4,
        "_ZN5nvllm23gemm_rowdir_loop_kernelILi1ELi16ELi6ELi0EEE": 4,
        "_ZN5nvllm18gemm_rowdir_kernelILi8ELi16ELi2ELi5EEE": 4,   # QKV of short prompts, norm, rotation and cache writes in it
        "_ZN5nvllm13lmhead_kernelILi4ELi5ELi4EEE": 2,             # LM head, 64 rows, vocabulary 151936, K 1024
        "_ZN5nvllm16gemm_tile_kernelILi8ELi2ELi0EEE": 2,              # prefill tile GEMM: 8-wave workgroups, two waves per SIMD
        "_ZN5nvllm16gemm_tile_kernelILi6ELi2ELi2EEE": 2,
        "_ZN5nvllm16gemm_tile_kernelILi8ELi2ELi3EEE": 2,              # ... with the q/k-norm + RoPE + KV-write epilogue
        "_ZN5nvllm16gemm_tile_kernelILi8ELi2ELi9EEE": 2,              # ... into a 24-bit cache
        "_ZN5nvllm19attn_prefill_kernelILi128ELi2ELi1ELi0EEE": 2,     # prompt attention, one and two sets of waves
        "_ZN5nvllm19attn_prefill_kernelILi128ELi2ELi2ELi0EEE": 2,
        "_ZN5nvllm17exact_rows_kernelILi1ELi8EEE": 4,                 # 32-bit products of few rows (8-wave workgroups) ...
        "_ZN5nvllm17exact_rows_kernelILi1ELi16EEE": 4,
        "_ZN5nvllm17exact_tile_kernelE": 2,                           # ... and of many
    }
    # with a 24-bit cache the fused attention kernels spill a few prologue values (outside the K/V loop)
    scratch = {"_ZN5nvllm17attn_paged_kernelILi128ELi4ELb1ELi1EEE": 52, "_ZN5nvllm17attn_paged_kernelILi128ELi4ELb1ELi2EEE": 116}
    for prefix, min_waves in want.items():
        hits = [(n, r) for n, r in res.items() if n.startswith(prefix)]
        assert len(hits) == 1, (prefix, [n for n, _ in hits])
        r = hits[0][1]
        assert r["Occupancy [waves/SIMD]"] >= min_waves, (prefix, r)
        assert r["ScratchSize [bytes/lane]"] <= scratch.get(prefix, 0), (prefix, r)


def test_kernels_that_read_lds_by_assembly_do_not_spill():
    # a destination spilled while its read is in flight would lose the data (the prompt products' reads are waited for in other statements)
    res = _kernel_resources()
    for part, count in (("gemm_tile_kernel", 27), ("attn_prefill_kernel", 8), ("gemm_stream_kernel", 128), ("gemm_rowdir_loop_kernel", 33)):
        hits = {n: r for n, r in res.items() if part in n}
        assert len(hits) == count, (part, len(hits))
        for n, r in hits.items():
            assert r["ScratchSize [bytes/lane]"] == 0, (n, r)


def test_latent_attention_kernels_stay_in_registers():
    # attention over the latent cache, the expansion and the prompt kernel: no scratch in any instance; two waves per SIMD for the
    # attention kernels (their LDS allows two workgroups per CU, or one of eight waves)
    res = {n: r for n, r in _kernel_resources().items() if "latent" in n}
    assert len([n for n in res if "latent_attn_kernel" in n]) == 16
    for n, r in res.items():
        assert r["ScratchSize [bytes/lane]"] == 0, (n, r)
        if "latent_attn_kernel" in n or "latent_prefill_kernel" in n:
            assert r["Occupancy [waves/SIMD]"] >= 2, (n, r)


def test_bias_attention_and_recurrence_kernels_stay_in_registers():
    # prompt kernels read LDS by inline asm: a destination spilled while its read is in flight would lose the data, so no instance may
    # use scratch; the token-by-token scan may for key sizes above 256
    res = _kernel_resources()
    for part, count in (("bias_prefill_kernel", 20), ("bias_decode_kernel", 20), ("piece_scan_kernel", 24), ("delta_pieces_kernel", 8)):
        hits = {n: r for n, r in res.items() if part in n}
        assert len(hits) == count, (part, len(hits))
        for n, r in hits.items():
            assert r["ScratchSize [bytes/lane]"] == 0, (n, r)
    for n, r in res.items():
        if "bias_prefill_kernelILi4ELi8" in n or "bias_decode_kernelILi4ELi8" in n:
            assert r["Occupancy [waves/SIMD]"] >= 2, (n, r)
        if "recurrence_decode_kernelILi2" in n:
            assert r["Occupancy [waves/SIMD]"] >= 4 and r["ScratchSize [bytes/lane]"] == 0, (n, r)


def test_scan_and_expert_kernels_stay_in_registers():
    res = _kernel_resources()
    for part, count in (("scan_prompt_kernel", 18), ("scan_decode_kernel", 9), ("conv_rows16_kernel", 3), ("group_gemm_kernel", 8), ("gemm_tile_kernelILi8ELi2ELi5", 1), ("gemm_tile_kernelILi8ELi2ELi6", 1),
                        ("gemm_tile_kernelILi8ELi2ELi7", 1), ("gemm_tile_kernelILi6ELi2ELi8", 1), ("conv_attn_rows16_kernel", 12), ("conv_attn_decode_kernel", 12)):
        hits = {n: r for n, r in res.items() if part in n and "piece_scan" not in n}
        assert len(hits) == count, (part, len(hits))
        for n, r in hits.items():
            assert r["ScratchSize [bytes/lane]"] == 0, (n, r)
    for n, r in res.items():
        if "scan_prompt_kernelILi4ELi4E" in n or "scan_decode_kernelILi4ELi4E" in n:
            assert r["Occupancy [waves/SIMD]"] >= 4, (n, r)


def test_later_kernels_keep_their_register_budget():
    # the eight-wave attention (one workgroup per CU), the products of two row blocks, the prompt product with the norm's preparation, which
    # reads LDS by assembly: no scratch in any, two waves per SIMD
    res = _kernel_resources()
    for part, count in (("attn_paged_kernelILi128ELi8E", 3), ("gemm_rowpair_kernel", 7), ("tile_resid_kernel", 4), ("exact_rows_loop_kernel", 1)):
        hits = {n: r for n, r in res.items() if part in n}
        assert len(hits) == count, (part, len(hits))
        for n, r in hits.items():
            assert r["ScratchSize [bytes/lane]"] == 0 and r["Occupancy [waves/SIMD]"] >= 2, (n, r)


def test_decode_attention_reads_its_block_table_by_scalar_loads(tmp_path):
    # A vector load of a block number in the tile loop waits for every tile that is in flight before it.  The code objects of this library, as
    # hipcc made them here.
    import shutil
    import subprocess

    from nano_vllm_candle_amd._lib import LIB_PATH

    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump")
    so = shutil.copy(LIB_PATH, tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", str(so)], cwd=tmp_path, check=True, capture_output=True)
    loops = 0
    for obj in sorted(tmp_path.glob("lib.so.*gfx950")):
        names = [l.split()[-1] for l in subprocess.run([objdump, "--syms", str(obj)], check=True, capture_output=True, text=True).stdout.splitlines() if "attn_paged_" in l and " F " in l]
        for name in names:
            asm = subprocess.run([objdump, "-d", f"--disassemble-symbols={name}", str(obj)], check=True, capture_output=True, text=True).stdout.splitlines()
            ops = [l.split()[0] for l in asm if l.startswith("\t")]
            mfma = [i for i, o in enumerate(ops) if "mfma" in o]
            loop = ops[mfma[0]:mfma[-1]]
            assert any(o.startswith("buffer_load") for o in loop) and any(o.startswith("s_load") for o in loop), name
            assert not [o for o in loop if o.startswith(("global_load", "flat_load"))], name
            loops += 1
    assert loops == 12  # head sizes, waves, prologue, forms of the cache, two tiles ahead of the prologue
