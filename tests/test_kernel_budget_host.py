"""CPU: the compiler's report on kernels that test_abi's lists do not name: no scratch (the tile product reads LDS by assembly whose waits stand in other statements: a
destination spilled while its read is in flight would lose the data), and the waves per SIMD that their launches count on."""
import pytest

from tests.test_abi import _kernel_resources


@pytest.mark.parametrize("part,count,waves", [
    ("gemm_tile_rows_kernel", 4, 2),        # QKV products in blocks of 128 and 192 rows, 16- and 24-bit caches: workgroups of eight waves
    ("attn_prefill_dealt_kernel", 4, 2),    # 128 with 16, 24 bits of V, 24 of both, 64: two workgroups of four waves on a CU
    ("gemm_rowsum_kernel", 6, 4),           # workgroups of sixteen waves
    ("gemm_rowslab_kernel", 1, 4),
    ("exact_rows16_kernel", 3, 4),          # ... and of eight, two on a CU
    ("copy_out_kernel", 1, 2),
])
def test_no_scratch(part, count, waves):
    hits = {n: r for n, r in _kernel_resources().items() if part in n}
    assert len(hits) == count, sorted(hits)
    for n, r in hits.items():
        assert r["ScratchSize [bytes/lane]"] == 0 and r["Occupancy [waves/SIMD]"] >= waves, (n, r)
