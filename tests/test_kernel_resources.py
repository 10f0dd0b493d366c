"""CPU check of the hot kernels' private (scratch) memory, from the
compiler's resource report for gfx950.

An index the compiler cannot resolve into the by-value MoeArgs kernel
argument makes it copy the whole struct to scratch in every thread (the
per-token kernels ran 4x slower that way); spills show up the same way.
The kernels listed here must use no scratch at all; where waits count
vector-memory instructions (the tile product, the LDS rings), a spill would
also break the count.
"""
import re

import pytest

from logan_amd import build

from _asm import compiled

HOT = {
    "gemm.hip": [r"affine_qmm_tile_kernelILi%dELi%dE" % (b, mi) for b in (4, 5, 6, 8) for mi in (1, 2, 4, 6, 8)],
    "moe.hip": [r"moe_gateup_kernelILi4ELi1E", r"moe_down_kernelILi4ELi16E", r"moe_route_tok_kernel",
                r"moe_group_kernel", r"moe_combine_kernel"],
    "moe_fused.hip": [r"moe_fused_b1_kernelILi4ELi1ELi16E"],
    "moe_mfma.hip": [r"moe_gateup_lds_kernel", r"moe_gateup_wide_kernel", r"moe_down_lds_kernel", r"moe_gateup_mfma_kernelILi4E",
                     r"moe_down_mfma_kernelILi4E", r"moe_mroute_kernel", r"moe_mgroup_kernel",
                     r"moe_mcombine_kernel"],
}


def test_hot_moe_kernels_use_no_scratch():
    try:
        build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    from concurrent.futures import ThreadPoolExecutor

    with ThreadPoolExecutor(len(HOT)) as ex:
        reps = dict(zip(sorted(HOT), ex.map(lambda s: compiled(s)[1], sorted(HOT))))
    for src, pats in HOT.items():
        for pat in pats:
            hits = {k: v for k, v in reps[src].items() if re.search(pat, k)}
            assert hits, f"no kernel matches {pat} in {src}"
            bad = {k: v for k, v in hits.items() if v["ScratchSize [bytes/lane]"] != 0}
            assert not bad, f"scratch in {src}: {bad}"


def test_tile_product_of_32_rows_fits_two_blocks_a_cu():
    """Products of few rows and 257 to 512 column tiles run in one round only
    if a CU holds two blocks: half of its LDS, and 128 registers a thread."""
    try:
        build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    ks = {k: v for k, v in compiled("gemm.hip")[1].items() if re.search(r"affine_qmm_tile_kernelILi\dELi1E", k)}
    assert len(ks) == 24
    bad = {k: v for k, v in ks.items() if v["LDS Size [bytes/block]"] > 81920 or v["VGPRs"] > 128}
    assert not bad


def test_tile_product_stores_whole_runs():
    """Aligned rows of y are stored 16 bytes a lane, the tile turned through
    LDS; 8-byte stores are those of the sums' own layout (bf16), 16 bytes in
    each of 32 rows per instruction."""
    try:
        build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    stores, kernel = {}, None
    with open(compiled("gemm.hip")[0]) as f:
        for line in f:
            m = re.match(r"(_ZN\S*affine_qmm_tile_kernel\S+):", line)
            if m:
                kernel = stores.setdefault(m[1], [])
            elif line.startswith(".Lfunc_end"):
                kernel = None
            elif kernel is not None:
                m = re.match(r"\s+(global_store\w+)", line)
                if m:
                    kernel.append(m[1])
    assert len(stores) == 119
    for name, ops in stores.items():
        assert "global_store_dwordx4" in ops and "global_store_dwordx2" not in ops, name
