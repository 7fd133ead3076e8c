"""What the kernels of the built library were compiled to need, from the metadata of its code objects."""
import os
import re
import shutil
import subprocess

import pytest

from quartet_amd import _lib

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled name: (vector registers, bytes of scratch per lane)}"""
    tools = [shutil.which(t, path=f"{LLVM}:{os.environ['PATH']}") for t in ("llvm-objdump", "llvm-readelf", "c++filt")]
    if not os.path.exists(_lib.LIB_PATH) or not all(tools):
        pytest.skip("needs the built library, ROCm's LLVM tools and c++filt")
    where = tmp_path_factory.mktemp("objects")
    lib = shutil.copy(_lib.LIB_PATH, where)
    subprocess.run([tools[0], "--offloading", lib], cwd=where, check=True, capture_output=True)
    found = {}
    for f in sorted(os.listdir(where)):
        if f.endswith("gfx950"):
            notes = subprocess.run([tools[1], "--notes", os.path.join(where, f)], check=True, capture_output=True, text=True).stdout
            for k in notes.split("  - .agpr_count:")[1:]:
                get = lambda key: re.search(rf"^    \.{key}:\s+(\S+)", k, re.M).group(1)
                found[get("name")] = (int(get("vgpr_count")), int(get("private_segment_fixed_size")))
    names = subprocess.run([tools[2]], input="\n".join(found), check=True, capture_output=True, text=True).stdout.split("\n")
    return dict(zip(names, found.values()))


def test_products_keep_nothing_in_memory(kernels):
    """A tile runs 5 to 30 K steps: what its prologue spills is not paid back.  With the rotation in the epilogue as without."""
    tiles = {n: v for n, v in kernels.items() if "tile_kernel<" in n}
    persistent = {n: v for n, v in kernels.items() if "gemm_mxfp4_tn_big4_kernel" in n}
    assert tiles and persistent
    assert {n: v for n, v in {**tiles, **persistent}.items() if v[1]} == {}


@pytest.mark.parametrize("name", ["gemm_mxfp4_tn_two_kernel<", "gemm_bf16_logits_kernel<", "gemm_mxfp4_tn_rows_kernel<", "linear_decode_kernel<", "gemm_mxfp4_tn_pair_kernel<",
                                  "gemm_mxfp4_e5m2_pair_kernel<", "gemm_mxfp4_tn_after_kernel<"])
def test_other_products_keep_nothing_in_memory(kernels, name):
    """The first two are within ten of the registers that two workgroups to a CU leave a lane."""
    found = {n: v for n, v in kernels.items() if name in n}
    assert found and {n: v for n, v in found.items() if v[1]} == {}
    if "two_kernel" in name or "logits" in name:
        assert all(v[0] <= 256 for v in found.values()), found


def test_a_rotation_in_the_epilogue_holds_no_registers_through_the_product(kernels):
    """The last template argument is the rotation.  Its lane constants belong to the epilogue: a few registers' difference, not 16."""
    tiles = {n: v[0] for n, v in kernels.items() if "tile_kernel<" in n}
    rotating = {n: v for n, v in tiles.items() if "true>(qm::TileProduct" in n}
    assert rotating
    for n, registers in rotating.items():
        plain = tiles[n.replace("true>(qm::TileProduct", "false>(qm::TileProduct")]
        assert registers <= plain + 4, (n, registers, plain)


def test_backward_quantizers_fit_their_waves_without_scratch(kernels):
    """The grid of the four quantizers of a backward pass: 512 registers a lane shared by five waves, four for wider blocks."""
    grids = {n: v for n, v in kernels.items() if "job_kernel<" in n and "TransposedJob<" in n and "RequantTiledJob<" in n}
    assert len(grids) >= 12
    for n, (registers, scratch) in grids.items():
        block = int(re.search(r"RequantTiledJob<\d+, (\d+),", n).group(1))
        assert scratch == 0 and registers <= (96 if block == 32 else 128), (n, registers, scratch)


def test_norm_producers_of_eight_elements_a_lane_have_no_scratch(kernels):
    """The RMSNorm in front of a quantizer of rows of up to 2048 elements, 2^24 in all: latency is what bounds it, so waves are what it wants, eight to a SIMD."""
    found = {n: v for n, v in kernels.items() if "RmsNormOctetsJob<" in n}
    assert len(found) >= 3
    for n, (registers, scratch) in found.items():
        assert scratch == 0, (n, scratch)
        if "RowmajorTiledJob" not in n:   # the weight's quantizer in the same grid has its own need
            assert registers <= 64, (n, registers)


def test_norm_producers_fit_four_waves_without_scratch(kernels):
    """The RMSNorm in front of a quantizer, fp32 rows with a bf16 residual summand, wider or more of them than eight elements a lane serve."""
    found = {n: v for n, v in kernels.items() if "RmsNormProducer<float, unsigned short>, true" in n}
    assert len(found) >= 6
    for n, (registers, scratch) in found.items():
        assert scratch == 0 and registers <= 128, (n, registers, scratch)
