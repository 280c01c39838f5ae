"""Which kernels store their results through the L2s (write_through.h), read off the generated code (no GPU needed, hipcc only)."""
import re

from test_asm_hazards import assembly

THROUGH = re.compile(r"global_store_dwordx[24] .* sc0 sc1$")


def kernels(source):
    """symbol -> (stores written through, plain stores) of every kernel of a source"""
    found, name = {}, None
    for line in assembly(source):
        m = re.match(r"(_Z\w+):", line)
        if m:
            name = m.group(1)
            found[name] = [0, 0]
        elif line.startswith("global_store"):
            found[name][0 if THROUGH.match(line) else 1] += 1
    return found


def test_rounding_to_bf16_stores_plainly():
    found = [n for k, n in kernels("ew_norm_ops.hip").items() if "13k_f32_to_bf16" in k]
    assert len(found) == 2 and all(through == 0 and plain > 0 for through, plain in found)


def test_tiles_of_a_product_are_stored_one_way_by_a_kernel():
    """f32 results and partial sums plainly or through, bf16 results plainly"""
    found = {k: n for k, n in kernels("gemm_tiles_gfx950.hip").items() if "12k_gemm_tiles" in k}
    f32 = [n for k, n in found.items() if "12k_gemm_tilesIf" in k]
    assert len(f32) == 16 and sum(through > 0 for through, _ in f32) == 8
    assert all((through > 0) != (plain > 0) for through, plain in f32)
    assert all(through == 0 and plain > 0 for k, (through, plain) in found.items() if "12k_gemm_tilesIf" not in k)
