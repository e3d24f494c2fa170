"""The check of the distances that inline matrix instructions need (csrc/check_products.py), on mistakes planted in listings and on the built extension."""

import glob
import importlib.util
import os

import pytest

import colossalai_amd

HERE = os.path.dirname(colossalai_amd.__file__)
_spec = importlib.util.spec_from_file_location("check_products", os.path.join(HERE, "csrc", "check_products.py"))
check = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(check)

M = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"
OTHER = "v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[4:7]"


def _listing(lines):
    """Instructions of four bytes from address 0x100 on; a branch's target is the index behind its `@`."""
    out = ["0000000000000100 <kernel>:"]
    for i, line in enumerate(lines):
        line, _, to = line.partition(" @")
        where = f" <kernel+0x{4 * int(to):x}>" if to else ""
        out.append(f"\t{line:<50} // {0x100 + 4 * i:012X}: BF800000{where}")
    return "\n".join(out)


@pytest.mark.parametrize("lines,wrong", [
    ([M, "s_nop 15", "v_accvgpr_read_b32 v9, a3", "s_endpgm"], 0),
    ([M, "s_nop 10", "v_accvgpr_read_b32 v9, a3", "s_endpgm"], 0),
    ([M, "s_nop 9", "v_accvgpr_read_b32 v9, a3", "s_endpgm"], 1),            # read too early
    ([M, "s_nop 9", "v_accvgpr_read_b32 v9, a4", "s_endpgm"], 0),
    ([M] + ["s_mov_b32 s0, 0"] * 5 + ["ds_write_b128 v8, a[0:3]", "s_endpgm"], 1),
    ([M, "s_nop 4", "v_accvgpr_write_b32 a2, v9", "s_endpgm"], 1),            # written too early
    ([M, "s_branch 2 @3", "v_accvgpr_read_b32 v9, a3", "s_endpgm"], 0),       # on no path
    ([M, "s_cbranch_scc1 2 @4", "s_nop 15", "s_nop 0", "v_accvgpr_read_b32 v9, a3", "s_endpgm"], 1),   # on one of two
    (["v_accvgpr_read_b32 v9, a0", "s_nop 15", M, "s_cbranch_scc1 65000 @0", "s_endpgm"], 1),          # round a loop
    (["v_mov_b32_e32 v5, v9", "s_nop 0", M, "s_endpgm"], 1),                  # an operand written just ahead
    (["v_mov_b32_e32 v5, v9", "s_nop 1", M, "s_endpgm"], 0),
    (["v_accvgpr_write_b32 a1, v9", M, "s_endpgm"], 1),
    (["v_swap_b32 v9, v5", M, "s_endpgm"], 1),
    (["v_mov_b32_e32 v9, v5", M, "s_endpgm"], 0),
    ([M, OTHER, OTHER.replace("a[4:7]", "a[8:11]"), "s_nop 0", M, "s_endpgm"], 0),
    ([M, OTHER, M, "s_endpgm"], 1),                                           # its own sum too early
    ([M, "s_nop 3", M.replace("a[0:3]", "a[2:5]"), "s_endpgm"], 1),           # a part of another's
    ([M, "s_nop 3", OTHER.replace("v[0:3]", "a[0:3]"), "s_endpgm"], 1),       # another's as a factor
])
def test_planted(lines, wrong):
    found, seen = check.problems(_listing(lines), "kernel")
    assert (len(found) > 0) == wrong, found
    assert seen == sum(line.startswith("v_mfma") for line in lines)


def test_the_built_extension():
    built = glob.glob(os.path.join(HERE, "_C.*.so"))
    if not built or check.objdump() is None:
        pytest.skip("no built extension, or no disassembler")
    check.check(built[0])
