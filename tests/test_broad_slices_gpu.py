"""Recurrences of 1025 to 1536 units with slices of 32 units (more rows than 16-row blocks of slices of 16 seat), against the CPU
oracle, 64-bit arithmetic and the kernels with 32-row blocks."""
import numpy as np
import pytest

from helpers import check_against, make_problem
from test_core_gpu import oracle_reference, run_core

pytestmark = pytest.mark.gpu

# the first row past slices of 16, all groups seated with and without a partial block, one row more than that (several blocks per
# group and step), three blocks; contractions of 33 (the shortest), 35, 40 (both forward kernels' ends), 44 and 48 k-steps
SHAPES = [(5, 49, 1025), (6, 112, 1056), (4, 100, 1120), (7, 81, 1280), (3, 97, 1281), (6, 33, 1400), (5, 80, 1536), (4, 81, 1536), (3, 161, 1536)]


NARROW_FORWARD = [(97, 1281), (81, 1536), (161, 1536), (165, 1280)]   # slices of 16 forward: as many turns a step with 32-row blocks


@pytest.mark.parametrize("T,B,H", SHAPES)
@pytest.mark.parametrize("stepwise", [False, True])
def test_slices_of_32_units_against_the_oracle(T, B, H, stepwise):
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    got, info = run_core(p, stepwise=stepwise, core=core)
    assert info["fallbacks"] == 0 and core.info("slice_bwd") == 32 and core.info("slice_fwd") == (16 if (B, H) in NARROW_FORWARD else 32)
    core.close()
    check_against(ref, got, label=f"B={B} H={H} stepwise={stepwise}")


# over enough steps that every slot of the rings is used again, no further from 64 bits than 32-row blocks with slices of 16
# (a sum's order flips roundings of dG: 5 %, as between the other layouts); and the option for those is honoured without packing again
@pytest.mark.parametrize("T,B,H", [(24, 48, 1536), (21, 80, 1400), (22, 165, 1280), (25, 100, 1100)])
def test_slices_of_32_units_against_64_bits_and_32_row_blocks(T, B, H):
    from flashlstm_poc_amd import LstmCore
    from helpers import reference_64, rell2
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref = {k: v.cpu().numpy() for k, v in reference_64(p).items()}
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    got, info = run_core(p, core=core)
    assert info["fallbacks"] == 0 and core.info("slice_bwd") == 32 and core.info("row_tiles_bwd") == 1
    assert core.info("slice_fwd") == (16 if (B, H) in NARROW_FORWARD else 32)
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 2)
    blocks, info = run_core(p, core=core)
    assert info["fallbacks"] == 0 and core.info("slice_bwd") == 16 and core.info("slice_fwd") == 16 and core.info("row_tiles_bwd") == 2
    for k in ref:
        assert rell2(got[k], ref[k]) <= 1.05 * rell2(blocks[k], ref[k]), (k, rell2(got[k], ref[k]), rell2(blocks[k], ref[k]))
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 0)
    again, _ = run_core(p, core=core)
    for k in got:
        assert np.array_equal(again[k], got[k]), k
    core.close()


# 33 to 48 rows where slices of 16 would seat them as well: forward alone; one row fewer keeps those
@pytest.mark.parametrize("T,B,H,forward", [(22, 33, 1056, 32), (21, 40, 1216, 32), (23, 48, 1344, 32), (21, 32, 1216, 16)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_forward_slices_where_both_kinds_are_seated(T, B, H, forward, stepwise):
    from flashlstm_poc_amd import LstmCore
    from helpers import reference_64, rell2
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref = {k: v.cpu().numpy() for k, v in reference_64(p).items()}
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    got, info = run_core(p, core=core, stepwise=stepwise)
    assert info["fallbacks"] == 0 and core.info("slice_fwd") == forward and core.info("slice_bwd") == 16
    core.set_option("row_tiles_fwd", 2)
    blocks, info = run_core(p, core=core)
    assert info["fallbacks"] == 0 and core.info("slice_fwd") == 16
    for k in ref:   # (as above)
        assert rell2(got[k], ref[k]) <= 1.05 * rell2(blocks[k], ref[k]), (k, rell2(got[k], ref[k]), rell2(blocks[k], ref[k]))
    core.close()


@pytest.mark.parametrize("T,B,H", [(21, 80, 1100), (23, 48, 1536), (20, 90, 1400)])
def test_slices_of_32_units_in_ranges_of_steps(T, B, H):
    from test_kernel_variants_gpu import test_wide_layers_in_ranges_of_steps as in_ranges
    in_ranges(T, B, H)
