"""Kernels and launch choices that a rule picks by size, each at the sizes where the rule or the kernel could go wrong
(both sides of a boundary, remainders, the smallest and the largest of a range), against the CPU oracle."""
import pytest

from helpers import check_against, make_problem
from test_core_gpu import oracle_reference, run_core

pytestmark = pytest.mark.gpu


# hidden sizes on both sides of every step of the contraction the recurrence kernels are built for; the batch decides
# between 16-row blocks (few rows), 32-row blocks (200 rows of 513 units) and the eight-wave kernel (300 rows of 512)
@pytest.mark.parametrize("B,H", [(3, 128), (17, 256), (5, 257), (40, 512), (300, 512), (200, 513), (9, 700), (33, 769), (2, 1024),
                                 (20, 1100), (40, 1536), (7, 1537)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_recurrence_kernels_by_contraction_length(B, H, stepwise):
    p = make_problem(5, B, 24, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    got, info = run_core(p, stepwise=stepwise)
    assert info["fallbacks"] == 0
    check_against(ref, got, label=f"B={B} H={H} stepwise={stepwise}")


# more hidden units than 2048: one kernel per 512 units of the contraction, batch rows in tiles of 16 (one tile, a partial
# second one, several), hidden sizes that are a multiple of nothing
@pytest.mark.parametrize("B,H", [(1, 2049), (16, 2560), (17, 2561), (40, 3072), (3, 3100), (33, 3585), (2, 4096), (18, 4096)])
def test_recurrence_kernels_for_wide_layers(B, H):
    p = make_problem(4, B, 24, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    got, info = run_core(p)
    assert info["fallbacks"] == 0 and info["persistent_fwd"] == 1
    check_against(ref, got, label=f"B={B} H={H}")


# short contractions: the smallest layer, both sides of the lines (64 | 65, 256 | 257, 384 | 385, 512 | 513 units), batches
# that take one, two and four waves per workgroup or just miss them, sequences of one, an odd and an even number of steps
@pytest.mark.parametrize("T,B,H", [(1, 1, 8), (2, 16, 32), (7, 17, 64), (8, 3, 65), (3, 1030, 40), (6, 129, 256), (5, 257, 256),
                                   (4, 513, 256), (9, 64, 257), (4, 130, 288), (5, 33, 384), (6, 130, 385), (4, 128, 512),
                                   (3, 129, 500)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_recurrence_kernels_for_short_contractions(T, B, H, stepwise):
    p = make_problem(T, B, 20, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    got, info = run_core(p, stepwise=stepwise)
    assert info["fallbacks"] == 0
    check_against(ref, got, label=f"T={T} B={B} H={H} stepwise={stepwise}")


# few rows of 32 and 64 units, backward: the two moments at which a step's operands are requested, on both sides of their line, over
# sequences of one, an odd and an even number of steps and some that reuse every slot of the ring
@pytest.mark.parametrize("T,B,H", [(1, 1, 32), (2, 4, 32), (3, 5, 32), (21, 4, 17), (40, 1, 64), (33, 2, 60), (34, 3, 64), (256, 2, 64), (257, 2, 64), (257, 4, 32)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_backward_of_few_rows_of_small_layers(T, B, H, stepwise):
    p = make_problem(T, B, 20, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    got, info = run_core(p, stepwise=stepwise)
    assert info["fallbacks"] == 0
    check_against(ref, got, label=f"T={T} B={B} H={H} stepwise={stepwise}")


# 32-row blocks asked for where the rule takes the kernels for short contractions, which have 16-row blocks: the option and
# a tuned entry are both honoured, after the weights were packed, and taken back without packing again.  One and several row
# blocks, a partial one, a hidden size per kernel family: both short kernels (256), the forward one alone (385, 512)
@pytest.mark.parametrize("T,B,H", [(6, 3, 40), (5, 33, 256), (4, 130, 288), (5, 17, 385), (4, 40, 512)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_row_tile_choice_where_short_contraction_kernels_are_the_rule(T, B, H, stepwise):
    import numpy as np
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 20, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    core = LstmCore(B, 20, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    by_rule, info = run_core(p, core=core, stepwise=stepwise)
    assert info["fallbacks"] == 0 and core.info("row_tiles_fwd") == 1
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 2)
    got, info = run_core(p, core=core, stepwise=stepwise)
    assert info["fallbacks"] == 0 and core.info("row_tiles_fwd") == 2 and core.info("row_tiles_bwd") == 2
    check_against(ref, got, label=f"T={T} B={B} H={H} stepwise={stepwise} 32-row blocks")
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 0)
    assert core.lib.flstm_core_set_tuned(core._h, T, 2, 2, int(stepwise), int(stepwise), 0, -1) == 0
    tuned, _ = run_core(p, core=core, stepwise=stepwise)
    assert core.info("row_tiles_fwd") == 2 and core.info("row_tiles_bwd") == 2
    core.set_option("clear_tuned", 1)
    again, _ = run_core(p, core=core, stepwise=stepwise)
    assert core.info("row_tiles_fwd") == 1
    for k in by_rule:   # the same kernels on the same fragments: the same bits
        assert np.array_equal(tuned[k], got[k]) and np.array_equal(again[k], by_rule[k]), k
    core.close()


# The partial sums that the workgroups of a column slice exchange keep all of their bits.  With one non-zero weight, a one, in
# every column of W_hh the closing product gives back single fp16 gate gradients, exactly: one tile, two, several
@pytest.mark.parametrize("T,B,H", [(1, 16, 2049), (3, 5, 2560), (2, 17, 3072), (4, 40, 3585), (3, 33, 4096)])
def test_wide_backward_exchanges_whole_sums(T, B, H):
    import torch
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    p["w_hh"] = torch.zeros(4 * H, H)
    p["w_hh"][(torch.arange(H) * 7919 + 13) % (4 * H), torch.arange(H)] = 1.0
    got, info = run_core(p)
    assert info["fallbacks"] == 0 and info["bwd_two_d"] == 1
    dh0 = torch.from_numpy(got["dh0"])
    normal = dh0.abs() >= 2.0 ** -14
    assert normal.float().mean() > 0.5
    assert torch.equal(dh0[normal], dh0[normal].half().double())


# more than 2048 units over enough steps that every slot of the rings is used again and again (eight of dG, three of partial
# sums): one tile, two, several.  No further from 64-bit arithmetic than one launch per step is; the two differ by which fp16
# roundings of dG their summation orders flip, 1.3 % in the error at the most over 64 measured pairs, hence 5 %
@pytest.mark.parametrize("T,B,H", [(24, 1, 2049), (21, 32, 4096), (20, 40, 3072), (22, 70, 2560), (33, 17, 3600)])
def test_wide_layers_against_64_bits(T, B, H):
    from helpers import reference_64, rell2
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref = {k: v.cpu().numpy() for k, v in reference_64(p).items()}
    got, info = run_core(p)
    assert info["fallbacks"] == 0 and info["persistent_fwd"] == 1 and info["persistent_bwd"] == 1 and info["bwd_two_d"] == 1
    check_against(ref, got, label=f"T={T} B={B} H={H}")
    steps, info = run_core(p, stepwise=True)
    assert info["persistent_bwd"] == 0
    for k in ref:
        assert rell2(got[k], ref[k]) <= 1.05 * rell2(steps[k], ref[k]), (k, rell2(got[k], ref[k]), rell2(steps[k], ref[k]))


# ... and fed in ranges of steps: what a launch leaves for the next one (the cell state, running dc, both rings, the delay
# hint) gives the bits of one launch.  Ranges of one step, shorter and longer than the rings
@pytest.mark.parametrize("T,B,H", [(21, 16, 2049), (23, 30, 3072), (20, 48, 4096), (26, 65, 2600)])
def test_wide_layers_in_ranges_of_steps(T, B, H):
    import numpy as np
    import torch
    from helpers import rell2, to_np
    from flashlstm_poc_amd import LstmCore
    I = 64
    p = make_problem(T, B, I, H, seed=B * 10000 + H)
    core = LstmCore(B, I, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    want, info = run_core(p, core=core)
    lib, s = core.lib, torch.cuda.current_stream().cuda_stream
    t16 = {k: p[k].cuda().half() for k in ("x", "dy", "h0", "c0", "d_hn", "d_cn")}
    ptr = {k: v.data_ptr() for k, v in t16.items()}
    F16 = 1
    hy, cy = torch.empty(B, H, device="cuda", dtype=torch.float16), torch.empty(B, H, device="cuda", dtype=torch.float16)
    assert lib.flstm_core_forward_begin(core._h, T, ptr["x"], F16, ptr["h0"], ptr["c0"], F16, s) == 0
    cuts = [0, 1, 2, 5, 14, T]
    for a, b in zip(cuts[:-1], cuts[1:]):
        assert lib.flstm_core_forward_steps(core._h, a, b - a, s) == 0
    assert lib.flstm_core_forward_end(core._h, hy.data_ptr(), cy.data_ptr(), F16, 1, s) == 0
    dx = torch.empty(T, B, I, device="cuda", dtype=torch.float16)
    out = {k: torch.empty(*n, device="cuda") for k, n in (("dw_ih", (4 * H, I)), ("dw_hh", (4 * H, H)), ("db", (4 * H,)),
                                                        ("db_hh", (4 * H,)), ("dh0", (B, H)), ("dc0", (B, H)))}
    assert lib.flstm_core_backward_begin(core._h, T, ptr["dy"], F16, ptr["d_hn"], ptr["d_cn"], F16, 1.0, dx.data_ptr(), F16, s) == 0
    for a, b in reversed(list(zip(cuts[:-1], cuts[1:]))):
        assert lib.flstm_core_backward_steps(core._h, b - 1, b - a, s) == 0
    assert lib.flstm_core_backward_end(core._h, ptr["x"], F16, *(out[k].data_ptr() for k in ("dw_ih", "dw_hh", "db", "db_hh", "dh0", "dc0")), s) == 0
    torch.cuda.synchronize()
    assert core.info("fallbacks") == 0 and core.info("persistent_bwd") == 1
    assert np.array_equal(to_np(hy), want["hn"]) and np.array_equal(to_np(cy), want["cn"])
    for k in ("dh0", "dc0", "dw_ih", "dw_hh"):
        assert np.array_equal(to_np(out[k]), want[k]), k
    assert rell2(to_np(dx), want["dx"]) <= 1e-5                # (products of other heights)
    assert rell2(to_np(out["db"]), want["db"]) <= 1e-6         # (summed range by range)
    core.close()


# four waves asked for where the rule runs the kernel for short contractions with one, two and four: the kernel that splits
# the contraction between its waves, on weights packed before, and back
@pytest.mark.parametrize("T,B,H,rule", [(5, 64, 256, 1), (4, 40, 512, 2), (3, 300, 256, 4), (6, 9, 65, 1)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_four_waves_where_short_contraction_kernels_are_the_rule(T, B, H, rule, stepwise):
    import numpy as np
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 20, H, seed=B * 10000 + H)
    ref, _ = oracle_reference(p)
    core = LstmCore(B, 20, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    assert core.info("waves_fwd") == rule and core.info("slice_fwd") == 8 * rule
    by_rule, _ = run_core(p, core=core, stepwise=stepwise)
    core.set_option("waves_fwd", 4)
    assert core.info("waves_fwd") == 4 and core.info("slice_fwd") == 32 and core.info("row_tiles_fwd") == 1
    got, info = run_core(p, core=core, stepwise=stepwise)
    assert info["fallbacks"] == 0
    check_against(ref, got, label=f"T={T} B={B} H={H} stepwise={stepwise} four waves")
    core.set_option("waves_fwd", 0)
    again, _ = run_core(p, core=core, stepwise=stepwise)
    assert core.info("waves_fwd") == rule
    for k in by_rule:
        assert np.array_equal(again[k], by_rule[k]), k
    core.close()
