"""Recurrences in blocks of few rows, fragments that hold several k-steps of them: against 64-bit arithmetic, the kernels with blocks of 32
rows, ranges of steps, launches per step, values that are not finite, and a layout that changes during a pass."""
import numpy as np
import pytest

from helpers import make_problem, reference_64, rell2, to_np
from test_core_gpu import run_core

pytestmark = pytest.mark.gpu

# T, B, H and the groups backward and forward (None: another kernel forward).  Slices that end a pack of two or four and slices that
# leave 1 to 3 of its k-steps without one; the first and last size of every kernel (4, 8, 12, 16, 24, 32 k-steps a wave); one row, a block that
# is not full, the last batch of blocks of 4 and the first of 8, of 8 and of another kernel; forward the last batch of 8 rows (the last three are
# another kernel's over so few steps)
SHAPES = [(9, 1, 32, 1, None), (9, 5, 100, 2, None), (7, 16, 128, 4, None), (6, 9, 130, 3, None), (8, 4, 256, 1, None), (7, 129, 256, 17, None),
          (9, 70, 257, 18, None), (6, 65, 384, 9, None), (6, 5, 385, 2, None), (7, 64, 512, 16, None), (6, 128, 512, 16, None), (5, 1, 513, 1, 1),
          (9, 20, 650, 5, 3), (6, 33, 768, 5, 5), (7, 32, 769, 8, 4), (6, 6, 800, 2, 1), (8, 32, 1024, 8, 4), (5, 33, 1000, 5, None), (5, 64, 1024, 8, None),
          (6, 65, 769, 5, 5), (6, 128, 1024, 8, 8), (4, 97, 801, 7, 7)]


@pytest.mark.parametrize("T,B,H,backward,forward", SHAPES)
@pytest.mark.parametrize("half", [True, False])
def test_few_rows_against_64_bits_and_32_row_blocks(T, B, H, backward, forward, half):
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref = {k: v.cpu().numpy() for k, v in reference_64(p).items()}
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    got, info = run_core(p, core=core, half=half)
    assert info["fallbacks"] == 0 and core.info("groups_bwd") == backward and (forward is None or core.info("groups_fwd") == forward)
    steps, _ = run_core(p, core=core, half=half, stepwise=True)
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 2)
    blocks, info = run_core(p, core=core, half=half)
    assert info["fallbacks"] == 0 and core.info("groups_bwd") == -(-B // 32)
    # What both kernels are off by is the rounding of h, dG and the outputs to fp16, 2^-11 at most and some 2^-12 in the mean, once or twice
    # in every sum.  Another order of an fp32 sum moves it by some 2^-20, which turns one rounding in a hundred the other way: the errors of
    # two right kernels differ by that hundredth (0.8 % at most over this table, 1.5 % of hn of five rows), a wrong term is more than all of it.
    for k in ref:
        assert rell2(blocks[k], ref[k]) <= 1e-3, k
        assert rell2(got[k], ref[k]) <= 1.05 * rell2(blocks[k], ref[k]), (k, rell2(got[k], ref[k]), rell2(blocks[k], ref[k]))
    # launches per step run the same kernel: the same bits but for db, whose sums of up to 9 steps and 129 rows a launch adds up by itself
    for k in ref:
        assert np.array_equal(steps[k], got[k]) if k != "db" else rell2(steps[k], got[k]) <= 1e-6, k
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 0)
    again, _ = run_core(p, core=core, half=half)
    for k in got:
        assert np.array_equal(again[k], got[k]), k
    core.close()


@pytest.mark.parametrize("T,B,H", [(21, 9, 100), (22, 40, 257), (20, 20, 650), (21, 33, 1000), (23, 80, 800)])
def test_few_rows_in_ranges_of_steps(T, B, H):
    from test_kernel_variants_gpu import test_wide_layers_in_ranges_of_steps as in_ranges
    in_ranges(T, B, H)


@pytest.mark.parametrize("shape", [(6, 8, 64, 250), (7, 20, 64, 650), (6, 32, 64, 1024), (6, 100, 64, 1000)])
def test_a_row_of_nans_stays_in_its_row(shape):
    from test_core_gpu import test_a_batch_row_of_nans_stays_in_its_row as stays
    stays(shape)


# a weight beyond fp16: every sum it enters is infinite and its gate saturated, and nothing else changes
@pytest.mark.parametrize("B,H", [(8, 250), (20, 650), (32, 1024), (100, 1000)])
def test_infinite_weights_give_what_the_other_kernels_give(B, H):
    from flashlstm_poc_amd import LstmCore
    p = make_problem(5, B, 24, H, seed=3)
    p["w_hh"] = p["w_hh"].clone()
    p["w_hh"][3, 7] = 1e6
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    got, info = run_core(p, core=core)
    assert info["fallbacks"] == 0
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 2)
    blocks, _ = run_core(p, core=core)
    for k in ("y", "hn", "cn", "dx", "dh0", "dc0"):
        assert np.array_equal(np.isfinite(got[k]), np.isfinite(blocks[k])), k
        there = np.isfinite(blocks[k])
        assert rell2(got[k][there], blocks[k][there]) <= 2e-3, k
    core.close()


# an option that changes the layout between two ranges of a forward pass: it goes on in the other layout's ring
@pytest.mark.parametrize("T,B,H", [(11, 20, 650), (9, 32, 1024)])
@pytest.mark.parametrize("name,value", [("row_tiles_fwd", 2), ("stepwise", 1)])
def test_layout_that_changes_during_a_pass(T, B, H, name, value):
    import torch
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 64, H, seed=5)
    core = LstmCore(B, 64, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    want, _ = run_core(p, core=core)
    lib, s = core.lib, torch.cuda.current_stream().cuda_stream
    t16 = {k: p[k].cuda().half() for k in ("x", "dy", "h0", "c0", "d_hn", "d_cn")}
    hy, cy = (torch.empty(B, H, device="cuda", dtype=torch.float16) for _ in range(2))
    for first, then in ((0, value), (value, 0)):
        core.set_option(name, first)
        assert lib.flstm_core_forward_begin(core._h, T, t16["x"].data_ptr(), 1, t16["h0"].data_ptr(), t16["c0"].data_ptr(), 1, s) == 0
        assert lib.flstm_core_forward_steps(core._h, 0, 6, s) == 0
        core.set_option(name, then)
        assert lib.flstm_core_forward_steps(core._h, 6, T - 6, s) == 0
        assert lib.flstm_core_forward_end(core._h, hy.data_ptr(), cy.data_ptr(), 1, 1, s) == 0
        torch.cuda.synchronize()
        assert core.info("fallbacks") == 0
        assert rell2(to_np(hy), want["hn"]) <= 1e-3 and rell2(to_np(cy), want["cn"]) <= 1e-3
        core.set_option(name, 0)
        grads = core.backward(t16["x"], t16["dy"], t16["d_hn"], t16["d_cn"])   # from the caches of all steps
        for k, g in zip(("dx", "dw_ih", "dw_hh", "db", "dh0", "dc0"), grads):
            assert rell2(to_np(g), want[k]) <= 1e-3, k
    core.close()


# ... of a backward pass, or behind the last of them: the pass keeps the layout it began with -- the ring, and the groups whose bias
# gradients its end adds up (2 to 17 groups become one, and one becomes as many)
@pytest.mark.parametrize("T,B,H,name,value", [(8, 9, 100, "row_tiles_bwd", 2), (8, 16, 650, "row_tiles_bwd", 2), (8, 32, 1024, "row_tiles_bwd", 2),
                                              (7, 129, 256, "row_tiles_bwd", 2), (8, 20, 650, "stepwise", 1), (6, 16, 2048, "bwd_two_d", 0)])
def test_a_backward_pass_keeps_its_layout(T, B, H, name, value):
    import torch
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 64, H, seed=6)
    core = LstmCore(B, 64, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    lib, s = core.lib, torch.cuda.current_stream().cuda_stream
    t16 = {k: p[k].cuda().half() for k in ("x", "dy", "h0", "c0")}
    core.forward(t16["x"], t16["h0"], t16["c0"])

    def in_two_ranges(first, between, behind):
        out = [torch.full(shape, float("nan"), device="cuda") for shape in ((T, B, 64), (4 * H, 64), (4 * H, H), (4 * H,), (B, H), (B, H))]
        dx, dw_ih, dw_hh, db, dh0, dc0 = (t.data_ptr() for t in out)
        core.set_option(name, first)
        assert lib.flstm_core_backward_begin(core._h, T, t16["dy"].data_ptr(), 1, None, None, 1, 1.0, dx, 0, s) == 0
        assert lib.flstm_core_backward_steps(core._h, T - 1, 3, s) == 0
        core.set_option(name, between)
        assert lib.flstm_core_backward_steps(core._h, T - 4, T - 3, s) == 0
        core.set_option(name, behind)
        assert lib.flstm_core_backward_end(core._h, t16["x"].data_ptr(), 1, dw_ih, dw_hh, db, None, dh0, dc0, s) == 0
        torch.cuda.synchronize()
        assert core.info("fallbacks") == 0
        return [to_np(t) for t in out]

    default = 1 if name == "bwd_two_d" else 0
    for first, other in ((default, value), (value, default)):
        want = in_two_ranges(first, first, first)
        assert all(np.isfinite(w).all() for w in want)
        for between, behind in ((first, other), (other, other), (other, first)):
            for w, g in zip(want, in_two_ranges(first, between, behind)):
                assert np.array_equal(w, g)
    core.close()


# The one-way kernel's weights, made when an option first asks for that kernel: those of the last packing, as a plan of more rows packs them
# (its blocks of 32 rows sum a row as these do)
@pytest.mark.parametrize("B,H", [(20, 650), (32, 1024), (5, 513), (70, 800)])
def test_weights_of_the_one_way_kernel_follow_the_packing(B, H):
    import torch
    from flashlstm_poc_amd import LstmCore
    few, other = LstmCore(B, 64, H), LstmCore(250, 64, H)
    for core in (few, other):
        core.set_option("waves_fwd", 4)
        core.set_option("row_tiles_fwd", 2)
    for k, (name, value) in enumerate((("row_tiles_fwd", 2), ("row_tiles_fwd", 0), ("waves_fwd", 0), ("row_tiles_fwd", 2))):
        p = make_problem(6, 250, 64, H, seed=80 + k)
        weights = [p[n].cuda() for n in ("w_ih", "w_hh", "b_ih", "b_hh")]
        x, h0, c0 = (p[n].cuda().half() for n in ("x", "h0", "c0"))
        small = [x[:, :B].contiguous(), h0[:B].contiguous(), c0[:B].contiguous()]
        few.pack(*weights)
        other.pack(*weights)
        want = other.forward(x, h0, c0)
        few.set_option(name, value)
        for again in range(2):
            got = few.forward(*small)
            if few.info("row_tiles_fwd") == 2:
                for g, w in zip(got, (want[0][:, :B], want[1][:B], want[2][:B])):
                    assert torch.equal(g, w)
            else:
                assert rell2(to_np(got[0]), to_np(want[0][:, :B])) <= 1e-3
    few.close()
    other.close()


# Blocks of 16 rows: from 512 steps on where the projection stands in front, from 2048 on beside it, and the bits of the one-way kernel, which
# takes the others.  The weights that the other kernel reads are made from the packed ones, for each packing anew.  (8 blocks of 7 and of 8
# k-steps a wave, the last one not full; 6 and 5 of 8)
@pytest.mark.parametrize("first,B,I,H,beside", [(512, 128, 24, 769, 0), (512, 113, 24, 1024, 0), (512, 90, 520, 1000, 0), (2048, 66, 24, 1000, 1)])
def test_many_steps_in_blocks_of_16(first, B, I, H, beside):
    import torch
    from flashlstm_poc_amd import LstmCore
    core, other = LstmCore(B, I, H), LstmCore(B, I, H)
    other.set_option("waves_fwd", 4)
    for seed, lengths in ((90, (first, first - 1)), (91, (5, first))):
        p = make_problem(first, B, I, H, seed=seed)
        weights = [p[n].cuda() for n in ("w_ih", "w_hh", "b_ih", "b_hh")]
        x, h0, c0 = (p[n].cuda().half() for n in ("x", "h0", "c0"))
        core.pack(*weights)
        other.pack(*weights)
        for T in lengths:
            got, want = core.forward(x[:T], h0, c0), other.forward(x[:T], h0, c0)
            assert core.info("few_rows_fwd") == (16 if T == first else 0) and other.info("few_rows_fwd") == 0
            assert core.info("fallbacks") == 0 and (T < first or core.info("projection_fwd") == beside)
            for g, w in zip(got, want):
                assert torch.equal(g, w)
    core.set_option("stepwise", 1)
    got = core.forward(x, h0, c0)
    assert core.info("few_rows_fwd") == 16 and all(torch.equal(g, w) for g, w in zip(got, want))
    core.close()
    other.close()


# Blocks of 16 rows asked for where the rule takes blocks of fewer: the one-way kernel above 512 units forward and 384 backward, by an option and by a
# tuned entry, step-wise as well; below, where 16-row blocks never were that kernel's, the rule's.  (First and last sizes of that kernel's
# instantiations; a block that is not full, one row, all rows that have blocks of 8)
@pytest.mark.parametrize("T,B,H", [(6, 65, 384), (6, 5, 385), (7, 64, 512), (5, 1, 513), (9, 20, 650), (7, 32, 769), (5, 33, 1000), (8, 32, 1024)])
@pytest.mark.parametrize("stepwise", [False, True])
def test_blocks_of_16_rows_where_fewer_are_the_rule(T, B, H, stepwise):
    from flashlstm_poc_amd import LstmCore
    p = make_problem(T, B, 24, H, seed=B * 10000 + H)
    ref = {k: v.cpu().numpy() for k, v in reference_64(p).items()}
    core = LstmCore(B, 24, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    runs = {}
    for tiles in (0, 2, 1):
        for name in ("row_tiles_fwd", "row_tiles_bwd"):
            core.set_option(name, tiles)
        runs[tiles], info = run_core(p, core=core, stepwise=stepwise)
        assert info["fallbacks"] == 0
    assert core.info("few_rows_fwd") == 0 and core.info("row_tiles_fwd") == 1 and core.info("row_tiles_bwd") == 1
    one_way = H > 384
    assert (core.info("few_rows_bwd") == 0) == one_way and (not one_way or core.info("groups_bwd") == -(-B // 16))
    assert H <= 512 or core.info("groups_fwd") == -(-B // 16)
    # (the error of blocks of 32 and the allowance for flipped roundings: test_few_rows_against_64_bits_and_32_row_blocks)
    for k in ref:
        assert rell2(runs[1][k], ref[k]) <= 1.05 * rell2(runs[2][k], ref[k]) <= 1.05e-3, k
        assert one_way or np.array_equal(runs[1][k], runs[0][k]), k
    # a tuned entry says the same, and one without a choice leaves the rule in force
    for name in ("row_tiles_fwd", "row_tiles_bwd"):
        core.set_option(name, 0)
    for tiles in (1, 0):
        assert core.lib.flstm_core_set_tuned(core._h, T, tiles, tiles, int(stepwise), int(stepwise), 0, -1) == 0
        tuned, _ = run_core(p, core=core, stepwise=stepwise)
        for k in tuned:
            assert np.array_equal(tuned[k], runs[tiles][k]), (tiles, k)
    core.close()


# The tuner has all three: what it keeps is a choice that can be put back, and no slower than either of the others
def test_tuner_tries_the_rule_beside_blocks_of_16_and_32_rows():
    from flashlstm_poc_amd import LstmCore, sweep
    T, B, I, H = 64, 20, 64, 650
    p = sweep.make_problem(T, B, I, H, seed=9)
    core = LstmCore(B, I, H)
    core.pack(p["w_ih"], p["w_hh"], p["b_ih"], p["b_hh"])
    least = {}
    for tiles in (0, 1, 2):
        core.set_option("row_tiles_bwd", tiles)
        core.forward(p["x"])
        for _ in range(8):
            core.backward(p["x"], p["dy"])
            least[tiles] = min(least.get(tiles, 1e9), core.last_ms("bwd_rec"))
    core.set_option("row_tiles_bwd", 0)
    t = core.tune(T, repeats=6)
    # (bwd_rec_ms is the device's own time; the three differ by more than a third: 1.3 us a step, 2.5 and more)
    assert t["row_tiles_bwd"] == min(least, key=least.get) == 0 and t["bwd_rec_ms"] < 1.2 * least[0]
    assert core.info("few_rows_bwd") == 4
    core.close()
