"""Forward passes whose outputs lie in their inputs -- a serving loop that carries its state in one pair of buffers, y over x -- give
the bits of the same passes with buffers of their own, and take the path that reads everything before it writes (asserted through
"outputs_behind": the race that the other path would be need not show)."""
import pytest

pytestmark = pytest.mark.gpu


def made(B, I, H, seed):
    import torch
    from flashlstm_poc_amd import LstmCore
    g = torch.Generator(device="cuda").manual_seed(seed)
    uniform = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * H ** -0.5
    core = LstmCore(B, I, H)
    core.pack(uniform(4 * H, I), uniform(4 * H, H), uniform(4 * H), uniform(4 * H))
    return core, lambda *s: torch.randn(*s, generator=g, device="cuda")


# one launch (up to 512 units; 33 and 130: h0 through the ring), separate launches (650: outputs copied, 1024 and 2048: y written by the
# recurrence where nothing overlaps), one row, several groups
@pytest.mark.parametrize("B,H", [(1, 256), (20, 64), (5, 33), (17, 130), (100, 512), (3, 650), (40, 1024), (16, 2048)])
@pytest.mark.parametrize("T", [1, 2, 3])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_state_carried_in_place(B, H, T, dtype):
    import torch
    kind = {"f16": torch.float16, "f32": torch.float32}[dtype]
    core, normal = made(B, 96, H, seed=B * 1000 + H)
    empty = lambda *s: torch.empty(*s, device="cuda", dtype=kind)
    h, c = normal(B, H).to(kind), normal(B, H).to(kind)
    hs, cs = h.clone(), c.clone()
    y = empty(T, B, H)
    for step in range(6):
        x = normal(T, B, 96).to(kind)
        want_y, want_h, want_c = empty(T, B, H), empty(B, H), empty(B, H)
        core.forward_static(x, hs, cs, want_y, want_h, want_c)
        assert core.info("outputs_behind") == 0
        hs, cs = want_h, want_c
        core.forward_static(x, h, c, y, h, c)
        assert core.info("outputs_behind") == 1
        assert torch.equal(y, want_y) and torch.equal(h, want_h) and torch.equal(c, want_c), step
    assert core.info("fallbacks") == 0
    core.close()


# y over x whole (the fp16 rows that the kernels read in place, and converted ones), y over h0, y over half of x, states of one element type over
# those of another, hy over c0 and cy over h0
@pytest.mark.parametrize("T,B,N", [(40, 20, 128), (100, 32, 1024), (1, 7, 128), (1, 40, 1024)])
@pytest.mark.parametrize("where", ["x", "x32", "half", "h0", "types", "crossed"])
def test_outputs_anywhere_in_the_inputs(T, B, N, where):
    import torch
    core, normal = made(B, N, N, seed=T + N)
    f16, f32 = torch.float16, torch.float32
    x, state = normal(T, B, N).to(f32 if where == "x32" else f16), f32 if where == "types" else f16
    h, c = normal(B, N).to(state), normal(B, N).to(state)
    out = x.dtype
    empty = lambda *s: torch.empty(*s, device="cuda", dtype=out)
    y, hy, cy = empty(T, B, N), empty(B, N), empty(B, N)
    core.forward(x, h, c, save_for_backward=False)   # (leaves the words of a projection beside the recurrence: a static call allocates none)
    core.forward_static(x, h, c, y, hy, cy)
    assert core.info("outputs_behind") == 0
    over_y, over_h, over_c = empty(T, B, N), empty(B, N), empty(B, N)
    if where in ("x", "x32"):
        over_y = x
    elif where == "half":   # x in the first T steps of a buffer of twice as many, y half of that further on
        room = empty(2 * T, B, N)
        room[:T].copy_(x)
        first = T * B * N // 2
        x, over_y = room[:T], room.view(-1)[first:first + T * B * N].view(T, B, N)
    elif where == "h0":
        room = empty(T, B, N)
        room[0].copy_(h)
        h, over_y = room[0], room
    elif where == "types":
        over_h, over_c = (t.view(-1).view(f16)[:B * N].view(B, N) for t in (h, c))
    else:
        over_h, over_c = c, h
    core.forward_static(x, h, c, over_y, over_h, over_c)
    assert core.info("outputs_behind") == 1 and core.info("fallbacks") == 0
    assert torch.equal(over_y, y) and torch.equal(over_h, hy) and torch.equal(over_c, cy)
    core.close()


@pytest.mark.parametrize("B,H", [(20, 64), (5, 33), (40, 1024)])
@pytest.mark.parametrize("T", [1, 3])
def test_repeat_after_a_give_up_reads_what_was_handed_over(B, H, T):
    import torch
    core, normal = made(B, H, H, seed=B * 1000 + H)
    x, h, c = normal(T, B, H).half(), normal(B, H).half(), normal(B, H).half()
    want = [torch.empty(*s, device="cuda", dtype=torch.float16) for s in ((T, B, H), (B, H), (B, H))]
    core.forward_static(x, h, c, *want)
    core.set_option("inject_stall", 1)
    core.forward_static(x, h, c, x, h, c)   # y over x as well
    assert core.info("fallbacks") == 1
    assert all(torch.equal(a, b) for a, b in zip((x, h, c), want))
    core.close()


def test_call_that_fails_leaves_the_state_in_place_alone():
    import torch
    core, normal = made(20, 96, 64, seed=1)
    x, h, c, y = normal(3, 20, 96).half(), normal(20, 64).half(), normal(20, 64).half(), torch.empty(3, 20, 64, device="cuda").half()
    before = h.clone(), c.clone()
    core.set_option("inject_stall", 2)   # the repeat fails too
    with pytest.raises(RuntimeError):
        core.forward_static(x, h, c, y, h, c)
    assert torch.equal(h, before[0]) and torch.equal(c, before[1])
    # in ranges of steps (as the host-streaming windows carry their state): the caller repeats the pass
    core.set_option("inject_stall", 1)
    core.set_option("stepwise", 1)
    lib, s = core.lib, torch.cuda.current_stream().cuda_stream
    assert lib.flstm_core_forward_begin(core._h, 3, x.data_ptr(), 1, h.data_ptr(), c.data_ptr(), 1, s) == 0
    assert lib.flstm_core_forward_steps(core._h, 0, 3, s) == 0
    assert lib.flstm_core_forward_end(core._h, h.data_ptr(), c.data_ptr(), 1, 0, s) == 2003
    assert torch.equal(h, before[0]) and torch.equal(c, before[1])
    core.close()


@pytest.mark.parametrize("B,N", [(20, 128), (5, 33), (40, 1024)])
@pytest.mark.parametrize("stall", [0, 1])
def test_gradients_in_place(B, N, stall):
    """dx over dY, dh0 over d_hn, dc0 over d_cn: with the caller's buffers still whole for the step-wise repeat."""
    import torch
    T = 5
    core, normal = made(B, N, N, seed=B * 1000 + N)
    x, dy = normal(T, B, N).half(), normal(T, B, N).half()
    d_hn, d_cn = normal(B, N), normal(B, N)
    core.forward(x)
    core.set_option("stepwise", stall)   # (as the repeat runs)
    want = core.backward(x, dy, d_hn, d_cn)
    core.set_option("stepwise", 0)
    core.set_option("inject_stall", stall)
    dW_ih, dW_hh, db = (torch.empty_like(t) for t in want[1:4])
    rc = core.lib.flstm_core_backward(core._h, T, x.data_ptr(), 1, dy.data_ptr(), 1, d_hn.data_ptr(), d_cn.data_ptr(), 0, 1.0, dy.data_ptr(), 1,
                                      dW_ih.data_ptr(), dW_hh.data_ptr(), db.data_ptr(), None, d_hn.data_ptr(), d_cn.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and core.info("fallbacks") == stall
    for k, (a, b) in enumerate(zip((dy, dW_ih, dW_hh, db, d_hn, d_cn), want)):
        assert torch.equal(a, b), k
    core.close()


@pytest.mark.parametrize("stalled", [None, 0, 1, 2])
def test_stack_in_place(stalled):
    """States in one pair of buffers, rows and gradients of every other layer in one buffer, and a layer that gave up."""
    import torch
    from flashlstm_poc_amd import LstmStack
    from flashlstm_poc_amd.stack import _pointers
    T, B, H, L = 4, 20, 64, 4
    g = torch.Generator(device="cuda").manual_seed(3)
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")
    stack = LstmStack(B, H, H, L)
    stack.pack([(normal(4 * H, H) * 0.1, normal(4 * H, H) * 0.1, normal(4 * H) * 0.1, normal(4 * H) * 0.1) for _ in range(L)])
    x, h, c, dy = normal(T, B, H).half(), normal(L, B, H).half(), normal(L, B, H).half(), normal(T, B, H).half()
    d_hn, d_cn = normal(L, B, H), normal(L, B, H)
    y, hy, cy = stack._forward(x, h, c)
    if stalled is not None:   # (as its repeat runs: the bias gradient is summed in another order)
        stack.layers[stalled].set_option("stepwise", 1)
    want = stack._backward(dy, 1.0, list(d_hn), list(d_cn), True)
    if stalled is not None:
        stack.layers[stalled].set_option("stepwise", 0)
    xs = [t.clone() for t in stack._inputs]

    def stall():
        if stalled is not None:
            stack.layers[stalled].set_option("inject_stall", 1)

    lib, s, plans = stack._lib, torch.cuda.current_stream().cuda_stream, stack._plans()
    rows = [torch.empty_like(x) for _ in range(2)]
    stall()
    assert lib.flstm_stack_forward(plans, L, T, x.data_ptr(), 1, h.data_ptr(), c.data_ptr(), 1, _pointers([rows[l % 2] for l in range(L)]), 1,
                                   h.data_ptr(), c.data_ptr(), s) == 0
    assert torch.equal(rows[(L - 1) % 2], y) and torch.equal(h, hy) and torch.equal(c, cy)
    for layer in stack.layers:
        assert layer.info("fallbacks") == (1 if layer is stack.layers[stalled or 0] and stalled is not None else 0)
    stall()
    grads = [[torch.empty_like(t) for t in triple] for triple in want[1]]
    assert lib.flstm_stack_backward(plans, L, T, _pointers(xs), 1, dy.data_ptr(), 1, 1.0, _pointers(list(d_hn)), _pointers(list(d_cn)), 0, 1.0,
                                    _pointers([rows[l % 2] for l in range(L)]), 1, *(_pointers([t[k] for t in grads]) for k in range(3)), None,
                                    _pointers(list(d_hn)), _pointers(list(d_cn)), s) == 0
    assert torch.equal(rows[0], want[0]) and torch.equal(d_hn, want[5]) and torch.equal(d_cn, want[6])
    for mine, theirs in zip(grads, want[1]):
        assert all(torch.equal(a, b) for a, b in zip(mine, theirs))
    stack.close()


# y apart from the inputs is written by the recurrence of separate launches, whatever becomes of the states
@pytest.mark.parametrize("T,B,I,H", [(100, 32, 512, 1024), (20, 40, 96, 640)])
def test_rows_apart_from_the_inputs_are_not_copied(T, B, I, H):
    import torch
    core, normal = made(B, I, H, seed=T + H)
    x, h, c = normal(T, B, I).half(), normal(B, H).half(), normal(B, H).half()
    empty = lambda *s: torch.empty(*s, device="cuda", dtype=torch.float16)
    want, y, rows = [empty(T, B, H), empty(B, H), empty(B, H)], empty(T, B, H), empty(T, B, H)
    core.forward(x, h, c, save_for_backward=False)   # (as in test_outputs_anywhere_in_the_inputs)
    core.forward_static(x, h, c, *want)
    assert core.info("outputs_behind") == 0 and core.info("rows_behind") == 0
    rows[-1].copy_(h)
    core.forward_static(x, rows[-1], c, rows, empty(B, H), empty(B, H))   # y over h0
    assert core.info("outputs_behind") == 1 and core.info("rows_behind") == 1 and torch.equal(rows, want[0])
    core.forward_static(x, h, c, y, h, c)
    assert core.info("outputs_behind") == 1 and core.info("rows_behind") == 0 and core.info("fallbacks") == 0
    assert all(torch.equal(a, b) for a, b in zip((y, h, c), want))
    core.close()
