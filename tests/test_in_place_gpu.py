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
