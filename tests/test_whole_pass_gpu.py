"""A whole forward pass as one launch (short contractions) against the same pass as separate launches -- the option "profile"
takes that path -- bit for bit: outputs, caches, and the gradients made from them."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def cached(core, which, rows, dtype):
    import torch
    from flashlstm_poc_amd import load_library
    ptr, ld = ctypes.c_void_p(), ctypes.c_size_t()
    assert core.lib.flstm_core_cache_ptr(core._h, which, ctypes.byref(ptr), ctypes.byref(ld)) == 0
    out = torch.empty(rows, ld.value, device="cuda", dtype=dtype)
    assert load_library() is core.lib
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipMemcpy(ctypes.c_void_p(out.data_ptr()), ptr, ctypes.c_size_t(out.numel() * out.element_size()), 3) == 0
    return out


# one to five steps (pairs and a single one left), row tiles of 1, 16 and 17 rows, rows of less than and exactly 64, 128 and 256
# features and of more, every length of the contraction, odd widths; T = 64 crosses the rule for few units, 33 the one for 256 features
SHAPES = [(1, 1, 128, 256), (2, 16, 64, 64), (3, 17, 65, 33), (4, 3, 1, 1), (5, 40, 256, 512), (33, 20, 200, 130), (32, 20, 200, 130),
          (70, 5, 128, 96), (64, 5, 128, 96), (45, 5, 128, 96), (9, 100, 300, 512), (12, 512, 20, 256), (7, 128, 64, 257), (6, 64, 129, 384), (37, 33, 100, 384)]
IN_FRONT = [(33, 20, 200, 130), (70, 5, 128, 96), (64, 5, 128, 96), (9, 100, 300, 512)]   # whose projection has a launch of its own


@pytest.mark.parametrize("T,B,I,H", SHAPES)
@pytest.mark.parametrize("dtype,state", [("f16", "f16"), ("f32", "f32"), ("f16", None), ("f32", "f16")])
def test_whole_pass_gives_the_bits_of_separate_launches(T, B, I, H, dtype, state):
    import torch
    from flashlstm_poc_amd import LstmCore
    types = {"f16": torch.float16, "f32": torch.float32}
    g = torch.Generator(device="cuda").manual_seed(T * 1000 + H)
    uniform = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * H ** -0.5
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")
    core = LstmCore(B, I, H)
    core.pack(uniform(4 * H, I), uniform(4 * H, H), uniform(4 * H), uniform(4 * H))
    x, dy = normal(T, B, I).to(types[dtype]), normal(T, B, H).to(types[dtype])
    h0 = c0 = None
    if state:
        h0, c0 = normal(B, H).to(types[state]), normal(B, H).to(types[state])

    def passed(save, want_y=True):
        out = list(core.forward(x, h0, c0, save_for_backward=save, want_y=want_y))
        if save:
            out += [cached(core, 0, (T + 1) * B, torch.float16), cached(core, 1, (T + 1) * B, torch.float32), cached(core, 2, T * B, torch.float16)]
            out += list(core.backward(x, dy))
        return out

    core.set_option("profile", 1)
    want = passed(True)
    assert core.info("whole_fwd") == 0
    core.set_option("profile", 0)
    for save, want_y in ((True, True), (False, True), (True, False), (True, True), (False, True)):   # (each leaves the ring to the next)
        for k, (a, b) in enumerate(zip(passed(save, want_y), want)):
            assert a is None or torch.equal(a, b), (save, k)
        assert core.info("whole_fwd") == 1 and core.info("projection_fwd") == (0 if (T, B, I, H) in IN_FRONT else 2)
    assert core.info("fallbacks") == 0
    core.close()


def test_whole_passes_of_a_plan_whose_launch_gave_up():
    """A pass that gives up leaves the ring in no known state: the next one prepares it anew."""
    import torch
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(16, 64, 128)
    core.pack(*(torch.randn(*s, device="cuda") * 0.1 for s in ((512, 64), (512, 128), (512,), (512,))))
    x = torch.randn(11, 16, 64, device="cuda").half()
    want = core.forward(x)
    core.set_option("inject_stall", 1)
    for _ in range(12):   # repeated step-wise, demoted for eight passes, whole again
        assert all(torch.equal(a, b) for a, b in zip(core.forward(x), want))
    assert core.info("whole_fwd") == 1
    assert core.info("demotions_fwd") == 1 and core.info("hold_fwd") == 0 and core.info("persistent_fwd") == 1
    core.close()


# enough steps for some wave to ask too early: of 11 steps of the first, half the passes went through without a reload
@pytest.mark.parametrize("T,B,I,H", [(250, 16, 64, 128), (200, 40, 300, 512), (250, 100, 20, 256)])
def test_whole_pass_that_gives_up_inside(T, B, I, H):
    """A bound of no reload at all: a wave finds the fragments unwritten and leaves, with the ring half written and the status in the
    host's memory.  The pass is repeated step-wise; with the bound taken back, whole passes over other rows follow, and their bits."""
    import torch
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(B, I, H)
    core.pack(*(torch.randn(*s, device="cuda") * 0.1 for s in ((4 * H, I), (4 * H, H), (4 * H,), (4 * H,))))
    xs = [torch.randn(T, B, I, device="cuda").half() for _ in range(12)]
    want = [core.forward(x) for x in xs]
    assert core.info("whole_fwd") == 1 and core.info("fallbacks") == 0
    core.set_option("spin_limit", 0)
    assert all(torch.equal(a, b) for a, b in zip(core.forward(xs[0]), want[0]))
    assert core.info("fallbacks") == 1 and core.info("persistent_fwd") == 0 and core.info("whole_fwd") == 0
    core.set_option("spin_limit", 1 << 30)
    for x, w in zip(xs, want):   # seven more of them step-wise
        assert all(torch.equal(a, b) for a, b in zip(core.forward(x), w))
    assert core.info("whole_fwd") == 1 and core.info("fallbacks") == 1
    core.close()


@pytest.mark.parametrize("T,B,I,H,save,whole", [(260, 16, 32, 64, True, 1), (270, 16, 32, 64, True, 0), (270, 16, 32, 64, False, 1), (540, 16, 32, 64, False, 0),
                                                (540, 1, 32, 64, False, 1), (300, 512, 32, 256, True, 1), (300, 20, 32, 384, True, 1)])
def test_long_passes_are_one_launch_where_that_is_the_faster_way(T, B, I, H, save, whole):
    """The rule's two sides, with the same bits."""
    import torch
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(B, I, H)
    core.pack(*(torch.randn(*s, device="cuda") * 0.1 for s in ((4 * H, I), (4 * H, H), (4 * H,), (4 * H,))))
    x = torch.randn(T, B, I, device="cuda").half()
    core.set_option("profile", 1)
    want = core.forward(x)
    core.set_option("profile", 0)
    got = core.forward(x, save_for_backward=save)
    assert core.info("whole_fwd") == whole and all(torch.equal(a, b) for a, b in zip(got, want))
    core.close()
