"""The x-projection formed by the idle workgroups of the recurrence's launch against the same projection in front of it -- the option
"profile" takes that path -- bit for bit."""
import pytest

pytestmark = pytest.mark.gpu

# one, two and four groups inside XCDs (what is idle: six whole XCDs, four, ...), groups across XCDs, slices of 16 units (two of them in
# a column of tiles), two row blocks; rows that end inside a tile, one tile of rows, rows of 64 features and many
SHAPES = [(600, 32, 1024, 1024), (300, 64, 512, 1024), (255, 33, 448, 640), (400, 7, 1024, 992), (130, 100, 2048, 640),
          (200, 16, 2048, 2048), (150, 48, 512, 1536), (333, 9, 256, 1400), (260, 100, 512, 640),
          (64, 200, 32, 512), (60, 200, 700, 512), (40, 100, 128, 1536)]
IN_FRONT = [(130, 100, 2048, 640), (64, 200, 32, 512), (60, 200, 700, 512)]   # so few workgroups take longer than the recurrence and the product apart


@pytest.mark.parametrize("T,B,I,H", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_projection_beside_the_recurrence_gives_the_bits_of_one_in_front(T, B, I, H, dtype):
    import torch
    from flashlstm_poc_amd import LstmCore
    kind = {"f16": torch.float16, "f32": torch.float32}[dtype]
    g = torch.Generator(device="cuda").manual_seed(T + H)
    uniform = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1) * H ** -0.5
    normal = lambda *s: torch.randn(*s, generator=g, device="cuda")
    core = LstmCore(B, I, H)
    core.pack(uniform(4 * H, I), uniform(4 * H, H), uniform(4 * H), uniform(4 * H))
    h0, c0 = normal(B, H).to(kind), normal(B, H).to(kind)
    dy = normal(T, B, H).to(kind)
    xs = [normal(T, B, I).to(kind) for _ in range(3)]

    def passed(x):
        return list(core.forward(x, h0, c0)) + list(core.backward(x, dy))

    core.set_option("profile", 1)
    want = [passed(x) for x in xs]
    assert core.info("projection_fwd") == 0
    core.set_option("profile", 0)
    for x, w in zip(xs + xs[:1], want + want[:1]):   # other rows every time: no tile of a pass before may be taken for this one's
        for k, (a, b) in enumerate(zip(passed(x), w)):
            assert torch.equal(a, b), k
        assert core.info("projection_fwd") == (0 if (T, B, I, H) in IN_FRONT else 1)
    short = xs[0][:T // 2].contiguous()
    core.set_option("profile", 1)
    y, _, _ = core.forward(short, h0, c0)
    core.set_option("profile", 0)
    assert torch.equal(core.forward(short, h0, c0)[0], y)
    assert core.info("fallbacks") == 0
    core.close()


def test_recurrence_that_waits_in_vain_for_its_projection_is_repeated():
    """A bound of no reload at all: the recurrence gives up before the first tile is there, the pass is repeated step-wise."""
    import torch
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(64, 512, 1024)
    core.pack(*(torch.randn(*s, device="cuda") * 0.03 for s in ((4096, 512), (4096, 1024), (4096,), (4096,))))
    x = torch.randn(128, 64, 512, device="cuda").half()
    want = core.forward(x)
    assert core.info("projection_fwd") == 1 and core.info("fallbacks") == 0
    core.set_option("spin_limit", 0)
    assert all(torch.equal(a, b) for a, b in zip(core.forward(x), want))
    assert core.info("fallbacks") >= 1 and core.info("persistent_fwd") == 0
    core.close()


def test_step_wise_passes_between_projections_beside_replay_one_graph():
    """The arguments of a step-wise launch are the key of its captured graph: what a pass with its projection beside left behind in them
    must not show."""
    import torch
    from flashlstm_poc_amd import LstmCore
    core = LstmCore(64, 512, 1024)
    core.pack(*(torch.randn(*s, device="cuda") * 0.03 for s in ((4096, 512), (4096, 1024), (4096,), (4096,))))
    x = torch.randn(128, 64, 512, device="cuda").half()
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):   # (the legacy default stream cannot be captured)
        want = core.forward(x)
        for again in range(5):
            core.set_option("stepwise", 1)
            assert all(torch.equal(a, b) for a, b in zip(core.forward(x), want))
            assert core.info("projection_fwd") == 0 and core.info("graph_captures") == 1 and core.info("graph_replays") == again
            core.set_option("stepwise", 0)
            assert all(torch.equal(a, b) for a, b in zip(core.forward(x), want))
            assert core.info("projection_fwd") == 1
    core.close()
