"""Phase times (flstm_core_last_ms) name what they hold, whichever way a pass took: the projection has a time of its own where a launch
in front of the recurrence forms it and none elsewhere, and the total holds every launch of the pass."""
import time

import pytest

pytestmark = pytest.mark.gpu


def timed(core, *args, **kwargs):
    """A call's own wall-clock milliseconds, the least of several, and the phase times of that call."""
    import torch
    best = None
    for _ in range(12):
        torch.cuda.synchronize()
        t = time.perf_counter()
        core.forward(*args, **kwargs)
        ms = (time.perf_counter() - t) * 1e3
        if best is None or ms < best[0]:
            best = ms, {k: core.last_ms(k) for k in ("fwd_proj", "fwd_rec", "fwd_total")}
    return best


# whole pass, projection inside, nothing in front; the same with converted rows; whole pass, projection in front (1024 features: as long as
# the recurrence; with rows used in place nothing else comes first); projection beside; in front of separate launches
@pytest.mark.parametrize("T,B,I,H,dtype,whole,projection", [
    (64, 16, 128, 256, "f16", 1, 2), (64, 512, 128, 256, "f32", 1, 2), (64, 256, 1024, 256, "f16", 1, 0), (64, 256, 1000, 256, "f32", 1, 0),
    (256, 64, 1024, 1024, "f16", 0, 1), (64, 256, 1024, 1024, "f16", 0, 0), (64, 256, 1000, 1000, "f32", 0, 0)])
def test_forward_phases(T, B, I, H, dtype, whole, projection):
    import torch
    from flashlstm_poc_amd import LstmCore
    kind = {"f16": torch.float16, "f32": torch.float32}[dtype]
    core = LstmCore(B, I, H)
    core.pack(*(torch.randn(*s, device="cuda") * 0.03 for s in ((4 * H, I), (4 * H, H), (4 * H,), (4 * H,))))
    x = torch.randn(T, B, I, device="cuda").to(kind)
    ms, phase = timed(core, x, save_for_backward=False)
    assert core.info("whole_fwd") == whole and core.info("projection_fwd") == projection and core.info("fallbacks") == 0
    # a product no faster than the matrix cores (2.5 PFLOP/s), rows converted no faster than memory (8 TB/s)
    product, converted = 8.0 * T * B * I * H / 2.5e12, (6.0 * T * B * I / 8e9 if dtype == "f32" else 0.0)
    if projection == 0:
        assert phase["fwd_proj"] >= product
    else:
        assert phase["fwd_proj"] < 0
    assert phase["fwd_rec"] > 0
    # (times are fp32 milliseconds: sums of two of them agree to 1e-6)
    assert max(phase["fwd_proj"], 0.0) + phase["fwd_rec"] <= phase["fwd_total"] * 1.000001 <= ms
    assert phase["fwd_total"] >= phase["fwd_rec"] + converted + (product if projection == 0 else 0.0)
    core.close()


def test_backward_total_holds_the_setup_and_the_outputs():
    import torch
    from flashlstm_poc_amd import LstmCore
    T, B, I, H = 64, 512, 100, 250   # fp32 rows of odd sizes: converted in the setup
    core = LstmCore(B, I, H)
    core.pack(*(torch.randn(*s, device="cuda") * 0.03 for s in ((4 * H, I), (4 * H, H), (4 * H,), (4 * H,))))
    x, dy = torch.randn(T, B, I, device="cuda"), torch.randn(T, B, H, device="cuda")
    core.forward(x)
    for _ in range(3):
        core.backward(x, dy)
    total, parts = core.last_ms("bwd_total"), [core.last_ms(k) for k in ("bwd_rec", "bwd_dx", "bwd_dw")]
    assert min(parts) >= 0 and total > sum(parts)
    core.close()
