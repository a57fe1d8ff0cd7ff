"""dX and the weight gradients of a whole backward pass share a launch where both products run with small tiles: the same bits as the
products of their own launches, which a pass in ranges of steps (here: one range of all of them) makes."""
import numpy as np
import pytest
import torch

from helpers import make_problem, to_np
from test_core_gpu import run_core

pytestmark = pytest.mark.gpu

# T, B, I, H: 64 x 64 tiles for both (one tile each, ragged, dX's last); 128 x 128 for the weight gradients (dX's tiles first, last), for
# dX, for both; tiles that keep a launch to themselves
SHAPES = [(1, 1, 1, 1), (8, 9, 65, 257), (20, 100, 1000, 64), (33, 9, 456, 950), (200, 70, 65, 257), (260, 50, 300, 72), (128, 100, 512, 256),
          (300, 64, 128, 64), (64, 256, 1024, 256)]
APART = [(300, 64, 128, 64), (64, 256, 1024, 256)]


@pytest.mark.parametrize("T,B,I,H", SHAPES)
@pytest.mark.parametrize("half", [True, False])
def test_shared_launch_gives_the_bits_of_two(T, B, I, H, half):
    from flashlstm_poc_amd import LstmCore
    from flashlstm_poc_amd.core import load_library
    p = make_problem(T, B, I, H, seed=T * 1000 + H)
    core = LstmCore(B, I, H)
    core.pack(*(p[k].cuda() for k in ("w_ih", "w_hh", "b_ih", "b_hh")))
    want, info = run_core(p, core=core, half=half)
    assert info["fallbacks"] == 0 and core.info("products_shared") == (0 if (T, B, I, H) in APART else 1)
    dt = torch.float16 if half else torch.float32
    code = 1 if half else 0
    dev = {k: p[k].cuda().to(dt) for k in ("x", "h0", "c0", "dy", "d_hn", "d_cn")}
    core.forward(dev["x"], dev["h0"], dev["c0"])
    f32 = lambda *s: torch.empty(*s, device="cuda")
    dx = torch.empty(T, B, I, device="cuda", dtype=dt)
    out = dict(dw_ih=f32(4 * H, I), dw_hh=f32(4 * H, H), db=f32(4 * H), db_hh=f32(4 * H), dh0=f32(B, H), dc0=f32(B, H))
    lib, s = load_library(), torch.cuda.current_stream().cuda_stream
    assert lib.flstm_core_backward_begin(core._h, T, dev["dy"].data_ptr(), code, dev["d_hn"].data_ptr(), dev["d_cn"].data_ptr(), code,
                                         1.0, dx.data_ptr(), code, s) == 0
    assert lib.flstm_core_backward_steps(core._h, T - 1, T, s) == 0
    assert lib.flstm_core_backward_end(core._h, dev["x"].data_ptr(), code,
                                       *(out[k].data_ptr() for k in ("dw_ih", "dw_hh", "db", "db_hh", "dh0", "dc0")), s) == 0
    torch.cuda.synchronize()
    assert core.info("products_shared") == 0
    for k, v in dict(out, dx=dx).items():
        if k != "db_hh":
            assert np.array_equal(to_np(v), want[k]), k
    core.close()
