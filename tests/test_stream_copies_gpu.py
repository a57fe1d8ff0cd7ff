"""Rows on their way to pinned host memory (beside the recurrence, on workgroups that have no part in it, or by a launch of
their own) at widths and alignments that no 16-byte access fits: the same bits as through the runtime's copies to pageable
memory, and nothing beside them touched."""
import numpy as np
import pytest
import torch

from helpers import make_problem
from test_v2_api_gpu import run_v2

pytestmark = pytest.mark.gpu

GUARD = 16   # elements in front of and behind an output


# odd widths of x and h, single columns, rows shorter than 16 bytes, recurrence workgroups of one, two and four waves, a layer
# that leaves none idle (128 rows of 1030 units); outputs that start at any element of 16 bytes
@pytest.mark.parametrize("T,B,I,H,R", [(200, 32, 257, 257, 8), (130, 9, 1, 511, 3), (150, 70, 650, 129, 50), (140, 128, 1023, 40, 1),
                                       (200, 3, 3, 5, 7), (130, 4, 2, 1, 3), (120, 20, 650, 650, 8), (100, 64, 512, 512, 8), (100, 128, 65, 1030, 8),
                                       (96, 5, 33, 2049, 8)])
@pytest.mark.parametrize("shift", [0, 1, 5])
def test_pinned_rows_of_any_width_and_alignment(T, B, I, H, R, shift, monkeypatch):
    p = make_problem(T, B, I, H, seed=T + B)
    want = run_v2(p, R=R, h_dtype=torch.float16, c_dtype=torch.float32, pin=False, fresh_backward=True)
    empty, guarded = torch.empty, []

    def shifted(*size, **kw):
        if not kw.get("pin_memory"):
            return empty(*size, **kw)
        shape = tuple(size[0]) if len(size) == 1 and not isinstance(size[0], int) else size
        n = int(np.prod(shape))
        flat = empty(GUARD + shift + n + GUARD, **kw).fill_(-7.0)
        guarded.append((flat, n))
        return flat[GUARD + shift:GUARD + shift + n].view(shape)

    monkeypatch.setattr(torch, "empty", shifted)
    got = run_v2(p, R=R, h_dtype=torch.float16, c_dtype=torch.float32, pin=True, fresh_backward=True)
    monkeypatch.undo()
    assert len(guarded) >= 4
    for flat, n in guarded:
        assert (flat[:GUARD + shift] == -7.0).all() and (flat[GUARD + shift + n:] == -7.0).all()
    for k in ("y", "ck_h", "ck_c", "hn", "cn", "dx", "dh0", "dc0", "dw_ih", "dw_hh"):
        assert np.array_equal(got[k], want[k]), k
