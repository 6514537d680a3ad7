"""``agmi_concat``: joins whose rows, pieces and borders fall on every side of the 16-byte vectors that large joins move, and small
ones, which move one element to a thread; a copy, so exact."""

import numpy as onp
import pytest

pytestmark = pytest.mark.gpu

# (outer, inner, extents); small joins: one vector more or less than a piece, empty pieces, and the most pieces one launch takes
SMALL = [
    (1, 1, (1,)), (1, 1, (3, 1)), (3, 1, (4, 5, 0, 3)), (256, 1, (128, 512, 1)), (35, 1, (128, 40, 1)), (7, 3, (1, 2, 5)),
    (1, 512, (2,) * 31 + (0,)), (2, 1, (1023, 1, 1025)), (5, 1, (2048, 2047)), (1, 1, (1,) * 32), (3, 17, (100, 1, 33)),
]
# large joins in 16-byte vectors: borders between vectors throughout; borders inside a vector, rows that start inside one and
# blocks of 1024 (512) elements across several rows; blocks within one row; empty pieces first, last and in between; totals
# that end one, two and three elements into a vector; rows of pieces short but aligned
WIDE = [
    (1, 641, (256,) * 32), (1401, 1, (300, 512, 1)), (3, 1, (400001, 0, 7, 100003)), (2, 1, (0, 33335) * 15 + (70002, 0)),
    (1, 1, (333335, 1, 700002, 20001)), (1, 3, (1, 400001, 7, 2)), (2100, 4, (16,) * 8), (530, 1, (2047, 1)), (66, 17, (999, 1)),
]
# joins as large whose vectors would cross borders all the time: one element to a thread
LARGE = [(4000, 17, (13, 1, 3)), (1000, 33, (1,) * 32), (400001, 1, (1, 2))]


@pytest.mark.parametrize("dtype", [onp.float32, onp.float64])
@pytest.mark.parametrize("form", ["plain", "columns", "outer_gap", "broadcast", "offset"])
@pytest.mark.parametrize("outer,inner,extents,wide", [j + (False,) for j in SMALL + LARGE] + [j + (True,) for j in WIDE])
def test_joins_are_copies(dtype, form, outer, inner, extents, wide):
    import torch

    from autograd_amd import _lib

    dev, code = _lib.device(), _lib.DTYPE_CODE[onp.dtype(dtype)]
    rs = onp.random.RandomState(outer + inner + len(extents))
    pieces, want = [], []
    for k, extent in enumerate(extents):
        shape = (outer, extent, inner)
        if form == "columns" and k % 2 == 0:  # stored with the joined axis innermost
            t = torch.from_numpy(rs.randn(outer, inner, extent).astype(dtype)).to(dev).transpose(1, 2)
        elif form == "outer_gap":  # gapless rows that lie apart
            t = torch.from_numpy(rs.randn(outer, extent + 1, inner).astype(dtype)).to(dev)[:, :extent]
        elif form == "broadcast" and k % 2 == 1:
            t = torch.from_numpy(rs.randn(1, 1, 1).astype(dtype)).to(dev).expand(shape)
        elif form == "offset":  # one element past a 16-byte border
            t = torch.from_numpy(rs.randn(1 + outer * extent * inner).astype(dtype)).to(dev)[1:].view(shape)
        else:
            t = torch.from_numpy(rs.randn(*shape).astype(dtype)).to(dev)
        pieces.append((t, extent) + tuple(t.stride()))
        want.append(t.cpu().numpy())
    want = onp.concatenate(want, axis=1)
    memory = torch.full((want.size + 2,), -7.0, dtype=pieces[0][0].dtype, device=dev)
    out = memory[1:-1]
    _lib.lib()
    _lib.concat(code, outer, inner, pieces, out)
    assert ("16 bytes" in _lib.lib().agmi_last_kernel().decode()) == wide
    got = memory.cpu().numpy()
    assert got[0] == -7.0 and got[-1] == -7.0  # nothing is written beside the result
    assert onp.array_equal(got[1:-1].reshape(want.shape), want)
