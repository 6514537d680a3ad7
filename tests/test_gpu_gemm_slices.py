"""Products of few tiles and a long K, cut along K across blocks: tiles x slices on both sides of the 256 CUs, slices with a
remainder, and the shortest K that is cut (float64; float32 up to K = 4096 has a kernel that cuts it within a block) and the longest
that is not; the oracle is NumPy in float64."""

import numpy as onp
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 4100), (641, 512, 4608), (513, 128, 5000), (704, 640, 4128), (65, 129, 8191), (1000, 8, 6001), (10, 10, 256), (127, 63, 255),
          (320, 256, 700), (10, 10, 128), (10, 10, 127), (33, 40, 4097), (33, 40, 4096), (1024, 512, 4200)]


@pytest.mark.parametrize("dtype", [onp.float32, onp.float64])
@pytest.mark.parametrize("left", ["N", "T"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products_cut_along_k(dtype, left, M, N, K):
    import autograd_amd.numpy as dnp
    from autograd_amd import _lib

    rs = onp.random.RandomState(M + N + K)
    a, b = rs.randn(M, K).astype(dtype), rs.randn(K, N).astype(dtype)
    got = (dnp.dot(dnp.array(a), dnp.array(b)) if left == "N" else dnp.dot(dnp.array(onp.ascontiguousarray(a.T)).T, dnp.array(b))).numpy()
    tiles = -(-M // 64) * -(-N // 64)
    cut = tiles < 128 and (K > 4096 if dtype == onp.float32 else K >= 128)
    assert ("+split" in _lib.lib().agmi_last_kernel().decode()) == cut
    a, b = a.astype("float64"), b.astype("float64")
    # the longest serial chain holds K terms at most, each sum rounded once; float64's oracle rounds as often
    bound = (2 if dtype == onp.float64 else 1) * (K + 64) * onp.finfo(dtype).eps / 2
    assert (abs(got - a @ b) <= bound * (abs(a) @ abs(b))).all()
    # and far closer on the whole: roundings of either sign add up like their square root
    assert onp.linalg.norm(got - a @ b) <= 4 * K ** 0.5 * onp.finfo(dtype).eps * onp.linalg.norm(a @ b)
