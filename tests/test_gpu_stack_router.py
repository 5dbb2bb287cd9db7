"""The picks of a layer stack's router (csrc/stack_ops.hip): the largest first, the first of equal ones, a NaN only where it is the first of what is left."""
import numpy as np
import pytest

from tests.util import BF16, F32, rng
from vllm_rs_amd import _lib, ops

pytestmark = pytest.mark.gpu


def picks(z, top):
    left, out = list(range(len(z))), []
    for _ in range(top):
        best = left[0]
        for e in left:
            if z[e] > z[best]:
                best = e
        out.append(best)
        left.remove(best)
    return out


# one output, rounds of one to five outputs a wave, up to and beyond one and two a lane, the largest that lanes keep marks for and one more (picked by one thread)
@pytest.mark.parametrize("dt", [BF16, F32])
@pytest.mark.parametrize("E,top", [(1, 1), (6, 2), (11, 2), (17, 3), (64, 64), (65, 6), (160, 8), (4096, 4), (4097, 4)])
@pytest.mark.parametrize("gate", [0, 1])
def test_picks(gate, E, top, dt):
    r = rng(E + gate)
    W, T = 64, 5
    x = np.zeros((T, W), np.float32)
    x[np.arange(T), np.arange(T)] = 8.0  # the norm of a row is its unit vector times 8 (whole rows, eps below the last bit): z is a column of the weights
    rw = r.permuted(np.tile(np.arange(E + 1, dtype=np.float32) % 97 - 48, (W, 1)), axis=1).T.copy()  # whole numbers, equal ones among them
    rw[E // 2:, 1] = np.nan  # not the first: never picked ahead of a number
    rw[0, 2] = np.nan        # the first of all: picked first, and the next by size
    rw[:, 3] = -np.inf       # all equal
    rw[E // 3, 4] = np.inf
    rw[E] = 0.5
    plain = np.isfinite(rw).all(0)  # (0 times an infinity is a NaN: a column with one is there for its own row only)
    w = np.ones(W, np.float32)

    def cast(v):
        return ops.dev((v.view(np.uint32) >> 16).astype(np.uint16) if dt == BF16 else v)
    for t in range(T):
        wt = rw.copy()
        wt[:, ~plain] = 0.0
        wt[:, t] = rw[:, t]
        z = wt[:E, t] * 8.0
        h, pe, pw, gt = ops.DevBuf(W * 4), ops.DevBuf(top * 4), ops.DevBuf(top * 4), ops.DevBuf(4)
        xd, wd, rd = ops.dev(x[t:t + 1].copy()), ops.dev(w), cast(wt[:E + gate])
        _lib.load().vra_stack_op_group_norm(xd.ptr, wd.ptr, h.ptr, 1, W, 1, 0.0, rd.ptr, E, top, gate, pe.ptr, pw.ptr, gt.ptr, dt, 0)
        ops.check_error()
        want = picks(z, top)
        assert pe.numpy(np.int32, (top,)).tolist() == want
        with np.errstate(over="ignore"):
            s = 1.0 / (1.0 + np.exp(-z[want].astype(np.float64)))
        # sigmoid in f32: an exponential, a sum and a quotient, each within 2 of the last place
        assert np.allclose(pw.numpy(np.float32, (top,)), s, rtol=6 * 2.0 ** -23, atol=1e-37, equal_nan=True)
        if gate:
            assert abs(float(gt.numpy(np.float32, (1,))[0]) - 1 / (1 + np.exp(-4.0))) < 6 * 2.0 ** -23
