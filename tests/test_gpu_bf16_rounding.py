"""Rounding of float32 to bfloat16 on the device (csrc/common.cuh BF16::from_f32, through vra_cast) against the oracle, bit for bit: every upper half, so
denormals, infinities and every NaN's, with the lower halves around a tie."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.util import BF16, F32
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("low", [0, 1, 0x7fff, 0x8000, 0x8001, 0xffff])
def test_every_upper_half_rounds_as_the_oracle(low):
    x = (np.arange(1 << 16, dtype=np.uint32) << 16 | np.uint32(low)).view(np.float32)
    src, out = ops.dev(x), ops.DevBuf(x.size * 2)
    ops.lib().vra_cast(src.ptr, out.ptr, x.size, F32, BF16, 0)
    np.testing.assert_array_equal(out.numpy(np.uint16, x.shape), orc.to_bf16(x))
