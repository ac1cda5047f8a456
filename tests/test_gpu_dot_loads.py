"""The scalar product's 16-byte loads and its rounding by one wave: vectors
that start at an odd entry of an allocation, lengths around the 8-byte tail,
a wave's 512 entries and the second pass over the grid, and sums whose digits
lie at either end of the accumulator.  The sum is exact and rounded once, so
it equals math.fsum's bit for bit."""
import ctypes as C
import math

import numpy as np
import pytest

import omodels_amd as om

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -1030, 2.0 ** 905, 2.0 ** 1000, -1.0])
@pytest.mark.parametrize("off_x,off_y", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_offsets_lengths_and_magnitudes(off_x, off_y, scale):
    rng = np.random.default_rng(11)
    lengths = [1, 2, 3, 127, 129, 511, 513, 4097]
    if scale == 1.0:
        lengths.append(256 * 8 * 512 + 513)
    for m in lengths:
        x = rng.standard_normal(m + off_x)
        y = rng.standard_normal(m + off_y)
        x[off_x + m // 2] += 3.0
        y *= scale
        dx, dy = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(y).to("cuda:0")
        out = torch.full((1,), float("nan"), dtype=torch.float64, device="cuda:0")
        stream = torch.cuda.current_stream(torch.device("cuda:0"))
        rc = om.lib().omodels_scalar_product_noalloc(m, C.c_void_p(dx.data_ptr() + 8 * off_x),
                                                     C.c_void_p(dy.data_ptr() + 8 * off_y),
                                                     C.c_void_p(out.data_ptr()), C.c_void_p(stream.cuda_stream))
        assert rc == 0, om.lib().omodels_last_error().decode()
        torch.cuda.synchronize()
        want = math.fsum((x[off_x:] * y[off_y:]).tolist())
        assert float(out.cpu().numpy()[0]) == want, (m, off_x, off_y, scale)
