"""The stream that operator calls run on, and the CFL check's paired maxima."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_calls_follow_the_current_stream(mlv):
    import torch

    L = mlv._lib
    assert (L.stream_handle().value or 0) == torch.cuda.current_stream().cuda_stream
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert L.stream_handle().value == s.cuda_stream
    assert L.stream_handle(s).value == s.cuda_stream
    assert (L.stream_handle().value or 0) == torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shape", [(1, 1), (33, 7), (256, 1024)])
def test_paired_maxima(mlv, dtype, shape):
    rng = np.random.default_rng(5)
    a, b = (-rng.random(shape).astype(dtype) for _ in range(2))
    assert mlv.hip.max_pair(a, mlv.hip.asarray(b).t()) == (float(a.max()), float(b.max()))
    b[-1, -1] = np.nan
    m, n = mlv.hip.max_pair(a, b)
    assert m == float(a.max()) and math.isnan(n)
