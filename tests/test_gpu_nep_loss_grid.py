"""The gradient of the NEP training loss for batches that fill the device once, several times and badly: each copy of a
structure has the gradient that the structure has in a batch of three, which is held against the oracle here.  Bars: the
loss within 1e-10 of the oracle; a copy's rows are the same sums in the same order, from residual forces that another
kernel may have summed in another order, so n = 70 terms of rounding each: 1e-11 in fp64 (70 * 2.2e-16 with three orders for
cancellation), 2e-4 in fp32 (the bar of fp32 against fp64)."""
import numpy as np
import pytest

from test_gpu_nep_loss import GRADS, close, gpu_loss, larger_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_dtype,bar", [(np.float64, 1e-11), (np.float32, 2e-4)])
@pytest.mark.parametrize("copies", [1, 21, 43, 44, 67, 86, 100, 171, 200])
def test_batches_of_any_size(oracle, np_dtype, bar, copies):
    m, nb, labels = larger_case(oracle, 3, (70, 45, 58))
    w = (0.9, 1.3, 0.4)
    few = gpu_loss(m, nb, labels, w)
    assert close(few["bloss"], oracle.nep_loss(m, nb, w, labels)[0])
    many = lambda d: {k: np.concatenate([v] * copies) if np.ndim(v) else v for k, v in d.items()}
    got = gpu_loss(m, many(nb), many(labels), w, np_dtype)
    for k in GRADS:
        assert got[k].shape[0] == 3 * copies
        for c in range(copies):
            assert close(got[k][3 * c:3 * c + 3], few[k], bar), (k, c)
