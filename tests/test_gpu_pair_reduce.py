"""Pair reduction (csrc/pair_reduce.hip) where segments run over: lists that name one atom more often than a row is long,
at row lengths around the entries a lane keeps in registers (4 of 16 lanes each) and the wavefront's width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
@pytest.mark.parametrize("U", [1, 9, 64, 65, 130])
@pytest.mark.parametrize("named", ["one", "few", "any"])
def test_force_of_lists_that_run_over(np_dtype, U, named):
    import torch
    from ai2pot_amd import ops
    B, P, nghost = 2, 23, 3
    rng = np.random.default_rng(U)
    binum = np.array([P, P - 6], np.int32)
    bilist = np.stack([rng.permutation(P) for _ in range(B)]).astype(np.int32)
    nn = rng.integers(0, U + 1, (B, P)).astype(np.int32)
    nn[:, 0] = U
    top = {"one": 1, "few": 3, "any": P + nghost}[named]
    fn = (rng.integers(0, top, (B, P, U)) + (P + nghost - top)).astype(np.int32)
    dei = (rng.normal(size=(B, P, U, 3)) * 10.0 ** rng.integers(-3, 3, (B, P, U, 1))).astype(np_dtype)
    want = np.zeros((B, P + nghost, 3))
    size = np.zeros_like(want)
    for b in range(B):
        for ii in range(binum[b]):
            for s in range(nn[b, ii]):
                g = dei[b, ii, s].astype(np.float64)
                want[b, bilist[b, ii]] += g
                want[b, fn[b, ii, s]] -= g
                size[b, bilist[b, ii]] += np.abs(g)
                size[b, fn[b, ii, s]] += np.abs(g)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    runs = [ops.ForceSrOp(d(binum), d(bilist), d(nn), d(fn), nghost, U, d(dei))[0].cpu().numpy() for _ in range(3)]
    # a row's own sum is made in the input's precision, the named pairs' in fixed point below its rounding
    bound = size * np.finfo(np_dtype).eps * (8 + U // 64)
    assert np.all(np.abs(runs[0] - want) <= bound)
    assert all(np.array_equal(r, runs[0]) for r in runs[1:])
