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


@pytest.mark.parametrize("np_dtype", [np.float64, np.float32])
def test_lists_that_run_over_take_linear_time(np_dtype):
    """An eighth of the atoms named by all pairs, seven of eight pairs beyond the segments, at 50,000 rows: the time stays
    within a few times that of a list that fits (1.4 times measured; 200 times when every target searched what ran over)."""
    import time
    import torch
    from ai2pot_amd import ops
    n, U = 50000, 32
    rng = np.random.default_rng(3)
    dei = rng.normal(size=(1, n, U, 3)).astype(np_dtype)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    head = (d(np.array([n], np.int32)), d(np.arange(n, dtype=np.int32)[None]), d(np.full((1, n), U, np.int32)))
    g = d(dei)
    best = {}
    for name, fn in (("fits", np.stack([rng.permutation(n) for _ in range(U)], 1)[None]),
                     ("over", rng.integers(0, n // 8, (1, n, U)))):
        f = d(fn.astype(np.int32))
        best[name] = np.inf
        for _ in range(5):
            torch.cuda.synchronize()
            begin = time.perf_counter()
            out = ops.ForceSrOp(*head, f, 0, U, g)[0]
            torch.cuda.synchronize()
            best[name] = min(best[name], time.perf_counter() - begin)
        want = dei[0].astype(np.float64).sum(1)
        size = np.abs(dei[0].astype(np.float64)).sum(1)
        np.subtract.at(want, fn[0].ravel(), dei[0].reshape(-1, 3).astype(np.float64))
        np.add.at(size, fn[0].ravel(), np.abs(dei[0].reshape(-1, 3).astype(np.float64)))
        # the row's own sum in the input's precision, the named pairs' in fixed point below its rounding
        assert np.all(np.abs(out[0].cpu().numpy() - want) <= size * np.finfo(np_dtype).eps * 8)
    assert best["over"] < 15 * best["fits"], best
