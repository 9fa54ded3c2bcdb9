"""Status words read back by polling pinned host memory (csrc/common.hip, read_back): behind an empty stream, behind a
queue longer than the polling limit of one millisecond, and from several host threads at once."""
import threading

import pytest

from ai2pot_amd import synth
from conftest import to_device

pytestmark = pytest.mark.gpu


def _call(oracle):
    import torch
    from ai2pot_amd import ops
    lat, pos = synth.random_packed(40, [9.0, 10.0, 9.5], 2.2, 5)
    ty = synth.rng_randint(6, 40, 2)
    nb = to_device(synth.pack_batch([oracle.nblist(lat, ty, pos, 5.0, 200)]), torch.float64)
    dei = torch.from_numpy(synth.rng_normal(7, nb["brcs"].numel()).reshape(nb["brcs"].shape)).to("cuda:0")

    def call(first):
        return ops.ForceSrOp(nb["binum"], nb["bilist"], nb["bnumneigh"], first, 0, 200, dei)[0]
    return call, nb["bfirstneigh"]


@pytest.mark.parametrize("queue_ms", [0, 20])
def test_status_behind_a_queue(oracle, queue_ms):
    import torch
    call, first = _call(oracle)
    bad = first.clone()
    bad[0, 3, 0] = 4000
    want = call(first)
    x = torch.zeros(1 << 26, device="cuda:0")
    for _ in range(3):
        for _ in range(queue_ms * 10):                 # about 0.1 ms each
            x.add_(1.0)
        with pytest.raises(RuntimeError, match="neighbour index"):
            call(bad)
        assert torch.equal(call(first), want)          # the word is cleared


def test_status_from_several_threads(oracle):
    """Each waiting thread holds a slot of the pinned page of its own."""
    import torch
    from ai2pot_amd import _lib
    call, first = _call(oracle)
    call(first)
    stream = torch.cuda.current_stream().cuda_stream
    failed = []

    def work():
        try:
            for _ in range(200):
                _lib.check_status(stream)
        except Exception as ex:
            failed.append(ex)
    threads = [threading.Thread(target=work) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
