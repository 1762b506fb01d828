"""The reverse mode where memory is short."""
import numpy as np
import pytest
import torch

import pymfc
from parity import equal

pytestmark = pytest.mark.gpu


def free_bytes():
    return torch.cuda.mem_get_info()[0]


def test_batch_gradient_with_little_memory_left():
    """The recorded secant results make the replay of a run faster, but nothing depends on them: a batch
    keeps them only where they leave room for what all its instances need. Here 512 MB are left
    beside that, and the first five would take more; the results are a single handle's."""
    def config(i):
        c = pymfc.cut_config(250, 80, 10.0, thermal="contact", jitter=0.01, seed=i + 1)
        c.promote_fp64, c.secant_tol = 1, 1e-14
        return c

    n, steps = 6, 750
    run = (steps, 30, 0, 200)
    alone = pymfc.Sim(config(0))
    before = free_bytes()
    F = alone.vjp_forward(*run)
    tape = 8 * alone.N * steps
    need = before - free_bytes() - tape  # an instance's, without its secant results
    assert need > tape and (n - 1) * tape > 512 << 20
    grad = alone.vjp_backward([1.0, 0.5])
    alone.close()
    batch = pymfc.Batch([config(i) for i in range(n)])
    fill = []
    try:
        while (spare := free_bytes() - n * need - (512 << 20)) > 4 << 20:
            fill.append(torch.empty(min(spare, 32 << 30), dtype=torch.uint8, device="cuda"))
        Fs = batch.vjp_forward(*run)
        gs = batch.vjp_backward(np.tile([1.0, 0.5], (n, 1)))
    finally:
        del fill
        torch.cuda.empty_cache()
        batch.close()
    assert equal(Fs[0], F) and equal(gs[0], grad)
    assert np.all(np.isfinite(Fs))
