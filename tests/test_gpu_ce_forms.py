"""The channel estimator's products in their 32-row and 128-row forms (a base's
rows: models x slots x Rx x DMRS symbols, the forms meeting at 256) give the
same bits: a batch's channel estimates and noise equal each slot's alone, at
slot counts on both sides, for every rank (one or two bases, one to four
models) and for 6 and 64 antennas (the time interpolation's antenna chunks)."""
import numpy as np
import pytest

from puschrx import abi, ops
from puschrx import profiles as P

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rx,rank,prb,slots", [(4, 4, 11, 7), (4, 4, 11, 8), (4, 3, 11, 16), (4, 2, 25, 33),
                                               (4, 1, 6, 33), (6, 4, 6, 5), (64, 2, 5, 2)])
def test_batch_equals_slots(gpu_stream, rx, rank, prb, slots):
    from puschrx.chain import ChainOptions, NativeChain
    fft = 128 if prb <= 9 else 512
    prof = P.Profile(name="t", rx=rx, rank=rank, num_rb=prb, fft=fft, qm=4, padded_subcarriers=P.align_up(12 * prb, 128),
                     code_rate=0.4)
    cfg = prof.config()
    g = ops.Geometry(cfg)
    plan = ops.tb_plan(ops.tbs(prb, 12 * g.ndata, 4, rank, 0.4), g.cw_symbols * 4, 4, rank)
    opts = ChainOptions(tau_s=200e-9, fd_hz=30.0, iq_format=abi.IQ_COMPLEX64)
    rng = np.random.default_rng(rx + rank + slots)
    iq = torch.from_numpy(rng.normal(0, 1, (slots, g.nr, g.samples, 2)).astype(np.float32)).cuda()
    per = g.nr * g.nl * 14 * g.pad
    batch = NativeChain(cfg, plan, max_slots=slots, opts=opts, use_graph=False)
    batch.enqueue(iq, slots)
    got = [batch.fetch(n, torch.float16, slots * k) for n, k in (("h_re", per), ("h_im", per), ("noise_ce", g.nr))]
    one = NativeChain(cfg, plan, max_slots=1, opts=opts, use_graph=False)
    for s in range(slots):
        one.enqueue(iq[s:s + 1].contiguous(), 1)
        want = [one.fetch(n, torch.float16, k) for n, k in (("h_re", per), ("h_im", per), ("noise_ce", g.nr))]
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            k = b.numel()
            assert torch.equal(a[s * k:(s + 1) * k].view(torch.int16), b.view(torch.int16)), s
    batch.close()
    one.close()
