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


def test_grouped_forms(gpu_stream):
    """A ragged batch of 20 grants of one rank-3 shape: its pair's base (320
    rows) takes the 128-row form and the single layer's (160) the 32-row form
    within one grouped launch."""
    from puschrx import grants as G
    from puschrx.chain import ChainOptions, NativeChain
    grants = [G.Grant(name=f"g{i}", rank=3, qm=4, num_rb=11, fft_size=256, code_rate=0.4, rnti=i + 1,
                      padded_subcarriers=256) for i in range(20)]
    compiled = G.compile_grants(G.Radio(), grants)
    batch = G.GrantBatch(compiled, dict(iq_format=abi.IQ_COMPLEX64, tau_s=200e-9, fd_hz=30.0), use_graph=False)
    assert batch.num_shapes == 1
    rng = np.random.default_rng(3)
    g = ops.Geometry(compiled[0][1])
    iqs = [rng.normal(0, 1, (g.nr, g.samples, 2)).astype(np.float32) for _ in compiled]
    batch.enqueue(batch.pack_iq(iqs))
    opts = ChainOptions(tau_s=200e-9, fd_hz=30.0, iq_format=abi.IQ_COMPLEX64)
    for i in (0, 7, 19):
        _, cfg, plan = compiled[i]
        n = cfg.qm * g.cw_stride
        got = batch.fetch("cw_llr", torch.int16, n, batch.layout[i].cw_offset)
        one = NativeChain(cfg, plan, max_slots=1, opts=opts, use_graph=False)
        one.enqueue(torch.from_numpy(iqs[i][None]).cuda(), 1)
        want = one.fetch("cw_llr", torch.int16, n)
        torch.cuda.synchronize()
        assert torch.equal(got, want), i
        one.close()
    batch.close()
