"""The fused detector's packed demapper (every modulation and layer count)
against the operators, which demap one axis at a time: the descrambled
codeword LLRs of the batched chain and of the ragged batch equal the
operator chain's bit for bit, on slots of random samples at three levels
(LLRs from saturated to a few units) and on a slot of zeros (no channel, no
noise: the NaN and infinity rules)."""
import numpy as np
import pytest

from puschrx import abi, ops
from puschrx import grants as G
from puschrx import profiles as P

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _iq(g, seed):
    rng = np.random.default_rng(seed)
    iq = rng.normal(0, 1, (4, g.nr, g.samples, 2)).astype(np.float32)
    iq *= np.array([1.0, 1e-3, 8.0, 0.0], np.float32)[:, None, None, None]
    # A channel that repeats from symbol to symbol, so that some REs detect
    # something: the slot's symbols are one symbol plus a little noise.
    n = g.fft + g.cp_short
    iq[0] = np.tile(iq[0][:, :n], (1, g.samples // n + 1, 1))[:, : g.samples] + 0.01 * iq[0]
    return np.ascontiguousarray(iq)


@pytest.mark.parametrize("qm", [2, 4, 6, 8])
@pytest.mark.parametrize("rank", [1, 2, 3, 4])
def test_fused_demap_matches_operators(gpu_stream, qm, rank):
    from puschrx.chain import ChainOptions, NativeChain, OpChain
    prof = P.Profile(name="t", rx=4, rank=rank, num_rb=6, fft=128, qm=qm, padded_subcarriers=128, code_rate=0.5)
    cfg = prof.config()
    g = ops.Geometry(cfg)
    plan = ops.tb_plan(ops.tbs(6, 12 * g.ndata, qm, rank, 0.5), g.cw_symbols * qm, qm, rank)
    opts = ChainOptions(tau_s=100e-9, fd_hz=10.0, iq_format=abi.IQ_COMPLEX64)
    iq = torch.from_numpy(_iq(g, 10 * qm + rank)).cuda()
    nat = NativeChain(cfg, plan, max_slots=4, opts=opts, use_graph=False)
    op = OpChain(cfg, plan, opts)
    nat.enqueue(iq, 4)
    cw = nat.fetch("cw_llr", torch.int16, 4 * qm * g.cw_stride)
    torch.cuda.synchronize()
    cw = cw.cpu().numpy().reshape(4, -1)
    for s in range(4):
        want = op.run_slot(iq[s].contiguous(), keep=True)["cw_nr"]
        torch.cuda.synchronize()
        assert np.array_equal(cw[s], want.cpu().numpy()), s
    nat.close()
    op.close()


def test_ragged_demap_matches_chain(gpu_stream):
    from puschrx.chain import ChainOptions, NativeChain
    grants = [G.Grant(name=f"g{qm}{rank}", rank=rank, qm=qm, num_rb=4 + rank, fft_size=128, code_rate=0.5,
                      padded_subcarriers=128) for qm in (2, 4, 6, 8) for rank in (1, 2, 3, 4)]
    compiled = G.compile_grants(G.Radio(), grants)
    batch = G.GrantBatch(compiled, dict(iq_format=abi.IQ_COMPLEX64, tau_s=100e-9, fd_hz=10.0), use_graph=False)
    iqs = [_iq(ops.Geometry(cfg), 3 + i)[i % 4] for i, (_, cfg, _) in enumerate(compiled)]
    batch.enqueue(batch.pack_iq(iqs))
    opts = ChainOptions(tau_s=100e-9, fd_hz=10.0, iq_format=abi.IQ_COMPLEX64)
    for (_, cfg, plan), lo, iq in zip(compiled, batch.layout, iqs):
        n = cfg.qm * ops.Geometry(cfg).cw_stride
        got = batch.fetch("cw_llr", torch.int16, n, lo.cw_offset)
        chain = NativeChain(cfg, plan, max_slots=1, opts=opts, use_graph=False)
        chain.enqueue(torch.from_numpy(iq[None]).cuda(), 1)
        want = chain.fetch("cw_llr", torch.int16, n)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), want.cpu().numpy()), (cfg.qm, cfg.num_layers)
        chain.close()
    batch.close()
