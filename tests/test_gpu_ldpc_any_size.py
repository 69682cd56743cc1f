"""Decoding of lifting sizes outside 24 << i (hand-made plans; the library's own
plans use 24 .. 384 by powers of two): the decoded bits and iteration counts
bit for bit against the oracle's rate dematch and decoder on the same codeword
LLRs, and the payloads of the device transmitter through a good channel.  Odd
sizes, halves that are no multiple of 4, the smallest and the largest size, two
blocks to a transport block, few and all active rows, repetition."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from oracle_lib import OrTbPlan, load_oracle, ptr
from puschrx import abi, ops
from puschrx import grants as G
from puschrx.synth import ChannelSpec
from puschrx.txgpu import GpuTransmitter, device_channel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

#        PRB, Qm, Z, C
SHAPES = [(4, 4, 25, 1), (4, 4, 36, 1), (4, 4, 45, 1), (4, 4, 72, 1), (4, 6, 100, 1), (4, 6, 120, 1), (6, 6, 45, 2),
          (10, 6, 150, 2), (20, 6, 383, 1), (11, 8, 340, 1), (12, 4, 192, 1)]


def any_size_plan(g, z, c):
    """A plan of c blocks of lifting size z filling one slot of geometry g."""
    kprime = 22 * z - (z // 2 + 3)
    crc_cb, crc_tb = (24 if c > 1 else 0), 16
    p = abi.AiranTbPlanV1(tbs=c * (kprime - crc_cb) - crc_tb, crc_tb=crc_tb, crc_cb=crc_cb, C=c, K=22 * z,
                          Kprime=kprime, Z=z, filler=22 * z - kprime, N=66 * z, Ncb=66 * z, G=g.cw_symbols * g.qm)
    units = p.G // (g.nl * g.qm)
    p.n_low = c - units % c
    p.E_low = g.nl * g.qm * (units // c)
    p.E_high = g.nl * g.qm * (-(-units // c))
    return p


def transmit(cfg, plan, payload, seed, snr_db=40.0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    tx = GpuTransmitter(cfg, plan, payload.shape[0])
    grid = tx.encode(torch.from_numpy(payload).cuda())
    gains, delays = device_channel(gen, cfg, ChannelSpec(taps=8, delay_spread_s=50e-9, doppler_hz=5.0, rx_corr=0.3,
                                                         snr_db=snr_db, sinusoids=8), payload.shape[0])
    iq = tx.channel(grid, gains, delays, snr_db, seed)
    torch.cuda.synchronize()
    tx.close()
    return iq


def oracle_decode(cfg, plan, cw, iterations, early):
    oracle, g = load_oracle(), ops.Geometry(cfg)
    op = OrTbPlan(**{f: getattr(plan, f) for f, _ in OrTbPlan._fields_ if hasattr(plan, f)})
    op.bg = 1
    lam = np.zeros(plan.C * 68 * plan.Z, np.int16)
    oracle.or_rate_dematch(C.byref(op), g.nl, g.qm, g.cw_symbols, g.cw_stride, 1, ptr(np.ascontiguousarray(cw)), ptr(lam))
    rows = ops.ldpc_active_rows(plan)
    bits, it = np.zeros(plan.C * plan.K, np.int8), np.zeros(plan.C, np.uint8)
    oracle.or_ldpc_decode(plan.Z, plan.C, ptr(lam), abi.LDPC_MODE_FP16, iterations, rows, plan.K, 1 if early else 0,
                          ptr(bits), ptr(it))
    return bits, it


@pytest.mark.parametrize("early", [True, False])
def test_ragged_batch(gpu_stream, early):
    rng = np.random.default_rng(11)
    grants = [dataclasses.replace(g, num_rb=prb, rank=1, qm=qm, code_rate=0.5, fft_size=G.fft_for(prb),
                                  padded_subcarriers=None)
              for g, (prb, qm, _, _) in zip(G.config4_grants(rng, len(SHAPES)), SHAPES)]
    compiled = [(rt, cfg, any_size_plan(ops.Geometry(cfg), z, c))
                for (rt, cfg, _), (_, _, z, c) in zip(G.compile_grants(G.Radio(), grants), SHAPES)]
    batch = G.GrantBatch(compiled, dict(iq_format=abi.IQ_COMPLEX64, ldpc_iterations=6, early_stop=early,
                                        tau_s=100e-9, fd_hz=10.0))
    payloads = [rng.integers(0, 2, (1, p.tbs), dtype=np.uint8) for _, _, p in compiled]
    iqs = [transmit(cfg, p, x, i)[0].cpu().numpy() for i, ((_, cfg, p), x) in enumerate(zip(compiled, payloads))]
    iqs[3] = rng.normal(0, 1, iqs[3].shape).astype(np.float32)  # a block that does not converge
    batch.enqueue(batch.pack_iq(iqs))
    tb_ok = batch.fetch("tb_ok", torch.uint8, batch.n)
    iters = batch.fetch("iterations", torch.uint8, batch.num_cb)
    torch.cuda.synchronize()
    tb_ok, iters = tb_ok.cpu().numpy(), iters.cpu().numpy()
    for i, ((_, cfg, p), lo) in enumerate(zip(compiled, batch.layout)):
        g = ops.Geometry(cfg)
        print(f"grant {i}: Z {p.Z}, C {p.C}, {ops.ldpc_active_rows(p)} rows", flush=True)
        cw = batch.fetch("cw_llr", torch.int16, g.qm * g.cw_stride, lo.cw_offset)
        bits = batch.fetch("bits", torch.int8, p.C * p.K, lo.bits_offset)
        torch.cuda.synchronize()
        want, it = oracle_decode(cfg, p, cw.cpu().numpy(), 6, early)
        bits = bits.cpu().numpy()
        assert np.array_equal(bits, want), i
        assert np.array_equal(iters[lo.first_cb: lo.first_cb + p.C], it), i
        got = bits.reshape(p.C, p.K)[:, : p.Kprime - p.crc_cb].reshape(-1)[: p.tbs]
        assert (tb_ok[i] == 1) == np.array_equal(got, payloads[i][0]), i
    assert tb_ok[3] == 0 and tb_ok.sum() >= 7
    batch.close()


@pytest.mark.parametrize("early", [1, 0])
@pytest.mark.parametrize("prb,qm,z", [(6, 2, 72), (11, 2, 120), (6, 4, 144), (10, 6, 360)])
def test_chain(gpu_stream, prb, qm, z, early):
    """Sizes that are a multiple of 24 and few rows: the decoder reads the
    chain's codeword LLRs itself."""
    from puschrx import profiles as P
    from puschrx.chain import ChainOptions, NativeChain
    cfg = P.Profile(name="t", rx=4, rank=1, num_rb=prb, fft=256, qm=qm, code_rate=0.5).config()
    g = ops.Geometry(cfg)
    plan = any_size_plan(g, z, 1)
    rows = ops.ldpc_active_rows(plan)
    print(f"Z {z}, {rows} rows", flush=True)
    assert rows <= 8
    n = 3
    payload = np.random.default_rng(z).integers(0, 2, (n, plan.tbs), dtype=np.uint8)
    iq = transmit(cfg, plan, payload, z, 45.0)
    opts = ChainOptions(tau_s=100e-9, fd_hz=10.0, iq_format=abi.IQ_COMPLEX64, early_stop=early)
    chain = NativeChain(cfg, plan, max_slots=n, opts=opts, use_graph=False)
    chain.enqueue(iq, n)
    cw = chain.fetch("cw_llr", torch.int16, n * qm * g.cw_stride).reshape(n, -1)
    bits = chain.fetch("bits", torch.int8, n * plan.K).reshape(n, -1)
    iters = chain.fetch("iterations", torch.uint8, n)
    tb_ok = chain.fetch("tb_ok", torch.uint8, n)
    torch.cuda.synchronize()
    cw, bits, iters, tb_ok = (x.cpu().numpy() for x in (cw, bits, iters, tb_ok))
    for t in range(n):
        want, it = oracle_decode(cfg, plan, cw[t], opts.ldpc_iterations, bool(early))
        assert np.array_equal(bits[t], want) and iters[t] == it[0], t
        assert (tb_ok[t] == 1) == np.array_equal(bits[t][: plan.tbs], payload[t]), t
    chain.close()
