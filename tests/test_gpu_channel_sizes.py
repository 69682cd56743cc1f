"""The device channel at every transform size, tap count and layer count at
which its work split changes, against numpy in 64 bits on the same gains:
transforms of 128 .. 4096 points (the last passes have radix 8, 16, 2, 4, 8,
16), 1 .. 32 taps (two halves of 16 to a wave), delays up to a cyclic prefix,
a grid as wide as its transform allows.

Bound: a sample is a sum of 16 to 4096 products in fp32, each rounded at
2^-24; the passes and the tap sums put some 30 roundings of independent sign
behind each other, 2^-24 sqrt(30) = 3.3e-7 (-129.7 dB).  Twice that: -123 dB."""
import numpy as np
import pytest

from puschrx import abi, ops, synth
from puschrx import profiles as P
from puschrx.txgpu import GpuTransmitter

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fft,rb,rank,taps", [(128, 1, 1, 1), (128, 10, 4, 17), (256, 21, 3, 16), (512, 42, 2, 32),
                                              (1024, 20, 4, 5), (1024, 85, 1, 24), (2048, 106, 3, 15), (2048, 170, 4, 32),
                                              (4096, 275, 4, 32), (4096, 25, 2, 2)])
def test_channel_sizes_match_numpy(gpu_stream, fft, rb, rank, taps):
    prof = P.Profile(name="t", rx=4, rank=rank, num_rb=rb, fft=fft, qm=4, padded_subcarriers=12 * rb + (-12 * rb) % 4)
    cfg = prof.config()
    g = ops.Geometry(cfg)
    plan = ops.tb_plan(ops.tbs(rb, 12 * g.ndata, 4, rank, 0.5), g.cw_symbols * 4, 4, rank)
    rng = np.random.default_rng(fft + taps)
    S = 2
    cplx = lambda *s: (rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)  # noqa: E731
    grid, gains = cplx(S, g.nl, 14, g.used), cplx(S, g.nr, g.nl, taps, 14) / np.float32(np.sqrt(taps))
    delays = rng.uniform(0, g.cp_short / (30e3 * fft), (S, taps)).astype(np.float32)
    tx = GpuTransmitter(cfg, plan, max_tbs=S)
    iq = tx.channel(*(torch.from_numpy(x).cuda() for x in (grid, gains.astype(np.complex64), delays)), float("inf"),
                    seed=1, iq_format=abi.IQ_COMPLEX64)
    torch.cuda.synchronize()
    tx.close()
    got = iq.cpu().numpy().astype(np.float64)
    freqs = (np.arange(g.used) - g.used // 2) * 30e3
    for s in range(S):
        steer = np.exp(-2j * np.pi * freqs[None, :] * delays[s].astype(np.float64)[:, None])
        H = np.einsum("rltk,tu->rlku", gains[s].astype(np.complex128), steer)
        y = np.einsum("rlku,lku->rku", H, grid[s].astype(np.complex128))
        bins = np.zeros((g.nr, 14, fft), np.complex128)
        bins[:, :, (np.arange(g.used) - g.used // 2) % fft] = y
        t = np.fft.ifft(bins, axis=-1) * np.sqrt(fft)
        want = np.concatenate([np.concatenate([t[:, k, fft - cp:], t[:, k]], axis=-1)
                               for k, cp in enumerate([g.cp_long] + 13 * [g.cp_short])], axis=-1)
        have = got[s, ..., 0] + 1j * got[s, ..., 1]
        assert have.shape == want.shape
        nmse = 10 * np.log10(np.sum(np.abs(have - want) ** 2) / np.sum(np.abs(want) ** 2))
        print(f"fft {fft} rb {rb} rank {rank} taps {taps}: {nmse:.1f} dB", flush=True)
        assert nmse <= -123.0
