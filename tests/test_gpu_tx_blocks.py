"""The device encoder's code blocks at the edges of its packing, against the
host transmitter bit for bit: lifting sizes below, at and off a multiple of
32, a transport block below one word, repetition (more bits sent than the
buffer holds), every redundancy version, filler, TB CRC bits in two words,
every modulation and layer count, and code blocks that end inside a slot."""
import numpy as np
import pytest

from puschrx import ops, synth
from puschrx import profiles as P
from puschrx.txgpu import GpuTransmitter

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# PRBs, layers, Qm, TB bits (None: from the rate), rate, slots per TB, rv
CASES = [
    (1, 1, 2, 24, None, 1, 0),       # smallest TB, wraps many times
    (1, 2, 4, None, 0.4, 1, 3),
    (3, 3, 6, None, 0.7, 1, 1),
    (6, 4, 8, None, 0.9, 1, 0),
    (11, 3, 8, None, 0.55, 1, 2),
    (24, 2, 2, None, 0.12, 1, 0),    # low rate: all 46 rows
    (24, 4, 6, None, 0.33, 3, 2),    # several slots to a TB
    (52, 1, 4, None, 0.95, 1, 0),
    (106, 3, 8, None, 0.8, 2, 0),    # many code blocks over two slots
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}prb_l{c[1]}_qm{c[2]}_T{c[5]}_rv{c[6]}")
def test_encoder_blocks_match_host(gpu_stream, case):
    rb, rank, qm, tbs, rate, T, rv = case
    fft = 128 if 12 * rb <= 128 else (512 if 12 * rb <= 384 else 2048)
    prof = P.Profile(name="t", rx=4, rank=rank, num_rb=rb, fft=fft, qm=qm)
    cfg = prof.config()
    g = ops.Geometry(cfg)
    if tbs is None:
        tbs = ops.tbs(rb, 12 * g.ndata * T, qm, rank, rate)
    plan = ops.tb_plan(tbs, T * g.cw_symbols * qm, qm, rank, rv)
    n = 2
    payload = synth.random_payload(np.random.default_rng(rb + qm), n, plan.tbs)
    want_grid, want_coded = synth.tx_grid(cfg, plan, payload, slots_per_tb=T, want_coded=True)
    print(f"TB of {plan.tbs} bits, C = {plan.C}, Z = {plan.Z}, filler {plan.filler}", flush=True)
    tx = GpuTransmitter(cfg, plan, max_tbs=n, slots_per_tb=T)
    # An odd start address: payload bytes are read 16 at a time.
    buf = torch.zeros(payload.size + 3, dtype=torch.uint8, device="cuda")
    dev = buf[3:].view(n, plan.tbs)
    dev.copy_(torch.from_numpy(payload))
    grid, coded = tx.encode(dev, want_coded=True)
    torch.cuda.synchronize()
    tx.close()
    assert np.array_equal(coded.cpu().numpy(), want_coded)
    assert np.array_equal(grid.cpu().numpy().view(np.uint32), want_grid.view(np.uint32))
