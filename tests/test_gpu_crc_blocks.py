"""The CRC check's two kernels against the oracle's remainders: a workgroup
per code block (any K and alignment, few blocks) and the matrix product (from
3000 blocks on), at code block sizes that are and are not multiples of the 16
and 32 positions a thread reads, with and without code-block CRCs, on both
sides of the dispatch."""
import numpy as np
import pytest

from oracle_lib import load_oracle, ptr
from puschrx import abi, ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _blocks(plan, rng):
    """One TB's code blocks [C, K] with both CRCs attached."""
    oracle = load_oracle()
    kind = 0 if plan.crc_tb == 24 else 2
    pay = rng.integers(0, 2, plan.tbs, dtype=np.uint8)
    r = oracle.or_crc(kind, ptr(pay), plan.tbs)
    msg = np.concatenate([pay, [(r >> (plan.crc_tb - 1 - i)) & 1 for i in range(plan.crc_tb)]]).astype(np.uint8)
    per = plan.Kprime - plan.crc_cb
    out = np.zeros((plan.C, plan.K), np.int8)
    for c in range(plan.C):
        seg = np.ascontiguousarray(msg[c * per:(c + 1) * per])
        out[c, :per] = seg
        if plan.crc_cb:
            rb = oracle.or_crc(1, ptr(seg), per)
            out[c, per:per + 24] = [(rb >> (23 - i)) & 1 for i in range(24)]
    return out


@pytest.mark.parametrize("tbs,ntb,offset", [(400, 5, 0), (400, 5, 1), (1000, 3, 0), (3824, 2, 4), (24072, 3, 0),
                                            (24072, 3, 1), (24072, 999, 0), (24072, 1000, 0)])
def test_crc_of_every_block(gpu_stream, tbs, ntb, offset):
    qm, layers = 4, 1
    plan = ops.tb_plan(tbs, 4 * ((tbs // 2) // 4 + 1) * qm * layers, qm, layers)
    rng = np.random.default_rng(tbs + ntb)
    tbs_bits = np.stack([_blocks(plan, rng) for _ in range(min(ntb, 7))])[np.arange(ntb) % 7 % min(ntb, 7)].copy()
    cb_want, tb_want = np.ones((ntb, plan.C), np.uint8), np.ones(ntb, np.uint8)
    # Flip one bit somewhere in every third TB: the first, the last and a
    # random checked position, and one beyond K' that no CRC covers.
    for t in range(0, ntb, 3):
        c = int(rng.integers(plan.C))
        pos = [0, plan.Kprime - 1, int(rng.integers(plan.Kprime)), plan.K - 1][t // 3 % 4]
        tbs_bits[t, c, pos] ^= 1
        if pos < plan.Kprime:
            cb_want[t, c] = 0 if plan.crc_cb else 1
            tb_want[t] = 0 if pos < plan.Kprime - plan.crc_cb else 1
    buf = torch.zeros(tbs_bits.size + offset, dtype=torch.int8, device="cuda")
    buf[offset:] = torch.from_numpy(tbs_bits.reshape(-1)).cuda()
    cb_ok, tb_ok, _ = ops.crc_check(plan, ntb, buf[offset:])
    torch.cuda.synchronize()
    assert np.array_equal(cb_ok.cpu().numpy().reshape(ntb, plan.C), cb_want)
    assert np.array_equal(tb_ok.cpu().numpy(), tb_want)


@pytest.mark.parametrize("z,c,ntb", [(25, 1, 5), (45, 2, 4), (383, 3, 3), (52, 1, 3001)])
def test_crc_of_odd_block_sizes(gpu_stream, z, c, ntb):
    """K = 22 z that is no multiple of 16 (plans made by hand), also at a count
    where blocks of another size would take the matrix product."""
    kprime, crc_cb = 22 * z - 7, 24 if c > 1 else 0
    plan = abi.AiranTbPlanV1(tbs=c * (kprime - crc_cb) - 16, crc_tb=16, crc_cb=crc_cb, C=c, K=22 * z, Kprime=kprime, Z=z)
    rng = np.random.default_rng(z)
    bits = np.repeat(_blocks(plan, rng)[None], ntb, axis=0)
    cb_want, tb_want = np.ones((ntb, c), np.uint8), np.ones(ntb, np.uint8)
    for t in range(0, ntb, 2):  # one checked payload bit of every other TB
        r = int(rng.integers(c))
        bits[t, r, int(rng.integers(kprime - crc_cb))] ^= 1
        cb_want[t, r], tb_want[t] = 1 if c == 1 else 0, 0
    cb_ok, tb_ok, _ = ops.crc_check(plan, ntb, torch.from_numpy(bits.reshape(-1)).cuda())
    torch.cuda.synchronize()
    assert np.array_equal(cb_ok.cpu().numpy().reshape(ntb, c), cb_want)
    assert np.array_equal(tb_ok.cpu().numpy(), tb_want)
