"""The decoder kernel of one code block per workgroup (Z = 384, REF mode, more
than 8 active rows, unaligned buffers) bit for bit against the oracle where it can go
wrong: every lifting size (the halves of 12 .. 192 words), the row counts at
which its unrolled rows, its two register arrays and its kernels end, buffers
of any alignment, a K that is no multiple of 4, and int16 inputs large enough
for REF mode's growing posteriors to reach infinity and NaN."""
import numpy as np
import pytest

from oracle_lib import load_oracle, ptr
from puschrx import abi, ops

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _check(lam, n, z, k, iters, rows, mode, early, offset=0, want_lam=True):
    oracle = load_oracle()
    ref = lam.copy()
    bits, it = np.zeros(n * k, np.int8), np.zeros(n, np.uint8)
    oracle.or_ldpc_decode(z, n, ptr(ref), mode, iters, rows, k, 1 if early else 0, ptr(bits), ptr(it))
    dev = torch.zeros(lam.size + offset, dtype=torch.int16, device="cuda")
    dev[offset:] = torch.from_numpy(lam).cuda()
    got, lam_out, git = ops.ldpc_decode(dev[offset:], n, z, k, iters, rows, mode, early, want_lam=want_lam)
    torch.cuda.synchronize()
    assert np.array_equal(git.cpu().numpy(), it)
    assert np.array_equal(got.cpu().numpy(), bits)
    if want_lam:
        assert np.array_equal(lam_out.cpu().numpy(), ref)


def _llrs(z, n, rows, ebno, seed):
    oracle, rng = load_oracle(), np.random.default_rng(seed)
    out = np.zeros((n, 68 * z), np.int16)
    var = 1.0 / (2.0 * 22 / (20 + rows) * 10 ** (0.1 * ebno))
    for row in out:
        info, cw = rng.integers(0, 2, 22 * z, dtype=np.uint8), np.zeros(68 * z, np.uint8)
        oracle.or_ldpc_encode(z, ptr(info), ptr(cw))
        y = 1.0 - 2.0 * cw + rng.normal(0, np.sqrt(var), cw.size)
        row[:] = np.clip(np.rint(2 * y / var * 256), -5120, 5120)
        row[: 2 * z] = 0
        row[(22 + rows) * z:] = 0
    return out.reshape(-1)


@pytest.mark.parametrize("mode", [abi.LDPC_MODE_REF, abi.LDPC_MODE_FP16])
@pytest.mark.parametrize("z,rows", [(24, 46), (48, 12), (96, 9), (192, 43), (384, 4), (384, 9), (384, 10), (384, 11),
                                    (384, 41), (384, 42), (384, 43)])
def test_rows_and_lifting_sizes(gpu_stream, mode, z, rows):
    for early, ebno in ((True, 3.0), (False, 1.0)):
        _check(_llrs(z, 5, rows, ebno, z + rows), 5, z, 22 * z, 6, rows, mode, early)


@pytest.mark.parametrize("offset", [1, 2])
@pytest.mark.parametrize("rows", [6, 17])
def test_alignment_and_odd_k(gpu_stream, offset, rows):
    z = 384
    _check(_llrs(z, 3, rows, 3.0, 5), 3, z, 22 * z - 3, 5, rows, abi.LDPC_MODE_FP16, True, offset=offset)


@pytest.mark.parametrize("mode", [abi.LDPC_MODE_REF, abi.LDPC_MODE_FP16])
@pytest.mark.parametrize("rows", [9, 46])
def test_full_range_inputs(gpu_stream, mode, rows):
    """Bits and iterations only: the clamped posterior of a NaN is no number."""
    rng = np.random.default_rng(rows)
    lam = rng.integers(-32768, 32768, (4, 68 * 96)).astype(np.int16)
    lam[3] = np.where(rng.integers(0, 2, 68 * 96), 32767, -32768)
    _check(lam.reshape(-1), 4, 96, 22 * 96, 20, rows, mode, True, want_lam=False)


@pytest.mark.parametrize("rows", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("n,early", [(3, True), (300, False), (300, True), (520, False)])
def test_few_rows_at_every_dispatch(gpu_stream, rows, n, early):
    """Z = 384 and at most 8 rows: one block per workgroup, or two between one
    and two blocks a compute unit without early stop.  Three distinct blocks,
    repeated: every repetition decodes alike."""
    z, k = 384, 22 * 384
    lam = _llrs(z, 3, rows, 4.0, rows)
    oracle = load_oracle()
    ref = lam.copy()
    bits, it = np.zeros(3 * k, np.int8), np.zeros(3, np.uint8)
    oracle.or_ldpc_decode(z, 3, ptr(ref), abi.LDPC_MODE_FP16, 4, rows, k, 1 if early else 0, ptr(bits), ptr(it))
    reps = -(-n // 3)
    dev = torch.from_numpy(np.tile(lam.reshape(3, -1), (reps, 1))[:n].copy()).cuda().reshape(-1)
    got, lam_out, git = ops.ldpc_decode(dev, n, z, k, 4, rows, abi.LDPC_MODE_FP16, early, want_lam=True)
    torch.cuda.synchronize()
    tile = lambda a: np.tile(a.reshape(3, -1), (reps, 1))[:n]  # noqa: E731
    assert np.array_equal(git.cpu().numpy(), tile(it).reshape(-1))
    assert np.array_equal(got.cpu().numpy().reshape(n, -1), tile(bits))
    assert np.array_equal(lam_out.cpu().numpy().reshape(n, -1), tile(ref))


@pytest.mark.parametrize("mode", [abi.LDPC_MODE_REF, abi.LDPC_MODE_FP16])
@pytest.mark.parametrize("z,rows,n", [(24, 46, 520), (48, 11, 520), (96, 43, 520), (24, 10, 1040), (96, 9, 1040)])
def test_many_small_blocks(gpu_stream, mode, z, rows, n):
    """Z <= 96 and more blocks than are resident at once with 192 lanes each:
    one wave per block, whose lanes are fewer than the columns' runs."""
    k = 22 * z - 2
    lam = _llrs(z, 3, rows, 3.0, z + rows)
    oracle = load_oracle()
    ref = lam.copy()
    bits, it = np.zeros(3 * k, np.int8), np.zeros(3, np.uint8)
    oracle.or_ldpc_decode(z, 3, ptr(ref), mode, 6, rows, k, 1, ptr(bits), ptr(it))
    tile = lambda a: np.tile(a.reshape(3, -1), (-(-n // 3), 1))[:n]  # noqa: E731
    for offset in (0, 1):
        dev = torch.zeros(n * 68 * z + offset, dtype=torch.int16, device="cuda")
        dev[offset:] = torch.from_numpy(tile(lam).reshape(-1).copy()).cuda()
        got, lam_out, git = ops.ldpc_decode(dev[offset:], n, z, k, 6, rows, mode, True, want_lam=True)
        torch.cuda.synchronize()
        assert np.array_equal(git.cpu().numpy(), tile(it).reshape(-1))
        assert np.array_equal(got.cpu().numpy().reshape(n, -1), tile(bits))
        assert np.array_equal(lam_out.cpu().numpy().reshape(n, -1), tile(ref))


@pytest.mark.parametrize("rank,qm,rate", [(4, 8, 0.85), (3, 6, 0.91), (2, 4, 0.93), (1, 8, 0.8)])
def test_chain_blocks_match_operators(gpu_stream, rank, qm, rate):
    """The decoder reading a chain's codeword LLRs itself against rate dematch
    + decoder as operators."""
    from puschrx import profiles as P
    from puschrx.chain import ChainOptions, NativeChain
    prof = P.Profile(name="t", rx=4, rank=rank, num_rb=51, fft=1024, qm=qm, code_rate=rate)
    cfg = prof.config()
    g = ops.Geometry(cfg)
    tbs = ops.tbs(51, 12 * g.ndata, qm, rank, rate)
    plan = ops.tb_plan(tbs, g.cw_symbols * qm, qm, rank)
    assert plan.Z == 384 and ops.ldpc_active_rows(plan) <= 8  # the fused decoder's shape
    n = 3
    rng = np.random.default_rng(rank)
    iq = torch.from_numpy(rng.normal(0, 1, (n, g.nr, g.samples, 2)).astype(np.float32)).cuda()
    for early in (1, 0):
        opts = ChainOptions(tau_s=100e-9, fd_hz=10.0, iq_format=abi.IQ_COMPLEX64, early_stop=early)
        chain = NativeChain(cfg, plan, max_slots=n, opts=opts, use_graph=False)
        chain.enqueue(iq, n)
        cw = chain.fetch("cw_llr", torch.int16, n * qm * g.cw_stride).reshape(n, -1)
        bits = chain.fetch("bits", torch.int8, 3 * plan.C * plan.K).cpu().numpy().reshape(3, -1)
        torch.cuda.synchronize()
        for t in range(3):
            lam = ops.rate_dematch(cfg, cw[t].contiguous(), 1, plan)
            want, _, _ = ops.ldpc_decode(lam, plan.C, plan.Z, plan.K, opts.ldpc_iterations, ops.ldpc_active_rows(plan),
                                         abi.LDPC_MODE_FP16, bool(early))
            torch.cuda.synchronize()
            assert np.array_equal(bits[t], want.cpu().numpy()), t
        chain.close()
