"""DMRS references whose Gold bits are derived a row at a time, against the
oracle bit for bit: one and a few pilots, the widest row, first resource
blocks up to the end of the carrier and, past the span that is derived from
index 0, with a jump to the first pilot."""
import ctypes as C

import numpy as np
import pytest

from puschrx import abi, ops
from puschrx import profiles as P
from oracle_lib import OracleGeom, cref, ptr

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _generate(cfg, re, im):
    lib = ops.load_library()
    rt = C.c_void_p()
    ops._check("dmrs CreateRuntime", lib.airan_mimo_dmrs_gen_CreateRuntime(C.byref(rt)))
    a = ops._hdr(abi.MimoDmrsGenOpArgsV1, dmrs_re=C.c_void_p(re.data_ptr()), dmrs_im=C.c_void_p(im.data_ptr()),
                 config=C.pointer(cfg), layout=C.pointer(ops.layout(cfg)), stream=C.c_void_p(ops.stream_ptr()))
    try:
        ops._check("dmrs Enqueue", lib.airan_mimo_dmrs_gen_Enqueue(rt, C.byref(a)))
        torch.cuda.synchronize()
    finally:
        lib.airan_mimo_dmrs_gen_DestroyRuntime(rt)


@pytest.mark.parametrize("rb,start", [(1, 0), (1, 274), (11, 100), (273, 2), (275, 0), (20, 900), (273, 911), (275, 60000)])
def test_dmrs_rows_match_oracle(oracle, gpu_stream, rb, start):
    prof = P.Profile(name="t", rx=4, rank=4, num_rb=rb, fft=128 if rb <= 10 else 4096, qm=4, n_scid=1)
    cfg = prof.config(7)
    cfg.rb_start = start
    g = OracleGeom(cfg)
    want = [np.zeros(g.nl * g.ndmrs * g.ref_pad, np.uint16) for _ in range(2)]
    oracle.or_dmrs_gen(cref(cfg), ptr(want[0]), ptr(want[1]))
    n = want[0].size
    for shift in (0, 1):  # 1: rows off 16 bytes, one value at a time
        buf = torch.full((2, n + 8), 77, dtype=torch.int16, device="cuda")
        _generate(cfg, buf[0, shift:], buf[1, shift:])
        for w, x in zip(want, buf.cpu().numpy()):
            assert np.array_equal(x[shift:shift + n].view(np.uint16), w), (rb, start, shift)
            assert np.all(x[:shift] == 77) and np.all(x[shift + n:] == 77)
