"""The chain holds no decoder workspace: its decoder keeps the message state in
registers, so a transport block more costs less than the workspace and input
of a separate decoder call for it."""
import pytest

from puschrx import abi, ops
from puschrx import profiles as P

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [abi.LDPC_MODE_REF, abi.LDPC_MODE_FP16])
def test_no_decoder_workspace(gpu_stream, mode):
    from puschrx.chain import ChainOptions, NativeChain
    cfg = P.Profile(name="t", rx=1, rank=1, num_rb=52, fft=1024, qm=8, code_rate=0.5).config()
    g = ops.Geometry(cfg)
    plan = ops.tb_plan(ops.tbs(52, 12 * g.ndata, 8, 1, 0.35), g.cw_symbols * 8, 8, 1)
    rows = ops.ldpc_active_rows(plan)
    assert plan.Z == 384 and rows > 8
    held = []
    for slots in (1, 9):
        chain = NativeChain(cfg, plan, max_slots=slots, use_graph=False,
                            opts=ChainOptions(receiver=abi.CHAIN_RX_LS_ZF, ldpc_mode=mode))
        held.append(chain.device_bytes())
        chain.close()
    per_tb = (held[1] - held[0]) // 8
    workspace = abi.load_library().airan_ldpc_decode_WorkspaceBytes(plan.C, plan.Z, rows)
    print(f"{per_tb} bytes a transport block, workspace {workspace}", flush=True)
    assert per_tb < workspace + plan.C * 68 * plan.Z * 2
