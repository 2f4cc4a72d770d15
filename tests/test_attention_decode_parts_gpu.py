"""GPU parity of decode attention whose parts the last workgroup of a head puts together (attention_decode.hip, arrive.h): key counts
at the edges of parts of 128 and of 256 keys, and workspaces of any content.  Bars as in test_attention_gpu.py."""
import numpy as np
import pytest
import torch

from oracle import oracle
from tests.util import NAME, TOL, as_f64, assert_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=lambda d: NAME[d])
@pytest.mark.parametrize("B,H,Sq,Skv,D", [(1, 3, 1, 512, 64), (2, 2, 16, 640, 128), (1, 2, 3, 1024, 64), (1, 2, 2, 1025, 64), (1, 1, 5, 2304, 128), (1, 1, 1, 16384, 64),
                                         (1, 2, 16, 8192, 128), (1, 1, 13, 16384, 64), (1, 5, 7, 4000, 128), (1, 3, 9, 1100, 64)],
                         ids=lambda v: str(v))
def test_parts_and_workspace_of_any_content(lib, B, H, Sq, Skv, D, dtype):
    from metalhlo_amd import kernels
    rng = np.random.default_rng(Skv)
    q, k, v = (to_dev(rng.standard_normal((B, H, n, D)), dtype) for n in (Sq, Skv, Skv))
    code = kernels.DTYPE_CODE[dtype]
    need = lib.mhip_flash_attention_workspace(B, H, Sq, Skv, D, 0, code)
    assert need > 0
    exp = oracle.attention(as_f64(q), as_f64(k), as_f64(v))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    want = None
    for fill in (0, 255, 128, None, None):
        if fill is not None:
            ws.fill_(fill)
        o = torch.full_like(q, float("nan"))
        assert lib.mhip_flash_attention_ws(torch.cuda.current_stream().cuda_stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, o.data_ptr(), B, H, Sq, Skv, D,
                                           D ** -0.5, 0, 0, 0, code, None, ws.data_ptr(), need) == 0
        assert_close(o, exp, TOL[dtype], f"parts {(B, H, Sq, Skv, D)}")
        want = o if want is None else want
        assert torch.equal(o, want), fill
