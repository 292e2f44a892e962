"""GPU parity of the streaming kernels at 17..32 rows on both sides of the
grid size (two workgroups per CU) where they change from three stages to two,
with one step, fewer steps than stages and an odd number of them: against the
CPU oracle (the bound of tests/test_gemm_gpu.py), and bit for bit against the
launch without a pair table, which loads the same plan's scales as windows."""

from __future__ import annotations

import pytest

from tests.conftest import from_dev
from tests.test_gemm_gpu import _case, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,Ns,gs,dtype", [
    (17, 512, (64,), 64, "bf16"), (32, 1024, (4,), 128, "f16"), (31, 1536, (200, 72), 64, "f16"),
    (32, 2560, (320, 64, 132), 64, "bf16"), (17, 12288, (256,), 128, "bf16"),
    (32, 512, (32768,), 64, "bf16"), (18, 512, (32772,), 64, "bf16"),
    (32, 1024, (16384, 16384), 128, "bf16"), (32, 1024, (16384, 16448), 128, "f16"),
])
def test_stages(dev, M, K, Ns, gs, dtype):
    import ctypes

    import torch

    from dflash_mlx_amd import _lib, _runtime, verify_qmm as vq

    lib = _lib.load()
    cases, mats, x = [], [], None
    for i, N in enumerate(Ns):
        case, (xi, w, s, b) = _case(dev, M, K, N, gs, 4, dtype, seed=60 + i)
        x, cx = (xi, case[0]) if x is None else (x, cx)
        cases.append((cx,) + case[1:])
        mats.append((w, s, b))
    n = len(mats)
    got = (vq.quantized_matmul_multi(x, mats, group_size=gs, bits=4) if n > 1 else
           [vq.quantized_matmul(x, *mats[0], group_size=gs, bits=4)])
    for y, case in zip(got, cases):
        _check(from_dev(y, dtype), case, gs, 4, dtype)
    plain = [torch.full_like(y, float("nan")) for y in got]
    segs = (_lib.QmmSegment * n)()
    for g, (w, s, b), y in zip(segs, mats, plain):
        g.w_q, g.scales, g.biases = w.data_ptr(), s.data_ptr(), b.data_ptr()
        g.y, g.N = y.data_ptr(), int(w.shape[0])
    need = int(lib.dfmi_qmm_multi_workspace_bytes(
        M, K, (ctypes.c_int64 * n)(*Ns), n, gs, 4))
    ws, ws_bytes = _runtime.workspace(x.device, need) if need else (0, 0)
    rc = lib.dfmi_qmm_affine_multi(x.data_ptr(), _runtime.dtype_code(x.dtype), segs, n, M, K, gs,
                                   4, ws, ws_bytes, _runtime.stream_ptr(x.device))
    assert rc == _lib.DFMI_OK, lib.dfmi_last_error()
    assert all(torch.equal(a, b) for a, b in zip(got, plain))
