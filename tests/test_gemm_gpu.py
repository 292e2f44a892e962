"""GPU parity of ``qmm_gemm_kernel`` (more than 32 activation rows) against the
CPU oracle at the edges of its tiles: 32-, 64- and 96-row blocks, 128- and
256-column blocks, 128-k steps with a remainder, one and several K splits.

Bound per output: one rounding to the output type (half an ulp: 2^-8 relative
in bf16, 2^-11 in f16) plus the fp32 sum's worst case, K 2^-24 of the sum of
the terms' magnitudes |x| (|q s| + |b|)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle
from tests.conftest import from_dev, make_qmm_case, to_dev

pytestmark = pytest.mark.gpu


def _case(dev, M, K, N, gs, bits, dtype, seed):
    x, w_q, s, b = make_qmm_case(M, K, N, gs, dtype=dtype, seed=seed, bits=bits)
    ten = (to_dev(x, dtype, dev), to_dev(w_q, "u32", dev), to_dev(s, dtype, dev),
           to_dev(b, dtype, dev))
    return (x, w_q, s, b), ten


def _check(got, case, gs, bits, dtype):
    x, w_q, s, b = case
    ref = oracle.quantized_matmul(x, w_q, s, b, group_size=gs, bits=bits, dtype=dtype)
    xf, sf, bf = (oracle.to_f32(a, dtype).astype(np.float64) for a in (x, s, b))
    q = oracle.qmm.unpack(w_q, bits).astype(np.float64)
    mag = np.abs(xf) @ (q * np.repeat(np.abs(sf), gs, 1) + np.repeat(np.abs(bf), gs, 1)).T
    g = oracle.to_f32(got, dtype).astype(np.float64)
    bound = (2.0 ** -8 if dtype == "bf16" else 2.0 ** -11) * np.abs(ref) + \
        x.shape[1] * 2.0 ** -24 * mag
    assert np.all(np.abs(g - ref) <= bound), float((np.abs(g - ref) / bound).max())


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,K,N,gs", [
    (33, 32, 1, 32), (33, 64, 4, 64), (64, 128, 127, 128), (65, 160, 128, 32),
    (77, 192, 129, 64), (96, 1088, 260, 64), (97, 1152, 1000, 128), (129, 320, 256, 32),
    (200, 576, 2501, 64), (65, 4096, 300, 64),
])
def test_tile_edges(dev, M, K, N, gs, bits, dtype):
    from dflash_mlx_amd import _lib, verify_qmm as vq

    assert _lib.load().dfmi_qmm_kernel_name(M, K, N, gs, bits, None) == b"qmm_gemm_kernel"
    case, (x, w, s, b) = _case(dev, M, K, N, gs, bits, dtype, seed=M + K + N + bits)
    y = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    _check(from_dev(y, dtype), case, gs, bits, dtype)
    again = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    assert np.array_equal(from_dev(y, dtype), from_dev(again, dtype))


def test_tables_and_workspaces(dev):
    """The same bits with the matrix's own table, a column slice of a wider
    one and the table the call builds in its workspace; within the bound
    without a workspace (general kernel), with one too small for a K split,
    and into an output that starts off a 16-byte boundary."""
    import torch

    from dflash_mlx_amd import _lib, _runtime

    lib = _lib.load()
    M, K, N, gs = 77, 2048, 520, 64
    case, (x, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=5)
    need = int(lib.dfmi_qmm_workspace_bytes(M, K, N, gs, 4))
    ws = torch.zeros(need + 256, dtype=torch.uint8, device=dev)
    own = _runtime.build_sb_pairs(s, b)
    wide = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // gs, N + 136), dtype=torch.int32, device=dev)
    wide[:, 128:128 + N] = own
    out = torch.empty(M * N + 8, dtype=torch.bfloat16, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)

    def run(pairs, stride, wsb, shift=0):
        out.fill_(float("nan"))
        y = out[shift:shift + M * N]
        ptr, args = y.data_ptr(), (M, K, N, gs, 4, ws.data_ptr() if wsb else None, wsb)
        if stride:
            rc = lib.dfmi_qmm_affine_pairs_strided(
                x.data_ptr(), _lib.DFMI_BF16, w.data_ptr(), s.data_ptr(), b.data_ptr(),
                pairs.data_ptr(), stride, ptr, *args, st)
        else:
            rc = lib.dfmi_qmm_affine_pairs(
                x.data_ptr(), _lib.DFMI_BF16, w.data_ptr(), s.data_ptr(), b.data_ptr(),
                pairs.data_ptr() if pairs is not None else None, ptr, *args, None, st)
        assert rc == _lib.DFMI_OK, lib.dfmi_last_error()
        torch.cuda.synchronize()
        return from_dev(y.clone().reshape(M, N), "bf16")

    ref = run(own, 0, need)
    _check(ref, case, gs, 4, "bf16")
    assert np.array_equal(run(wide[:, 128:128 + N], N + 136, need), ref)
    assert np.array_equal(run(None, 0, need), ref)
    assert np.array_equal(run(own, 0, need, shift=1), ref)
    for pairs, wsb in ((own, 0), (None, 0), (own, 65536 + 4096), (None, 65536 + 4096)):
        _check(run(pairs, 0, wsb), case, gs, 4, "bf16")
    assert not ws[:65536].any()  # the counters' region is left as it was


def test_rows_with_infinities_stay_apart(dev):
    """A row holding infinities or NaN changes no other row."""
    import torch

    from dflash_mlx_amd import verify_qmm as vq

    M, K, N, gs = 70, 448, 256, 64
    _, (x, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=9)
    ref = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=4)
    x[11, 5], x[40, 447], x[69, 0] = float("inf"), float("nan"), -float("inf")
    got = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=4)
    rows = [r for r in range(M) if r not in (11, 40, 69)]
    assert torch.equal(got[rows], ref[rows])
    assert not torch.isfinite(got[[11, 40, 69]]).any()


def test_module_many_rows(dev):
    """A verify module's many-row call equals the stock operator bit for bit,
    alone and as a sibling, also after its scales change in place."""
    import torch
    from torch import nn

    from dflash_mlx_amd import verify_linear as vl, verify_qmm as vq

    K, gs, M = 512, 64, 45
    root = nn.Module()
    root.mlp = nn.Module()
    x = None
    for i, (name, N) in enumerate((("gate_proj", 384), ("up_proj", 640), ("down_proj", 256))):
        _, (xi, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=20 + i)
        x = xi if x is None else x
        setattr(root.mlp, name, vl.QuantizedLinear(w, s, b, group_size=gs, bits=4))
    vl.install_verify_linears(root, enable_qmm=True)
    for change in (False, True):
        for name in ("gate_proj", "up_proj", "down_proj"):
            m = getattr(root.mlp, name)
            if change:
                m.scales.mul_(1.5)
            want = vq.quantized_matmul(x, m.weight, m.scales, m.biases, group_size=gs, bits=4)
            assert torch.equal(m(x), want), name
