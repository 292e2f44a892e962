"""GPU parity of ``qmm_gemm_kernel`` (more than 32 activation rows; small
products with K up to 4096 stay on the general kernels).  The shapes of few
rows and columns, against the CPU oracle, are planned on its 32 x 128 tile;
``test_every_tile`` takes each of the three tiles (32 x 128, 96 x 128, 64 x
256), with one and several K splits, ragged rows, columns and K, against
float64 sums, and checks which tile the plan took.

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
    (33, 4128, 1, 32), (33, 4160, 4, 64), (64, 4224, 127, 128), (65, 4256, 128, 32),
    (77, 4288, 129, 64), (96, 5184, 260, 64), (97, 5248, 1000, 128), (129, 4416, 256, 32),
    (200, 4672, 2501, 64), (65, 8192, 300, 64),
])
def test_tile_edges(dev, M, K, N, gs, bits, dtype):
    from dflash_mlx_amd import _lib, verify_qmm as vq

    assert _lib.load().dfmi_qmm_kernel_name(M, K, N, gs, bits, None) == b"qmm_gemm_kernel"
    case, (x, w, s, b) = _case(dev, M, K, N, gs, bits, dtype, seed=M + K + N + bits)
    y = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    _check(from_dev(y, dtype), case, gs, bits, dtype)
    again = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    assert np.array_equal(from_dev(y, dtype), from_dev(again, dtype))


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("M,K,N,gs", [
    (33, 32, 1, 32), (33, 64, 4, 64), (64, 128, 127, 128), (77, 192, 129, 64), (97, 1152, 1000, 128),
    (333, 4096, 40, 64), (64, 4096, 1024, 64), (64, 4096, 1028, 64), (256, 512, 2048, 32),
])
def test_small_products_on_the_general_kernels(dev, M, K, N, gs, bits, dtype):
    """Up to the line of the dispatch, and past it at 8 bits: one launch without
    a workspace, the bits of the forced general plan."""
    import torch

    from dflash_mlx_amd import _lib, verify_qmm as vq

    lib, rows = _lib.load(), -(-M // 16) * 16 if bits == 8 else -(-M // 32) * 32
    small = rows * K * N <= (1 << 28 if bits == 8 else 1 << 29)
    name = lib.dfmi_qmm_kernel_name(M, K, N, gs, bits, None)
    assert (name != b"qmm_gemm_kernel") == small
    assert (lib.dfmi_qmm_workspace_bytes(M, K, N, gs, bits) == 0) == small
    case, (x, w, s, b) = _case(dev, M, K, N, gs, bits, dtype, seed=M + K + N + bits)
    y = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits)
    _check(from_dev(y, dtype), case, gs, bits, dtype)
    if small:
        assert torch.equal(y, vq.quantized_matmul(x, w, s, b, group_size=gs, bits=bits,
                                                  tuning=_lib.QmmTuning(1, 0, 0, 0)))


def _plan(M, K, Ns, gs, bits):
    from dflash_mlx_amd import _lib

    ns, out = (ctypes.c_int64 * len(Ns))(*Ns), [ctypes.c_int() for _ in range(3)]
    rc = _lib.load().dfmi_qmm_gemm_plan(M, K, ns, len(Ns), gs, bits,
                                        *[ctypes.byref(v) for v in out])
    assert rc == _lib.DFMI_OK
    return tuple(v.value for v in out)


def _random_weights(dev, gen, N, K, gs, bits, dt):
    """Any codes; scales and biases of a weight of about 0.02."""
    import torch

    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K * bits // 32), generator=gen, device=dev,
                      dtype=torch.int32)
    s = (torch.rand((N, K // gs), generator=gen, device=dev) + 0.5) * (0.08 / 2 ** bits)
    b = (torch.rand((N, K // gs), generator=gen, device=dev) - 1.5) * 0.04
    return w, s.to(dt), b.to(dt)


def _within(y, x, mat, gs, bits):
    """y against float64 sums, by blocks of columns, to the bound above."""
    import torch

    w, s, b = mat
    K, half = x.shape[1], 2.0 ** (-8 if y.dtype == torch.bfloat16 else -11)
    shifts = torch.arange(32 // bits, device=w.device, dtype=torch.int32) * bits
    for n in range(0, w.shape[0], 4096):
        q = ((w[n:n + 4096, :, None] >> shifts) & (2 ** bits - 1)).reshape(-1, K).double()
        sd, bd = (a[n:n + 4096].double().repeat_interleave(gs, 1) for a in (s, b))
        ref = x.double() @ (q * sd + bd).T
        mag = x.double().abs() @ (q * sd.abs() + bd.abs()).T
        bound = half * ref.abs() + K * 2.0 ** -24 * mag
        assert bool(((y[:, n:n + 4096].double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("tile,split,M,K,Ns", [
    ((32, 128), False, 1000, 576, (1000,)), ((32, 128), False, 97, 1088, (4100,)),
    ((32, 128), True, 65, 4288, (136,)), ((32, 128), True, 500, 4160, (644, 4, 640)),
    ((64, 256), False, 103, 320, (16388,)), ((64, 256), False, 1000, 320, (2504,)),
    ((64, 256), False, 1000, 576, (2501,)), ((64, 256), True, 97, 2112, (8200,)),
    ((64, 256), True, 500, 4160, (1284,)), ((64, 256), False, 1000, 192, (1028, 4, 1480)),
    ((96, 128), False, 229, 192, (16388,)), ((96, 128), False, 500, 192, (8200,)),
    ((96, 128), True, 77, 4160, (12296,)), ((96, 128), True, 65, 4160, (6148, 4, 6148)),
])
def test_every_tile(dev, tile, split, M, K, Ns, gs, bits, dtype):
    import torch

    from dflash_mlx_amd import verify_qmm as vq

    # the same steps of 128 at every group size: K - 32, K and K + 64
    K += {32: -32, 64: 0, 128: -K % 128}[gs]
    rows, cols, kp = _plan(M, K, Ns, gs, bits)
    assert (rows, cols) == tile and (kp > 1) == split
    print(f"case: {M} x {K} x {Ns} gs {gs} {bits}-bit {dtype}", flush=True)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    gen = torch.Generator(device=dev)
    gen.manual_seed(M + K + gs + bits)
    x = torch.randn((M, K), generator=gen, device=dev).to(dt)
    mats = [_random_weights(dev, gen, N, K, gs, bits, dt) for N in Ns]
    if len(Ns) > 1:
        ys = vq.quantized_matmul_multi(x, mats, group_size=gs, bits=bits)
    else:
        ys = [vq.quantized_matmul(x, *mats[0], group_size=gs, bits=bits)]
    for y, mat in zip(ys, mats):
        _within(y, x, mat, gs, bits)


def test_tables_and_workspaces(dev):
    """The same bits with the matrix's own table, a column slice of a wider
    one and the table the call builds in its workspace; within the bound
    without a workspace (general kernel), with one too small for a K split,
    and into an output that starts off a 16-byte boundary."""
    import torch

    from dflash_mlx_amd import _lib, _runtime

    lib = _lib.load()
    M, K, N, gs = 77, 6144, 520, 64
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

    M, K, N, gs = 70, 4544, 256, 64
    _, (x, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=9)
    ref = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=4)
    x[11, 5], x[40, 4543], x[69, 0] = float("inf"), float("nan"), -float("inf")
    got = vq.quantized_matmul(x, w, s, b, group_size=gs, bits=4)
    rows = [r for r in range(M) if r not in (11, 40, 69)]
    assert torch.equal(got[rows], ref[rows])
    assert not torch.isfinite(got[[11, 40, 69]]).any()


@pytest.mark.parametrize("M,K,Ns,gs,bits,dtype", [
    (33, 64, (4, 260, 4), 32, 4, "bf16"), (77, 800, (4, 260), 32, 4, "bf16"), (77, 1152, (132, 4, 388), 64, 4, "f16"),
    (200, 640, (512, 128), 128, 8, "bf16"), (65, 4096, (256, 260, 64), 64, 4, "bf16"),
])
def test_matrices_in_one_launch(dev, M, K, Ns, gs, bits, dtype):
    """Two and three matrices, their tables side by side, in one launch: each
    within the bound, with partial column tiles at the seams, also without a
    workspace (no K split); the launch beside it, one per matrix, too."""
    import torch

    from dflash_mlx_amd import _lib, _runtime, verify_qmm as vq

    cases, mats, x = [], [], None
    for i, N in enumerate(Ns):
        case, (xi, w, s, b) = _case(dev, M, K, N, gs, bits, dtype, seed=40 + i)
        x, cx = (xi, case[0]) if x is None else (x, cx)
        cases.append((cx,) + case[1:])
        mats.append((w, s, b))

    def check(ys):
        for y, case in zip(ys, cases):
            _check(from_dev(y, dtype), case, gs, bits, dtype)

    one = vq.quantized_matmul_multi(x, mats, group_size=gs, bits=bits)
    check(one)
    check([vq.quantized_matmul(x, *m, group_size=gs, bits=bits) for m in mats])
    fused = torch.cat([_runtime.build_sb_pairs(s, b) for _, s, b in mats], dim=1).contiguous()
    outs = [torch.full_like(y, float("nan")) for y in one]
    segs = (_lib.QmmSegment * len(mats))()
    for g, (w, s, b), y in zip(segs, mats, outs):
        g.w_q, g.scales, g.biases = w.data_ptr(), s.data_ptr(), b.data_ptr()
        g.y, g.N = y.fill_(float("nan")).data_ptr(), int(w.shape[0])
    rc = _lib.load().dfmi_qmm_affine_multi_fused(
        x.data_ptr(), _runtime.dtype_code(x.dtype), segs, len(mats), fused.data_ptr(), M, K, gs,
        bits, None, 0, _runtime.stream_ptr(x.device))
    assert rc == _lib.DFMI_OK
    check(outs)
    ns = (ctypes.c_int64 * len(mats))(*Ns)
    need = int(_lib.load().dfmi_qmm_multi_workspace_bytes(M, K, ns, len(mats), gs, bits))
    ws, ws_bytes = _runtime.workspace(x.device, need)
    for y in outs:
        y.fill_(float("nan"))
    rc = _lib.load().dfmi_qmm_affine_multi(  # tables into the workspace, for the call
        x.data_ptr(), _runtime.dtype_code(x.dtype), segs, len(mats), M, K, gs, bits, ws, ws_bytes,
        _runtime.stream_ptr(x.device))
    assert rc == _lib.DFMI_OK and all(torch.equal(a, b) for a, b in zip(one, outs))
    for y in outs:
        y.fill_(float("nan"))
    rc = _lib.load().dfmi_qmm_affine_multi_fused(
        x.data_ptr(), _runtime.dtype_code(x.dtype), segs, len(mats), fused.data_ptr(), M, K, gs,
        bits, ws, ws_bytes, _runtime.stream_ptr(x.device))
    assert rc == _lib.DFMI_OK and all(torch.equal(a, b) for a, b in zip(one, outs))


def test_many_rows_in_inference_mode(dev):
    """Tensors that count no versions (made under inference mode) are taken,
    by the operators and by modules, and weights changed in place between two
    siblings' calls are seen."""
    import torch
    from torch import nn

    from dflash_mlx_amd import verify_linear as vl, verify_qmm as vq

    M, K, N, gs = 45, 512, 256, 64
    case, (x, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=31)
    with torch.inference_mode():
        xi, wi, si, bi = (t.clone() for t in (x, w, s, b))
        _check(from_dev(vq.quantized_matmul(xi, wi, si, bi, group_size=gs, bits=4), "bf16"),
               case, gs, 4, "bf16")
        for y in vq.quantized_matmul_multi(xi, [(w, s, b), (wi, si, bi)], group_size=gs, bits=4):
            _check(from_dev(y, "bf16"), case, gs, 4, "bf16")
    root = nn.Module()
    root.mlp = nn.Module()
    for name in ("gate_proj", "up_proj"):
        setattr(root.mlp, name, vl.QuantizedLinear(w.clone(), s.clone(), b.clone(),
                                                   group_size=gs, bits=4))
    vl.install_verify_linears(root, enable_qmm=True)
    gate, up = root.mlp.gate_proj, root.mlp.up_proj
    with torch.inference_mode():
        for m in (gate, up):
            _check(from_dev(m(x.clone()), "bf16"), case, gs, 4, "bf16")
    gate(x)
    up.weight.zero_()
    want = vq.quantized_matmul(x, up.weight, up.scales, up.biases, group_size=gs, bits=4)
    assert torch.equal(up(x), vq.quantized_matmul_multi(
        x, [(m.weight, m.scales, m.biases) for m in (gate, up)], group_size=gs, bits=4)[1])
    assert torch.allclose(up(x).float(), want.float(), rtol=2 ** -7, atol=0)


def test_module_many_rows(dev):
    """A verify module's many-row call: alone it equals the stock operator bit
    for bit, siblings the shared launch of quantized_matmul_multi (each within
    the bound), also with rows split over workgroups, in any call order, under
    graph replay, and after scales change in place (then the stock route)."""
    import torch
    from torch import nn

    from dflash_mlx_amd import verify_linear as vl, verify_qmm as vq

    K, gs = 2048, 64
    names = (("gate_proj", 384), ("up_proj", 644), ("down_proj", 256))
    for M in (45, 200):
        root, cases, x = nn.Module(), {}, None
        root.mlp = nn.Module()
        for i, (name, N) in enumerate(names):
            case, (xi, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=20 + i)
            x, cx = (xi, case[0]) if x is None else (x, cx)
            cases[name] = (cx,) + case[1:]
            setattr(root.mlp, name, vl.QuantizedLinear(w, s, b, group_size=gs, bits=4))
        vl.install_verify_linears(root, enable_qmm=True)
        gate, up, down = (getattr(root.mlp, n) for n, _ in names)
        want = vq.quantized_matmul_multi(
            x, [(m.weight, m.scales, m.biases) for m in (gate, up)], group_size=gs, bits=4)
        for first, second in ((0, 1), (1, 0)):
            mods = (gate, up)
            got = {first: mods[first](x), second: mods[second](x)}
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        for m, name in ((gate, "gate_proj"), (up, "up_proj")):
            _check(from_dev(m(x), "bf16"), cases[name], gs, 4, "bf16")
        stock = vq.quantized_matmul(x, down.weight, down.scales, down.biases, group_size=gs,
                                    bits=4)
        assert torch.equal(down(x), stock)
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            gate(x), up(x)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            g, u = gate(x), up(x)
        for _ in range(3):
            g.zero_(), u.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(g, want[0]) and torch.equal(u, want[1])
        gate.scales.mul_(1.5)
        for m in (gate, up, down):
            want1 = vq.quantized_matmul(x, m.weight, m.scales, m.biases, group_size=gs, bits=4)
            assert torch.equal(m(x), want1)


@pytest.mark.parametrize("route", ["operator", "siblings", "module", "group"])
def test_scales_are_read_at_each_call(dev, route):
    """Beyond 32 rows the product is of the scales as they are: after an
    update that counts no version, and in a graph replayed after one, also
    when eager calls and other allocations came between."""
    import torch
    from torch import nn

    from dflash_mlx_amd import verify_linear as vl, verify_qmm as vq

    M, K, Ns, gs = 45, 6144, (384, 256), 64
    mats, x = [], None
    for i, N in enumerate(Ns):
        _, (xi, w, s, b) = _case(dev, M, K, N, gs, 4, "bf16", seed=70 + i)
        x = xi if x is None else x
        mats.append((w, s, b))
    root = nn.Module()
    root.mlp = nn.Module()
    for name, (w, s, b) in zip(("gate_proj", "up_proj"), mats):
        setattr(root.mlp, name, vl.QuantizedLinear(w, s, b, group_size=gs, bits=4))
    vl.install_verify_linears(root, enable_qmm=True, fuse_siblings=route == "group")

    def run(a):
        if route == "operator":
            return [vq.quantized_matmul(a, *m, group_size=gs, bits=4) for m in mats]
        if route == "siblings":
            return vq.quantized_matmul_multi(a, mats, group_size=gs, bits=4)
        return [root.mlp.gate_proj(a), root.mlp.up_proj(a)]

    def want():  # the same values in tensors the library has not seen
        fresh = [tuple(t.clone() for t in m) for m in mats]
        if route in ("siblings", "group"):
            return vq.quantized_matmul_multi(x.clone(), fresh, group_size=gs, bits=4)
        return [vq.quantized_matmul(x, *m, group_size=gs, bits=4) for m in fresh]

    def same(got, ref):
        torch.cuda.synchronize()
        assert all(torch.equal(g, r) for g, r in zip(got, ref))

    same(run(x.clone()), want())
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        ys = run(x)
    for step in range(3):
        for _, s, b in mats:
            for t in (s, b):
                t.data.copy_(torch.roll(t, 1 + step, 0))  # counts no version of s, b
        ref = want()
        graph.replay()
        same(ys, ref)
        same(run(x.clone()), ref)
        junk = [torch.full((m[1].numel(),), float("nan"), device=dev) for m in mats * 8]
        graph.replay()
        same(ys, ref)
        del junk
