"""GPU parity of the routed experts beyond 256 pairs (``moe_gemm_kernel``, and the
gathers that take the smaller of them) and of the device sort of ``switch_glu``, against a float64 torch restatement that
rounds where mlx-lm's operators do.  Tolerance: the reference's own metric,
max|d| / (max|ref| + 1e-3) <= 1e-2 (tests/test_verify_qmm_parity.py:69-70)."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _experts(torch, gen, E, N, K, gs, dtype, dev):
    from dflash_mlx_amd.quantize import quantize

    w = torch.randn((E * N, K), generator=gen, device=dev) * 0.05
    q, s, b = quantize(w, gs, 4, dtype)
    return q.reshape(E, N, -1), s.reshape(E, N, -1), b.reshape(E, N, -1)


def _dense(torch, trip, e, gs):
    from dflash_mlx_amd.quantize import dequantize

    return dequantize(trip[0][e], trip[1][e], trip[2][e], gs, 4).double()


def _reference(torch, x, inds, gate, up, down, gs):
    T, k = inds.shape
    flat = inds.reshape(-1).long()
    token = torch.arange(T * k, device=x.device) // k
    E, dt = gate[0].shape[0], x.dtype
    h = torch.full((T * k, gate[0].shape[1]), float("nan"), dtype=dt, device=x.device)
    y = torch.full((T * k, down[0].shape[1]), float("nan"), dtype=dt, device=x.device)
    for e in flat.unique().tolist():
        if not 0 <= e < E:
            continue
        at = (flat == e).nonzero().reshape(-1)
        xe = x[token[at]].double()
        g = (xe @ _dense(torch, gate, e, gs).T).to(dt).double()
        u = (xe @ _dense(torch, up, e, gs).T).to(dt).double()
        sig = torch.sigmoid(g).to(dt).double()
        h[at] = ((g * sig).to(dt).double() * u).to(dt)
        y[at] = (h[at].double() @ _dense(torch, down, e, gs).T).to(dt)
    return h, y


def _close(torch, got, ref):
    nan = torch.isnan(ref)
    assert torch.equal(torch.isnan(got), nan)
    g, r = got.double()[~nan], ref.double()[~nan]
    if r.numel():
        rel = float((g - r).abs().max() / (r.abs().max() + 1e-3))
        assert rel <= 1e-2, rel


# (tokens, top-k, experts, D, I, group size): tables and 32-row tiles with
# runs of 1, 32, 33 and hundreds of pairs; then shapes without a table, one
# for each of the plain gathers
SHAPES = [
    (1, 1, 1, 256, 128, 64), (33, 8, 7, 256, 128, 64), (40, 8, 300, 512, 256, 64),
    (300, 2, 3, 256, 128, 128), (129, 8, 1023, 256, 384, 64), (257, 1, 8, 2048, 512, 64),
    (70, 4, 9, 96, 160, 32), (60, 5, 6, 1024, 96, 32), (60, 5, 6, 1280, 96, 32),
]


@pytest.fixture
def pays(monkeypatch):
    """Decide for the rule whether many pairs get a table."""
    from dflash_mlx_amd import moe

    return lambda answer: monkeypatch.setattr(moe, "_table_pays", lambda *a: answer)


@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("T,k,E,D,I,gs", SHAPES)
def test_switch_glu(dev, pays, T, k, E, D, I, gs, dtype, table):
    import torch

    from dflash_mlx_amd import moe

    pays(table)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    gen = torch.Generator(device=dev)
    gen.manual_seed(T + E + D)
    gate, up = (_experts(torch, gen, E, I, D, gs, dt, dev) for _ in range(2))
    down = _experts(torch, gen, E, D, I, gs, dt, dev)
    x = torch.randn((T, D), generator=gen, device=dev).to(dt)
    inds = torch.randint(0, E, (T, k), generator=gen, device=dev)
    if T == 300:
        inds[:] = 1        # one expert for all
        inds[5, 0] = -1    # invalid ids: NaN rows, no others
        inds[290, 1] = E
    h, y = moe.switch_glu(x, inds, gate, up, down, group_size=gs)
    hr, yr = _reference(torch, x, inds, gate, up, down, gs)
    _close(torch, h, hr)
    _close(torch, y, yr)
    h2, y2 = moe.switch_glu(x, inds.to(torch.int32), gate, up, down, group_size=gs)
    assert torch.equal(h.view(torch.int16), h2.view(torch.int16))
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("ordered", [False, True])
def test_gathers_many_pairs(dev, pays, ordered, table):
    """gather_swiglu / gather_qmm on 1100 pairs, sorted and not, with row ids
    out of range: each pair's row as the reference has it."""
    import torch

    from dflash_mlx_amd import moe

    pays(table)
    gen = torch.Generator(device=dev)
    gen.manual_seed(3)
    E, D, I, P, R, gs = 20, 512, 256, 1100, 90, 64
    gate, up = (_experts(torch, gen, E, I, D, gs, torch.bfloat16, dev) for _ in range(2))
    down = _experts(torch, gen, E, D, I, gs, torch.bfloat16, dev)
    x = torch.randn((R, D), generator=gen, device=dev).to(torch.bfloat16)
    rhs = torch.randint(0, E, (P,), generator=gen, device=dev, dtype=torch.int32)
    if ordered:
        rhs = rhs.sort().values
    lhs = torch.randint(0, R, (P,), generator=gen, device=dev, dtype=torch.int32)
    lhs[7], lhs[1099] = -3, R
    ok = (lhs >= 0) & (lhs < R)
    xs = x[lhs.long().clamp(0, R - 1)]
    hr, yr = _reference(torch, xs, rhs.reshape(-1, 1), gate, up, down, gs)
    hr[~ok] = float("nan")
    h = moe.gather_swiglu(x, gate, up, rhs, lhs_indices=lhs, group_size=gs)
    _close(torch, h, hr)
    good = torch.where(ok[:, None], h, torch.zeros_like(h))
    y = moe.gather_qmm(good, *down, rhs, group_size=gs)
    _close(torch, y[ok], yr[ok])


def test_switch_glu_captured(dev, pays):
    """Captured before and after the stream has its tables and workspaces,
    replayed with new routing: the eager results."""
    import torch

    from dflash_mlx_amd import moe

    pays(True)
    gen = torch.Generator(device=dev)
    gen.manual_seed(8)
    E, D, I, gs = 16, 256, 128, 64
    gate, up = (_experts(torch, gen, E, I, D, gs, torch.bfloat16, dev) for _ in range(2))
    down = _experts(torch, gen, E, D, I, gs, torch.bfloat16, dev)
    x = torch.randn((50, D), generator=gen, device=dev).to(torch.bfloat16)
    inds = torch.randint(0, E, (50, 8), generator=gen, device=dev)
    for warm in (False, True):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        if warm:
            with torch.cuda.stream(stream):
                moe.switch_glu(x, inds, gate, up, down, group_size=gs)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            h, y = moe.switch_glu(x, inds, gate, up, down, group_size=gs)
        for i in range(3):
            inds.copy_(torch.randint(0, E, (50, 8), generator=gen, device=dev))
            graph.replay()
            torch.cuda.synchronize()
            hr, yr = _reference(torch, x, inds, gate, up, down, gs)
            _close(torch, h, hr)
            _close(torch, y, yr)


@pytest.mark.parametrize("table", [True, False])
def test_scales_are_read_at_each_call(dev, pays, table):
    """Beyond 256 pairs the results are of the scales as they are: after an
    update that counts no version, and in a graph replayed after one."""
    import torch

    from dflash_mlx_amd import moe

    pays(table)
    gen = torch.Generator(device=dev)
    gen.manual_seed(12)
    E, D, I, gs = 16, 256, 128, 64
    gate, up = (_experts(torch, gen, E, I, D, gs, torch.bfloat16, dev) for _ in range(2))
    down = _experts(torch, gen, E, D, I, gs, torch.bfloat16, dev)
    x = torch.randn((50, D), generator=gen, device=dev).to(torch.bfloat16)
    inds = torch.randint(0, E, (50, 8), generator=gen, device=dev)
    rhs, lhs = inds.reshape(-1), torch.arange(400, device=dev) // 8

    def run():
        h = moe.gather_swiglu(x, gate, up, rhs, lhs_indices=lhs, group_size=gs)
        return (*moe.switch_glu(x, inds, gate, up, down, group_size=gs), h,
                moe.gather_qmm(h, *down, rhs, group_size=gs))

    run()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        ys = run()
    for step in range(3):
        for t in (*gate[1:], *up[1:], *down[1:]):
            t.data.copy_(torch.roll(t, 1 + step, 0))
        hr, yr = _reference(torch, x, inds, gate, up, down, gs)
        graph.replay()
        torch.cuda.synchronize()
        for got in (ys, run()):
            for g, r in zip(got, (hr, yr, hr, yr)):
                _close(torch, g, r)


def test_expert_weights_off_the_gpu_are_refused(dev):
    import torch

    from dflash_mlx_amd import moe

    gen = torch.Generator(device=dev)
    gen.manual_seed(1)
    gate = _experts(torch, gen, 4, 128, 256, 64, torch.bfloat16, dev)
    down = _experts(torch, gen, 4, 256, 128, 64, torch.bfloat16, dev)
    x = torch.randn((3, 256), generator=gen, device=dev).to(torch.bfloat16)
    inds = torch.zeros((3, 2), dtype=torch.int32, device=dev)
    for i in range(3):
        host = tuple(t.cpu() if j == i else t for j, t in enumerate(down))
        with pytest.raises(ValueError):
            moe.switch_glu(x, inds, gate, gate, host)
    with pytest.raises(ValueError):
        moe.switch_glu(x, inds.cpu(), gate, gate, down)
