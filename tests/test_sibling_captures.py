"""Pending outputs of a sibling group and graph captures: a member takes what
its group's launch computed only where that launch runs in the same place --
both calls eager, or both in one capture -- at every row count."""

from __future__ import annotations

import pytest
import torch

from dflash_mlx_amd import _runtime, verify_linear as vl


class _State:
    N, K, gs, bits = 8, 64, 64, 4

    def __init__(self, value):
        self.w = self.s = self.b = torch.full((1,), float(value))


@pytest.mark.parametrize("M", [4, 16, 32, 33])
def test_outputs_stay_with_their_launch(monkeypatch, M):
    grp = vl.SiblingGroup([_State(0), _State(1)], None, 0)
    launches = []

    class Record:
        def run(self, x2, ys, st):
            launches.append(where[0])
            for y in ys:
                y.fill_(len(launches))

    monkeypatch.setattr(grp, "_record", lambda *a: Record())
    monkeypatch.setattr(grp, "_takes_many", lambda active: True)
    monkeypatch.setattr(vl, "qmm_multi_launch", lambda x2, mats, gs, bits, outs:
                        Record().run(x2, outs, 0))
    where = [0]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: where[0] != 0)
    monkeypatch.setattr(_runtime, "capture_key", lambda st: where[0], raising=False)
    x = torch.zeros((M, 64))
    # eager q, then k in a capture, q in another one, k eager, q eager
    for step, (w, member) in enumerate([(0, 0), (7, 1), (9, 0), (0, 1), (0, 0)]):
        where[0] = w
        y = grp.product(member, x, M, 5)
        want = min(step + 1, 4)  # the last one is the eager launch before it
        assert len(launches) == want and torch.all(y == want)
    assert launches == [0, 7, 9, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("M", [16, 40])
def test_siblings_over_eager_calls_and_two_captures(dev, M):
    """gate eager and up captured, then gate captured by a second graph: each
    replay is of its own graph's input."""
    from torch import nn

    gen = torch.Generator(device=dev)
    gen.manual_seed(M)
    K, gs = 1024, 64
    root = nn.Module()
    root.mlp = nn.Module()
    for name, N in (("gate_proj", 512), ("up_proj", 512)):
        lin = nn.Linear(K, N, bias=False, device=dev)
        setattr(root.mlp, name, vl.QuantizedLinear.from_linear(lin, gs, 4, torch.bfloat16))
    vl.install_verify_linears(root, enable_qmm=True)
    vl.prewarm_verify_kernels(root)
    gate, up = root.mlp.gate_proj, root.mlp.up_proj
    stream = torch.cuda.Stream()
    x = torch.randn((M, K), generator=gen, device=dev).to(torch.bfloat16)
    stream.wait_stream(torch.cuda.current_stream())
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    with torch.cuda.stream(stream):
        for m in (gate, up):
            m(x.clone())  # workspace and prepared launch of this stream
        root.mlp.gate_proj._verify_state.group.reset()
        gate(x)
    torch.cuda.synchronize()
    with torch.cuda.graph(graphs[0], stream=stream):
        u = up(x)
    with torch.cuda.graph(graphs[1], stream=stream):
        g = gate(x)
    for _ in range(3):
        x.copy_(torch.randn((M, K), generator=gen, device=dev).to(torch.bfloat16))
        want_g, want_u = gate(x.clone()), up(x.clone())
        for graph, y, want in ((graphs[1], g, want_g), (graphs[0], u, want_u)):
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
