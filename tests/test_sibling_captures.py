"""Verify modules over streams and graph captures.  A member of a sibling group
takes what its group's launch computed only where that launch runs in the same
place -- both calls eager, or both in one capture -- at every row count; and a
launch on another stream than the install's waits for the tables."""

from __future__ import annotations

import copy

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


def test_each_launch_prepared_waits_for_its_table(monkeypatch):
    monkeypatch.setattr(vl, "LaunchRecord", lambda *a, **k: object())
    gets = []

    class Built:
        def __init__(self, name):
            self.name = name

        def get(self):
            gets.append(self.name)

    bf = torch.bfloat16
    states = []
    for name in "ab":
        w, s = torch.zeros((64, 32), dtype=torch.int32), torch.zeros((64, 4), dtype=bf)
        q = vl._VerifyState(w, s, s, 64, 256, 64, 4)
        q.pairs, q.built = torch.zeros(1), Built(name)
        states.append(q)
    x = torch.zeros((16, 256), dtype=bf)
    for st in (5, 5, 6):
        states[0].record(16, st, x)
    assert gets == ["a", "a"]
    gets.clear()
    grp = vl.SiblingGroup(states, torch.zeros(1), 128)
    for st in (5, 5, 6):
        grp._record(16, st, x, (0, 1))
    assert gets == ["a", "b"] * 2


@pytest.mark.gpu
def test_deepcopy_of_an_installed_model(dev):
    """A model is copied with its tables, also after calls of every kind."""
    from torch import nn

    root = nn.Module()
    root.mlp = nn.Module()
    for name in ("gate_proj", "up_proj"):
        setattr(root.mlp, name, vl.QuantizedLinear.from_linear(
            nn.Linear(1024, 256, bias=False, device=dev), 64, 4, torch.bfloat16))
    vl.install_verify_linears(root, enable_qmm=True)
    x = torch.randn((16, 1024), device=dev).to(torch.bfloat16)
    want = root.mlp.gate_proj(x), root.mlp.up_proj(x)
    twin = copy.deepcopy(root)
    got = twin.mlp.gate_proj(x), twin.mlp.up_proj(x)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    state = twin.mlp.gate_proj._verify_state
    assert torch.equal(state.built.get()[:, :256], state.pairs)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [16, 40])
@pytest.mark.parametrize("fuse", [False, True])
def test_call_on_another_stream_right_after_install(dev, M, fuse):
    """Installed behind a long-running kernel of one stream, called on another
    at once: the result of the finished tables."""
    from torch import nn

    gen = torch.Generator(device=dev)
    gen.manual_seed(M)
    K, N, gs = 1024, 512, 64
    x = torch.randn((M, K), generator=gen, device=dev).to(torch.bfloat16)
    got, streams = {}, [torch.cuda.Stream(), torch.cuda.Stream()]
    mats = [vl.QuantizedLinear.from_linear(nn.Linear(K, N, bias=False, device=dev), gs, 4,
                                           torch.bfloat16) for _ in range(2)]
    for late in (False, True):
        root = nn.Module()
        root.mlp = nn.Module()
        for name, q in zip(("gate_proj", "up_proj"), mats):
            setattr(root.mlp, name, vl.QuantizedLinear(
                q.weight.clone(), q.scales.clone(), q.biases.clone(), group_size=gs, bits=4))
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            if late:
                torch.cuda._sleep(100_000_000)
            vl.install_verify_linears(root, enable_qmm=True, fuse_siblings=fuse)
        if not late:
            torch.cuda.synchronize()
        with torch.cuda.stream(streams[1]):
            got[late] = [root.mlp.gate_proj(x), root.mlp.up_proj(x)]
        torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got[False], got[True]))


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
        same = x.clone()  # one shared launch for both
        want_g, want_u = gate(same), up(same)
        for graph, y, want in ((graphs[1], g, want_g), (graphs[0], u, want_u)):
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
