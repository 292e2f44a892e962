"""Host side of the calls that enqueue several kernels and pass data between
them through scratch (more than 32 rows, more than 256 routed pairs, the expert
sort): two calls in flight on one stream share no byte of it, and none of them
brings a table kept from an earlier call.  On the CPU a stand-in library
records what each call brings and holds the first call inside the library
until the second one has been there; on the GPU two threads call on one
stream."""

from __future__ import annotations

import copy
import threading

import pytest
import torch

from dflash_mlx_amd import _lib, _runtime, moe, verify_qmm as vq


class _Library:
    """Answers as libdfmi does, launching nothing."""

    def __init__(self, entry, ws):
        self.entry, self.ws = entry, ws  # entry point looked at; positions of (ptr, bytes) pairs
        self.seen = []
        self.second = threading.Event()

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("workspace_bytes") or name.endswith("workspace_bytes_ex"):
                return 65536 + 4096
            if name == self.entry:
                self.seen.append([(args[i], args[i + 1]) for i in self.ws])
                if len(self.seen) == 1:
                    self.second.wait(10)
                else:
                    self.second.set()
            return _lib.DFMI_OK
        return call


@pytest.fixture
def library(monkeypatch):
    def use(entry, ws):
        lib = _Library(entry, ws)
        monkeypatch.setattr(_lib, "load", lambda: lib)
        return lib

    monkeypatch.setattr(_runtime, "require_device", lambda t, name: None)
    monkeypatch.setattr(_runtime, "_raw_stream", lambda i: 0)
    monkeypatch.setattr(vq, "_raw_stream", lambda i: 0)
    monkeypatch.setattr(_runtime, "stream_ptr", lambda dev: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_runtime.PAIRS, "get", lambda *a, **k: torch.zeros(1))
    monkeypatch.setattr(_runtime, "WORKSPACES", _runtime._WorkspaceCache())
    monkeypatch.setattr(moe, "_table_pays", lambda *a: True)
    return use


def _weights(N, K, gs=64, lead=()):
    bf = torch.bfloat16
    return (torch.zeros((*lead, N, K // 8), dtype=torch.int32),
            torch.zeros((*lead, N, K // gs), dtype=bf), torch.zeros((*lead, N, K // gs), dtype=bf))


def _two_at_once(lib, call):
    first = threading.Thread(target=call)
    first.start()
    while not lib.seen:
        first.join(0.01)
        assert first.is_alive() or lib.seen
    call()
    first.join()
    a, b = lib.seen
    for (pa, na), (pb, nb) in zip(a, b):
        assert pa and pb and na and nb
        assert pa + na <= pb or pb + nb <= pa, "two calls in flight share scratch"


@pytest.mark.parametrize("route", ["single", "siblings", "general", "record"])
def test_many_rows(library, route):
    x, w = torch.zeros((40, 256), dtype=torch.bfloat16), _weights(128, 256)
    if route == "single":
        lib = library("dfmi_qmm_affine_pairs", (12,))
        _two_at_once(lib, lambda: vq.quantized_matmul(x, *w))
    elif route == "siblings":
        lib = library("dfmi_qmm_affine_multi", (8,))
        _two_at_once(lib, lambda: vq.quantized_matmul_multi(x, [w, w]))
    elif route == "general":
        lib = library("dfmi_qmm_general", (13,))
        _two_at_once(lib, lambda: vq._general(x, *w, True, 64, 4))
    else:
        lib = library("dfmi_qmm_affine_multi", (8,))
        rec = vq.LaunchRecord(40, 256, x.dtype, x.device, [w], 64, 4)
        _two_at_once(lib, lambda: rec.run(x, [torch.empty((40, 128), dtype=x.dtype)], 0))


def test_many_pairs(library):
    E, D = 4, 256
    w = _weights(128, D, lead=(E,))
    x = torch.zeros((300, D), dtype=torch.bfloat16)
    ids = torch.zeros(300, dtype=torch.int32)
    lib = library("dfmi_gather_qmm_affine_pairs", (16,))
    _two_at_once(lib, lambda: moe.gather_qmm(x, *w, ids))
    lib = library("dfmi_gather_qmm_swiglu_pairs", (19,))
    _two_at_once(lib, lambda: moe.gather_swiglu(x, w, w, ids))


def test_expert_sort(library):
    E, D, I = 4, 256, 128
    gate, down = _weights(I, D, lead=(E,)), _weights(D, I, lead=(E,))
    x = torch.zeros((16, D), dtype=torch.bfloat16)
    ids = torch.zeros((16, 8), dtype=torch.int32)
    lib = library("dfmi_switch_glu", (24,))
    _two_at_once(lib, lambda: moe._switch_glu(x, ids, gate, gate, down, 64, 4))


def _from_two_threads(calls, check):
    errors = []

    def work(i):
        try:
            for _ in range(60):
                check(i, calls[i]())
        except Exception as exc:  # reported by the main thread
            errors.append(exc)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_where_a_table_for_many_pairs_pays():
    """The rule's lines: the persistent gather's shapes, the others by size, and
    long runs of few experts."""
    pays = moe._table_pays
    assert not pays(1024, 2048, 512, 256, 64, True) and pays(1025, 2048, 512, 256, 64, True)
    assert not pays(512, 2048, 768, 64, 64, True) and pays(1024, 2048, 768, 64, 64, True)
    assert not pays(511, 512, 2048, 256, 64, False) and pays(512, 512, 2048, 256, 64, False)
    assert pays(512, 512, 1024, 8, 64, False) and not pays(512, 512, 1024, 64, 64, False)
    assert not pays(257, 256, 128, 1, 64, False)


def test_tables_are_waited_for_once_per_stream(monkeypatch):
    """A table is waited for on the device by the first call on each stream but
    the one that built it, never while capturing, and its event not queried."""
    waits, at = [], {"stream": 1, "capturing": False}

    class Event:
        def record(self, stream):
            waits.append(("record", stream))

        def query(self):
            raise AssertionError("queried")

    class Stream:
        def wait_event(self, event):
            waits.append(at["stream"])

    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: Stream())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: at["capturing"])
    monkeypatch.setattr(_runtime, "_raw_stream", lambda d: at["stream"])
    table = torch.zeros(4)
    built = _runtime._Built(table)
    waits.clear()
    for stream, capturing in ((1, False), (2, False), (2, False), (3, True), (3, False), (1, False),
                              (2, False), (3, False)):
        at.update(stream=stream, capturing=capturing)
        assert built.get() is table
    assert waits == [2, 3]
    twin = copy.deepcopy(built)  # (as with the module that holds it)
    assert twin.table is not table and torch.equal(twin.get(), table)


def test_expert_tensors_on_another_device(library):
    """switch_glu refuses expert ids or weights that are not where x is, before
    anything reaches the library."""
    class Elsewhere(torch.Tensor):
        def get_device(self):
            return 1

    gate, down = _weights(128, 256, lead=(4,)), _weights(256, 128, lead=(4,))
    x, ids = torch.zeros((16, 256), dtype=torch.bfloat16), torch.zeros((16, 8), dtype=torch.int32)
    for at in range(10):
        lib = library("dfmi_switch_glu", ())
        lib.second.set()
        ts = [t.as_subclass(Elsewhere) if i == at else t
              for i, t in enumerate((ids, *gate, *gate, *down))]
        with pytest.raises(ValueError, match="expert ids or weights on"):
            moe._switch_glu(x, ts[0], ts[1:4], ts[4:7], ts[7:10], 64, 4)
        assert not lib.seen


def test_no_kept_tables(library, monkeypatch):
    """More than 32 rows bring no pair table, more than 256 pairs one built in
    the call; 32 rows and 256 pairs take the cached ones."""
    kept = torch.zeros(1)
    monkeypatch.setattr(_runtime.PAIRS, "get", lambda *a, **k: kept)
    tables = []

    class Lib(_Library):
        def __getattr__(self, name):
            def call(*args):
                if name.endswith("bytes") or name.endswith("bytes_ex"):
                    return 65536 + 4096
                tables.append(name)
                if name == "dfmi_qmm_affine_pairs":
                    tables.append(args[5])
                elif name == "dfmi_qmm_affine_multi":
                    tables.extend(args[2][i].sb_pairs for i in range(args[3]))
                elif name in ("dfmi_gather_qmm_affine_pairs", "dfmi_moe_pairs"):
                    tables.append(args[6] if "gather" in name else args[8])
                return _lib.DFMI_OK
            return call

    monkeypatch.setattr(_lib, "load", lambda: Lib("", ()))
    monkeypatch.setattr(_runtime.FUSED_PAIRS, "get", lambda tables: None)
    w = _weights(128, 512)
    for M in (33, 32):
        x = torch.zeros((M, 512), dtype=torch.bfloat16)
        vq.quantized_matmul(x, *w)
        vq.quantized_matmul_multi(x, [w, w])
        t = kept.data_ptr() if M == 32 else None
        assert [a or None for a in tables] == ["dfmi_qmm_affine_pairs", t, "dfmi_qmm_affine_multi",
                                               t, t]
        tables.clear()
    e = _weights(128, 512, lead=(4,))
    for P in (257, 256):
        x = torch.zeros((P, 512), dtype=torch.bfloat16)
        moe.gather_qmm(x, *e, torch.zeros(P, dtype=torch.int32))
        if P == 257:
            assert tables == ["dfmi_moe_pairs", tables[1], "dfmi_gather_qmm_affine_pairs",
                              tables[1]] and tables[1] not in (None, kept.data_ptr())
        else:
            assert tables == ["dfmi_gather_qmm_affine_pairs", kept.data_ptr()]
        tables.clear()


@pytest.mark.gpu
@pytest.mark.parametrize("shared", [False, True])
def test_threads_on_one_stream(dev, shared):
    """K splits (product, then sum) from two threads on one stream, through
    the operator and through the C ABI with one workspace for both: each call
    has its own result."""
    M, K, Ns, gs = 40, 8192, (256, 512), 64
    gen = torch.Generator(device=dev)
    gen.manual_seed(2)

    def rand(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(torch.bfloat16)

    xs = [rand(M, K) for _ in Ns]
    mats = [(torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=gen, device=dev,
                           dtype=torch.int32), rand(N, K // gs), rand(N, K // gs)) for N in Ns]
    want = [vq.quantized_matmul(x, *w, group_size=gs) for x, w in zip(xs, mats)]
    lib = _lib.load()
    need = max(int(lib.dfmi_qmm_workspace_bytes(M, K, N, gs, 4)) for N in Ns)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    st = _runtime.stream_ptr(dev)
    torch.cuda.synchronize()

    def through_abi(i):
        y = torch.empty((M, Ns[i]), dtype=torch.bfloat16, device=dev)
        w, s, b = mats[i]
        rc = lib.dfmi_qmm_affine(xs[i].data_ptr(), _lib.DFMI_BF16, w.data_ptr(), s.data_ptr(),
                                 b.data_ptr(), y.data_ptr(), M, K, Ns[i], gs, 4, ws.data_ptr(),
                                 int(lib.dfmi_qmm_workspace_bytes(M, K, Ns[i], gs, 4)), st)
        assert rc == _lib.DFMI_OK
        return y

    def through_operator(i):
        return vq.quantized_matmul(xs[i], *mats[i], group_size=gs)

    call = through_abi if shared else through_operator

    def check(i, y):
        torch.cuda.synchronize()
        assert torch.equal(y, want[i])

    _from_two_threads([lambda i=i: call(i) for i in range(2)], check)


@pytest.mark.gpu
def test_expert_routing_from_two_threads(dev):
    """The sorted pairs of two threads' SwitchGLU calls on one stream stay
    apart, with few and many pairs."""
    from dflash_mlx_amd.quantize import quantize

    E, D, I, gs = 8, 256, 128, 64
    gen = torch.Generator(device=dev)
    gen.manual_seed(4)

    def experts(N, K):
        w = torch.randn((E * N, K), generator=gen, device=dev) * 0.05
        return tuple(t.reshape(E, N, -1) for t in quantize(w, gs, 4, torch.bfloat16))

    gate, up, down = experts(I, D), experts(I, D), experts(D, I)
    args = []
    for T in (90, 16):
        x = torch.randn((T, D), generator=gen, device=dev).to(torch.bfloat16)
        args.append((x, torch.randint(0, E, (T, 4), generator=gen, device=dev)))
    want = [moe.switch_glu(x, ids, gate, up, down, group_size=gs) for x, ids in args]
    torch.cuda.synchronize()

    def check(i, got):
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want[i]))

    _from_two_threads([lambda i=i: moe.switch_glu(*args[i], gate, up, down, group_size=gs)
                       for i in range(2)], check)
