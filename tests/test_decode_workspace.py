"""The memory that decode layers are launched with, on the CPU (the descriptors are looked at, nothing is launched): the two launches of a layer that
goes row by row get memory of the call's own, so that a captured graph's belongs to the graph, and the single launch's workspace, which keeps
counters between calls, stays where a graph has its address."""
import pytest
import torch

from triton_amd import _native as nt
from triton_amd import moe_decode


class _Library:
    def __init__(self, real):
        self.real, self.given, self.capture = real, [], 0

    def __getattr__(self, name):
        return getattr(self.real, name)

    def tk_stream_capture_id(self, stream):
        return self.capture

    def tk_moe_decode_layer(self, d, stream):
        self.given.append(d.workspace)
        return 0


class _Weights:  # a tiled tensor, its storage and its scales, as far as the call looks at them
    def __init__(self, e, k, n):
        self.shape = (e, k, n)
        self.storage = self
        self.data = self.b_mx_scale = torch.zeros((e, 16), dtype=torch.uint8)


@pytest.fixture
def layer(monkeypatch):
    """layer(T, k, dims): a decode layer on CPU tensors with a library that only notes the workspace; layer.given: those."""
    lib = _Library(nt.lib())
    nt.rules()
    monkeypatch.setattr(nt, "lib", lambda: lib)
    monkeypatch.setattr(nt, "stream_ptr", lambda device=None: 0)
    monkeypatch.setattr(moe_decode, "one_launch_reason", lambda *a: None)
    monkeypatch.setattr(moe_decode, "_swiglu_args", lambda act: (1.702, 7.0, 1))
    monkeypatch.setattr(moe_decode, "_WORKSPACES", {})
    monkeypatch.setattr(moe_decode, "_CAPTURED", {})

    class PC:
        def __init__(self, w):
            self.b_mx_scale = w

    def call(T, k, dims=2880, E=128):
        w1, w2 = _Weights(E, dims, 2 * dims), _Weights(E, dims, dims)
        return moe_decode.moe_decode_layer(torch.zeros((T, dims), dtype=torch.bfloat16), torch.zeros((T, E)), k, w1, None, w2, None, PC(w1), PC(w2), None)

    call.given = lib.given
    return call


@pytest.mark.parametrize("T, k, dims", [(1, 1, 2880), (1, 4, 2880), (8, 1, 2880), (64, 1, 512)])
def test_row_by_row_memory_is_the_calls_own(layer, T, k, dims):
    assert nt.rules().decode_by_rows(T, k, dims, dims)
    layer(T, k, dims)
    assert len(layer.given) == 1 and layer.given[0] and moe_decode._WORKSPACES == {}


@pytest.mark.parametrize("T, k, dims", [(16, 4, 2880), (65, 1, 512), (4, 16, 512)])
def test_the_single_launch_keeps_its_counters(layer, T, k, dims):
    assert not nt.rules().decode_by_rows(T, k, dims, dims)
    layer(T, k, dims)
    layer(T, k, dims)
    ((ws, _), ) = moe_decode._WORKSPACES.values()
    assert layer.given == [ws.data_ptr()] * 2


@pytest.fixture
def capturing(layer):
    """capturing(id): the current stream counts as being captured, 0 = no longer."""
    return lambda capture: setattr(nt.lib(), "capture", capture)


def _others(n):
    for t in range(n):
        moe_decode._workspace(torch.device("cpu"), 1 + t, 32, 512, 64, 64)


def test_a_captured_workspace_is_never_dropped(layer, capturing):
    """Warmed up, captured, then more other shapes than are kept: the graph's address is still this workspace's, and no other one's."""
    layer(16, 4)
    capturing(7)
    layer(16, 4)
    capturing(0)
    warm, captured = layer.given
    assert warm == captured
    ws = moe_decode._workspace(torch.device("cpu"), 16, 4, 128, 2880, 2880)
    assert ws.data_ptr() == captured
    _others(150)
    assert len(moe_decode._WORKSPACES) <= 64
    assert moe_decode._workspace(torch.device("cpu"), 16, 4, 128, 2880, 2880) is ws
    layer(16, 4)
    assert layer.given[-1] == captured


def test_workspaces_without_a_graph_are_dropped(layer):
    import weakref
    first = weakref.ref(moe_decode._workspace(torch.device("cpu"), 16, 4, 128, 2880, 2880))
    _others(64)
    assert first() is None and len(moe_decode._WORKSPACES) == 64


def test_a_workspace_made_in_a_capture_is_that_captures_own(layer, capturing):
    """Its counters are zero only once that graph has run, so neither an eager call nor another capture may be given it."""
    get = lambda: moe_decode._workspace(torch.device("cpu"), 16, 4, 128, 2880, 2880)
    capturing(7)
    first = get()
    assert get() is first
    capturing(8)
    second = get()
    assert second is not first and get() is second
    capturing(0)
    eager = get()
    assert eager is not first and eager is not second and get() is eager


@pytest.mark.parametrize("T, k, d_ff, d_model, by_rows", [
    (1, 4, 2880, 2880, True), (7, 1, 3072, 3072, True), (2, 4, 2880, 2880, True), (9, 1, 2880, 2880, True), (5, 2, 2880, 2880, True),
    (3, 4, 2880, 2880, False), (12, 1, 2880, 2880, False), (4, 4, 2880, 2880, False),
    (16, 1, 2048, 2048, True), (10, 2, 2048, 2048, True), (21, 1, 2048, 2048, False), (13, 2, 2048, 2048, False),
    (24, 1, 1536, 1536, True), (4, 8, 1536, 1536, True), (32, 1, 1536, 1536, False), (20, 2, 1536, 1536, False),
    (32, 1, 1024, 1024, True), (24, 2, 1024, 1024, True), (8, 8, 1024, 1024, True), (48, 1, 1024, 1024, False), (64, 1, 1024, 1024, False),
    (32, 2, 1024, 1024, False), (16, 2, 2048, 1024, True), (32, 1, 2048, 1024, False), (64, 1, 512, 512, True), (4, 16, 512, 512, False),
])
def test_which_layers_go_row_by_row(T, k, d_ff, d_model, by_rows):
    """Both sides of the line, at sizes where each form of launch was measured to be the faster one (or, in the end, is the only one)."""
    assert nt.rules().decode_by_rows(T, k, d_ff, d_model) == by_rows
