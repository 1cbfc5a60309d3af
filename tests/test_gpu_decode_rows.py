"""The decode layer row by row (two launches, small streams of weights) against the CPU oracle and against the single launch on the same
arguments, which a caller gets by naming a spin limit: one token and the most rows, one expert a token and the most, experts met by several
tokens, fragments and stages that are partly filled, the largest K, both router widths, 16-bit logits, with and without biases."""
import pytest
import torch

from oracle import moe as omoe
from oracle import mxfp as omx
from oracle import routing as ort
from oracle.checks import assert_close, assert_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T, E, k, d_model, d_ff, bias_dtype, limit, logits_dtype", [
    (1, 4, 1, 8, 8, torch.bfloat16, 7.0, torch.float32),
    (1, 6, 4, 2880, 2880, torch.bfloat16, 7.0, torch.float32),
    (1, 8, 8, 3072, 3072, torch.float32, None, torch.bfloat16),
    (3, 5, 2, 136, 264, torch.float32, 7.0, torch.bfloat16),
    (64, 130, 1, 360, 248, None, 7.0, torch.float32),
    (16, 6, 4, 520, 1144, torch.bfloat16, None, torch.float32),
    (8, 512, 8, 144, 96, torch.bfloat16, 7.0, torch.float32),
    (5, 8, 2, 2880, 2880, torch.bfloat16, 7.0, torch.float32),
    # (k that does not divide the second launch's sixteen waves: some have no expert, and the others uneven shares of the stages)
    (5, 9, 3, 264, 392, torch.bfloat16, 7.0, torch.float32),
    (4, 7, 5, 520, 1656, torch.float32, 7.0, torch.bfloat16),
    (2, 140, 6, 136, 3072, torch.bfloat16, None, torch.float32),
    (9, 7, 7, 128, 640, None, 7.0, torch.float32),
    (2, 8, 7, 1032, 2440, torch.bfloat16, 7.0, torch.float32),
])
def test_rows_against_oracle_and_single_launch(device, monkeypatch, T, E, k, d_model, d_ff, bias_dtype, limit, logits_dtype):
    from bench import to_matmul_layout
    from triton_amd import _native as nt
    from triton_kernels import moe_decode
    from triton_kernels.matmul import FnSpecs, FusedActivation, PrecisionConfig
    from triton_kernels.swiglu import swiglu_fn
    g = torch.Generator().manual_seed(T * 131 + E)
    x = torch.randn((T, d_model), generator=g).to(torch.bfloat16)
    logits = torch.randn((T, E), generator=g).to(logits_dtype)
    dev = lambda t: None if t is None else t.to(device)
    w = [(torch.randn(s, generator=g) / s[1]**0.5).to(torch.bfloat16) for s in ((E, d_model, 2 * d_ff), (E, d_ff, d_model))]
    q = []
    for m in w:  # K is no multiple of the block in some cases: padded with zeros, as a loader does
        pad = -m.shape[1] % 32
        q += omx.downcast_to_mxfp(torch.nn.functional.pad(m, (0, 0, 0, pad)), torch.uint8, axis=1)
    b1 = b2 = None
    if bias_dtype is not None:
        b1, b2 = (torch.randn((E, n), generator=g).mul(0.1).to(bias_dtype) for n in (2 * d_ff, d_model))
    tiled = to_matmul_layout({n: dev(t) for n, t in dict(w1=q[0], w1s=q[1], w2=q[2], w2s=q[3], b1=b1, b2=b2).items()})
    for name, m in (("w1", w[0]), ("w2", w[1])):
        tiled[name].shape[-2] = m.shape[1]
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, limit))
    args = (dev(x), dev(logits), k, tiled["w1"], tiled["b1"], tiled["w2"], tiled["b2"], PrecisionConfig(b_mx_scale=tiled["w1s"]),
            PrecisionConfig(b_mx_scale=tiled["w2s"]), act)
    assert moe_decode.one_launch_reason(*args) is None
    out, indx, vals = moe_decode.moe_decode_layer(*args, return_routing=True)
    assert torch.equal(moe_decode.moe_mlp(*args), out)

    class Bounded(nt.DecodeLayerDesc):
        def __init__(self):
            super().__init__()
            self.spin_limit = 1 << 22

    with monkeypatch.context() as p:
        p.setattr(nt, "DecodeLayerDesc", Bounded)
        one, one_indx, one_vals = moe_decode.moe_decode_layer(*args, return_routing=True)
    r = ort.routing(logits.float(), k)  # (both launches keep the gate values in fp32)
    assert_equal(r.indx, indx.to(torch.int32), "indx")
    assert torch.equal(indx, one_indx)
    assert_close(r.vals.float(), vals, what="gate values")
    xp = torch.nn.functional.pad(x, (0, -d_model % 32))
    h = omoe.matmul(xp, q[0], b1, r.meta.col_sum, gather_indx=r.gather_indx, w_mx_scale=q[1])
    a = torch.nn.functional.pad(omoe.swiglu(h, 1.702, limit), (0, -d_ff % 32))
    y = omoe.matmul(a, q[2], b2, r.meta.col_sum, scatter_indx=r.scatter_indx, gammas=r.gammas, w_mx_scale=q[3])
    # (the oracle rounds the pre-activations to bf16, which the kernels keep in fp32: these layers in 64 bits, rounded only where the kernels
    # round, are 3.5e-3 to 4.02e-3 away from it)
    assert_close(omoe.reduce_k(y, k), out, maxtol=3e-2, rmstol=4.5e-3, what="row by row against the oracle")
    # the two kernels sum K in different groupings: an ulp of a hidden value here and there
    assert_close(one.cpu(), out, maxtol=2e-2, what="row by row against the single launch")


def test_a_k_that_routing_refuses_stays_refused(device):
    from triton_kernels.moe_decode import moe_mlp
    from bench import make_moe_weights, to_matmul_layout
    from triton_kernels.matmul import FnSpecs, FusedActivation, PrecisionConfig
    from triton_kernels.swiglu import swiglu_fn
    W = to_matmul_layout(make_moe_weights(8, 128, 256, seed=1, device=device)[0])
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    x, logits = torch.zeros((2, 128), dtype=torch.bfloat16, device=device), torch.zeros((2, 8), device=device)
    with pytest.raises(ValueError):
        moe_mlp(x, logits, 3, W["w1"], W["b1"], W["w2"], W["b2"], PrecisionConfig(b_mx_scale=W["w1s"]), PrecisionConfig(b_mx_scale=W["w2s"]), act)


@pytest.fixture(scope="module")
def small_layer(device):
    """call(x, logits): a layer of 8 experts through `moe_mlp`, top 4, row by row at the sizes below."""
    from bench import make_moe_weights, to_matmul_layout
    from triton_kernels import moe_decode
    from triton_kernels.matmul import FnSpecs, FusedActivation, PrecisionConfig
    from triton_kernels.swiglu import swiglu_fn
    W = to_matmul_layout(make_moe_weights(8, 256, 512, seed=4, device=device)[0])
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    pc1, pc2 = PrecisionConfig(b_mx_scale=W["w1s"]), PrecisionConfig(b_mx_scale=W["w2s"])
    return lambda x, logits: moe_decode.moe_mlp(x, logits, 4, W["w1"], W["b1"], W["w2"], W["b2"], pc1, pc2, act)


def _inputs(T, device, g):
    return torch.randn((T, 256), generator=g).to(torch.bfloat16).to(device), torch.randn((T, 8), generator=g).to(device)


@pytest.mark.parametrize("T", [1, 3])
def test_a_graph_owns_its_memory(device, small_layer, T):
    """Warmed up and captured on one stream, replayed with new inputs after the workspaces of more shapes than are kept, with other tensors in
    whatever memory they have left: bit for bit the eager layer's result."""
    from triton_kernels import moe_decode
    g = torch.Generator().manual_seed(T)
    x, logits = _inputs(T, device, g)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        small_layer(x, logits)
        with torch.cuda.graph(graph, stream=side):
            got = small_layer(x, logits)
        for t in range(1, 71):
            moe_decode._workspace(device, t, 2, 8, 256, 256)
    torch.cuda.synchronize()
    for rep in range(3):
        a, b = _inputs(T, device, g)
        x.copy_(a), logits.copy_(b)
        others = [torch.full((n, ), 0x7F, dtype=torch.uint8, device=device) for n in (512, 4096, 65536, 1 << 20)]
        graph.replay()
        torch.cuda.synchronize()
        assert all(bool((o == 0x7F).all()) for o in others)
        assert torch.equal(got, small_layer(x, logits)), f"replay {rep}"


def test_graphs_of_one_stream_replayed_side_by_side(device, small_layer):
    """Two graphs captured on one stream at one shape share no memory: replayed on two streams at a time each gives its own result."""
    g = torch.Generator().manual_seed(9)
    side, ins, graphs, outs = torch.cuda.Stream(), [], [], []
    for _ in range(2):
        x, logits = _inputs(4, device, g)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            small_layer(x, logits)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                out = [small_layer(x, logits) for _ in range(4)]
        torch.cuda.synchronize()
        ins.append((x, logits)), graphs.append(graph), outs.append(out)
    want = [small_layer(*i) for i in ins]
    assert not torch.equal(*want)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for rep in range(20):
        for s, graph in zip(streams, graphs):
            with torch.cuda.stream(s):
                graph.replay()
        torch.cuda.synchronize()
        for w, out in zip(want, outs):
            assert all(torch.equal(w, o) for o in out), f"replay {rep}"


def test_threads_of_one_stream_may_share_a_workspace(device, monkeypatch):
    """The two launches of a call are enqueued together: calls of two threads on one stream with one workspace give what each gives alone."""
    import threading

    from bench import make_moe_weights, to_matmul_layout
    from triton_amd import _native as nt
    from triton_kernels import moe_decode
    from triton_kernels.matmul import FnSpecs, FusedActivation, PrecisionConfig
    from triton_kernels.swiglu import swiglu_fn
    W = to_matmul_layout(make_moe_weights(8, 256, 512, seed=4, device=device)[0])
    act = FusedActivation(FnSpecs("swiglu", swiglu_fn, ("alpha", "limit"), reduction_n=2), (1.702, 7.0))
    pc1, pc2 = PrecisionConfig(b_mx_scale=W["w1s"]), PrecisionConfig(b_mx_scale=W["w2s"])
    layer = lambda x, logits: moe_decode.moe_decode_layer(x, logits, 4, W["w1"], W["b1"], W["w2"], W["b2"], pc1, pc2, act)
    g = torch.Generator().manual_seed(13)
    ins = [_inputs(2, device, g) for _ in range(2)]
    want = [layer(*i) for i in ins]
    real = nt.rules()

    class Rules:  # (the workspace of the single launch, which calls of one stream and shape share, for the same two launches)
        def __getattr__(self, name):
            return (lambda *a: False) if name == "decode_by_rows" else getattr(real, name)

    monkeypatch.setattr(nt, "rules", lambda: Rules())
    outs, errors = [[], []], []

    def work(i):
        try:
            outs[i] += [layer(*ins[i]) for _ in range(200)]
        except Exception as e:
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i, )) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i in range(2):
        assert len(outs[i]) == 200 and all(torch.equal(o, want[i]) for o in outs[i])
