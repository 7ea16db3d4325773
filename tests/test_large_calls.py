"""Calls of more than 1024 tokens: the one large workspace that a device's layers share (its size,
its order over streams, its absence under graph capture), and calls of several chunks, whose token
ids, gate logits, residual rows and outputs start at each chunk's own offset."""

import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from urbilateria_amd import configs as C
from urbilateria_amd import native as N
from urbilateria_amd import synth

from .gpu_helpers import REL_L2_BAR, ids_match, rel_l2
from .test_gpu_parity import (_dsv4_hash_layer, _oracle, _qwen_shared_layer, _scores,
                              _small_layer, moe_mod)

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu(require_gpu):
    torch.cuda.set_device(0)
    yield


class Call:
    """One kind of layer call on fixed inputs: run(stream) enqueues it into self.out."""

    def __init__(self, kind, T):
        self.kind, self.T = kind, T
        self.host = {"glm": lambda: _small_layer("c3_mxfp4_decode"),
                     "qwen_block": _qwen_shared_layer,
                     "dsv4_hash": _dsv4_hash_layer}[kind]()
        H, k = self.host.spec.hidden, self.host.spec.top_k
        self.x_np = synth.activations(f"x.large.{kind}.{T}", T, H)
        self.x = torch.from_numpy(self.x_np).cuda()
        self.norm_np = synth.activations(f"norm.{kind}", 1, H)[0] * np.float32(0.125)
        self.norm = torch.from_numpy(self.norm_np).cuda()
        self.tok_np = (synth.splitmix64(synth.stream_seed(f"tok.{T}"), 0, T) % 50).astype(np.uint32)
        self.tok = torch.from_numpy(self.tok_np.view(np.int32)).cuda()
        self.out = [torch.empty((T, H), dtype=torch.float32, device="cuda"),
                    torch.empty((T, k), dtype=torch.int32, device="cuda"),
                    torch.empty((T, k), dtype=torch.float32, device="cuda")]
        self.layer = moe_mod().MoeLayer(self.host, max_tokens=T)

    def run(self, stream=None, tokens=None):
        lib, T = N.moe_lib(), tokens or self.T
        s = ctypes.c_void_p((stream or torch.cuda.current_stream()).cuda_stream)
        p = lambda t: ctypes.c_void_p(t.data_ptr())
        ctx, out = self.layer._ctx, [p(t) for t in self.out]
        if self.kind == "glm":
            st = lib.urb_moe_forward(ctx, p(self.x), T, *out, s)
        elif self.kind == "dsv4_hash":
            st = lib.urb_moe_forward_tokens(ctx, p(self.x), p(self.tok), T, *out, s)
        else:
            st = lib.urb_moe_forward_block(ctx, p(self.x), p(self.norm), 1e-6, T, *out, s)
        N.check(st, self.kind)

    def results(self):
        torch.cuda.synchronize()
        self.layer.sync()
        return [t.clone() for t in self.out]

    def check(self, got):
        y, ids, w = [t.cpu().numpy() for t in got]
        host = self.host
        if self.kind == "qwen_block":
            ref = _oracle(host, O.zc_rms_norm(self.x_np, self.norm_np, 1e-6))
            want, y = O.add_residual_bf16(self.x_np, ref.output) - self.x_np, y - self.x_np
            assert np.array_equal(ids, ref.ids)
        else:
            ref = _oracle(host, self.x_np,
                          token_ids=self.tok_np if self.kind == "dsv4_hash" else None)
            want = ref.output
            assert ids_match(ids, ref.ids, _scores(host.spec, ref, host.correction_bias))
        assert rel_l2(y, want) < REL_L2_BAR
        assert np.allclose(w, ref.weights, rtol=1e-5, atol=1e-7)


KINDS = ["glm", "qwen_block", "dsv4_hash"]


@pytest.mark.parametrize("kind", KINDS)
def test_calls_of_several_chunks_match_oracle(kind):
    call = Call(kind, 4101)   # two chunks: 2051 and 2050 tokens
    call.run()
    call.check(call.results())
    call.layer.close()


@pytest.mark.parametrize("kind", KINDS)
def test_captured_large_calls_keep_to_the_layers_own_workspace(kind):
    # 2101 tokens in three chunks of the layer's own workspace; between the replays the same call
    # runs eagerly in the large one
    call = Call(kind, 2101)
    call.run(tokens=701)
    call.run()
    eager = call.results()
    call.check(eager)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call.run(stream)
    first = None
    for _ in range(3):
        for t in call.out:
            t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        got = call.results()
        if first is None:
            call.check(got)
            first = got
        assert all(torch.equal(a, b) for a, b in zip(got, first))
        call.run()
        assert all(torch.equal(a, b) for a, b in zip(call.results(), eager))
    del graph
    call.layer.close()


@pytest.mark.parametrize("first", ["default stream", "stream"])
def test_layers_on_two_streams_take_turns_in_the_large_workspace(first):
    calls = [Call("glm", 3000), Call("qwen_block", 3500)]
    want = []
    for c in calls:
        c.run()
        want.append(c.results())
    streams = [torch.cuda.default_stream() if first == "default stream" else torch.cuda.Stream(),
               torch.cuda.Stream()]
    for _ in range(4):
        for c in calls:
            for t in c.out:
                t.zero_()
        torch.cuda.synchronize()
        for _ in range(3):
            for c, s in zip(calls, streams):
                c.run(s)
        for c, ref in zip(calls, want):
            assert all(torch.equal(a, b) for a, b in zip(c.results(), ref))
    for c in calls:
        c.layer.close()


def test_layers_share_one_large_workspace_and_give_it_back():
    spec = C.small_spec(C.workload("c5_mxfp4_zipf_prefill").spec, hidden=2048, n_experts=16,
                        intermediate=128)
    host = C.make_host_layer(spec, bias=C.zipf_bias(16, 1.1, 0.05))
    make = lambda T: moe_mod().MoeLayer(host, max_tokens=T)
    short = make(1024)
    weights, own = short.memory()
    torch.cuda.synchronize()
    free = lambda: torch.cuda.mem_get_info()[0]
    before = free()
    layers = [make(4096) for _ in range(4)]
    # a layer that may be called with 4096 tokens holds no more than one of 1024 tokens does ...
    assert all(l.memory()[1] == own for l in layers)
    # ... and the four share one workspace of four times that (64 MiB: allocation granularity)
    slack = 64 << 20
    taken = before - free()
    assert 4 * own < taken < 4 * (own + weights) + 4.2 * own + slack, (taken, own, weights)
    for l in layers[:3]:
        l.close()
    assert before - free() > 4 * own
    layers[3].close()
    assert before - free() < slack
    short.close()


@pytest.mark.parametrize("name", ["c2_bf16_prefill", "qwen36_release", "c4_mxfp8_mx_activation",
                                  "c5_mxfp4_dsv41"])
def test_layers_that_round_to_bf16_keep_16_bit_rows(name):
    # where the routed outputs are stored as BF16, the whole workspace of a 1024-token layer is
    # smaller than those outputs in f32 would be
    T, H, k = 1024, 2048, 8
    host = _small_layer(name, hidden=H)
    assert host.spec.top_k == k
    layer = moe_mod().MoeLayer(host, max_tokens=T)
    assert layer.memory()[1] < T * k * H * 4, layer.memory()
    x = synth.activations(f"x.rows16.{name}", T, H)
    y, ids, _ = layer.forward(torch.from_numpy(x).cuda())
    ref = _oracle(host, x)
    assert ids_match(ids.cpu().numpy(), ref.ids, _scores(host.spec, ref, host.correction_bias))
    assert rel_l2(y.cpu().numpy(), ref.output) < REL_L2_BAR
    layer.close()
