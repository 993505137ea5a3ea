"""fmx_attention_decode against a NumPy restatement of FreeMoe's decode
attention loop (engine.cpp:1360-1420, engine.cpp:378-393 softmax): per head,
scores float(double dot * scale) with the dot summed in index order, the
float maximum, double exponentials summed in position order,
p = float(e / sum), values summed in double in position order. The sums are
restated with np.add.accumulate (sequential, in order). Both sides use their
own exp (the device's and NumPy's, each within an ulp), so results are
compared within 1e-6 relative and most elements are expected bit for bit."""
import numpy as np
import pytest

from freemoe_amd import fmx

pytestmark = pytest.mark.gpu


def reference(q, kv, kv_heads, head_dim, v_offset, scale):
    heads = q.shape[0] // head_dim
    group = heads // kv_heads
    P = kv.shape[0]
    out = np.empty(heads * head_dim, np.float32)
    for h in range(heads):
        kvh = h // group
        qd = q[h * head_dim:(h + 1) * head_dim].astype(np.float64)
        k = kv[:, kvh * head_dim:(kvh + 1) * head_dim].astype(np.float64)
        dots = np.add.accumulate(k * qd, axis=1)[:, -1]
        s = (dots * scale).astype(np.float32)
        m = np.float64(s.max())
        e = np.exp(s.astype(np.float64) - m)
        total = np.add.accumulate(e)[-1]
        p = (e / total).astype(np.float32)
        v = kv[:, v_offset + kvh * head_dim:v_offset + (kvh + 1) * head_dim].astype(np.float64)
        acc = np.add.accumulate(p.astype(np.float64)[:, None] * v, axis=0)[-1]
        out[h * head_dim:(h + 1) * head_dim] = acc.astype(np.float32)
    return out


CASES = {
    # name: (heads, kv_heads, head_dim, positions, row padding floats)
    "one_position": (4, 4, 64, 1, 0),
    "mha_32x128_513": (32, 32, 128, 513, 0),
    "gqa_8_of_2_300": (8, 2, 64, 300, 8),
    "long_4000": (4, 4, 128, 4000, 0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_attention_decode_vs_engine_restatement(gpu, name):
    import torch
    heads, kvh, D, P, pad = CASES[name]
    rng = np.random.default_rng(hash(name) & 0xFFFF)
    kv_dim = kvh * D
    stride = 2 * kv_dim + pad
    kv = (rng.standard_normal((P, stride)) * 0.5).astype(np.float32)
    q = (rng.standard_normal(heads * D) * 0.5).astype(np.float32)
    scale = 1.0 / np.sqrt(float(D))
    want = reference(q, kv, kvh, D, kv_dim, scale)
    qd = torch.from_numpy(q).to(gpu)
    kvd = torch.from_numpy(kv).to(gpu)
    out = torch.empty(heads * D, dtype=torch.float32, device=gpu)
    ws = torch.zeros(256, dtype=torch.uint8, device=gpu)
    fmx.call("fmx_attention_decode", qd.data_ptr(), kvd.data_ptr(), stride, kv_dim, heads, kvh, D, P, scale,
             out.data_ptr(), ws.data_ptr(), 256, fmx.stream_handle())
    torch.cuda.synchronize()
    assert fmx.lib().fmx_moe_status(ws.data_ptr(), fmx.stream_handle()) == 0
    got = out.cpu().numpy()
    err = np.abs(got.astype(np.float64) - want) / np.maximum(np.abs(want).max(), 1e-30)
    assert err.max() <= 1e-6, err.max()
    same = np.mean(got.view(np.uint32) == want.view(np.uint32))
    print(f"{name}: {same:.4%} of outputs bit for bit")
    assert same >= 0.9


def test_attention_decode_reports_nonfinite_scores(gpu):
    import torch
    heads, kvh, D, P = 2, 2, 32, 5
    kv = np.zeros((P, 2 * kvh * D), np.float32)
    kv[3, 0] = np.inf
    q = np.ones(heads * D, np.float32)
    qd, kvd = torch.from_numpy(q).to(gpu), torch.from_numpy(kv).to(gpu)
    out = torch.empty(heads * D, dtype=torch.float32, device=gpu)
    ws = torch.zeros(256, dtype=torch.uint8, device=gpu)
    fmx.call("fmx_attention_decode", qd.data_ptr(), kvd.data_ptr(), 2 * kvh * D, kvh * D, heads, kvh, D, P, 0.5,
             out.data_ptr(), ws.data_ptr(), 256, fmx.stream_handle())
    assert fmx.lib().fmx_moe_status(ws.data_ptr(), fmx.stream_handle()) == 4  # FMX_ERR_INTERNAL


ORDERED = {
    # name: (heads, kv_heads, head_dim, positions): one and several slices and
    # groups of four heads, ragged head dims, thread counts and their edges,
    # scores in the value kernel and in the score kernel
    "one": (1, 1, 4, 1),
    "two": (3, 1, 36, 2),
    "tile_edge_64": (8, 8, 64, 64),
    "tile_edge_65": (10, 2, 64, 65),
    "ragged_dim_997": (12, 2, 100, 997),
    "wide_edge_1024": (8, 2, 96, 1024),
    "wide_edge_1025": (8, 2, 96, 1025),
    "gqa_32_of_8_2000": (32, 8, 128, 2000),
    "mqa_6_of_1x256_4099": (6, 1, 256, 4099),
    "longest_8192": (32, 32, 128, 8192),
    "beyond_the_slot": (72, 8, 64, 8192),
    # one workgroup per head and either side of that rule: the shortest caches,
    # more slices than CUs, more scores than a buffer holds
    "heads_71": (4, 2, 64, 71),
    "slices_72": (4, 2, 64, 72),
    "heads_260_slices": (65, 65, 64, 449),
    "slices_260_slices": (65, 65, 64, 450),
    "heads_ragged_dim": (180, 2, 100, 691),
    "slices_ragged_dim": (180, 2, 100, 693),
    "heads_beyond_the_slot": (260, 4, 64, 2100),
}


def ordered_on_exp(q, kv, kv_heads, head_dim, v_offset, scale, gpu):
    """reference() with the device's exp, so that every bit is determined."""
    import torch
    heads = q.shape[0] // head_dim
    out = np.empty(heads * head_dim, np.float32)
    for h in range(heads):
        kvh = h // (heads // kv_heads)
        qd = q[h * head_dim:(h + 1) * head_dim].astype(np.float64)
        k = kv[:, kvh * head_dim:(kvh + 1) * head_dim].astype(np.float64)
        s = (np.add.accumulate(k * qd, axis=1)[:, -1] * scale).astype(np.float32).astype(np.float64)
        e = torch.exp(torch.from_numpy(s - s.max()).to(gpu)).cpu().numpy()
        p = (e / np.add.accumulate(e)[-1]).astype(np.float32).astype(np.float64)
        v = kv[:, v_offset + kvh * head_dim:v_offset + (kvh + 1) * head_dim].astype(np.float64)
        with np.errstate(invalid="ignore"):
            out[h * head_dim:(h + 1) * head_dim] = np.add.accumulate(p[:, None] * v, axis=0)[-1]
    return out


@pytest.mark.parametrize("spread", ["normal", "flat", "peaked"])
@pytest.mark.parametrize("name", list(ORDERED))
def test_attention_decode_keeps_the_ordered_sums(gpu, name, spread):
    """Bit for bit the sums in position order, whichever of the certified and
    the ordered way an element takes; cancelling, zero and infinite values,
    and scores whose exponentials tie, lie far apart or are all alike."""
    import torch
    heads, kvh, D, P = ORDERED[name]
    rng = np.random.default_rng(P * 31 + heads + len(spread))
    kv_dim = kvh * D
    kv = (rng.standard_normal((P, 2 * kv_dim)) * 0.5).astype(np.float32)
    q = (rng.standard_normal(heads * D) * {"normal": 0.5, "flat": 0.0, "peaked": 6.0}[spread]).astype(np.float32)
    kv[1::2, kv_dim] = -kv[:P - P % 2:2, kv_dim]  # element 0 cancels (where the weights allow)
    kv[:, kv_dim + 1] = 0.0
    kv[P // 2, kv_dim + 2] = np.inf
    kv[:, kv_dim + 3] *= np.float32(1e-38)
    scale = 1.0 / np.sqrt(float(D))
    want = ordered_on_exp(q, kv, kvh, D, kv_dim, scale, gpu)
    qd, kvd = torch.from_numpy(q).to(gpu), torch.from_numpy(kv).to(gpu)
    ws = torch.zeros(256, dtype=torch.uint8, device=gpu)
    for _ in range(2):
        out = torch.full((heads * D,), 7.0, dtype=torch.float32, device=gpu)
        fmx.call("fmx_attention_decode", qd.data_ptr(), kvd.data_ptr(), 2 * kv_dim, kv_dim, heads, kvh, D, P, scale,
                 out.data_ptr(), ws.data_ptr(), 256, fmx.stream_handle())
        assert fmx.lib().fmx_moe_status(ws.data_ptr(), fmx.stream_handle()) == 0
        assert np.array_equal(out.cpu().numpy(), want, equal_nan=True)


def test_attention_decode_calls_in_flight_share_no_scores(gpu):
    """Twelve calls on streams of their own, each with its own inputs and
    workspace (as many run at once as the process has hardware queues)."""
    import torch
    heads, kvh, D, P = 8, 2, 64, 1500
    calls = []
    for i in range(12):
        g = torch.Generator(device=gpu).manual_seed(100 + i)
        calls.append(dict(q=torch.randn(heads * D, generator=g, device=gpu),
                          kv=torch.randn(P, 2 * kvh * D, generator=g, device=gpu),
                          ws=torch.zeros(256, dtype=torch.uint8, device=gpu), stream=torch.cuda.Stream(),
                          out=torch.empty(heads * D, device=gpu)))

    def run(c, out, stream):
        fmx.call("fmx_attention_decode", c["q"].data_ptr(), c["kv"].data_ptr(), 2 * kvh * D, kvh * D, heads, kvh, D, P,
                 0.125, out.data_ptr(), c["ws"].data_ptr(), 256, stream)

    want = []
    for c in calls:
        run(c, c["out"], fmx.stream_handle())
        torch.cuda.synchronize()
        want.append(c["out"].clone())
    torch.cuda.synchronize()
    for _ in range(5):
        for c in calls:
            c["out"].zero_()
        torch.cuda.synchronize()
        for c in calls:
            run(c, c["out"], c["stream"].cuda_stream)
        torch.cuda.synchronize()
        for c, w in zip(calls, want):
            assert torch.equal(c["out"], w)


def test_attention_decode_captured_and_replayed(gpu):
    """A captured call, replayed between eager ones: its ticket names one score
    buffer for every replay, and each replay gives the eager call's bits."""
    import torch
    heads, kvh, D, P = 8, 2, 64, 1500
    g = torch.Generator(device=gpu).manual_seed(9)
    q = torch.randn(heads * D, generator=g, device=gpu)
    kv = torch.randn(P, 2 * kvh * D, generator=g, device=gpu)
    ws = torch.zeros(256, dtype=torch.uint8, device=gpu)
    out, eager = torch.empty(heads * D, device=gpu), torch.empty(heads * D, device=gpu)

    def run(o):
        fmx.call("fmx_attention_decode", q.data_ptr(), kv.data_ptr(), 2 * kvh * D, kvh * D, heads, kvh, D, P, 0.125,
                 o.data_ptr(), ws.data_ptr(), 256, fmx.stream_handle())

    run(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(out)
    for i in range(12):
        q.normal_(generator=g)
        run(eager)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {i}"


class _Captured:
    """Long calls of one shape, each captured on its own (its ticket is fixed
    there), with its own inputs and workspace, to be run at once."""
    heads, kvh, D, P = 32, 8, 128, 8192

    def __init__(self, gpu, n):
        import ctypes
        import torch
        self.hip, self.calls, self.execs = ctypes.CDLL("libamdhip64.so.7"), [], []
        for i in range(n):
            g = torch.Generator(device=gpu).manual_seed(300 + i)
            c = dict(q=torch.randn(self.heads * self.D, generator=g, device=gpu),
                     kv=torch.randn(self.P, 2 * self.kvh * self.D, generator=g, device=gpu),
                     ws=torch.zeros(256, dtype=torch.uint8, device=gpu), out=torch.empty(self.heads * self.D, device=gpu))
            self.run(c)
            torch.cuda.synchronize()
            self.calls.append(dict(c, want=c["out"].clone()))

    def run(self, c):
        fmx.call("fmx_attention_decode", c["q"].data_ptr(), c["kv"].data_ptr(), 2 * self.kvh * self.D, self.kvh * self.D,
                 self.heads, self.kvh, self.D, self.P, 0.125, c["out"].data_ptr(), c["ws"].data_ptr(), 256,
                 fmx.stream_handle())

    def capture(self, c):
        import torch
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            self.run(c)
        return graph

    def instantiate(self, graph):
        import ctypes
        e = ctypes.c_void_p()
        assert self.hip.hipGraphInstantiate(ctypes.byref(e), ctypes.c_void_p(graph.raw_cuda_graph()), None, None,
                                            ctypes.c_size_t(0)) == 0
        self.execs.append(e)
        return e

    def together(self, *execs):
        """Runs the instantiated graphs on a stream each, let go at once by an
        event behind a pause, and checks every call's output."""
        import ctypes
        import torch
        for c in self.calls:
            c["out"].copy_(c["want"])
        for c, _ in execs:
            c["out"].zero_()
        torch.cuda.synchronize()
        go, gate, streams = torch.cuda.Event(), torch.cuda.Stream(), [torch.cuda.Stream() for _ in execs]
        with torch.cuda.stream(gate):
            torch.cuda._sleep(2_000_000)
            go.record()
        for (_, e), s in zip(execs, streams):
            s.wait_event(go)
            assert self.hip.hipGraphLaunch(e, ctypes.c_void_p(s.cuda_stream)) == 0
        torch.cuda.synchronize()
        for i, c in enumerate(self.calls):
            assert torch.equal(c["out"], c["want"]), i

    def close(self):
        for e in self.execs:
            assert self.hip.hipGraphExecDestroy(e) == 0


@pytest.mark.parametrize("between", range(8))
def test_attention_decode_two_calls_meet_in_one_score_buffer(gpu, between):
    """Two long calls at once, `between` other calls apart: for some of those
    both write the same score buffer, and each value workgroup that finds the
    other's scores there forms its own."""
    k = _Captured(gpu, 2)
    a, b = k.calls
    graphs = [k.capture(a)] + [k.capture(a) for _ in range(between)] + [k.capture(b)]
    ea, eb = k.instantiate(graphs[0]), k.instantiate(graphs[-1])
    for _ in range(4):
        k.together((a, ea), (b, eb))
        k.together((b, eb), (a, ea))
    k.close()


@pytest.mark.parametrize("between", range(8))
def test_attention_decode_one_capture_twice_at_once(gpu, between):
    """One captured call instantiated twice and both run at once, beside a
    third call `between` calls later. The two executions share a ticket and
    all their memory; neither disturbs the third."""
    k = _Captured(gpu, 2)
    a, b = k.calls
    graphs = [k.capture(a)] + [k.capture(a) for _ in range(between)] + [k.capture(b)]
    e1, e2, eb = k.instantiate(graphs[0]), k.instantiate(graphs[0]), k.instantiate(graphs[-1])
    for _ in range(4):
        k.together((a, e1), (a, e2), (b, eb))
        k.together((a, e1), (b, eb), (a, e2))
    k.close()
