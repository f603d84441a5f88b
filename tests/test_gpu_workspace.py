"""The per-stream workspace of the calls that take one (kg_gfx950_entry.hip, split_workspace): the
fp32 partial sums of a K split over workgroups, packed operands, a conv's channel-last copy, the
partial outputs of split keys. One call of each kind, its route checked by its cost record, is run
from two threads on one stream, on more streams than buffers are kept for, with buffers that are
replaced by larger ones meanwhile, in recorded graphs, and while another thread records one. A
call's sums are in a fixed order, so its bits are compared with those of a call by itself."""

from __future__ import annotations

import threading

import pytest

from kernelcode_generate_amd import native

pytestmark = pytest.mark.gpu

# name: (operation, dtype, sizes, MFMA instructions of the route meant)
CALLS = {
    # matmul (M, K, N): 6 tiles of 128 x 256 and 46 slices of 32, in 5 K chunks
    "matmul_split": ("matmul", "bfloat16", (371, 1472, 328), 6 * 46 * 128),
    # 15 tiles of 128 x 256 and 80 slices, in 10 chunks (16.3 MB of partials)
    "matmul_split_large": ("matmul", "bfloat16", (384, 2560, 1064), 15 * 80 * 128),
    # odd rows: 6 tiles of 64 x 64 and 63 slices of 64, in 7 chunks
    "matmul_packed": ("matmul", "float16", (170, 4001, 99), 6 * 63 * 32),
    "matmul_packed_f32": ("matmul", "float32", (170, 4001, 99), 6 * 126 * 128),
    # conv (images, filters, stride, pad, memory_stage): the row-piece kernel, 14 tiles of 64 x 128, split
    "conv_rowvec": ("conv2d", "float16", ((1, 128, 28, 28), (128, 128, 3, 3), 1, 1, None), 7 * 24 * 16 * 3),
    # the gathering kernel (a set stage count), 4 tiles and 144 slices, in 36 chunks
    "conv_gather": ("conv2d", "bfloat16", ((2, 512, 7, 7), (512, 512, 3, 3), 1, 1, 2), 4 * 144 * 4 * 2 * 2 * 2),
    # the channel-last copy, 8 tiles of 64 x 64 and 45 slices, split; 1568 of 128 x 64 and 4 slices (13.5 MB)
    "conv_copy": ("conv2d", "bfloat16", ((2, 300, 15, 15), (64, 300, 3, 3), 1, 1, None), 8 * 45 * 32),
    "conv_copy_large": ("conv2d", "float16", ((16, 3, 224, 224), (64, 3, 7, 7), 2, 3, None), 1568 * 4 * 64),
    # attention (B, H, S_q, S_kv, D): 8 heads of one query and 128 steps of 32 keys, 16 ranges of keys
    "attention_bf16": ("attention", "bfloat16", (1, 8, 1, 4096, 128), 8 * 128 * 17),
    "attention_f32": ("attention", "float32", (1, 2, 16, 2000, 64), 2 * 125 * 32),
}
NAMES = [n for n in CALLS if not n.endswith("_large")]


def make(name, device, seed=0):
    """(call, output shape, dtype) of CALLS[name]: call(out) runs it on fixed inputs."""

    import torch

    op, dtype_name, size, mfma = CALLS[name]
    dt = getattr(torch, dtype_name)
    gen = torch.Generator(device=device).manual_seed(seed + len(name))

    def draw(*shape, scale=1.0):
        return (torch.randn(shape, generator=gen, device=device) * scale).to(dt)

    if op == "matmul":
        m, k, n = size
        args = (draw(m, k), draw(k, n, scale=k**-0.5), draw(n))
        shape, scalars = (m, n), ()
        entry = "kg_gfx950_matmul_entry"
    elif op == "conv2d":
        xs, ws, stride, pad, stage = size
        args = (draw(*xs), draw(*ws, scale=(ws[1] * ws[2] * ws[3]) ** -0.5), draw(ws[0]))
        side = [(xs[i] + 2 * pad - ws[i]) // stride + 1 for i in (2, 3)]
        shape = (xs[0], ws[0], *side)
        scalars = (stride, stride, 1, 1, pad, pad, pad, pad) + (() if stage is None else (1, 1, 1, 1, 1, stage))
        entry = "kg_gfx950_conv2d_entry"
    else:
        b, h, s_q, s_kv, d = size
        args = (draw(b, h, s_q, d), draw(b, h, s_kv, d), draw(b, h, s_kv, d))
        shape, scalars = (b, h, s_q, d), (64, 64, d**-0.5, 0)
        entry = "kg_gfx950_flash_attention_entry"
    family = {"attention": "flash_attention"}.get(op, op)
    specs = [native.TensorSpec(shape, dtype_name), *(native.TensorSpec.of(a) for a in args)]
    model = native.cost(family, [*specs, *scalars])
    assert model["MFMA"] == mfma, f"{name} takes another route: {model['MFMA']} MFMAs"
    torch.cuda.synchronize()

    def call(out):
        native.call_entry(entry, (out, *args, *scalars))

    return call, shape, dt


def alone(name, device, seed=0):
    """(call, a function that makes an output, the call's result by itself)."""

    import torch

    call, shape, dt = make(name, device, seed)

    def output():
        return torch.full(shape, float("nan"), dtype=dt, device=device)

    expected = output()
    torch.cuda.synchronize()
    native.set_launch_mode(True, None)
    call(expected)
    assert torch.isfinite(expected).all()
    return call, output, expected


def run_threads(workers):
    errors: list[BaseException] = []
    start = threading.Barrier(len(workers))

    def guarded(worker):
        try:
            start.wait()
            worker()
        except BaseException as exc:  # noqa: BLE001 - reported by the main thread
            errors.append(exc)

    threads = [threading.Thread(target=guarded, args=(w,)) for w in workers]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in threads), "a worker did not finish"
    assert not errors, errors


@pytest.mark.parametrize(
    "first,second",
    [("matmul_split", "conv_copy"), ("matmul_packed", "attention_bf16"), ("conv_rowvec", "matmul_packed_f32"),
     ("conv_gather", "attention_f32"), ("conv_copy", "conv_rowvec")],
)
def test_two_threads_on_one_stream(device, first, second):
    """Two synchronous threads on the default stream: a call's launches are not parted by another
    call that writes the same workspace."""

    import torch

    made = [alone(n, device) for n in (first, second)]
    wrong: list[tuple[str, int]] = []

    def worker(name, call, output, expected):
        native.set_launch_mode(True, None)
        for r in range(30):
            out = output()
            call(out)
            if not torch.equal(out, expected):
                wrong.append((name, r))

    print(f"[workspace] two threads: {first}, {second}", flush=True)
    run_threads([lambda n=n, m=m: worker(n, *m) for n, m in zip((first, second), made)])
    assert not wrong, wrong


def test_larger_requests_from_another_thread(device):
    """On each of ten streams one thread enqueues small calls while another's calls ask for ever
    larger workspaces, so a buffer with work still enqueued on it is replaced."""

    import torch

    small = alone("matmul_split", device)
    growing = [alone(n, device) for n in ("attention_bf16", "conv_copy", "conv_copy_large", "matmul_split_large")]
    for trial in range(10):
        stream = torch.cuda.Stream(device=device)
        small_out = [small[1]() for _ in range(12)]
        growing_out = [m[1]() for m in growing]
        torch.cuda.synchronize()
        print(f"[workspace] growing requests, stream {trial}", flush=True)

        def enqueue(calls):
            native.set_launch_mode(False, stream.cuda_stream)
            for call, out in calls:
                call(out)

        run_threads([lambda: enqueue([(small[0], o) for o in small_out]),
                     lambda: enqueue([(m[0], o) for m, o in zip(growing, growing_out)])])
        torch.cuda.synchronize()
        for out in small_out:
            assert torch.equal(out, small[2]), f"trial {trial}"
        for m, out in zip(growing, growing_out):
            assert torch.equal(out, m[2]), f"trial {trial}"


def test_more_streams_than_buffers(device):
    """Two rounds over 11 streams, every kind of call on each: the ninth and later streams take
    over the least recently used buffer (8 are kept per device)."""

    import torch

    streams = [torch.cuda.Stream(device=device) for _ in range(11)]
    made = {n: alone(n, device) for n in NAMES}
    results = []
    outputs = {(r, i, n): made[n][1]() for r in range(2) for i in range(len(streams)) for n in NAMES}
    torch.cuda.synchronize()
    try:
        for rnd in range(2):
            for i, stream in enumerate(streams):
                print(f"[workspace] round {rnd} stream {i}", flush=True)
                native.set_launch_mode(False, stream.cuda_stream)
                for n in NAMES:
                    out = outputs[rnd, i, n]
                    made[n][0](out)
                    results.append((rnd, i, n, out))
    finally:
        native.set_launch_mode(True, None)
    torch.cuda.synchronize()
    for rnd, i, n, out in results:
        assert torch.equal(out, made[n][2]), f"{n}, round {rnd} stream {i}"


def capture(stream, *calls):
    """A graph of calls [(call, out)] recorded on stream."""

    import torch

    graph = torch.cuda.CUDAGraph()
    try:
        with torch.cuda.graph(graph, stream=stream):
            native.set_launch_mode(False, stream.cuda_stream)
            for call, out in calls:
                call(out)
    finally:
        native.set_launch_mode(True, None)
    return graph


@pytest.mark.parametrize("warm", [True, False], ids=["warm", "cold"])
@pytest.mark.parametrize("name", NAMES)
def test_captured_calls_have_a_workspace_of_their_own(device, name, warm):
    """A graph recorded on a stream that has a workspace (warm) or has not (where allocating as usual
    would invalidate the recording) holds none of it: after a larger call on that stream has
    replaced the buffer, and while others write to the new one, every replay gives the call's bits."""

    import torch

    call, output, expected = alone(name, device)
    larger, larger_output, larger_expected = alone("conv_copy_large", device)
    stream = torch.cuda.Stream(device=device)
    eager, out, big = output(), output(), larger_output()
    torch.cuda.synchronize()
    try:
        native.set_launch_mode(False, stream.cuda_stream)
        if warm:
            call(eager)
            stream.synchronize()
        print(f"[workspace] capture {name} warm={warm}", flush=True)
        graph = capture(stream, (call, out))
        native.set_launch_mode(False, stream.cuda_stream)
        larger(big)
        stream.synchronize()
        assert torch.equal(big, larger_expected) and (not warm or torch.equal(eager, expected))
        for _ in range(3):
            for t in (out, eager, big):
                t.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            larger(big)
            call(eager)
            torch.cuda.synchronize()
            assert torch.equal(out, expected) and torch.equal(eager, expected) and torch.equal(big, larger_expected)
    finally:
        native.set_launch_mode(True, None)


def test_graphs_of_one_stream_replayed_together(device):
    """Two graphs recorded on one stream, of all kinds of call each in another order (so buffers
    are shared within a graph and outgrown), replayed at once on two streams."""

    import torch

    made = [alone(n, device) for n in CALLS]
    recording = torch.cuda.Stream(device=device)
    replaying = [torch.cuda.Stream(device=device) for _ in range(2)]
    outs = [[m[1]() for m in made] for _ in range(2)]
    torch.cuda.synchronize()
    orders = [list(range(len(made))), list(range(len(made)))[::-1]]
    print("[workspace] two graphs at once", flush=True)
    graphs = [capture(recording, *((made[i][0], outs[g][i]) for i in orders[g])) for g in range(2)]
    for _ in range(5):
        for row in outs:
            for out in row:
                out.fill_(float("nan"))
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, replaying):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        for row in outs:
            for m, out, n in zip(made, row, CALLS):
                assert torch.equal(out, m[2]), n


def test_graphs_give_their_workspaces_back(device):
    """The buffers of dropped graphs are freed: ten times eight graphs of 13.5 MB each, replayed and
    dropped, take no more of the device's memory in the end than after the first eight; a graph
    replays correctly after others are gone."""

    import torch

    call, output, expected = alone("conv_copy_large", device)
    stream = torch.cuda.Stream(device=device)
    kept_out, out, eager = output(), output(), output()
    torch.cuda.synchronize()
    kept = capture(stream, (call, kept_out))
    free = []
    for turn in range(10):
        print(f"[workspace] turn {turn} of graphs", flush=True)
        graphs = [capture(stream, (call, out)) for _ in range(8)]
        for graph in graphs:
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, expected)
        del graphs, graph
        call(eager)  # (takes a workspace outside a recording)
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info(device)[0])
    assert free[-1] >= free[0] - (32 << 20), free
    kept_out.fill_(float("nan"))
    kept.replay()
    torch.cuda.synchronize()
    assert torch.equal(kept_out, expected)


def test_first_call_while_another_thread_records(device):
    """A stream's first call that takes a workspace, made while another thread records a graph (in
    the mode that refuses other threads' allocations): the call's bits are those it has otherwise,
    and the recording is not disturbed."""

    import torch

    streams = [torch.cuda.Stream(device=device) for _ in range(11)]
    call, output, expected = alone("matmul_packed_f32", device)
    recorded, recorded_output, recorded_expected = alone("matmul_split", device)
    fresh, recording = streams[0], streams[10]
    for s in streams[1:10]:  # nine other streams: whatever buffer `fresh` had has gone to one of them
        out = output()
        torch.cuda.synchronize()
        native.set_launch_mode(False, s.cuda_stream)
        call(out)
        s.synchronize()
    out, graph_out = output(), recorded_output()
    torch.cuda.synchronize()
    print("[workspace] a first call while another thread records", flush=True)

    def from_another_thread(_):
        def worker():
            native.set_launch_mode(False, fresh.cuda_stream)
            call(out)

        run_threads([worker])

    graph = capture(recording, (recorded, graph_out), (from_another_thread, None))
    torch.cuda.synchronize()
    assert torch.equal(out, expected)
    for _ in range(3):
        graph_out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(graph_out, recorded_expected)
