"""Consecutive forwards overlap: with plain launches the model runtime runs the last, small operators
of a forward on a second stream, so that the next forward's first operators need not wait for them.
The results must be those of forwards run strictly one after the other: under the runtime's own memory
plan (which gives what those operators touch bytes of its own) and under a plan that does not (the
reference planner's, where their tensors share bytes with early layers' and the next forward has to
wait for them)."""
import numpy as np
import pytest

import cases
import mobilenet
from megcc_amd import abi, runtime

pytestmark = pytest.mark.gpu

BATCH = 32  # (kernels average over 6 us: the runtime uses two streams without asking)


class PlannedModel(runtime.Model):
    """runtime.Model that installs the reference planner's offsets for the operators' own lifetimes
    (no operator chains, no overlap: what a compiled model file carries) before it finalizes"""

    def __init__(self, net):
        super().__init__()
        lt = mobilenet.Lifetimes()
        net.build_gpu(model=lt)
        tids, begin, end, size = lt.requests()
        off, arena, _ = runtime.plan_memory(begin, end, size, 256)
        self.offsets = [0] * len(lt.sizes)
        for t, o in zip(tids, off):
            self.offsets[t] = int(o)
        self.arena = int(arena)

    def finalize(self):
        self.set_plan(self.offsets, self.arena)
        super().finalize()


def build(net, planned, keep_all=False, **options):
    for k, v in options.items():
        runtime.set_option(k, v)
    try:
        model, ids = net.build_gpu(keep_all=keep_all, model=PlannedModel(net) if planned else None)
        if options.get("no_graph"):  # (asked at the first forward: plain launches from then on)
            model.set_input(ids["image"], np.zeros((net.batch, 3, 224, 224), np.float32))
            model.forward()
            assert model.launch_mode()[0] == -1
        return model, ids
    finally:
        for k in options:
            runtime.set_option(k, 0)


@pytest.mark.parametrize("planned", [False, True], ids=["own_plan", "reference_plan"])
def test_overlapped_forwards_equal_forwards_run_one_after_the_other(planned):
    net = mobilenet.Net(BATCH)
    images = [mobilenet.draw_input(BATCH, seed=s) for s in (1, 2, 3, 4, 5)]
    # (no_graph: plain launches, no measuring phase)
    pipe, ids = build(net, planned, no_graph=1)
    serial, _ = build(net, planned, no_graph=1, nopipeline=1)
    assert pipe.nr_tail_kernel >= 2 and serial.nr_tail_kernel == 0
    assert pipe.nr_kernel - pipe.nr_tail_kernel >= 4
    if not planned:
        assert pipe.arena_bytes > serial.arena_bytes  # the tail's tensors have bytes of their own
    else:
        assert pipe.arena_bytes == serial.arena_bytes
    want = []
    for img in images:
        serial.set_input(ids["image"], img)
        serial.forward()
        want.append(serial.get(ids["softmax"]).copy())
    assert not np.array_equal(want[0], want[1])
    # forward, copy of its result and the next input enqueued without the host waiting for anything
    outs = [np.zeros((BATCH, 1000), np.float32) for _ in images]
    for img, out in zip(images, outs):
        pipe.set_input(ids["image"], img)
        pipe.forward()
        pipe.get_async(ids["softmax"], out)
    runtime.wait()
    for k, (o, w) in enumerate(zip(outs, want)):
        np.testing.assert_array_equal(o, w, err_msg="forward %d" % k)
    # forwards with nothing read in between, then the blocking read; and a forward read at once
    for _ in range(3):
        for img in images:
            pipe.set_input(ids["image"], img)
            pipe.forward()
    np.testing.assert_array_equal(pipe.get(ids["softmax"]), want[-1])
    pipe.set_input(ids["image"], images[0])
    pipe.forward()
    np.testing.assert_array_equal(pipe.get(ids["softmax"]), want[0])
    # the serial results themselves against the oracle (first input)
    ref, _ = mobilenet.Net(2).run_oracle(images[0][:2])  # (same weights: they do not depend on the batch)
    assert cases.max_rel_err(want[0][:2], ref) <= 1e-4
    pipe.close()
    serial.close()


def test_asynchronous_read_of_a_tensor_the_first_stream_writes():
    """every layer's result kept as an output: a layer far from the end is read between two forwards
    (that copy goes to the library stream, between this forward's operators and the next one's), the
    last layer's behind the second stream"""
    net = mobilenet.Net(BATCH)
    images = [mobilenet.draw_input(BATCH, seed=s) for s in (7, 8)]
    pipe, ids = build(net, False, keep_all=True, no_graph=1)
    serial, _ = build(net, False, keep_all=True, no_graph=1, nopipeline=1)
    assert pipe.nr_tail_kernel >= 2
    mid = np.zeros(pipe.shapes[ids["pw3"]][0], np.int8)
    last = np.zeros((BATCH, 1000), np.float32)
    pipe.set_input(ids["image"], images[0])
    pipe.forward()
    for img in images:
        pipe.set_input(ids["image"], img)
        pipe.forward()
        if img is images[0]:
            pipe.get_async(ids["pw3"], mid)
            pipe.get_async(ids["softmax"], last)
    runtime.wait()
    serial.set_input(ids["image"], images[0])
    serial.forward()
    np.testing.assert_array_equal(mid, serial.get(ids["pw3"]))
    np.testing.assert_array_equal(last, serial.get(ids["softmax"]))
    serial.set_input(ids["image"], images[1])
    serial.forward()
    np.testing.assert_array_equal(pipe.get(ids["softmax"]), serial.get(ids["softmax"]))
    pipe.close()
    serial.close()


def test_a_network_of_a_few_operators_keeps_one_stream():
    """fewer than four operators in front and two behind: nothing to overlap"""
    from cases import MultiTypeCase
    m = runtime.Model()
    x = m.tensor("x", (4, 64, 56, 56), abi.QINT8, 0.05)
    m.mark_input(x)
    t = x
    for k in range(5):
        y = m.tensor("relu%d" % k, (4, 64, 56, 56), abi.QINT8, 0.05)
        m.opr(MultiTypeCase(abi.Q_RELU, (4, 64, 56, 56), (0.05, 0.01, 0.05)).symbol(), [t], [y])
        t = y
    m.mark_output(t)
    runtime.set_option("no_graph", 1)
    try:
        m.finalize()
    finally:
        runtime.set_option("no_graph", 0)
    m.set_input(x, np.zeros((4, 64, 56, 56), np.int8))
    m.forward()
    assert m.nr_kernel == 5 and m.nr_tail_kernel == 0 and m.launched_tail_kernel == 0
    m.close()


def test_the_measuring_forwards_of_a_two_stream_model():
    """default options: forwards 2 + 3 and 7 + 8 are plain launches on two streams, 4 captures a graph
    (the tail of forward 3 still pending when the capture begins), 5 + 6 and 9 + 10 replay it, then the
    faster way runs. Same bytes throughout."""
    net = mobilenet.Net(BATCH)
    images = [mobilenet.draw_input(BATCH, seed=s) for s in (11, 12)]
    model, ids = build(net, False)
    serial, _ = build(net, False, no_graph=1, nopipeline=1)
    assert model.nr_tail_kernel >= 2
    want = []
    for img in images:
        serial.set_input(ids["image"], img)
        serial.forward()
        want.append(serial.get(ids["softmax"]).copy())
    model.set_input(ids["image"], images[0])
    for k in range(1, 13):
        model.forward()
        if k >= 4 and k % 2 == 0:
            np.testing.assert_array_equal(model.get(ids["softmax"]), want[0], err_msg="forward %d" % k)
    assert model.launch_mode()[0] in (1, -1)
    for img, w in zip(images[::-1], want[::-1]):
        model.set_input(ids["image"], img)
        model.forward()
        model.forward()
        np.testing.assert_array_equal(model.get(ids["softmax"]), w)
    model.close()
    serial.close()


@pytest.mark.parametrize("planned", [False, True], ids=["own_plan", "reference_plan"])
def test_two_hundred_overlapped_forwards(planned):
    """three inputs in rotation, every result copied out asynchronously, the host waits once at the
    end: each of the 200 results is the one of its input"""
    net = mobilenet.Net(BATCH)
    images = [mobilenet.draw_input(BATCH, seed=s) for s in (21, 22, 23)]
    pipe, ids = build(net, planned, no_graph=1)
    serial, _ = build(net, planned, no_graph=1, nopipeline=1)
    assert pipe.nr_tail_kernel >= 2
    want = []
    for img in images:
        serial.set_input(ids["image"], img)
        serial.forward()
        want.append(serial.get(ids["softmax"]).copy())
    outs = [np.zeros((BATCH, 1000), np.float32) for _ in range(200)]
    for k, out in enumerate(outs):
        pipe.set_input(ids["image"], images[k % 3])
        pipe.forward()
        pipe.get_async(ids["softmax"], out)
    runtime.wait()
    bad = [k for k, out in enumerate(outs) if not np.array_equal(out, want[k % 3])]
    assert not bad, bad[:10]
    pipe.close()
    serial.close()


@pytest.mark.parametrize("batch,forced,planned", [(32, True, False), (32, True, True), (112, False, False)],
                         ids=["32_forced_own_plan", "32_forced_reference_plan", "112_as_chosen"])
def test_forwards_with_a_run_of_blocks_as_one_kernel(batch, forced, planned):
    """the five blocks of 512 channels as one kernel among the others, on either stream and at the boundary between them: forwards back to
    back, a graph, the operators one by one. At 112 images whole forwards choose it, and memory is planned again without the run's tensors"""
    net = mobilenet.Net(batch)
    images = [mobilenet.draw_input(batch, seed=s) for s in (41, 42, 43)]
    serial, sids = build(net, False, no_graph=1, nopipeline=1)
    want = []
    for img in images:
        serial.set_input(sids["image"], img)
        serial.forward()
        want.append(serial.get(sids["softmax"]).copy())
    serial.close()
    assert not np.array_equal(want[0], want[1])
    for options in (dict(no_graph=1), {}):
        pipe, ids = build(net, planned, fuseblocks=int(forced), **options)
        without, _ = build(net, planned, nofuseblocks=1, no_graph=1)
        print(batch, "kernels", pipe.nr_kernel, "on the second stream", pipe.nr_tail_kernel, "without", without.nr_kernel)
        if not planned:
            assert pipe.nr_kernel <= without.nr_kernel - 4
        without.close()
        outs = [np.zeros((batch, 1000), np.float32) for _ in range(30)]
        for k, out in enumerate(outs):
            pipe.set_input(ids["image"], images[k % 3])
            pipe.forward()
            pipe.get_async(ids["softmax"], out)
        runtime.wait()
        bad = [k for k, out in enumerate(outs) if not np.array_equal(out, want[k % 3])]
        assert not bad, bad
        pipe.set_input(ids["image"], images[1])
        for i in range(pipe.nr_opr):
            pipe.run_opr(i)
        np.testing.assert_array_equal(pipe.get(ids["softmax"]), want[1])
        pipe.forward()
        np.testing.assert_array_equal(pipe.get(ids["softmax"]), want[1])
        pipe.close()


def test_a_forward_behind_a_wait_runs_on_one_stream():
    """whichever way the host has waited for the last forward - a blocking read, wait() after it, an asynchronous read and
    wait(), wait() and join() in either order with the next input in between -, the next one finds nothing to overlap; without a
    wait it uses the second stream. Every result is the one of its input"""
    net = mobilenet.Net(BATCH)
    images = [mobilenet.draw_input(BATCH, seed=s) for s in (31, 32, 33)]
    pipe, ids = build(net, False, no_graph=1)
    serial, _ = build(net, False, no_graph=1, nopipeline=1)
    tail = pipe.nr_tail_kernel
    assert tail >= 2
    want = []
    for img in images:
        serial.set_input(ids["image"], img)
        serial.forward()
        want.append(serial.get(ids["softmax"]).copy())
    out = np.zeros((BATCH, 1000), np.float32)

    def get():
        np.testing.assert_array_equal(pipe.get(ids["softmax"]), want[at])

    def get_async():
        pipe.get_async(ids["softmax"], out)

    def check():
        np.testing.assert_array_equal(out, want[at])

    ways = {  # what the caller does between two forwards: whether the second one's tail may overlap
        "nothing": ([], False), "get": ([get], True), "wait": ([runtime.wait], True), "async, wait": ([get_async, runtime.wait, check], True),
        "async": ([get_async], False), "join": ([pipe.join], False), "join, wait": ([pipe.join, runtime.wait], True),
        "wait, join": ([runtime.wait, pipe.join], True), "get, async": ([get, get_async], True), "wait, get": ([runtime.wait, get], True),
        # a read of another model waits for the library stream, on which this one's head is
        "other's get": ([lambda: serial.get(ids["softmax"])], False), "join, other's get": ([pipe.join, lambda: serial.get(ids["softmax"])], True),
    }
    at, before = 0, None
    for order in (list(ways), list(ways)[::-1], list(ways)[::2] * 2):
        for name in order:
            calls, waited = ways[name]
            # two forwards in front, the second one on two streams unless the first one's caller has waited
            at = (at + 1) % 3
            pipe.set_input(ids["image"], images[at])
            pipe.forward()
            pipe.forward()
            assert pipe.launched_tail_kernel == tail, (name, before)
            for call in calls:
                call()
            pipe.forward()
            assert pipe.launched_tail_kernel == (0 if waited else tail), (name, before)
            at = (at + 1) % 3
            pipe.set_input(ids["image"], images[at])
            pipe.forward()
            get()
            before = name
    pipe.close()
    serial.close()


def residual_net(n):
    """27 operators: four stages of two blocks (3x3, 3x3, addition), 64 channels at 56 x 56 to 512 at 7 x 7"""
    from cases import ConvCase, MultiTypeCase
    m = runtime.Model()
    names = iter(range(100))

    def tensor(shape):
        return m.tensor("t%d" % next(names), shape, abi.QINT8, 0.02)

    def conv(x, ic, oc, h, k, stride):
        case = ConvCase(abi.FMT_NCHW44, abi.DENSE, n, ic, h, h, oc, k, stride, k // 2, abi.RELU, scales=(0.02, 0.01, 0.02), flt_range=(-15, 15))
        arrays = case.gen(seed=oc + k)
        name = "w%d" % next(names)
        y = tensor(case.dst_shape())
        m.opr(case.symbol(), [x, m.weight(name, arrays["flt"], abi.QINT8, 0.01),
                              m.weight(name + "b", arrays["bias"], abi.QINT32, float(np.float32(0.02) * np.float32(0.01)))], [y])
        return y

    src = x = tensor((n, 16, 56, 56, 4))
    m.mark_input(x)
    c, h = 64, 56
    for stage in range(4):
        for block in range(2):
            stride, oc = (2 if stage and not block else 1), 64 << stage
            y = conv(x, c, oc, h, 3, stride)
            if stride == 2:
                x = conv(x, c, oc, h, 1, 2)
                h //= 2
            y = conv(y, oc, oc, h, 3, 1)
            shape = (n, oc // 4, h, h, 4)
            z = tensor(shape)
            m.opr(MultiTypeCase(abi.Q_FUSE_ADD_RELU, shape, (0.02, 0.02, 0.02)).symbol(), [x, y], [z])
            x, c = z, oc
    m.mark_output(x)
    m.finalize()
    return m, src, x


def test_two_streams_only_where_forwards_gain():
    """kernels of under 5 us on average and more of them than the host enqueues on two streams in the time they take: forwards one
    behind the other take no longer than on the one stream "nopipeline" keeps (two took 1.1 to 1.2 times as long)"""
    import time
    model, src, out = residual_net(1)
    runtime.set_option("nopipeline", 1)
    try:
        serial, ssrc, sout = residual_net(1)
    finally:
        runtime.set_option("nopipeline", 0)
    x = np.random.default_rng(5).integers(-128, 128, (1, 16, 56, 56, 4)).astype(np.int8)
    best = {}
    for m, i, o in ((model, src, out), (serial, ssrc, sout)):
        m.set_input(i, x)
        for _ in range(20):
            m.forward()
        best[m] = 1e9
    for _ in range(10):  # (in turn)
        for m in (model, serial):
            runtime.wait()
            t = time.perf_counter()
            for _ in range(60):
                m.forward()
            runtime.wait()
            best[m] = min(best[m], time.perf_counter() - t)
    np.testing.assert_array_equal(model.get(out), serial.get(sout))
    print("us a forward", best[model] / 60 * 1e6, "on one stream", best[serial] / 60 * 1e6)
    assert best[model] <= 1.07 * best[serial]
    model.close()
    serial.close()


def test_loading_a_network_of_many_images_costs_few_forwards():
    """at 80 images, where a run of blocks as one kernel wins nothing, no whole forwards are spent on the question (300 forwards with it, 200 without)"""
    import time
    net = mobilenet.Net(80)
    lengths = []
    for k in range(4):
        model, ids = net.build_gpu(model=Timed(lengths))
        if k < 3:
            model.close()
    model.set_input(ids["image"], mobilenet.draw_input(80, seed=1))
    forward = 1e9
    for _ in range(5):
        runtime.wait()
        t = time.perf_counter()
        for _ in range(20):
            model.forward()
        runtime.wait()
        forward = min(forward, (time.perf_counter() - t) / 20)
    print("finalize ms", [round(1e3 * v, 1) for v in lengths], "forward us", 1e6 * forward, "ratio", min(lengths) / forward)
    assert min(lengths) <= 250 * forward
    model.close()


class Timed(runtime.Model):
    def __init__(self, lengths):
        super().__init__()
        self.lengths = lengths

    def finalize(self):
        import time
        t = time.perf_counter()
        super().finalize()
        self.lengths.append(time.perf_counter() - t)


def test_loading_a_small_network_costs_few_forwards():
    """what finalize tries on a network of 5 us kernels takes less time than 130 of its forwards (seven boundaries between
    the streams: 160)"""
    import time
    net = mobilenet.Net(1)
    lengths = []
    for _ in range(5):  # (the first one loads the kernels)
        model, ids = net.build_gpu(model=Timed(lengths))
        model.set_input(ids["image"], mobilenet.draw_input(1, seed=1))
        for _ in range(20):
            model.forward()
        if len(lengths) < 5:
            model.close()
    forward = 1e9
    for _ in range(5):
        runtime.wait()
        t = time.perf_counter()
        for _ in range(20):
            model.forward()
            runtime.wait()
        forward = min(forward, (time.perf_counter() - t) / 20)
    print("finalize ms", [round(1e3 * v, 1) for v in lengths], "forward us", 1e6 * forward)
    assert min(lengths[1:]) <= 130 * forward
    model.close()
