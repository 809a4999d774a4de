"""Recorded batches: a decode step captured once into a HIP graph and replayed with new inputs and
positions must give, replay after replay, the bits of the same step issued eagerly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layer(pkg, ctx, g, pld=0, n_layers=1, idx=0, **kw):
    dims = dict(hidden_size=512, intermediate_size=1024, num_attention_heads=4, num_key_value_heads=1, head_dim=256)
    t = pkg.synth.decoder_layer_tensors(512, 1024, 4, 1, 256, pld, g, **kw)
    params = pkg.layer.LayerParams(layer_idx=idx, per_layer_dim=pld, **dims)
    return pkg.layer.TransformerLayer(params, pkg.layer.LayerWeights.from_host(ctx, t))


@pytest.mark.parametrize("n_lanes", [1, 3, 40])
def test_captured_decode_step_replays_like_eager(pkg, gpu, n_lanes):
    ctx, K = gpu
    g = pkg.synth.rng(950, n_lanes)
    pld, n_layers, lane_cap = 256, 2, 64
    layers = [_layer(pkg, ctx, g, pld, n_layers, i, output_scale=0.5 + 0.25 * i) for i in range(n_layers)]
    pools = [[pkg.QuantizedUnifiedKvPool(ctx, n_lanes, lane_cap, 1, 256, 2, 0) for _ in range(n_layers)] for _ in range(2)]
    for side in pools:
        for p in side:
            p.reset()
    bs = pkg.layer.BatchScratch(ctx, n_lanes, 512, 1024, 4, 1, 256, pld, n_layers)
    ones = pkg.Buffer.from_slice(ctx, np.ones(256, np.float16))
    xin = pkg.Buffer.empty(ctx, n_lanes * 1024)
    ple = pkg.Buffer.empty(ctx, n_lanes * n_layers * pld * 2)
    pos_buf = pkg.Buffer.empty(ctx, n_lanes * 4)
    outs = [pkg.Buffer.empty(ctx, n_lanes * 1024) for _ in range(2)]
    mids = [pkg.Buffer.empty(ctx, n_lanes * 1024) for _ in range(2)]

    def encode(batch, side):
        layers[0].forward_decode_batch_turbo(batch, K, n_lanes, pos_buf, xin, mids[side], bs, ones, pools[side][0], (ple, n_layers))
        layers[1].forward_decode_batch_turbo(batch, K, n_lanes, pos_buf, mids[side], outs[side], bs, ones, pools[side][1],
                                             (ple, n_layers))

    batch = pkg.CommandBatch(ctx)
    batch.begin_capture()
    encode(batch, 0)
    graph = batch.end_capture()
    assert graph.dispatch_count() >= 16          # two layers of 8 - 10 encoded steps each
    ctx.synchronize()
    assert not outs[0].as_array(np.uint16).any()          # recording runs nothing

    positions = (np.arange(n_lanes, dtype=np.uint32) * 5) % 23
    for step in range(7):
        xin.copy_from_bytes(g.standard_normal(n_lanes * 512, dtype=np.float32).astype(np.float16))
        ple.copy_from_bytes(g.standard_normal(n_lanes * n_layers * pld, dtype=np.float32).astype(np.float16))
        pos_buf.copy_from_bytes(positions)
        graph.launch()
        ctx.synchronize()
        got = outs[0].as_array(np.uint16)
        eager = pkg.CommandBatch(ctx)
        encode(eager, 1)
        eager.commit_and_wait()
        want = outs[1].as_array(np.uint16)
        assert np.isfinite(want.view(np.float16).astype(np.float32)).all() and want.any()
        assert np.array_equal(got, want), f"replay {step}"
        for a, b in zip(pools[0], pools[1]):
            assert np.array_equal(a.keys_q.as_array(np.uint8), b.keys_q.as_array(np.uint8))
            assert np.array_equal(a.value_norms.as_array(np.uint16), b.value_norms.as_array(np.uint16))
        positions += 1


def test_capture_refuses_what_a_graph_cannot_hold(pkg, gpu):
    ctx, K = gpu
    buf = pkg.Buffer.empty(ctx, 256)
    a, b = pkg.Buffer.from_slice(ctx, np.ones(64, np.float16)), pkg.Buffer.from_slice(ctx, np.ones(64, np.float16))
    batch = pkg.CommandBatch(ctx)
    batch.begin_capture()
    try:
        with pytest.raises(pkg.InvalidArgument):
            pkg.CommandBatch(ctx).begin_capture()
        with pytest.raises(pkg.InvalidArgument):
            pkg.Buffer.empty(ctx, 16)
        with pytest.raises(pkg.InvalidArgument):
            pkg.Buffer.from_slice(ctx, np.zeros(4, np.float32))
        with pytest.raises(pkg.InvalidArgument):
            buf.as_array(np.uint8)
        with pytest.raises(pkg.InvalidArgument):
            buf.copy_from_bytes(np.zeros(4, np.uint8))
        with pytest.raises(pkg.InvalidArgument):
            buf.fill_zero()
        with pytest.raises(pkg.InvalidArgument):
            batch.commit_and_wait()
        with pytest.raises(pkg.InvalidArgument):
            ctx.synchronize()
        K.residual_add_into(batch, a, b, buf, 64)
    finally:
        graph = batch.end_capture()
    with pytest.raises(pkg.InvalidArgument):
        batch.end_capture()
    assert graph.dispatch_count() == 1
    assert not buf.as_array(np.uint16, 64).any()
    graph.launch()
    ctx.synchronize()
    assert (buf.as_array(np.float16, 64) == 2.0).all()
    graph.free()
    assert pkg.Buffer.empty(ctx, 16).length() == 16       # the context is usable again


def test_buffer_released_during_capture_lives_as_long_as_the_graph(pkg, gpu):
    """A scratch buffer that a recorded dispatch writes and a later one reads is released by its owner while the
    capture is still open (as a Rust scope would drop it).  The graph keeps the allocation: several replays, with
    other allocations made in between (which would reuse a freed block), still give the right sums."""
    ctx, K = gpu
    n = 4096
    a = pkg.Buffer.from_slice(ctx, np.full(n, 1.5, np.float16))
    b = pkg.Buffer.from_slice(ctx, np.full(n, 2.0, np.float16))
    out = pkg.Buffer.empty(ctx, n * 2)
    scratch = pkg.Buffer.empty(ctx, n * 2)          # created before the capture: allocation is refused inside one
    batch = pkg.CommandBatch(ctx)
    batch.begin_capture()
    K.residual_add_into(batch, a, b, scratch, n)          # scratch = a + b
    K.residual_add_into(batch, scratch, b, out, n)        # out = scratch + b
    scratch.free()                                         # dropped while the capture is open
    graph = batch.end_capture()
    filler = []
    for step in range(4):
        # allocations of the same size between replays: a block freed too early would be handed out here and overwritten
        filler.append(pkg.Buffer.from_slice(ctx, np.full(n, 100.0 + step, np.float16)))
        a.copy_from_bytes(np.full(n, 1.5 + step, np.float16))
        out.fill_zero()
        graph.launch()
        ctx.synchronize()
        got = out.as_array(np.float16, n).astype(np.float32)
        assert (got == 1.5 + step + 4.0).all(), f"replay {step}: {got[:4]}"
    graph.free()


def test_graph_released_during_capture_does_not_disturb_it(pkg, gpu):
    """An older graph may be collected at any time, also while another is being recorded."""
    ctx, K = gpu
    n = 4096
    a, out = pkg.Buffer.from_slice(ctx, np.full(n, 1.5, np.float16)), pkg.Buffer.empty(ctx, n * 2)
    batch = pkg.CommandBatch(ctx)
    batch.begin_capture()
    K.residual_add_into(batch, a, a, out, n)
    old = batch.end_capture()
    batch.begin_capture()
    K.residual_add_into(batch, a, a, out, n)
    old.free()
    K.residual_add_into(batch, out, a, out, n)
    graph = batch.end_capture()
    for step in range(3):
        a.copy_from_bytes(np.full(n, 1.0 + step, np.float16))
        graph.launch()
        ctx.synchronize()
        assert (out.as_array(np.float16, n) == 3.0 + 3 * step).all()
    graph.free()


@pytest.mark.parametrize("size", [1, 3, 4, 63, 64, 65, 1028, 2047, 2048, 2049, 5001])
@pytest.mark.parametrize("offset", [0, 1, 4, 6])
def test_host_bytes_in_the_order_of_the_batch(pkg, gpu, size, offset):
    """CommandBatch.write: as kernel arguments up to 2 KB and copied beyond, in order with the dispatches around it, from a source that
    is overwritten at once; what lies around the range stays, and it is refused past the end and while a graph is recorded."""
    ctx, K = gpu
    g = pkg.synth.rng(5, size + offset)
    first, second = (g.integers(0, 256, size, dtype=np.uint8) for _ in range(2))
    a, b, batch = pkg.Buffer.from_slice(ctx, np.full(6000, 7, np.uint8)), pkg.Buffer.empty(ctx, 6000), pkg.CommandBatch(ctx)
    src = first.copy()
    batch.write(a, src, offset)
    src[:] = second
    batch.blit_copy(a, 0, b, 0, 6000)
    batch.write(a, src, offset)
    batch.commit_and_wait()
    for buf, want in ((a, second), (b, first)):
        got, around = buf.as_array(np.uint8), np.full(6000, 7, np.uint8)
        around[offset:offset + size] = want
        assert np.array_equal(got, around)
    with pytest.raises(pkg.InvalidArgument):
        batch.write(a, src, 6001 - size)
    batch.begin_capture()
    with pytest.raises(pkg.InvalidArgument):
        batch.write(a, src, 0)
    batch.end_capture()
    batch.write(a, src, 0)
    batch.commit_and_wait()


@pytest.mark.parametrize("size", [4, 64, 68, 2048, 2052, 2050, 8192, 9001, 65536, 65540])
@pytest.mark.parametrize("offset", [0, 4])
def test_writes_in_stream_order(pkg, gpu, size, offset):
    """Host data of every route -- launch arguments, staging memory, a copy -- lands in the order of the dispatches around it, more
    writes in a row than there are staging slots, and the source may change as soon as the call is back."""
    ctx, K = gpu
    g, batch = np.random.default_rng(size + offset), pkg.CommandBatch(ctx)
    dst, copies = pkg.Buffer.empty(ctx, offset + size + 16), [pkg.Buffer.empty(ctx, size) for _ in range(7)]
    dst.copy_from_bytes(np.full(offset + size + 16, 7, np.uint8))
    want = []
    for c in copies:
        src = g.integers(0, 256, size, dtype=np.uint8)
        want.append(src.copy())
        batch.write(dst, src, offset)
        src[:] = 0
        if offset % 16 == 0 or size % 4 == 0:
            batch.blit_copy(dst, offset, c, 0, size)
    batch.commit_and_wait()
    got = dst.as_array(np.uint8)
    assert (got[:offset] == 7).all() and (got[offset + size:] == 7).all() and np.array_equal(got[offset:offset + size], want[-1])
    for c, w in zip(copies, want):
        if offset % 16 == 0 or size % 4 == 0:
            assert np.array_equal(c.as_array(np.uint8, size), w)


def test_writes_of_several_threads(pkg, gpu):
    """Staged writes of threads that share a context each carry their own bytes."""
    import threading
    ctx, K = gpu
    size, bad = 40000, []

    def work(i):
        g, batch, dst = np.random.default_rng(i), pkg.CommandBatch(ctx), pkg.Buffer.empty(ctx, 40000)
        for _ in range(40):
            src = g.integers(0, 256, size, dtype=np.uint8)
            batch.write(dst, src)
            if not np.array_equal(dst.as_array(np.uint8), src):
                bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("size", [1, 15, 4097, 16384, 16385, 131072, 262144, 262145])
@pytest.mark.parametrize("offset", [0, 1, 4, 16])
@pytest.mark.parametrize("behind", [False, True])
def test_reads_of_every_route(pkg, gpu, size, offset, behind):
    """Through pinned memory or by the runtime's copy, behind work that is still to run or with nothing to wait for: the bytes asked for, and
    nothing around them."""
    ctx, K = gpu
    src = np.random.default_rng(size + offset).integers(0, 256, size + 64, dtype=np.uint8)
    a, b, batch = pkg.Buffer.from_slice(ctx, src), pkg.Buffer.empty(ctx, size + 64), pkg.CommandBatch(ctx)
    batch.blit_copy(a, 0, b, 0, size + 64)
    if not behind:
        batch.commit_and_wait()
    out = np.full(size + 32, 7, np.uint8)
    b.read_into(out[16:size + 16], offset)
    assert np.array_equal(out[16:size + 16], src[offset:offset + size]) and (out[:16] == 7).all() and (out[size + 16:] == 7).all()


def test_pinned_buffers_take_what_device_buffers_take(pkg, gpu):
    """Writes of every size and way, views, copies from and to device memory, zeros."""
    ctx, K = gpu
    data = np.random.default_rng(5).integers(0, 256, 200003, dtype=np.uint8)
    p, d = pkg.Buffer.pinned(ctx, data.size), pkg.Buffer.empty(ctx, data.size)
    assert not p.as_array(np.uint8).any()
    p.copy_from_bytes(data)
    assert np.array_equal(p.as_array(np.uint8), data) and np.array_equal(p.view(77, 1000).as_array(np.uint8), data[77:1077])
    batch = pkg.CommandBatch(ctx)
    batch.blit_copy(p, 16, d, 0, 100000)
    for at, n in ((3, 60), (100, 2000), (4096, 5000), (20000, 100000)):
        batch.write(p.view(at, n), data[:n])
        assert np.array_equal(p.as_array(np.uint8)[at:at + n], data[:n]), n
    assert np.array_equal(d.as_array(np.uint8)[:100000], data[16:100016])
    batch.blit_copy(d, 0, p, 0, data.size)
    assert np.array_equal(p.as_array(np.uint8)[:100000], data[16:100016])
    p.fill_zero()
    assert not p.as_array(np.uint8).any()


def test_replays_write_a_pinned_buffer_and_keep_one_that_was_freed(pkg, gpu):
    """A recorded product with results in pinned memory, replayed on new inputs between eager work; a buffer that went while it was recorded lives as long."""
    ctx, K = gpu
    g = pkg.synth.rng(8, 1)
    rows, cols = 66001, 2048
    w = pkg.QuantWeight.from_bytes(ctx, pkg.synth.weights("q4_0", rows, cols, g), pkg.Q4_0, rows, cols)
    xs = [pkg.synth.activations(1, cols, g)[0].astype(np.float16) for _ in range(4)]
    x, y, eager = pkg.Buffer.from_slice(ctx, xs[0]), pkg.Buffer.empty(ctx, rows * 4), pkg.Buffer.empty(ctx, rows * 4)
    kept, gone = pkg.Buffer.pinned(ctx, rows * 4), pkg.Buffer.pinned(ctx, rows * 4)
    batch = pkg.CommandBatch(ctx)
    w.matvec_copied_into(batch, K, x, y, kept, 0.0)
    batch.commit_and_wait()
    batch.begin_capture()
    w.matvec_copied_into(batch, K, x, y, gone, 30.0)
    w.matvec_copied_into(batch, K, x, y, kept, 0.0)
    gone.free()
    graph = batch.end_capture()
    for v in xs:
        x.copy_from_bytes(v)
        graph.launch()
        got = kept.as_array(np.uint32)
        w.matvec_f32out_into(batch, K, x, eager)
        batch.commit_and_wait()
        assert np.array_equal(got, eager.as_array(np.uint32)) and np.array_equal(got, y.as_array(np.uint32))
