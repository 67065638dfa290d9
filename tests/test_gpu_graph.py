"""HIP graph capture of the encoder path.

A serving loop captures the encoder once and replays it (hipGraphLaunch),
which removes the per-kernel host launch cost.  That works when a run, once
its runtime's workspaces exist, issues only kernel launches on the runtime's
stream: no allocation, no synchronisation, no memset (the balanced tail's
arrival counters are cleared by the kernels themselves).  The test warms
the runtime with one eager run, captures a block run (and a 3-layer encoder
run) on the runtime's stream through the HIP runtime API, and replays each
graph several times, alternating with the same run issued eagerly on a
second copy of the input and synchronising in between; every replay must
equal the eager result bit for bit.
"""
import ctypes

import numpy as np
import pytest

from conftest import assert_bits_equal
from vestra_hip import da3, seeded

pytestmark = pytest.mark.gpu

_CAPTURE_RELAXED = 2  # hipStreamCaptureModeRelaxed


def _hip():
    h = ctypes.CDLL("libamdhip64.so")
    vp, pvp = ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)
    for name, args in (("hipStreamBeginCapture", [vp, ctypes.c_int]),
                       ("hipStreamEndCapture", [vp, pvp]),
                       ("hipGraphInstantiate", [pvp, vp, pvp, ctypes.c_char_p, ctypes.c_size_t]),
                       ("hipGraphLaunch", [vp, vp]),
                       ("hipStreamSynchronize", [vp]),
                       ("hipGraphExecDestroy", [vp]),
                       ("hipGraphDestroy", [vp])):
        getattr(h, name).argtypes = args
        getattr(h, name).restype = ctypes.c_int
    return h


def _capture(hip, stream, run):
    """The kernels `run` issues on `stream`, as an instantiated graph."""
    assert hip.hipStreamBeginCapture(stream, _CAPTURE_RELAXED) == 0
    try:
        run()
    finally:
        graph = ctypes.c_void_p()
        rc = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert rc == 0 and graph.value
    exe = ctypes.c_void_p()
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
    return graph, exe


@pytest.mark.parametrize("layers, q8", [(1, False), (3, False), (2, True)],
                         ids=["block", "encoder3", "q8_encoder2"])
def test_encoder_graph_replays_equal_eager(rt, layers, q8):
    hip = _hip()
    stream = ctypes.c_void_p(rt.stream())
    blocks = [rt.prepare_block(da3.block_weights(seed=90 + i, layerscale="uniform"), q8_0=q8)
              for i in range(layers)]
    pos = da3.positions_yx(24, 36)
    x0 = seeded.normal(9000 + layers, 865 * 768)
    x, y = rt.upload_f32(x0), rt.upload_f32(x0)

    def run(t):
        if layers == 1:
            rt.vit_block_run(blocks[0], t, 1, 865, pos)
        else:
            rt.encoder_run(blocks, t, 1, 865, pos)

    run(y)  # warm-up: workspaces and the RoPE table exist before the capture
    rt.synchronize()
    x_ref = rt.download_f32(y)
    y = rt.upload_f32(x0)
    rt.synchronize()
    graph, exe = _capture(hip, stream, lambda: run(x))
    try:
        # The capture recorded the kernels without running them.
        assert np.array_equal(rt.download_f32(x), x0)
        for replay in range(3):
            assert hip.hipGraphLaunch(exe, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            run(y)  # the same run, eagerly, between the replays
            rt.synchronize()
            got, exp = rt.download_f32(x), rt.download_f32(y)
            assert_bits_equal(got, exp, f"replay {replay}")
            if replay == 0:
                assert_bits_equal(got, x_ref, "first replay against the warm-up run")
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


def test_graph_keeps_its_workspace_when_a_later_run_needs_a_larger_one(rt):
    """The workspace a capture was given outlives the graph's use of it: an
    eager run of more rows gets a larger one and the replays stay right."""
    hip = _hip()
    stream = ctypes.c_void_p(rt.stream())
    k = n = 768
    lin = rt.prepare_linear_f32(k, n, seeded.normal(9500, k * n, 0.02), seeded.normal(9501, n))
    x = rt.upload_f32(seeded.normal(9502, 865 * k))
    r0 = seeded.normal(9503, 865 * n)
    res, ref = rt.upload_f32(r0), rt.upload_f32(r0)
    lin.run_residual(x, 865, ref)
    rt.synchronize()
    exp = rt.download_f32(ref)
    graph, exe = _capture(hip, stream, lambda: lin.run_residual(x, 865, res))
    try:
        many = 40000
        big, acc = rt.upload_f32(seeded.normal(9504, many * k)), rt.upload_f32(np.zeros(many * n, np.float32))
        lin.run_residual(big, many, acc)
        rt.synchronize()
        assert hip.hipGraphLaunch(exe, stream) == 0
        assert hip.hipStreamSynchronize(stream) == 0
        assert_bits_equal(rt.download_f32(res), exp, "replay after the growth")
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("kind", ["f32", "late", "q8", "fp32_kernels", "wide"])
def test_graph_of_a_block_outlives_larger_runs(rt, monkeypatch, kind):
    """A captured block keeps every workspace that it was given (intermediates,
    Q8_0 rows, attention, split-K partials, counters): after an eager run of a
    larger size has grown them all, the replays are still right, and a size
    that no run has prepared is refused under capture, not allocated."""
    import vestra_hip as vh

    rt = vh.Runtime(0)  # its own, whose workspaces are still small
    hip = _hip()
    stream = ctypes.c_void_p(rt.stream())
    if kind == "fp32_kernels":
        monkeypatch.setenv("VESTRA_HIP_GEMM_TILE", "64x128x64x2x4x3")
        monkeypatch.setenv("VESTRA_HIP_FLASH_SPLITS", "4")
    w = da3.block_weights(seed=97, layerscale="uniform", qk_norm=kind == "late")
    if kind == "wide":  # one product at a time (the block's split form does not hold it)
        w["b_qkv"][2 * 768 + 70] = 1e12
        w["w_proj"].reshape(768, 768)[70] = 0.0
    block = rt.prepare_block(w, q8_0=kind == "q8")
    pos, more = da3.positions_yx(16, 20), da3.positions_yx(40, 40)
    x0 = seeded.normal(9600, 321 * 768)
    x, y = rt.upload_f32(x0), rt.upload_f32(x0)
    rt.vit_block_run(block, y, 1, 321, pos)
    rt.synchronize()
    exp = rt.download_f32(y)
    big = rt.upload_f32(seeded.normal(9601, 1601 * 768))
    graph, exe = _capture(hip, stream, lambda: rt.vit_block_run(block, x, 1, 321, pos))
    try:
        def refused():
            with pytest.raises(vh.UploadError):
                rt.vit_block_run(block, big, 1, 1601, None)

        other, other_exe = _capture(hip, stream, refused)
        hip.hipGraphExecDestroy(other_exe)
        hip.hipGraphDestroy(other)
        for replay in range(3):
            rt.vit_block_run(block, big, 1, 1601, more)
            rt.synchronize()
            rt.copy_segment_into_f32(x, 0, rt.upload_f32(x0), 0, x0.size)
            assert hip.hipGraphLaunch(exe, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            assert_bits_equal(rt.download_f32(x), exp, f"replay {replay}")
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


def test_graph_of_a_projection_that_no_run_has_prepared(rt):
    """Without a workspace for its split rows a captured projection takes the
    fp32 GEMM: the replays are right, and the same every time."""
    import vestra_hip as vh

    rt = vh.Runtime(0)  # its own, without workspaces
    hip = _hip()
    stream = ctypes.c_void_p(rt.stream())
    m, k, n = 500, 770, 768
    w = seeded.normal(9650, k * n, 0.02)
    lin = rt.prepare_linear_f32(k, n, w, np.zeros(n, np.float32))
    x, r0 = seeded.normal(9651, m * k), seeded.normal(9652, m * n)
    xt, res = rt.upload_f32(x), rt.upload_f32(r0)
    graph, exe = _capture(hip, stream, lambda: lin.run_residual(xt, m, res))
    try:
        got = []
        for replay in range(3):
            rt.copy_segment_into_f32(res, 0, rt.upload_f32(r0), 0, r0.size)
            assert hip.hipGraphLaunch(exe, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            got.append(rt.download_f32(res))
            res2 = rt.upload_f32(r0)
            lin.run_residual(xt, m, res2)  # eagerly, on split rows, between the replays
        exp = r0 + (x.reshape(m, k).astype(np.float64) @ w.reshape(k, n)).reshape(-1)
        for g in got:
            assert_bits_equal(g, got[0])
            assert np.linalg.norm(g - exp) <= 1e-6 * np.linalg.norm(exp)
        assert (rt.download_f32(res2) != got[0]).any()
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


def _free_bytes(hip):
    hip.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t)] * 2
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_failed_allocation_takes_back_the_split_rows(rt):
    """The workspace of the largest projection that a runtime has run goes back
    where an allocation needs it, unless a graph holds it; later calls get a
    new one."""
    import vestra_hip as vh

    rt = vh.Runtime(0)
    hip = _hip()
    stream = ctypes.c_void_p(rt.stream())
    m, k, n = 200000, 389, 128  # 333 MB of split rows
    lin = rt.prepare_linear_f32(k, n, seeded.normal(9750, k * n, 0.05), seeded.normal(9751, n))
    x, r0 = rt.upload_f32(seeded.normal(9752, 4096 * k)), seeded.normal(9753, 4096 * n)
    big, acc, res = rt.alloc_f32(m * k), rt.alloc_f32(m * n), rt.upload_f32(r0)
    for i in range(0, m, 4096):
        rows = min(4096, m - i)
        rt.copy_segment_into_f32(big, i * k, x, 0, rows * k)
        rt.copy_segment_into_f32(acc, i * n, res, 0, rows * n)

    def refused():
        with pytest.raises(vh.UploadError):
            rt.alloc_f32(1 << 45)

    lin.run_residual(x, 4096, res)
    exp = rt.download_f32(res)
    refused()
    before = _free_bytes(hip)
    lin.run_residual(big, m, acc)
    rt.synchronize()
    assert _free_bytes(hip) <= before - m * k * 4
    refused()
    assert _free_bytes(hip) >= before - (16 << 20)  # (but for small first-use workspaces)
    res = rt.upload_f32(r0)
    lin.run_residual(x, 4096, res)
    assert_bits_equal(rt.download_f32(res), exp, "after it went back")
    graph, exe = _capture(hip, stream, lambda: lin.run_residual(x, 4096, res))
    try:
        for replay in range(3):
            refused()
            rt.copy_segment_into_f32(res, 0, rt.upload_f32(r0), 0, r0.size)
            assert hip.hipGraphLaunch(exe, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            assert_bits_equal(rt.download_f32(res), exp, f"replay {replay}")
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)


def test_a_failed_allocation_takes_back_what_other_runtimes_hold(rt):
    """The blocks that another runtime of the device has kept go back to the
    device; a capture that its thread has begun meanwhile is not disturbed (no
    free becomes part of its graph, and the blocks it uses stay)."""
    import vestra_hip as vh

    hip = _hip()
    other = vh.Runtime(0)
    stream = ctypes.c_void_p(other.stream())

    def fill():
        for t in [other.alloc_f32((16 << 20) + 1024 * i) for i in range(4)]:
            t.free()
        other.synchronize()

    def refused():
        with pytest.raises(vh.UploadError):
            rt.alloc_f32(1 << 45)

    fill()
    before = _free_bytes(hip)
    refused()
    assert _free_bytes(hip) >= before + 4 * (64 << 20)

    lin = other.prepare_linear_f32(256, 256, seeded.normal(9700, 256 * 256, 0.05), seeded.normal(9701, 256))
    x, r0 = other.upload_f32(seeded.normal(9702, 300 * 256)), seeded.normal(9703, 300 * 256)
    res = other.upload_f32(r0)
    lin.run_residual(x, 300, res)
    exp = other.download_f32(res)
    res = other.upload_f32(r0)
    fill()

    def run():
        lin.run_residual(x, 300, res)
        refused()

    graph, exe = _capture(hip, stream, run)
    try:
        for replay in range(3):
            fill()
            other.copy_segment_into_f32(res, 0, other.upload_f32(r0), 0, r0.size)
            assert hip.hipGraphLaunch(exe, stream) == 0
            assert hip.hipStreamSynchronize(stream) == 0
            assert_bits_equal(other.download_f32(res), exp, f"replay {replay}")
    finally:
        hip.hipGraphExecDestroy(exe)
        hip.hipGraphDestroy(graph)
