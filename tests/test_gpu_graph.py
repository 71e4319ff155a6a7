"""GPU tests of the batched-submission (HIP graph) part of the C ABI: the node limit of one captured graph, the node
count query, and that executable graphs stay valid when the library's workspace grows after they were captured."""
import numpy as np
import pytest

from marmot_amd import capi
from oracle.pyoracle import KIND_Q4_0, KIND_Q4_1, KIND_Q4_K, KIND_Q6_K, KIND_Q8_0
from tests.util import assert_matmul_parity, bits, gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture()
def hip():
    from marmot_amd import HipBackend

    b = HipBackend(0)  # a device object of its own: the workspace starts empty
    yield b
    b.close()


def test_node_limit_and_count(hip):
    limit = hip.graph_max_nodes()
    assert limit == 1024
    buf = hip.alloc(4096)
    try:
        g = hip.graph_capture(lambda: [hip.lib.marmot_hip_memset(hip.dev, buf.ptr, i & 0xFF, 4096) for i in range(7)])
        assert hip.graph_last_capture_nodes() == 7
        hip.graph_launch(g)
        hip.synchronize()
        assert np.all(buf.download(np.uint8, (4096,)) == 6)
        hip.graph_destroy(g)

        with pytest.raises(capi.MarmotHipError) as err:
            hip.graph_capture(lambda: [hip.lib.marmot_hip_memset(hip.dev, buf.ptr, 1, 4096) for _ in range(limit + 1)])
        assert err.value.code == -5  # INVALID_OPERATION
        assert "limit is 1024" in err.value.detail
        assert hip.graph_last_capture_nodes() == limit + 1
        # the device object is usable afterwards: exactly the limit is accepted
        g = hip.graph_capture(lambda: [hip.lib.marmot_hip_memset(hip.dev, buf.ptr, 9, 4096) for _ in range(limit)])
        hip.graph_launch(g)
        hip.synchronize()
        assert np.all(buf.download(np.uint8, (4096,)) == 9)
        hip.graph_destroy(g)
    finally:
        buf.free()


def test_graph_survives_workspace_growth(hip, oracle):
    """A captured small-batch matmul reads packed activations and K-split partials in the workspace. A later eager call
    with a larger shape makes the workspace grow; the old one must stay allocated while the graph lives, and replays
    give the same bits as before."""
    kind = KIND_Q4_K
    M, K, N = 256, 1024, 8
    blocks = oracle.quantize(kind, gaussian(800, (M, K), 0.02))
    x = gaussian(801, (N, K))
    d_w, d_x = hip.to_device(blocks), hip.to_device(x)
    d_out = hip.alloc(N * M * 4)
    hip.linear_d(kind, d_w, d_x, capi.DT_F32, N, K, M, d_out, capi.DT_F32)  # sizes the workspace for this shape
    eager = d_out.download(np.float32, (N, M))
    g = hip.graph_capture(lambda: hip.linear_d(kind, d_w, d_x, capi.DT_F32, N, K, M, d_out, capi.DT_F32))
    try:
        # much larger activations: the workspace is outgrown several times over
        big_blocks = oracle.quantize(kind, gaussian(802, (64, 16384), 0.02))
        for n_big in (64, 512):
            big = hip.linear(gaussian(803, (n_big, 16384)), big_blocks, kind, 64)
            assert big.shape == (n_big, 64)
        for rep in range(3):
            d_out.upload(np.full(N * M * 4, 0xFF, dtype=np.uint8))
            hip.graph_launch(g)
            hip.synchronize()
            assert np.array_equal(bits(d_out.download(np.float32, (N, M))), bits(eager)), f"replay {rep}"
    finally:
        hip.graph_destroy(g)
        for b in (d_w, d_x, d_out):
            b.free()


@pytest.mark.parametrize("kind", [KIND_Q8_0, KIND_Q4_0, KIND_Q4_1])
def test_prepacked_prompt_is_captured_whatever_the_workspace(hip, oracle, kind):
    """A 32-value format at 160 tiles splits K where the workspace holds the partial sums (14.7 MB). A call that cannot grow
    the workspace gives the same bits without them: on a fresh device object, which has none, with a workspace too small for
    them, and with one that holds them."""
    N, K, M = 300, 4096, 4096
    blocks = oracle.quantize(kind, gaussian(810, (M, K), 0.02))
    x = gaussian(811, (N, K))
    some = np.r_[0, 1, 63, 64, 127, 128, 255, 256, 298, 299]
    ref = oracle.matmul(kind, blocks, np.ascontiguousarray(x[some]), M)
    d_w, d_x, d_out = hip.to_device(blocks), hip.to_device(x), hip.alloc(N * M * 4)
    d_p = hip.alloc(hip.packed_activation_bytes(kind, N, K))
    hip.pack_activations_d(kind, d_x, capi.DT_F32, N, K, d_p)
    hip.synchronize()

    def captured(kernels):
        """The captured call's output, the same on every one of three replays. Without partial sums it is one kernel."""
        g = hip.graph_capture(lambda: hip.linear_prepacked_d(kind, d_w, d_p, N, K, M, d_out))
        assert hip.graph_last_capture_nodes() == kernels
        outs = []
        try:
            for _ in range(3):
                d_out.upload(np.full(N * M * 4, 0xFF, dtype=np.uint8))
                hip.graph_launch(g)
                hip.synchronize()
                outs.append(d_out.download(np.float32, (N, M)))
        finally:
            hip.graph_destroy(g)
        assert all(np.array_equal(bits(o), bits(outs[0])) for o in outs)
        return outs[0]

    try:
        no_room = captured(1)
        # an eager call that needs between 4 and 8 MB of it: 600 packed rows
        small = oracle.quantize(kind, gaussian(812, (64, 8192), 0.02))
        hip.linear(gaussian(813, (600, 8192)), small, kind, 64)
        some_room = captured(1)
        hip.linear_prepacked_d(kind, d_w, d_p, N, K, M, d_out)
        eager = d_out.download(np.float32, (N, M))
        assert_matmul_parity(eager[some], ref, what="eager")
        assert np.array_equal(bits(no_room), bits(eager))
        assert np.array_equal(bits(some_room), bits(eager))
        assert np.array_equal(bits(captured(2)), bits(eager))
    finally:
        for b in (d_w, d_x, d_p, d_out):
            b.free()


def test_q6k_small_batch_needs_no_room_for_partial_sums(hip, oracle):
    """16 rows x 14336: the packed activations fit a workspace of 1 MiB, K-split partial sums (2 MB) would not. The row-group
    kernel has none, so the call is captured without an eager run of its own."""
    kind = KIND_Q6_K
    N, K, M = 16, 14336, 4096
    hip.linear(gaussian(820, (5, 512)), oracle.quantize(kind, gaussian(821, (16, 512), 0.02)), kind, 16)
    d_w, d_x = hip.to_device(oracle.quantize(kind, gaussian(822, (M, K), 0.02))), hip.to_device(gaussian(823, (N, K)))
    d_out = hip.alloc(N * M * 4)
    g = None
    try:
        g = hip.graph_capture(lambda: hip.linear_d(kind, d_w, d_x, capi.DT_F32, N, K, M, d_out, capi.DT_F32))
        hip.linear_d(kind, d_w, d_x, capi.DT_F32, N, K, M, d_out, capi.DT_F32)
        eager = d_out.download(np.float32, (N, M))
        for rep in range(3):
            d_out.upload(np.full(N * M * 4, 0xFF, dtype=np.uint8))
            hip.graph_launch(g)
            hip.synchronize()
            assert np.array_equal(bits(d_out.download(np.float32, (N, M))), bits(eager)), f"replay {rep}"
    finally:
        if g is not None:
            hip.graph_destroy(g)
        for b in (d_w, d_x, d_out):
            b.free()
