"""The shapes on either side of the lines where the automatic choice turns to
the matrix-core kernels, each with the kernel that is expected there (on 256
CUs): short rows, rounds of tiles that are full or not, rows longer than 5120
values over few rows per CU, columns that fill the LDS, odd rows and counts that
are no multiple of a tile, two to eight columns, both weight types.  Each
against the oracle within its derived tolerance (every sampled output), and the
F32 route against the pre-quantised one bit for bit, with a workspace and
without.  Then the calls that reach those kernels without a usable workspace or
with strides beyond their offsets."""
import numpy as np
import pytest

import _common
from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14


TILE, STAGED, SPLIT, GA = 1, 4, 5, 6  # SPLIT: K-split or one-column channels


@pytest.mark.parametrize("wtype,M,K,N,kernel", [
    # one or two super-blocks
    (Q4, 4081, 256, 2, TILE), (Q4, 4593, 256, 2, STAGED), (Q4, 4080, 512, 3, TILE), (Q4, 4081, 512, 3, STAGED),
    (Q4, 65160, 512, 7, STAGED),
    # 3 to 13; 257 tiles of 256 CUs fill half of two rounds
    (Q4, 4081, 768, 5, STAGED), (Q4, 4080, 1280, 8, TILE), (Q4, 4081, 3328, 6, STAGED), (Q4, 4097, 3328, 6, TILE),
    (Q4, 6129, 2816, 5, STAGED), (Q4, 6001, 2816, 5, TILE),
    (Q4, 40960, 2304, 5, STAGED), (Q4, 20480, 2304, 5, TILE), (Q4, 45056, 2304, 4, STAGED), (Q4, 24576, 2304, 4, TILE),
    # three and four columns
    (Q4, 16369, 2304, 4, STAGED), (Q4, 16368, 2304, 4, TILE), (Q4, 18944, 3072, 4, TILE), (Q4, 32753, 2304, 3, STAGED),
    (Q4, 32753, 2816, 3, STAGED),
    (Q4, 32753, 3072, 3, TILE),
    # long rows: one-column channels, the tile kernel, staged
    (Q4, 2049, 5376, 6, SPLIT), (Q4, 2048, 5376, 8, SPLIT), (Q4, 2561, 5376, 6, STAGED), (Q4, 8177, 5888, 5, STAGED),
    (Q4, 3072, 8192, 5, SPLIT), (Q4, 2560, 6144, 5, SPLIT), (Q4, 2816, 6144, 5, TILE), (Q4, 2817, 8192, 6, SPLIT),
    (Q4, 3585, 8192, 6, STAGED), (Q4, 4609, 8192, 6, TILE),
    # A from the Q8_1 copy; eight columns of 14336 values beside eight waves
    (Q4, 2049, 9472, 7, GA), (Q4, 2048, 9472, 7, SPLIT), (Q4, 3001, 22272, 5, GA), (Q4, 2560, 9472, 5, SPLIT),
    (Q4, 2561, 9472, 5, GA), (Q4, 8177, 14336, 8, STAGED),
    (Q6, 4081, 512, 5, STAGED), (Q6, 14333, 768, 8, STAGED), (Q6, 8177, 5376, 7, STAGED), (Q6, 2934, 22272, 7, GA),
    (Q6, 16369, 2304, 4, STAGED), (Q6, 4081, 3328, 6, STAGED), (Q6, 2049, 5888, 5, STAGED), (Q6, 2050, 8192, 5, STAGED),
    (Q6, 2063, 9472, 5, GA), (Q6, 4096, 512, 3, STAGED), (Q6, 4097, 9472, 5, TILE), (Q6, 6144, 5376, 5, TILE),
    (Q6, 2048, 8192, 5, SPLIT), (Q6, 18944, 3072, 5, TILE),
])
def test_choice_against_oracle_and_between_routes(Q, O, gpu, wtype, M, K, N, kernel):
    assert Q.geometry(K, M, N, wtype)["kernel"] == kernel
    import torch
    quant = Q.quantize_rows_q4_K if wtype == Q4 else Q.quantize_rows_q6_K
    rng = np.random.default_rng(M + K + N)
    wq = quant(_common.weights(min(M, 2048), K, 61), nthreads=16)
    wq = wq[rng.integers(0, wq.shape[0], M)]  # many rows of few
    x = _common.activations(N, K, 62)
    rows = np.unique(np.concatenate([[0, 1, 15, 16, M // 2, M - 17, M - 2, M - 1], rng.choice(M, 200, replace=False)]))
    ref = (O.gemv_q4K_q8_1 if wtype == Q4 else O.gemv_q6K_q8_1)(wq[rows], K, O.quantize_q8_1(x), want_sums=False)
    wd, xd = to_dev(wq, gpu), to_dev(x, gpu)
    y = Q.mul_mat_vec_q(wd, K, xd, wtype=wtype)
    _common.assert_within_tolerance(O, y.cpu().numpy()[:, rows], ref, f"{wtype} {M}x{K} N={N}")
    ws = torch.empty(Q.q8_1_bytes(K, N), dtype=torch.uint8, device=gpu)
    assert torch.equal(Q.mul_mat_vec_q(wd, K, xd, workspace=ws, wtype=wtype), y)
    assert torch.equal(Q.op_mul_mat_vec_q(wd, K, Q.quantize_row_q8_1(xd), N, wtype=wtype), y)


def test_q6_waves_follow_full_rounds(Q, gpu):
    """Q6_K takes 16 waves where their rounds of sixteen tiles are full (256 CUs)."""
    for M, K, waves in [(64128, 4096, 16), (61440, 4096, 8), (65536, 4096, 16), (73728, 4096, 8), (98304, 5120, 8),
                        (128256, 4096, 16), (62900, 5120, 16), (18944, 7168, 16), (14336, 4096, 8)]:
        g = Q.geometry(K, M, 8, Q6)
        assert (g["kernel"], g["waves_per_wg"]) == (STAGED, waves), (M, K)


def _weights(Q, wtype, M, K, seed):
    quant = Q.quantize_rows_q4_K if wtype == Q4 else Q.quantize_rows_q6_K
    wq = quant(_common.weights(min(M, 512), K, seed), nthreads=16)
    return wq[np.random.default_rng(seed).integers(0, wq.shape[0], M)]


def _node_types(call):
    """The types of the graph nodes that call(stream) records (0: a kernel)."""
    import ctypes
    import torch
    hip = ctypes.CDLL("libamdhip64.so")
    stream = torch.cuda.Stream()
    sp, graph, n = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t(0)
    assert hip.hipStreamBeginCapture(sp, 1) == 0  # thread-local capture mode
    call(stream)
    assert hip.hipStreamEndCapture(sp, ctypes.byref(graph)) == 0
    try:
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
        nodes = (ctypes.c_void_p * n.value)()
        assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
        types = []
        for nd in nodes:
            t = ctypes.c_int(-1)
            assert hip.hipGraphNodeGetType(ctypes.c_void_p(nd), ctypes.byref(t)) == 0
            types.append(t.value)
        return types
    finally:
        hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("wtype,M,K,N,one_launch", [
    (Q4, 2049, 9472, 7, True), (Q4, 3001, 14336, 8, True), (Q4, 2817, 22272, 7, False), (Q4, 4080, 8448, 5, True),
    (Q6, 2063, 9472, 5, True), (Q6, 3001, 11008, 6, True), (Q6, 2934, 22272, 7, False), (Q6, 8192, 14336, 5, True)])
def test_no_usable_workspace(Q, O, gpu, wtype, M, K, N, one_launch):
    """Activations that a launch can quantise by itself: a workspace that is too
    small or not aligned is not needed, and without one the call allocates
    nothing where one launch holds the columns.  Same bits as with one."""
    import torch
    assert Q.geometry(K, M, N, wtype)["kernel"] == GA
    wd, xd = to_dev(_weights(Q, wtype, M, K, 63), gpu), to_dev(_common.activations(N, K, 64), gpu)
    need = Q.q8_1_bytes(K, N)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    y = Q.mul_mat_vec_q(wd, K, xd, workspace=ws, wtype=wtype)
    assert torch.equal(Q.mul_mat_vec_q(wd, K, xd, workspace=ws[: need - 4], wtype=wtype), y), "too small"
    odd = torch.empty(need + 8, dtype=torch.uint8, device=gpu)[1:]
    assert torch.equal(Q.mul_mat_vec_q(wd, K, xd, workspace=odd, wtype=wtype), y), "not aligned"
    assert torch.equal(Q.mul_mat_vec_q(wd, K, xd, wtype=wtype), y), "none"
    out = torch.empty_like(y)
    if one_launch:
        assert _node_types(lambda st: Q.mul_mat_vec_q(wd, K, xd, out=out, wtype=wtype, stream=st)) == [0]


def test_workspace_that_the_route_needs(Q, gpu):
    """256 row tiles and more of long rows: the buffer is part of the route, and one
    that cannot hold the Q8_1 copy is refused."""
    import torch
    M, K, N = 4096, 14336, 6
    assert Q.geometry(K, M, N)["kernel"] == GA
    wd, xd = to_dev(_weights(Q, Q4, M, K, 65), gpu), to_dev(_common.activations(N, K, 66), gpu)
    with pytest.raises(Q.Q4KError) as e:
        Q.mul_mat_vec_q(wd, K, xd, workspace=torch.empty(Q.q8_1_bytes(K, N) - 4, dtype=torch.uint8, device=gpu))
    assert e.value.status == Q.Q4K_EINVAL


@pytest.mark.parametrize("wtype", [Q4, Q6])
def test_q8_1_columns_beyond_one_buffer(Q, O, gpu, wtype):
    """Q8_1 columns so far apart that eight of them span 2^31 bytes: more than the
    matrix-core kernel on the Q8_1 copy addresses at once, not more than the others
    do."""
    import torch
    M, K, N = 3073, 8448, 8
    assert Q.geometry(K, M, N, wtype, route="q8_1")["kernel"] == GA
    wq = _weights(Q, wtype, M, K, 67)
    x = _common.activations(N, K, 68)
    wd = to_dev(wq, gpu)
    blocks = (1 << 31) // (8 * 36) + 1
    far = torch.empty((N, blocks, 36), dtype=torch.uint8, device=gpu)
    q8 = Q.quantize_row_q8_1(to_dev(x, gpu)).view(N, -1, 36)[:, : K // 32]
    far[:, : K // 32] = q8
    dst = torch.empty((N, M), dtype=torch.float32, device=gpu)
    name = "q4k_op_mul_mat_vec_q" if wtype == Q4 else "q6k_op_mul_mat_vec_q"
    assert getattr(Q.lib(), name)(Q._ptr(wd), K, 0, M, Q._ptr(far), N, 32 * blocks, Q._ptr(dst), M,
                                  Q._stream()) == Q.Q4K_OK
    rows = np.unique(np.random.default_rng(69).choice(M, 200, replace=False))
    ref = (O.gemv_q4K_q8_1 if wtype == Q4 else O.gemv_q6K_q8_1)(wq[rows], K, O.quantize_q8_1(x), want_sums=False)
    _common.assert_within_tolerance(O, dst.cpu().numpy()[:, rows], ref, f"{wtype} columns far apart")
