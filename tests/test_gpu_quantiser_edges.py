"""The quantiser's branches at their edges: block maxima on either side of 2^-100
(below, the exact division) down to the subnormals whose d is not 0, NaN in one lane and infinities
among ordinary blocks of the same wave (which start again with it), and values
next to the ties of block scales that are no power of two.

Bar: the Q8_1 bytes of quantize_row_q8_1 equal the oracle's (with a NaN or an
infinite maximum the q8 alone: there the oracle's ds is not defined), and every
kernel that quantises inside its launch gives the outputs of the launch on those
bytes."""
import numpy as np
import pytest

import _common
from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu


def _blocks(kind, rng, n):
    """float32 [n, 32]; every fourth block is an ordinary one."""
    x = rng.standard_normal((n, 32)).astype(np.float32)
    edge = np.arange(n) % 4 != 3
    if kind == "tiny":
        amax = np.float32(2.0) ** rng.integers(-142, -96, n).astype(np.float32)
        at = np.array([2.0 ** -100, np.nextafter(np.float32(2.0 ** -100), np.float32(0)),
                       np.nextafter(np.float32(2.0 ** -100), np.float32(1)), 2.0 ** -126, 2.0 ** -142], np.float32)
        amax[: min(n, 8 * len(at))] = np.tile(at, 8)[:n]
        t = (rng.uniform(-1, 1, (n, 32)) * amax[:, None]).astype(np.float32)
        t[np.arange(n), rng.integers(0, 32, n)] = amax
    elif kind == "ties":
        t = np.empty((n, 32), np.float32)
        for b in range(n):
            amax = np.float32(2.0 ** rng.uniform(-20, 20))
            d = np.float32(amax / np.float32(127))
            v = ((rng.integers(-126, 126, 32) + 0.5) * np.float64(d)).astype(np.float32)
            steps = rng.integers(-4, 5, 32)
            for k in range(32):
                for _ in range(abs(steps[k])):
                    v[k] = np.nextafter(v[k], np.float32(np.inf if steps[k] > 0 else -np.inf))
            v[rng.integers(0, 32)] = amax
            t[b] = v
    elif kind == "nan":
        t = x.copy()
        t[np.arange(n), rng.integers(0, 32, n)] = np.nan
        t[n // 2] = np.nan
    else:
        t = x.copy()
        t[np.arange(n), rng.integers(0, 32, n)] = np.where(rng.random(n) < 0.5, np.inf, -np.inf)
    x[edge] = t[edge]
    return x


def _q(b):
    """roundf(x / d) of float32 blocks; 0 for a NaN, of all zeros and under an infinite maximum."""
    with np.errstate(all="ignore"):
        a = np.abs(np.where(np.isnan(b), np.float32(0), b)).max(1, keepdims=True)
        r = (b / (a / np.float32(127))).astype(np.float32)
        q = np.sign(r) * np.floor(np.abs(r).astype(np.float64) + 0.5)
    return np.where(np.isfinite(q) & (a > 0) & np.isfinite(a), q, 0).astype(np.int8)


@pytest.mark.parametrize("kind", ["tiny", "ties", "nan", "inf"])
def test_quantised_bytes(Q, O, gpu, kind):
    rng = np.random.default_rng(len(kind) * 7)
    N, K = 3, 2048
    b = _blocks(kind, rng, N * K // 32)
    x = b.reshape(N, K)
    got = Q.quantize_row_q8_1(to_dev(x, gpu)).cpu().numpy().reshape(-1, 36)
    assert np.array_equal(got[:, 4:].view(np.int8), _q(b)), kind
    if kind in ("tiny", "ties"):
        assert np.array_equal(got, O.quantize_q8_1(x).reshape(-1, 36)), kind


# the kernels that quantise inside their launch (Q4_K, Q6_K): one column of 4096
# and 8192 values in registers, of other lengths and short rows in LDS, several
# columns in short teams and in registers, the tile kernel, the matrix-core kernel
@pytest.mark.parametrize("wtype", [12, 14])
@pytest.mark.parametrize("M,K,N,kernel", [(300, 4096, 1, 0), (300, 8192, 1, 0), (300, 5120, 1, 0), (300, 1024, 1, 0),
                                          (300, 1024, 2, 0), (300, 1536, 4, 0), (300, 4096, 2, 5), (300, 5120, 1, 1),
                                          (300, 2304, 5, 1), (300, 1280, 8, 4), (300, 4352, 3, 4)])
def test_in_launch_equals_pre_quantised(Q, gpu, wtype, M, K, N, kernel):
    quant = Q.quantize_rows_q4_K if wtype == 12 else Q.quantize_rows_q6_K
    wd = to_dev(quant(_common.weights(M, K, 81), nthreads=16), gpu)
    for kind in ("tiny", "ties", "nan", "inf"):
        x = to_dev(_blocks(kind, np.random.default_rng(K + N), N * K // 32).reshape(N, K), gpu)
        try:
            Q.set_geometry_override(kernel=kernel)
            y = Q.mul_mat_vec_q(wd, K, x, wtype=wtype).cpu().numpy()
            if kernel == 5:  # (on the F32 route only; its bits are the tile kernel's)
                Q.set_geometry_override(kernel=1)
            y8 = Q.op_mul_mat_vec_q(wd, K, Q.quantize_row_q8_1(x), N, wtype=wtype).cpu().numpy()
        finally:
            Q.set_geometry_override()
        assert np.array_equal(y, y8, equal_nan=True), kind
