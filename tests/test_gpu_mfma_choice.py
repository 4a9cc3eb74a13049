"""The shapes on either side of the lines where the automatic choice turns to
the matrix-core kernels: short rows, rows longer than 5120 values over few
rows per CU, odd rows and counts that are no multiple of a tile, three to
eight columns, both weight types.  Each against the oracle within its derived
tolerance (every sampled output), and the F32 route against the pre-quantised
one bit for bit, with a workspace and without."""
import numpy as np
import pytest

import _common
from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14


@pytest.mark.parametrize("wtype,M,K,N", [
    (Q4, 4081, 256, 2), (Q4, 4080, 512, 3), (Q4, 4081, 512, 2), (Q4, 65160, 512, 7),  # one or two super-blocks
    (Q4, 4081, 768, 5), (Q4, 4080, 1280, 8), (Q4, 4097, 3328, 6),                      # 3 to 13
    (Q4, 16369, 2304, 4), (Q4, 16368, 2304, 4), (Q4, 32753, 3328, 3),                  # three and four columns
    (Q4, 2049, 5376, 6), (Q4, 2048, 5376, 8), (Q4, 8177, 5888, 5),                     # long rows, staged
    (Q4, 2049, 9472, 7), (Q4, 2048, 9472, 7), (Q4, 3001, 22272, 5),                    # A from the Q8_1 copy
    (Q6, 4081, 512, 5), (Q6, 14333, 768, 8), (Q6, 8177, 5376, 7), (Q6, 2934, 22272, 7),
    (Q6, 16369, 2304, 4), (Q6, 4081, 3328, 6), (Q6, 2049, 5888, 5), (Q6, 2050, 8192, 5), (Q6, 2063, 9472, 5),
    (Q6, 4096, 512, 3),
])
def test_choice_against_oracle_and_between_routes(Q, O, gpu, wtype, M, K, N):
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


def test_staged_kernel_up_to_the_end_of_the_lds(Q, gpu):
    """Eight columns of 14336 values fit beside eight waves (163456 of 163840 bytes)."""
    assert Q.geometry(14336, 8192, 8)["kernel"] == 4
