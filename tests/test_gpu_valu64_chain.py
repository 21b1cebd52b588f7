"""The valu64 tile's fmaf chains, computed by the fp32 matrix instructions:
bit-identical to the sequential chain also where the two could differ --
cancellation, wide exponent ranges, denormal operands, results and sums,
signed zeros, infinite operands and overflow -- for one k-stage and several."""
import numpy as np
import pytest

import oracle
from gpu_util import run_persistent, say

pytestmark = pytest.mark.gpu


def _operands(kind, M, N, K):
    rng = np.random.default_rng(11)
    A, B = oracle.fill_uniform_pm1(13, M, N, K)
    if kind == "wide":
        A *= np.exp2(rng.integers(-30, 30, A.shape)).astype(np.float32)
        B *= np.exp2(rng.integers(-30, 30, B.shape)).astype(np.float32)
    elif kind == "cancel":
        A[:, 1::2], B[1::2] = A[:, ::2], -B[::2]
    elif kind == "denormal_sums":
        A *= np.float32(2.0 ** -70)
        B *= np.float32(2.0 ** -70)
    elif kind == "denormal_operands":
        A *= np.float32(2.0 ** -130)
    elif kind == "zeros":
        A[:, ::2] = -0.0
        B[::3] = 0.0
    elif kind == "overflow":
        A[5] *= np.float32(2.0 ** 120)
        B[:, 40] *= np.float32(2.0 ** 20)
    elif kind == "inf":
        A[33, K - 1] = np.inf
        B[0, 63] = -np.inf
    return A, B


@pytest.mark.parametrize("K", [32, 96])
@pytest.mark.parametrize("kind", ["wide", "cancel", "denormal_sums", "denormal_operands", "zeros",
                                  "overflow", "inf"])
def test_valu64_bit_exact_chain(torch_gpu, apk, kind, K):
    say(f"valu64 {kind} M=128 N=64 K={K}")
    A, B = _operands(kind, 128, 64, K)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_VALU64, A, B, K, blocks=3, with_log=False)
    with np.errstate(all="ignore"):
        chain = oracle.gemm_f32_chain(A, B)
    nan = np.isnan(chain)
    assert np.array_equal(np.isnan(C), nan)
    assert np.array_equal(C.view(np.uint32)[~nan], chain.view(np.uint32)[~nan])
