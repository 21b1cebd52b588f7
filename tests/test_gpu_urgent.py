"""apk_urgent_gemm, the reference's urgent_tile (src/urgent_baseline.cu:
100-112): one block per tile, no queue, start stamped at block 0's first
instruction, end raised by every block. Its C must be bit-identical to the
persistent GEMM's (same engine, same per-element k order), the fp32 tile
bit-identical to the fmaf-chain oracle, and the stamps ordered."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, run_persistent, say

pytestmark = pytest.mark.gpu


def run_urgent(torch, apk, eng, A, B):
    M, K = A.shape
    N = B.shape[0] if apk.geometry(eng).b_transposed else B.shape[1]
    dA, dB = dev(torch, A), dev(torch, B)
    dC = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
    t = torch.zeros(2, dtype=torch.int64, device="cuda")
    apk.urgent_gemm(eng, dA.data_ptr(), dB.data_ptr(), dC.data_ptr(), M, N, K,
                    t.data_ptr(), t.data_ptr() + 8, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    start, end = t.cpu().numpy().tolist()
    return dC.cpu().numpy(), start, end


@pytest.mark.parametrize("name", ["valu64", "mfma128"])
def test_urgent_fp32_matches_persistent(torch_gpu, apk, name):
    eng = apk.ENGINES[name]
    g = apk.geometry(eng)
    M, N, K = 2 * g.tile_m, 2 * g.tile_n, 256
    say(f"urgent_gemm {name} {M}x{N}x{K} vs persistent_gemm")
    A, B = oracle.fill_uniform_pm1(21, M, N, K)
    C, start, end = run_urgent(torch_gpu, apk, eng, A, B)
    # records at every k-stage: the persistent GEMM's one-stage-per-barrier
    # loop, against the urgent kernel's (stage pairs for the fp32 MFMA tile)
    Cp, _, _ = run_persistent(torch_gpu, apk, eng, A, B, g.k_stage, blocks=3)
    assert np.array_equal(C.view(np.uint32), Cp.view(np.uint32))
    if name == "valu64":
        assert np.array_equal(C.view(np.uint32), oracle.gemm_f32_chain(A, B).view(np.uint32))
    assert oracle.rel_frobenius(C, oracle.gemm_f64(A, B, threads=8)) <= 1e-5
    assert 0 < start <= end


@pytest.mark.parametrize("name", ["bf16x256", "bf16x128", "bf16x256x128"])
def test_urgent_bf16_matches_persistent(torch_gpu, apk, name):
    eng = apk.ENGINES[name]
    g = apk.geometry(eng)
    M, N, K = 2 * g.tile_m, g.tile_n, 512
    say(f"urgent_gemm {name} {M}x{N}x{K} vs persistent_gemm")
    A_bits, A, B_bits, B = oracle.fill_normal_bf16(9, M, N, K)
    Bt = np.ascontiguousarray(B_bits.T)
    C, start, end = run_urgent(torch_gpu, apk, eng, A_bits.view(np.int16), Bt.view(np.int16))
    dA, dB = dev(torch_gpu, A_bits.view(np.int16)), dev(torch_gpu, Bt.view(np.int16))
    dC = torch_gpu.empty((M, N), dtype=torch_gpu.float32, device="cuda")
    q = torch_gpu.zeros(apk.QUEUE_WORDS, dtype=torch_gpu.int32, device="cuda")
    apk.persistent_gemm(eng, dA.data_ptr(), dB.data_ptr(), dC.data_ptr(), M, N, K, K,
                        q.data_ptr(), None, 2, torch_gpu.cuda.current_stream().cuda_stream)
    torch_gpu.cuda.synchronize()
    assert np.array_equal(C.view(np.uint32), dC.cpu().numpy().view(np.uint32))
    assert oracle.rel_frobenius(C, oracle.gemm_f64(A, B, threads=8)) <= 1e-5
    assert 0 < start <= end


# Jobs of at most 64 128x128 parts are computed part by part: the smallest
# (one part row, the least K), odd numbers of load regions, the last size on
# the parts and the first on the engine's own tile.
@pytest.mark.parametrize("name,M,N,K", [
    ("bf16x256", 256, 256, 64), ("bf16x256", 256, 768, 192), ("bf16x256", 2048, 512, 128),
    ("bf16x256", 2304, 512, 128), ("bf16x256x128", 256, 128, 32),
    ("bf16x256x128", 512, 384, 160), ("bf16x256x128", 1024, 1024, 96),
    ("bf16x256x128", 256, 4224, 96),
    # tile counts that leave surplus blocks: 5 and 9 of 8 and 16, 21 of 24
    ("bf16x256", 256, 1280, 64), ("bf16x256", 768, 768, 64), ("bf16x256x128", 768, 896, 96)])
def test_urgent_bf16_parts(torch_gpu, apk, name, M, N, K):
    torch = torch_gpu
    eng = apk.ENGINES[name]
    say(f"urgent_gemm {name} {M}x{N}x{K}: parts vs persistent_gemm")
    gen = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=gen).to(torch.bfloat16)
    Bt = torch.randn(N, K, generator=gen).to(torch.bfloat16)
    C, start, end = run_urgent(torch, apk, eng, A.view(torch.int16).numpy(),
                               Bt.view(torch.int16).numpy())
    dA, dB = A.cuda(), Bt.cuda()
    dC = torch.full((M, N), float("nan"), device="cuda")
    q = torch.zeros(apk.QUEUE_WORDS, dtype=torch.int32, device="cuda")
    apk.persistent_gemm(eng, dA.data_ptr(), dB.data_ptr(), dC.data_ptr(), M, N, K, K,
                        q.data_ptr(), None, 64, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    # the same products in the same order: not one bit may differ
    assert np.array_equal(C.view(np.uint32), dC.cpu().numpy().view(np.uint32))
    ref = oracle.gemm_f64(A.float().numpy(), np.ascontiguousarray(Bt.float().numpy().T), threads=8)
    # exact products; at most K roundings of 2^-24 of a partial sum, whose rms is at
    # most the result's
    assert oracle.rel_frobenius(C, ref) <= 2.0 ** -24 * K
    assert 0 < start <= end


@pytest.mark.parametrize("M,N,K", [(768, 896, 1568), (512, 2048, 2080)])
def test_urgent_bf16_parts_share_an_l2(torch_gpu, apk, M, N, K):
    """Each part of a job has a CU of its own, so a job of many parts takes
    about as long as one of two, as long as an XCD's L2 (4 MiB) holds what its
    blocks read. It does where a tile's parts run on one XCD; dealt row by row
    (in runs per XCD) the first (second) job took 2.1 times as long."""
    torch, eng = torch_gpu, apk.ENGINES["bf16x256x128"]
    say(f"urgent_gemm bf16x256x128 {M}x{N}x{K}: time against 256x128x{K}")
    A = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    B = torch.randn(N, K, device="cuda").to(torch.bfloat16)
    C = torch.empty(M, N, device="cuda")
    st = torch.cuda.current_stream().cuda_stream

    def us(m, n):
        best = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(20):
                apk.urgent_gemm(eng, A.data_ptr(), B.data_ptr(), C.data_ptr(), m, n, K, None,
                                None, st)
            e1.record()
            torch.cuda.synchronize()
            best.append(50 * e0.elapsed_time(e1))
        return min(best)

    us(M, N)
    many, two = us(M, N), us(256, 128)
    say(f"  {many:.1f} us, two parts {two:.1f}")
    assert many <= 1.6 * two


def test_urgent_rejects_bad_shape(torch_gpu, apk):
    # M = 100 is not a multiple of the 128-row tile: refused before any launch
    buf = torch_gpu.zeros(128 * 128, dtype=torch_gpu.float32, device="cuda")
    with pytest.raises(apk.ApkError):
        apk.urgent_gemm(apk.ENGINE_MFMA128, buf.data_ptr(), buf.data_ptr(), buf.data_ptr(),
                        100, 128, 128)
