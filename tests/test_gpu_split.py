"""The fp32 MFMA tile's split products (three bf16 parts per operand) on the
GPU: no less exact than the fp32 chain over the range of K, and operands that
the parts cannot carry (infinite, NaN, above bf16's range, bits below 2^-133)
computed with exact products -- from their k-stage on, or the whole tile --,
also through checkpoint, resume and retreat, and as preemptible as the others.

Bound for finite results: each C element sums K products in fp32, at most K
roundings of 2^-24 each, and three products of parts below 2^-24 of a b are
left out, so |C - C64| <= (K + 4) 2^-24 (|A| |B|) + (K + 1) 2^-149 (the last
term where sums are denormal)."""
import numpy as np
import pytest

import oracle
from gpu_util import run_persistent, say
from test_gpu_retreat import RetreatJob, _check
from test_gpu_yield import Job, _bits, _blocks

pytestmark = pytest.mark.gpu


def _bound(A, B):
    K = A.shape[1]
    mag = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    return (K + 4) * 2.0 ** -24 * mag + (K + 1) * 2.0 ** -149


@pytest.mark.parametrize("K", [32, 64, 96, 128, 992])
def test_split_no_less_exact_than_the_chain(torch_gpu, apk, K):
    """One stage (pipeline filled and drained at once), two, an odd number, many."""
    say(f"mfma128 split error, M=256 N=384 K={K}")
    A, B = oracle.fill_uniform_pm1(17, 256, 384, K)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, K, blocks=5, with_log=False)
    ref = oracle.gemm_f64(A, B, threads=8)
    chain = oracle.gemm_f32_chain(A, B)
    err, err_chain = oracle.rel_frobenius(C, ref), oracle.rel_frobenius(chain, ref)
    say(f"  rel-Frobenius {err:.2e}, fp32 chain {err_chain:.2e}")
    assert (np.abs(C - ref) <= _bound(A, B)).all()
    assert err <= 1.1 * err_chain  # two independent samples of rounding noise


def _special(kind):
    A, B = oracle.fill_uniform_pm1(5, 256, 256, 96)
    if kind == "tiny":        # all of A: lowest parts would be denormal or lost
        A *= np.float32(2.0 ** -118)
        B *= np.float32(2.0 ** 60)
    elif kind == "tiny_one":  # one element of one row
        A[200, 70] = np.float32(1.2345678 * 2.0 ** -120)
        A[200, :70] = A[200, 71:] = 0
    elif kind == "denormal":
        A[:, 5] = np.float32(2.0 ** -140)
        B[5, :] *= np.float32(2.0 ** 100)
    elif kind == "huge":      # above bf16's largest value, finite products
        A[7, 3] = np.float32(3.4028e38)
        B[3, :] *= np.float32(2.0 ** -20)
    elif kind == "inf":
        A[130, 95] = np.inf
    elif kind == "inf_zero":  # inf * 0 = NaN, in one row only
        A[1, 2] = np.inf
        B[2, 9] = 0
    elif kind == "nan":
        B[31, 200] = np.nan
    elif kind == "overflow":  # finite operands, infinite sums
        A[64] = np.float32(2.0 ** 100)
        B[:, 64] = np.float32(2.0 ** 100)
    elif kind == "zeros":     # signed zeros are ordinary operands
        A[:, ::2] = -0.0
        B[1::3] = 0.0
    return A, B


KINDS = ["tiny", "tiny_one", "denormal", "huge", "inf", "inf_zero", "nan", "overflow", "zeros"]


@pytest.mark.parametrize("kind", KINDS)
def test_split_special_operands(torch_gpu, apk, kind):
    say(f"mfma128 special operands: {kind}")
    A, B = _special(kind)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, 96, blocks=3,
                             with_log=False)
    with np.errstate(all="ignore"):
        chain = oracle.gemm_f32_chain(A, B)
        finite = np.isfinite(chain)
        assert np.array_equal(np.isnan(C), np.isnan(chain))
        assert np.array_equal(C[~finite & ~np.isnan(chain)], chain[~finite & ~np.isnan(chain)])
        ref = A.astype(np.float64) @ B.astype(np.float64)
        A0, B0 = np.nan_to_num(A, posinf=0.0), np.nan_to_num(B)
        bound = _bound(A0, B0)
        assert (np.abs(C - ref)[finite] <= bound[finite]).all()


@pytest.mark.parametrize("kind", ["tiny_one", "inf", "zeros"])
@pytest.mark.parametrize("resume", [0, 1])
def test_split_special_operands_through_yields(torch_gpu, apk, kind, resume):
    """The small operand lies in the first stages of a tile that is then
    checkpointed: the resumed tile must still be computed exactly."""
    say(f"mfma128 special operands through yields: {kind} resume={resume}")
    E = apk.ENGINE_MFMA128
    j = Job(torch_gpu, apk, E, 256, 256, 1024, 32, 128, 128, 64, events=30,
            blocks=min(8, _blocks(apk, E, apk.POLL_STAGE)), passes=20)
    if kind == "tiny_one":
        j.A[:, 8:] = 0
        j.A[:, :8] *= np.float32(2.0 ** -120)
    elif kind == "inf":
        j.A[200, 3] = np.inf
    else:
        j.A[:, ::3] = -0.0
    j.dA.copy_(torch_gpu.from_numpy(j.A))
    off = j.run(apk.POLL_OFF, events=0)
    r = j.run(apk.POLL_STAGE, resume=resume, gap_ticks=1000)
    assert int(r["stats"][:, apk.ST_YIELDS].sum()) >= 5
    assert (_bits(r["C"]) == _bits(off["C"])).all()
    assert (r["task_hash"] == off["task_hash"]).all()
    if kind == "tiny_one":
        ref = j.A.astype(np.float64) @ j.B.astype(np.float64)
        assert (np.abs(off["C"] - ref) <= _bound(j.A[:, :8], j.B[:8])).all()


# An operand alone in its row (column): all that its outputs hold. 2^-134 and
# below round to a bf16 zero; from 2^-110 on the three parts hold every bit.
@pytest.mark.parametrize("exp", [-149, -141, -135, -134, -133, -127, -112, -109, -90])
@pytest.mark.parametrize("side", ["A", "B"])
def test_split_small_operand_alone(torch_gpu, apk, side, exp):
    say(f"mfma128 small operand 2^{exp} alone in {side}")
    A, B = oracle.fill_uniform_pm1(7, 256, 256, 96)
    x = np.float32(-1.2345678 * 2.0 ** exp)
    if side == "A":
        A[200] = 0
        A[200, 70] = x
        B *= np.float32(2.0 ** 100)
    else:
        B[:, 33] = 0
        B[5, 33] = x
        A *= np.float32(2.0 ** 100)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, 96, blocks=3,
                             with_log=False)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    alone = ref[200] if side == "A" else ref[:, 33]
    assert (np.abs(alone) > 0).all()  # a lost operand leaves zeros, far outside the bound
    assert (np.abs(C - ref) <= _bound(A, B)).all()


# Ordinary operands whose products and sums (or only the parts' products) are
# denormal, and operands over a wide range of exponents.
@pytest.mark.parametrize("ea,eb", [(-62, -62), (-70, -70), (-72, -73), (-100, -20)])
def test_split_denormal_sums(torch_gpu, apk, ea, eb):
    say(f"mfma128 operands of 2^{ea} and 2^{eb}")
    A, B = oracle.fill_uniform_pm1(9, 256, 256, 96)
    A *= np.float32(2.0 ** ea)
    B *= np.float32(2.0 ** eb)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, 96, blocks=3,
                             with_log=False)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    assert (np.abs(C - ref) <= _bound(A, B)).all()


@pytest.mark.parametrize("K", [64, 992])
def test_split_wide_exponents(torch_gpu, apk, K):
    say(f"mfma128 wide exponents K={K}")
    rng = np.random.default_rng(3)
    A, B = oracle.fill_uniform_pm1(11, 256, 256, K)
    A *= np.exp2(rng.integers(-30, 30, A.shape)).astype(np.float32)
    B *= np.exp2(rng.integers(-30, 30, B.shape)).astype(np.float32)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, K, blocks=3,
                             with_log=False)
    ref = oracle.gemm_f64(A, B, threads=8)
    err, err_chain = oracle.rel_frobenius(C, ref), oracle.rel_frobenius(
        oracle.gemm_f32_chain(A, B), ref)
    say(f"  rel-Frobenius {err:.2e}, fp32 chain {err_chain:.2e}")
    assert (np.abs(C - ref) <= _bound(A, B)).all()


# The stage from which a tile is exact, at every place in the pipeline: both
# k-steps of the first, the second, a middle and the last stage.
LOSSY_K = [0, 15, 16, 31, 32, 63, 240, 263, 480, 496, 511]


@pytest.mark.parametrize("k", LOSSY_K)
def test_split_exact_from_any_stage(torch_gpu, apk, k):
    say(f"mfma128 small operand at k={k} of 512")
    A, B = oracle.fill_uniform_pm1(19, 256, 256, 512)
    A[77] = 0
    A[77, k] = np.float32(1.2345678 * 2.0 ** -136)
    B *= np.float32(2.0 ** 100)
    C, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, 512, blocks=3,
                             with_log=False)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    assert (np.abs(ref[77]) > 0).all()
    assert (np.abs(C - ref) <= _bound(A, B)).all()
    # the other tiles' rows are those of a run without the small operand
    A[77, k] = 0
    C0, _, _ = run_persistent(torch_gpu, apk, apk.ENGINE_MFMA128, A, B, 512, blocks=3,
                              with_log=False)
    assert (_bits(C[128:]) == _bits(C0[128:])).all()


def _lossy_job(torch, apk, poll, K, k, blocks, **kw):
    j = Job(torch, apk, apk.ENGINE_MFMA128, 512, 512, K, 32, 128, 128, 64,
            blocks=min(blocks, _blocks(apk, apk.ENGINE_MFMA128, poll)), **kw)
    j.A[::50, k] = np.float32(2.0 ** -141)
    j.A[9, 1] = np.inf  # the first row of tiles has to start again
    j.dA.copy_(torch.from_numpy(j.A))
    return j


@pytest.mark.parametrize("poll,resume", [(1, 0), (1, 1), (1, 2), (2, 0), (2, 1), (2, 2), (3, 0),
                                         (3, 1), (3, 2)])
def test_split_modes_through_yields(torch_gpu, apk, poll, resume):
    """Tiles with parts, exact from a middle stage on, and exact throughout,
    yielding at chunk, stage and issue sites in every resume mode."""
    say(f"mfma128 modes through yields: poll={poll} resume={resume}")
    j = _lossy_job(torch_gpu, apk, poll, 1024, 500, 16, events=30, passes=12)
    off = j.run(apk.POLL_OFF, events=0)
    r = j.run(poll, resume=resume, gap_ticks=1000, use_oracle=True)
    assert int(r["stats"][:, apk.ST_YIELDS].sum()) >= 5
    assert (_bits(r["C"]) == _bits(off["C"])).all()
    assert (r["task_hash"] == off["task_hash"]).all()
    assert (r["exec"] == 1).all() and (r["u_exec"][r["set_gt"] != 0] == j.U).all()
    assert int(r["stats"][:, apk.ST_STALE].sum()) == 0


@pytest.mark.parametrize("poll,resume", [(1, 0), (1, 1), (2, 0), (2, 1), (2, 2)])
def test_split_modes_through_retreat(torch_gpu, apk, poll, resume):
    say(f"mfma128 modes through retreat: poll={poll} resume={resume}")
    job = RetreatJob(torch_gpu, apk, apk.ENGINE_MFMA128, 1024, 1024, 2048, 128, 128, 128, 256,
                     passes=16, retreat=4)
    job.dA[::50, 100] = 2.0 ** -141
    job.dA[300, 1] = float("inf")
    ref = job.run(apk.POLL_STAGE, apk.RESUME_CKPT_FULL, preempt=False)
    assert (ref["exec"] == 1).all()
    _check(job, ref, job.run(poll, resume))


def test_split_exact_tiles_are_polled(torch_gpu, apk):
    """Exact products at every poll site: no block goes without one for as long
    as a tile's exact pass takes (K = 8192: about 490 us). A stage and the
    work of one event take some 20 us."""
    say("mfma128 observation latency over exact tiles")
    j = _lossy_job(torch_gpu, apk, apk.POLL_STAGE, 8192, 8190, 16, events=20, passes=4)
    r = j.run(apk.POLL_STAGE, resume=1, gap_ticks=10000)
    lat = (r["obs"] - r["set_gt"][:, None])[(r["set_gt"] != 0)[:, None] & (r["obs"] != 0)]
    say(f"  {lat.size} observations, latest {lat.max() / 100:.1f} us after its event")
    assert lat.size >= 10 * j.blocks and lat.max() < 15000


@pytest.mark.parametrize("kind", ["all", "last_stage"])
def test_split_exact_tiles_cost_one_pass(torch_gpu, apk, kind):
    """Operands with bits below 2^-133 cost at most a pass at the fp32 matrix
    rate: 1.25 of the ordinary time, where computing tiles twice takes 2.2."""
    say(f"mfma128 time of exact tiles: {kind}")
    T, n = torch_gpu, 2048
    A, B = T.rand(n, n, device="cuda") + 0.5, T.rand(n, n, device="cuda") + 0.5
    C = T.empty(n, n, device="cuda")
    q = T.zeros(apk.QUEUE_WORDS, dtype=T.int32, device="cuda")
    st = T.cuda.current_stream().cuda_stream

    def best():
        out = []
        for _ in range(8):
            q.zero_()
            e0, e1 = T.cuda.Event(enable_timing=True), T.cuda.Event(enable_timing=True)
            e0.record()
            apk.persistent_gemm(apk.ENGINE_MFMA128, A.data_ptr(), B.data_ptr(), C.data_ptr(),
                                n, n, n, n, q.data_ptr(), None, 256, st)
            e1.record()
            T.cuda.synchronize()
            out.append(e0.elapsed_time(e1))
        return min(out)

    best()
    plain = best()
    if kind == "all":
        A *= 1e-35
    else:
        A[:, n - 1] = 1e-37
    exact = best()
    say(f"  {1000 * plain:.0f} us, exact {1000 * exact:.0f}")
    assert exact <= 1.6 * plain
