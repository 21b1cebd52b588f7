"""The calls whose time matters, as a user's program makes them.

Five kinds of work go through the public entry points of apk_amd:

urgent   apk_urgent_gemm: the urgent job, one small GEMM whose latency counts
gemm     apk_persistent_gemm: one whole GEMM on a grid of resident workers
         (the caller clears the queue counters first)
noalloc  apk_persistent_gemm_noalloc: the same for callers that cannot
         allocate (serving loops)
yield    apk_persistent_yield: the preemptible GEMM, with an urgent GEMM
         arriving several times while it runs (device-set events)
tiny     apk_tiny_oracle: the scheduler's exactly-once check on tiny tasks

Operands are those of the measurement binaries: uniform in [-1, 1) for the
fp32 engines, N(0, 1) cast to bf16 for the bf16 ones (Bt = B transposed).
Time stamps (event times, per-tile records) differ from run to run and are
not among the outputs; every computed buffer and every count is.
"""
import math

import numpy as np
import torch

import apk_amd as apk

# Engine name -> (tile rows, tile columns, multiple that K must have).
TILE = {"valu64": (64, 64, 32), "mfma128": (128, 128, 32), "bf16x256": (256, 256, 64),
        "bf16x256x128": (256, 128, 32), "bf16x128": (128, 128, 32)}
# Blocks per CU that an engine's grids are sized for (at most).
PER_CU = {"valu64": 3, "mfma128": 1, "bf16x256": 1, "bf16x256x128": 2, "bf16x128": 4}
POLL = {"off": apk.POLL_OFF, "chunk": apk.POLL_CHUNK, "stage": apk.POLL_STAGE}
RESUME = {"full": apk.RESUME_CKPT_FULL, "acc": apk.RESUME_CKPT_ACC,
          "restart": apk.RESUME_RESTART}
GOLDEN, SALT = 0x9E3779B97F4A7C15, 0xD1B54A32D192ED03


def listed():
    def gemm(name, kind, engine, M, N, K, k_chunk=None, log=False):
        return dict(name=name, kind=kind, engine=engine, M=M, N=N, K=K,
                    k_chunk=K if k_chunk is None else k_chunk, log=log)

    def pre(name, engine, M, N, K, k_chunk, poll, resume, tasks, U, events, gap_us):
        return dict(name=name, kind="yield", engine=engine, M=M, N=N, K=K, k_chunk=k_chunk,
                    poll=poll, resume=resume, tasks=tasks, Mu=U[0], Nu=U[1], Ku=U[2],
                    events=events, gap_us=gap_us)

    return [
        # The urgent job itself, 256x256x256 fp32: the smallest call there is,
        # and the one somebody is waiting for.
        gemm("urgent_fp32", "urgent", "mfma128", 256, 256, 256),
        # A wider urgent job of a bf16 model.
        gemm("urgent_bf16", "urgent", "bf16x256", 512, 512, 512),
        # The reference's own tile and arithmetic (one fmaf chain per output):
        # the parity configuration, with its per-chunk timing records.
        gemm("valu64_parity", "gemm", "valu64", 1024, 1024, 128, 64, True),
        # The headline calibration: 4096^3 fp32, K walked in 32-deep chunks.
        gemm("fp32_4096", "gemm", "mfma128", 4096, 4096, 4096, 32),
        # A mid-size fp32 GEMM of a serving loop: tile counts that do not
        # divide over the CUs and an odd number of k-stages.
        gemm("fp32_ragged_noalloc", "noalloc", "mfma128", 1920, 1408, 992),
        # The large bf16 GEMM, one block per CU.
        gemm("bf16_8192", "gemm", "bf16x256", 8192, 8192, 8192),
        # bf16 at two blocks per CU, an ordinary layer's size.
        gemm("bf16_2cu", "gemm", "bf16x256x128", 4096, 4096, 2048),
        # bf16 at four blocks per CU, ragged in every direction.
        gemm("bf16_4cu_ragged", "gemm", "bf16x128", 2176, 1664, 1056),
        # The preemptible GEMM at the reference's defaults: 48x48 tiles of
        # 64x64, K = 64, 200,000 tasks, polls at every tile boundary. Short
        # tasks: queue pops and epilogues weigh as much as the sums.
        pre("yield_valu64", "valu64", 3072, 3072, 64, 64, "chunk", "full", 200000,
            (128, 128, 64), 8, 20),
        # The preemption study's background job, polls at k-chunk boundaries.
        pre("yield_fp32", "mfma128", 8192, 8192, 4096, 128, "chunk", "full", 4096,
            (256, 256, 256), 8, 20),
        # Its bf16 counterpart, polls at every pair of k-stages.
        pre("yield_bf16", "bf16x256", 8192, 8192, 4096, 256, "stage", "acc", 1024,
            (512, 512, 256), 4, 15),
        # The scheduler check: 4 million one-MFMA tasks, one id per pop.
        dict(name="tiny_oracle", kind="tiny", tasks=4_000_000, batch=1, pa=8, pb=8, events=16,
             per_event=64, gap_us=10, per_cu=2),
    ]


def _log_between(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _multiple(x, m):
    return max(1, round(x / m)) * m


def draw(rng):
    kind = rng.choice(["urgent", "gemm", "gemm", "noalloc", "yield", "yield", "tiny"])
    if kind == "tiny":
        return dict(kind=kind, tasks=int(_log_between(rng, 2_000_000, 4_000_000)),
                    batch=rng.choice([1, 2, 4]), pa=rng.randint(1, 12), pb=rng.randint(1, 12),
                    events=rng.randint(1, 16), per_event=rng.randint(1, 64), gap_us=10, per_cu=rng.choice([1, 2, 4]))
    engine = rng.choice(sorted(TILE))
    tm, tn, ka = TILE[engine]
    if kind == "urgent":
        M = _multiple(_log_between(rng, tm, 1024), tm)
        N = _multiple(_log_between(rng, tn, 1024), tn)
        K = _multiple(_log_between(rng, 64, 4096), ka)
        return dict(kind=kind, engine=engine, M=M, N=N, K=K, k_chunk=K, log=False)
    if kind in ("gemm", "noalloc"):
        top = 3072 if engine == "valu64" else 4096 if engine == "mfma128" else 8192
        M = _multiple(_log_between(rng, 256, top), tm)
        N = _multiple(_log_between(rng, 256, top), tn)
        K = _multiple(_log_between(rng, 64, top), ka)
        parts = [c for c in (32, 64, 96, 128, 160, 224, 256) if K % c == 0 and c % TILE[engine][2] == 0]
        return dict(kind=kind, engine=engine, M=M, N=N, K=K,
                    k_chunk=rng.choice(parts + [K]), log=kind == "gemm" and rng.random() < 0.25)
    # Preemptible jobs long enough for their events (4 at 15 us): passes over
    # the tile grid until the work is at least `least`.
    top = 3072 if engine == "valu64" else 8192
    M = _multiple(_log_between(rng, 1024, top), tm)
    N = _multiple(_log_between(rng, 1024, top), tn)
    k_chunk = _multiple(_log_between(rng, 64, 256), TILE[engine][2])
    K = k_chunk * rng.randint(1, 512 // k_chunk if engine == "valu64" else 4096 // k_chunk)
    K = _multiple(K, math.lcm(k_chunk, ka))
    task = 2.0 * tm * tn * K
    least = {"valu64": 55e9, "mfma128": 110e9}.get(engine, 330e9)
    tasks = max((M // tm) * (N // tn), math.ceil(least / task))
    return dict(kind="yield", engine=engine, M=M, N=N, K=K, k_chunk=k_chunk,
                poll=rng.choice(["off", "chunk", "stage"]),
                resume=rng.choice(["full", "acc", "restart"]), tasks=tasks,
                Mu=tm * rng.randint(1, 2), Nu=tn * rng.randint(1, 2), Ku=64 * rng.randint(1, 4),
                events=rng.randint(1, 4), gap_us=15)


def _operands(engine, M, N, K, gen):
    if engine.startswith("bf16"):
        A = torch.randn(M, K, generator=gen, device="cuda").to(torch.bfloat16)
        B = torch.randn(N, K, generator=gen, device="cuda").to(torch.bfloat16)  # transposed
    else:
        A = torch.rand(M, K, generator=gen, device="cuda") * 2 - 1
        B = torch.rand(K, N, generator=gen, device="cuda") * 2 - 1
    return A, B


def _inputs(case, seed):
    """The operands of a case, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "tiny":  # small integers: every sum is exact
        pool = lambda n: torch.randint(-4, 5, (n, 16, 16), generator=gen, device="cuda").to(torch.bfloat16)
        return pool(case["pa"]), pool(case["pb"])
    ops = _operands(case["engine"], case["M"], case["N"], case["K"], gen)
    if case["kind"] == "yield":
        ops += _operands(case["engine"], case["Mu"], case["Nu"], case["Ku"], gen)
    return ops


def _fill(params, **values):
    for k, v in values.items():
        setattr(params, k, v.data_ptr() if torch.is_tensor(v) else v)


def prepare(case, seed):
    ops = _inputs(case, seed)
    st = dict(case=case, ops=ops, stream=torch.cuda.current_stream().cuda_stream)
    cus = apk.device_info().cu_count
    zeros32 = lambda n: torch.zeros(n, dtype=torch.int32, device="cuda")
    zeros64 = lambda n: torch.zeros(n, dtype=torch.int64, device="cuda")
    if case["kind"] == "tiny":
        return _prepare_tiny(case, st, cus, zeros32, zeros64)
    engine = st["engine"] = apk.ENGINES[case["engine"]]
    M, N = case["M"], case["N"]
    st["C"] = torch.zeros(M, N, device="cuda")
    per_cu = PER_CU[case["engine"]]
    if case["kind"] in ("urgent", "gemm", "noalloc"):
        st["blocks"] = cus * min(per_cu, apk.occupancy(engine))
        st["next"] = zeros32(apk.QUEUE_WORDS)
        tm, tn, _ = TILE[case["engine"]]
        records = (M // tm) * (N // tn) * (case["K"] // case["k_chunk"])
        st["log"] = zeros64(records * 3) if case["log"] else None
        return st
    # The preemptible job: everything that is cleared before a launch lies in
    # one buffer, so that one fill clears it.
    E, poll = case["events"], POLL[case["poll"]]
    blocks = st["blocks"] = cus * min(per_cu, apk.yield_occupancy(engine, poll))
    st["poll"] = poll
    names = dict(next_task=8, uq_next=E, flag=1, claim=E, claim_site=E, u_end_max=E, set_gt=E,
                 u_gt=2 * E, obs_gt=E * blocks, u_exec=E, exec=(case["tasks"] + 1) // 2)
    # 8-byte words; the flag alone on a line of its own
    offsets, total = {}, 0
    for k, n in names.items():
        offsets[k] = total
        total += (n + 15) // 16 * 16
    clear = st["clear"] = zeros64(total)
    part = {k: clear[offsets[k]:offsets[k] + n] for k, n in names.items()}
    Cu = st["Cu"] = torch.zeros(E, case["Mu"], case["Nu"], device="cuda")
    st["sched"] = torch.arange(1, E + 1, dtype=torch.int64, device="cuda") * (case["gap_us"] * 100)
    st["ckpt"] = torch.zeros(blocks * apk.ckpt_floats(engine), device="cuda")
    A, B, Au, Bu = ops
    p = st["params"] = apk.YieldParams()
    _fill(p, A=A, B=B, C=st["C"], M=M, N=N, K=case["K"], k_chunk=case["k_chunk"],
          num_tasks=case["tasks"], next_task=part["next_task"], Au=Au, Bu=Bu, Cu=Cu,
          Mu=case["Mu"], Nu=case["Nu"], Ku=case["Ku"], uq_next=part["uq_next"],
          flag=part["flag"], flag_copies=1, flag_set=part["flag"], sched=st["sched"],
          num_events=E, poll_every=1, set_gt=part["set_gt"], obs_gt=part["obs_gt"],
          claim=part["claim"], claim_site=part["claim_site"], u_gt=part["u_gt"],
          u_end_max=part["u_end_max"], resume=RESUME[case["resume"]], ckpt=st["ckpt"],
          cu_event_stride=case["Mu"] * case["Nu"], exec_count=part["exec"],
          u_exec_count=part["u_exec"])
    st["exec"] = part["exec"].view(torch.int32)[:case["tasks"]]
    st["u_exec"] = part["u_exec"].view(torch.int32)[:E]
    return st


def _prepare_tiny(case, st, cus, zeros32, zeros64):
    E, n = case["events"], case["tasks"]
    blocks = st["blocks"] = cus * case["per_cu"]
    offsets, total = {}, 0
    names = dict(next_task=8, checksum=2, stats=2, flag=1, set_gt=E, uq_next=E, u_exec=E,
                 exec=(n + 1) // 2)
    for k, m in names.items():
        offsets[k] = total
        total += (m + 15) // 16 * 16
    clear = st["clear"] = zeros64(total)
    part = {k: clear[offsets[k]:offsets[k] + m] for k, m in names.items()}
    st["sched"] = torch.arange(1, E + 1, dtype=torch.int64, device="cuda") * (case["gap_us"] * 100)
    st["ckpt"] = torch.zeros(blocks * 4 * 256, device="cuda")
    p = st["params"] = apk.TinyParams()
    _fill(p, num_tasks=n, next_task=part["next_task"], batch=case["batch"], A=st["ops"][0],
          Bt=st["ops"][1], pa=case["pa"], pb=case["pb"], exec_count=part["exec"],
          checksum=part["checksum"], flag=part["flag"], sched=st["sched"], num_events=E,
          set_gt=part["set_gt"], uq_next=part["uq_next"], urgent_per_event=case["per_event"],
          u_exec_count=part["u_exec"], ckpt=st["ckpt"], stats=part["stats"])
    st["exec"] = part["exec"].view(torch.int32)[:n]
    st["u_exec"] = part["u_exec"].view(torch.int32)[:E]
    st["checksum"] = part["checksum"]
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "tiny":
        st["clear"].zero_()
        apk.tiny_oracle(st["params"], st["blocks"], st["stream"])
        return st["exec"], st["u_exec"], st["checksum"]
    if kind == "yield":
        st["clear"].zero_()
        apk.persistent_yield(st["engine"], st["poll"], True, st["params"], st["blocks"],
                             st["stream"])
        # without polls the events are never raised and Cu stays as it was
        return st["C"], st["Cu"], st["exec"], st["u_exec"]
    A, B = st["ops"]
    args = (st["engine"], A.data_ptr(), B.data_ptr(), st["C"].data_ptr(), case["M"], case["N"],
            case["K"])
    if kind == "urgent":
        apk.urgent_gemm(*args, None, None, st["stream"])
        return st["C"]
    log = None if st["log"] is None else st["log"].data_ptr()
    if kind == "noalloc":
        apk.persistent_gemm_noalloc(*args, case["k_chunk"], log, st["blocks"], st["stream"])
        return st["C"]
    st["next"].zero_()
    apk.persistent_gemm(*args, case["k_chunk"], st["next"].data_ptr(), log, st["blocks"],
                        st["stream"])
    return st["C"]


def work(case):
    if case["kind"] == "tiny":
        # one 16x16x16 product a task; its execution counter is written once
        done = case["tasks"] + case["events"] * case["per_event"]
        return {"bytes": 4 * case["tasks"] + 512 * (case["pa"] + case["pb"]), "flops": 8192 * done}
    M, N, K = case["M"], case["N"], case["K"]
    elem = 2 if case["engine"].startswith("bf16") else 4
    nbytes, flops = elem * (M * K + K * N) + 4 * M * N, 2 * M * N * K
    if case["kind"] == "yield":
        tm, tn, _ = TILE[case["engine"]]
        E = 0 if case["poll"] == "off" else case["events"]
        Mu, Nu, Ku = case["Mu"], case["Nu"], case["Ku"]
        flops = 2 * tm * tn * K * case["tasks"] + E * 2 * Mu * Nu * Ku
        nbytes += 4 * case["tasks"] + elem * (Mu * Ku + Ku * Nu) + 4 * E * Mu * Nu
    if case.get("log"):
        tm, tn, _ = TILE[case["engine"]]
        nbytes += 24 * (M // tm) * (N // tn) * (K // case["k_chunk"])
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # valu64 promises one fmaf chain per output in k order, and the tiny
    # tasks multiply small integers: nothing may differ.
    if case["kind"] == "tiny" or case["engine"] == "valu64":
        return "exact"
    # fp32 accumulation over K terms; four times the error against 64 bits
    # (1.15e-6 at K = 4096 for fp32 operands, 5.7e-7 at K = 8192 for bf16).
    return {"rel": 5e-6 if case["engine"] == "mfma128" else 2.5e-6}


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _exact_tiny(case, seed):
    A, Bt = (x.to(torch.float32).cpu().numpy() for x in _inputs(case, seed))
    pa, pb, E, U, n = case["pa"], case["pb"], case["events"], case["per_event"], case["tasks"]
    lane = np.arange(64)
    value = np.zeros((pa, pb), dtype=np.uint64)
    with np.errstate(over="ignore"):
        for a in range(pa):
            for b in range(pb):
                C = A[a] @ Bt[b].T
                for j in range(4):
                    bits = C[4 * (lane // 16) + j, lane % 16].astype(np.float32).view(np.uint32)
                    place = (4 * lane + j).astype(np.uint64) << np.uint64(32)
                    value[a, b] += _mix(bits.astype(np.uint64) + place).sum(dtype=np.uint64)
        t = np.arange(n, dtype=np.uint64)
        v = value[t % np.uint64(pa), (t // np.uint64(pa)) % np.uint64(pb)]
        background = _mix(v + t * np.uint64(GOLDEN)).sum(dtype=np.uint64)
        i = np.arange(E * U, dtype=np.uint64)
        v = value[(i * np.uint64(7) + np.uint64(3)) % np.uint64(pa),
                  (i * np.uint64(13) + np.uint64(5)) % np.uint64(pb)]
        urgent = _mix(v + i * np.uint64(GOLDEN) + np.uint64(SALT)).sum(dtype=np.uint64)
    return (np.ones(n, dtype=np.int32), np.full(E, U, dtype=np.int32),
            np.array([background, urgent], dtype=np.uint64).view(np.int64))


def exact(case, seed):
    if case["kind"] == "tiny":
        return _exact_tiny(case, seed)
    ops = _inputs(case, seed)

    def product(A, B):
        B = B.double()
        return A.double() @ (B.t().contiguous() if case["engine"].startswith("bf16") else B)

    C = product(ops[0], ops[1])
    if case["kind"] != "yield":
        return C
    E = case["events"]
    tm, tn, _ = TILE[case["engine"]]
    counts = torch.ones(case["tasks"], dtype=torch.int32)
    if case["poll"] == "off":
        return (C, torch.zeros(E, case["Mu"], case["Nu"], dtype=torch.float64), counts,
                torch.zeros(E, dtype=torch.int32))
    Cu = product(ops[2], ops[3])
    tiles = (case["Mu"] // tm) * (case["Nu"] // tn)
    return (C, Cu.expand(E, -1, -1).contiguous(), counts,
            torch.full((E,), tiles, dtype=torch.int32))
