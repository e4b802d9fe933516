"""The path plan of ssd_chunk_scan_fwd against the clock.  The library decides from a cost model (time per tile and
workgroup of the one-pass kernel, time per unit-tile of the staged kernels, cost of a launch) whether a shape runs on
the staged kernels, as one launch of the one-pass kernel, or on the one-pass kernel over segments of the sequence.
The model's constants are measurements that every kernel change moves; this test times, either side of the model's
cross-overs, the plan's choice beside the alternatives a caller can force -- the one-pass kernel
(ssd_chunk_scan_onepass_fwd), the staged kernels through their own entry points, and a batch of more than a round of
workgroups as two calls, its whole rounds as one launch and the rest as the plan says for it -- and asserts that what the
plan picked is within a quarter of the fastest of them, but for 5 us of launches in all but the shortest calls (a wrong side of a
cross-over costs a factor of about two).

Timing: the best of three means over twenty calls, HIP events on the launch stream, after a spin of the same work."""
from ctypes import byref

import pytest
import torch

from trading_bot_0_amd import ssd
from trading_bot_0_amd.synthetic import Workload, make_inputs

pytestmark = pytest.mark.gpu


def best_of(fn, reps=3, calls=20):
    for _ in range(5):
        fn()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(reps):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(calls):
            fn()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / calls * 1e3)
    return best   # microseconds


SHAPES = [
    # (nheads, headdim, dstate, ngroups, seqlen, batches either side of the cross-overs)
    (8, 32, 64, 1, 2048, "bf16", (4, 16, 32, 64, 128, 160, 256, 272)),   # staged | segments | one launch | whole rounds + a rest
    (8, 32, 64, 1, 512, "bf16", (16, 64, 128, 256)),
    (8, 32, 64, 1, 64, "bf16", (1, 16, 40)),                             # as short as the launches themselves
    (4, 32, 64, 1, 96, "bf16", (1, 16, 40)),
    (8, 32, 32, 1, 128, "bf16", (1, 16, 40)),
    (8, 32, 32, 1, 64, "f32", (1, 16, 40)),
    (8, 32, 64, 1, 8192, "bf16", (24, 130, 170, 250)),                   # more than half a round of long sequences: uncut
    (4, 32, 64, 1, 2048, "bf16", (32, 64, 128, 192, 256, 512)),          # four units per group: staged | four-wave one-pass
    (16, 64, 128, 2, 4096, "bf16", (1, 4, 8, 16)),                       # 128-wide state
    (8, 32, 64, 1, 300, "f32", (3, 30, 60, 100, 285)),                   # staged | one launch | whole rounds + a rest
    (8, 32, 64, 1, 2000, "f32", (2, 10, 20, 60, 96, 130, 200, 272)),     # staged | segments | one launch | whole rounds + a rest
    (8, 32, 32, 1, 6000, "f32", (2, 6, 20, 104, 150)),
]


@pytest.mark.parametrize("H,P,N,G,L,dtype,batches", SHAPES)
def test_plan_picks_a_path_within_a_quarter_of_the_fastest(H, P, N, G, L, dtype, batches):
    lib = ssd.load_library()
    report = []
    code, td = (ssd.SSD_DTYPE_BF16, torch.bfloat16) if dtype == "bf16" else (ssd.SSD_DTYPE_F32, torch.float32)
    for Bsz in batches:
        w = Workload("plan", Bsz, L, H, P, N, G, 128 if dtype == "bf16" else 64, dtype=dtype)
        inp = make_inputs(w, seed=1, device="cuda")
        x, dt, A, Bm, Cm, D = (inp[k] for k in ("x", "dt", "A", "B", "C", "D"))
        plan = ssd.PreparedChunkScan(x, dt, A, Bm, Cm, D, chunk=w.chunk)
        t_plan = best_of(plan)
        times = {}
        y = torch.empty_like(x)
        fin = torch.empty(Bsz, H, P, N, device="cuda")
        dims = ssd.SsdDims(Bsz, L, H, P, N, G, w.chunk)
        stream = torch.cuda.current_stream().cuda_stream

        def onepass(batch=Bsz):
            return lib.ssd_chunk_scan_onepass_fwd(byref(ssd.SsdDims(batch, L, H, P, N, G, w.chunk)), code, x.data_ptr(), dt.data_ptr(),
                                                  A.data_ptr(), Bm.data_ptr(), Cm.data_ptr(), D.data_ptr(), None, None, y.data_ptr(),
                                                  fin.data_ptr(), stream)

        per_round = 256 // (G * max(1, (H // G) * (P // 32) // (4 if N == 128 and dtype == "bf16" else 8)))
        if onepass() == 0:
            times["one-pass"] = best_of(onepass)
            whole = Bsz // per_round * per_round
            if 0 < whole < Bsz and H // G * (P // 32) % 8 == 0:
                rest = ssd.PreparedChunkScan(x[whole:], dt[whole:], A, Bm[whole:], Cm[whole:], D, chunk=w.chunk)
                times["whole rounds, then the rest"] = best_of(lambda: (onepass(whole), rest()))
                del rest
        else:
            ssd.last_error(lib)   # (clear the message of a shape the one-pass kernel does not take)
        dtcs = ssd.chunk_cumsum(dt, A, w.chunk)
        prev, _ = ssd.chunk_state_passing(x, Bm, dtcs)

        def staged():
            lib.ssd_chunk_cumsum_fwd(byref(dims), code, dt.data_ptr(), A.data_ptr(), dtcs.data_ptr(), stream)
            lib.ssd_chunk_state_passing_fwd(byref(dims), code, x.data_ptr(), Bm.data_ptr(), dtcs.data_ptr(), None,
                                            prev.data_ptr(), fin.data_ptr(), stream)
            lib.ssd_chunk_scan_stage_fwd(byref(dims), code, x.data_ptr(), Bm.data_ptr(), Cm.data_ptr(),
                                         dtcs.data_ptr(), prev.data_ptr(), D.data_ptr(), y.data_ptr(), stream)

        times["staged"] = best_of(staged)
        fastest = min(times.values())
        segs = ssd.chunk_scan_segments(Bsz, L, H, P, N, G, w.chunk, td)
        one = ssd.chunk_scan_is_onepass(Bsz, L, H, P, N, G, w.chunk, td)
        chosen = "one launch" if one else (f"{segs} segments" if segs > 1 else "staged / split")
        report.append(f"batch {Bsz}: plan ({chosen}) {t_plan:.0f} us; " + ", ".join(f"{k} {v:.0f}" for k, v in times.items()))
        assert t_plan <= 1.25 * fastest + (5.0 if L > 128 else 1.0), "\n".join(report)
        del plan, inp, x, dt, Bm, Cm, y, fin, dtcs, prev
    print("\n".join(report))


@pytest.mark.parametrize("H,P,N,L,few,more", [(4, 32, 64, 320, 1, 2), (4, 64, 64, 300, 3, 4), (4, 16, 16, 290, 5, 6)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_fewer_sequences_take_no_longer(H, P, N, L, few, more, dtype):
    """Staged calls whose tiles all have a workgroup of their own: a number of tiles that is no multiple of the eight XCDs (12, 36 and 60 or
    100) takes what the next one that is takes (24, 48 and 72 or 120), a tenth and half a microsecond allowed, not one more tile of 6 us."""
    times = []
    for Bsz in (few, more):
        w = Workload("plan", Bsz, L, H, P, N, 1, 128 if P * N > 2048 or dtype == "bf16" and P > 16 else 64, dtype=dtype)
        inp = make_inputs(w, seed=1, device="cuda")
        times.append(best_of(ssd.PreparedChunkScan(*(inp[k] for k in ("x", "dt", "A", "B", "C", "D")), chunk=w.chunk)))
        assert ssd.chunk_scan_segments(Bsz, L, H, P, N, 1, w.chunk, w.torch_dtype) == 1
        assert not ssd.chunk_scan_is_onepass(Bsz, L, H, P, N, 1, w.chunk, w.torch_dtype)
    print(times)
    assert times[0] <= 1.1 * times[1] + 0.5
