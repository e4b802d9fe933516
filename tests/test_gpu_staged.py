"""The staged forward in two or three launches (stages 2 and 4 work out the decays themselves; stage 4 runs the recurrence over
the chunks where they are few) at the edges of its dispatch, against the float64 sequential oracle and against the stages
called one by one, which share the same arithmetic up to the order of float32 sums."""
from ctypes import byref

import pytest
import torch

from trading_bot_0_amd import ssd, ssd_chunk_scan
from trading_bot_0_amd.synthetic import Workload, make_inputs

from _util import assert_close, check_y, np64, oracle_scan, to_dev
from oracle import c_oracle

pytestmark = pytest.mark.gpu
POLICY, LONG = (8, 32, 64, 1, 128), (16, 64, 128, 2, 256)  # heads, head dimension, state, groups, chunk


# (batch, seqlen, heads, headdim, dstate, groups, chunk): one chunk; a batch of the recurrence and one over (2, 3, 4, 5 chunks);
# the last chunk of one step; heads of 8, 24 and 64; every state width; more chunks than are folded (33), than one round of the
# separate recurrence holds (65) and a run of it that is cut short (18); more tiles, and more bytes, than are folded; one sequence's chunks
# one after the other as fast as a launch (4 and 6 of 16 KB) and slower (7 and 12)
SHAPES = [(1, 1, 1, 8, 16, 1, 32), (3, 70, 4, 24, 16, 1, 128), (2, 129, 2, 64, 128, 1, 64), (2, 161, 8, 32, 64, 1, 32),
          (2, 320, 4, 16, 32, 2, 64), (1, 130, 3, 40, 128, 3, 128), (2, 33 * 32, 2, 16, 16, 1, 32), (1, 65 * 32 - 5, 2, 32, 64, 1, 32),
          (2, 18 * 64 - 63, 2, 8, 64, 2, 64), (70, 8 * 64, 8, 16, 16, 1, 64), (3, 256 * 3 + 1, 16, 64, 128, 2, 256),
          (3, 290, 8, 32, 64, 1, 128), (1, 250, 8, 64, 64, 1, 64), (1, 380, 8, 64, 64, 1, 64), (1, 400, 8, 64, 64, 1, 64),
          (1, 12 * 64, 8, 64, 64, 1, 64)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_against_the_oracle(shape, dtype):
    B, L, H, P, N, G, Q = shape
    if dtype == "f32" and P * N * Q > 64 * 128 * 64:
        Q = 64   # (float32 tiles of the largest head sizes do not fit the LDS)
    w = Workload("staged", B, L, H, P, N, G, Q, dtype=dtype, init_std=0.5)
    cpu = make_inputs(w, seed=L)
    dev = to_dev(cpu)
    g = torch.Generator().manual_seed(L)
    mask = torch.rand(B, L, generator=g) < 0.02
    mask[0, 0] = True                                   # a row whose initial state is not read ...
    dev["init"][0] = float("nan")                       # ... whatever it holds
    cpu["init"][0] = 0.0
    yr, fr = c_oracle_reset(cpu, mask)
    finals = []

    def call(yd):
        y, f = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=Q, initial_states=dev["init"],
                              reset=mask.cuda(), y_dtype=yd)
        finals.append(f)
        return y

    check_y(call, yr, w.torch_dtype, f"{shape} y")
    assert_close(finals[0], fr, w.torch_dtype, f"{shape} final")
    y0, f0 = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=Q, initial_states=dev["init"],
                            reset=mask.cuda(), return_final_states=False)
    assert f0 is None and torch.equal(y0, call(None))   # (a final state that is not asked for changes nothing)


def c_oracle_reset(cpu, mask):
    """Row by row and episode by episode through the sequential oracle."""
    import numpy as np

    x, dt, A, Bm, Cm, D, init = (np64(cpu[k]) for k in ("x", "dt", "A", "B", "C", "D", "init"))
    Bsz, L = mask.shape
    y, fin = np.zeros_like(x), np.zeros((Bsz,) + init.shape[1:])
    for b in range(Bsz):
        cuts = [0] + [t for t in range(1, L) if mask[b, t]] + [L]
        state = init[b:b + 1] * 0.0 if mask[b, 0] else init[b:b + 1]
        for t0, t1 in zip(cuts, cuts[1:]):
            yb, state = c_oracle.ssd_sequential_c(x[b:b + 1, t0:t1].copy(), dt[b:b + 1, t0:t1].copy(), A, Bm[b:b + 1, t0:t1].copy(),
                                                  Cm[b:b + 1, t0:t1].copy(), D, state.copy(), nthreads=1)
            y[b, t0:t1] = yb[0]
            last = state
            state = np.zeros_like(state)
        fin[b] = last[0]
    return y, fin


@pytest.mark.parametrize("batch,seqlen,dims", [(3, 100, POLICY), (3, 400, POLICY), (3, 2000, POLICY), (90, 1024, POLICY), (60, 1000, POLICY),
                                               (8, 2060, LONG)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_final_state_written_over_the_initial_state(batch, seqlen, dims, dtype):
    """A stream's prefix that continues a state in place: the same buffer as initial and final state, at lengths whose separate
    buffers would take the recurrence inside stage 4, or on segments, inside their prologues."""
    if dtype == "f32" and dims is LONG:
        dims = (16, 64, 128, 2, 64)   # (float32 tiles of the largest head sizes do not fit the LDS)
    w = Workload("inplace", batch, seqlen, *dims, dtype=dtype, init_std=0.5)
    cpu = make_inputs(w, seed=3)
    dev = to_dev(cpu)
    yr, fr = oracle_scan(cpu)
    for _ in range(4):
        state = dev["init"].clone()
        y, f = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=dims[4], initial_states=state,
                              final_out=state, y_dtype=torch.float32)
        assert f.data_ptr() == state.data_ptr()
        assert_close(y, yr, w.torch_dtype, "y")
        assert_close(state, fr, w.torch_dtype, "final")


@pytest.mark.parametrize("nc", [1, 7, 8, 9, 15, 17, 63, 64, 65, 129, 200])
def test_state_passing_runs(nc):
    """The recurrence over the chunks in parallel runs: numbers of chunks around the runs' lengths and whole rounds, in place and
    not, against float64 (float32 sums of terms that decay: 1e-5 of the largest is four times what it shows)."""
    g = torch.Generator().manual_seed(nc)
    B, H, P, N, Q = 2, 3, 8, 16, 32
    S = torch.randn(B, nc, H, P, N, generator=g)
    init = torch.randn(B, H, P, N, generator=g)
    dt = torch.rand(B, nc * Q, H, generator=g) * 0.05
    A = -torch.rand(H, generator=g) - 0.1
    dtcs = ssd.chunk_cumsum(dt.cuda(), A.cuda(), Q)
    dec = torch.exp2((dtcs[:, :, :, 0, -1].double() + dtcs[:, :, :, 1, -1].double()).cpu())   # [B,H,nc]
    st, ref = init.double(), []
    for c in range(nc):
        ref.append(st)
        st = dec[:, :, c, None, None] * st + S[:, c].double()
    ref = torch.stack(ref, 1)
    for in_place in (False, True):
        prev, fin = ssd.state_passing(S.cuda(), dtcs, init.cuda(), in_place=in_place)
        assert (prev.cpu().double() - ref).abs().max() <= 1e-5 * ref.abs().max()
        assert (fin.cpu().double() - st).abs().max() <= 1e-5 * st.abs().max()


@pytest.mark.parametrize("batch,seqlen,dims", [(40, 2000, (16, 64, 128, 2, 256)), (300, 1024, (8, 32, 64, 1, 64))])
def test_forward_without_a_workspace_past_the_scratch_array(batch, seqlen, dims):
    """Shapes whose own path (whole rounds of workgroups and a rest on the staged kernels) needs more than the library's scratch array:
    one launch of the one-pass kernel, and so its bits."""
    w = Workload("noalloc", batch, seqlen, *dims, init_std=0.5)
    assert not ssd.chunk_scan_is_onepass(batch, seqlen, *dims, w.torch_dtype)
    assert ssd.workspace_bytes(batch, seqlen, *dims) > 64 << 20
    i = make_inputs(w, seed=7, device="cuda")
    lib, d, code = ssd.load_library(), ssd.SsdDims(batch, seqlen, *dims), ssd.SSD_DTYPE_BF16
    got = []
    for entry in (lib.ssd_chunk_scan_noalloc_fwd, lib.ssd_chunk_scan_onepass_fwd):
        y, fin = torch.empty_like(i["x"]), torch.empty_like(i["init"])
        rc = entry(byref(d), code, i["x"].data_ptr(), i["dt"].data_ptr(), i["A"].data_ptr(), i["B"].data_ptr(), i["C"].data_ptr(),
                   i["D"].data_ptr(), i["init"].data_ptr(), None, y.data_ptr(), fin.data_ptr(), None)
        assert rc == 0, ssd.last_error(lib)
        got.append((y, fin))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("batch,seqlen,dtype,dims", [(24, 2100, "bf16", POLICY), (16, 4100, "bf16", POLICY), (90, 1030, "bf16", POLICY),
                                                     (90, 2500, "bf16", POLICY), (20, 4000, "f32", POLICY), (96, 1999, "f32", POLICY),
                                                     (60, 1001, "f32", POLICY), (24, 2100, "f32", POLICY), (28, 2907, "f32", POLICY),
                                                     (12, 2700, "f32", (8, 32, 32, 1, 64)), (16, 4100, "f32", (8, 32, 32, 1, 64)), (4, 4000, "bf16", LONG), (8, 2060, "bf16", LONG),
                                                     (7, 4097, "bf16", LONG), (30, 2500, "bf16", (4, 32, 128, 1, 64))])
def test_forward_on_segments(batch, seqlen, dtype, dims):
    """Cuts into a few segments (states entering them worked out in the prologues), into eight and more (in a launch of their own; in
    float32 from nine, or fourteen of a 32-wide state) and over two rounds of workgroups, a 128-wide state (two waves per unit), with restarts, a row whose initial state is not read, and
    ragged last segments."""
    w = Workload("segments", batch, seqlen, *dims, dtype=dtype, init_std=0.5)
    assert ssd.chunk_scan_segments(batch, seqlen, *dims, w.torch_dtype) > 1
    cpu = make_inputs(w, seed=seqlen)
    dev = to_dev(cpu)
    mask = torch.rand(batch, seqlen, generator=torch.Generator().manual_seed(5)) < 0.002
    mask[0, 0] = True
    dev["init"][0] = float("nan")
    rows = [0, batch // 2, batch - 1]
    y, f = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=dims[4], initial_states=dev["init"],
                          reset=mask.cuda(), y_dtype=torch.float32)
    sub = {k: (v if k in ("A", "D") else v[rows].clone()) for k, v in cpu.items()}
    sub["init"][0] = 0.0
    yr, fr = c_oracle_reset(sub, mask[rows])
    assert_close(y[rows], yr, w.torch_dtype, "y")
    assert_close(f[rows], fr, w.torch_dtype, "final")


@pytest.mark.parametrize("batch,seqlen,dtype,dims", [(90, 1024, "bf16", POLICY), (33, 2907, "bf16", POLICY), (50, 3001, "bf16", (16, 32, 32, 2, 128)),
                                                     (33, 2100, "bf16", (8, 64, 64, 2, 64)), (96, 1999, "f32", POLICY), (42, 2907, "f32", POLICY),
                                                     (33, 2907, "f32", (8, 32, 32, 1, 64)), (40, 2500, "f32", (8, 64, 64, 2, 64))])
def test_state_continued_in_place_on_few_segments(batch, seqlen, dtype, dims):
    """Where the prologues work out the entering states, a call that writes its final state over its initial one reads a copy of it: the
    same bits as with separate buffers, several workgroups per sequence among them, with rows whose initial state is not read."""
    w = Workload("inplace", batch, seqlen, *dims, dtype=dtype, init_std=0.5)
    assert 1 < ssd.chunk_scan_segments(batch, seqlen, *dims, w.torch_dtype) < 8
    dev = to_dev(make_inputs(w, seed=seqlen))
    mask = torch.rand(batch, seqlen, generator=torch.Generator().manual_seed(6)) < 0.002
    mask[0, 0] = True
    dev["init"][0] = float("nan")
    args = [dev[k] for k in ("x", "dt", "A", "B", "C", "D")]
    y0, f0 = ssd_chunk_scan(*args, chunk=dims[4], initial_states=dev["init"], reset=mask.cuda())
    assert bool(torch.isfinite(f0).all())
    for _ in range(3):
        state = dev["init"].clone()
        y, f = ssd_chunk_scan(*args, chunk=dims[4], initial_states=state, final_out=state, reset=mask.cuda())
        assert f.data_ptr() == state.data_ptr()
        assert torch.equal(y, y0) and torch.equal(state, f0)


@pytest.mark.parametrize("batch,seqlen,dims", [(3, 300, POLICY), (20, 1000, POLICY), (3, 300, (8, 16, 16, 1, 256)), (2, 700, (8, 64, 64, 1, 128))])
def test_float32_result_does_not_depend_on_the_scratch(batch, seqlen, dims):
    """Float32 on the staged kernels: the same bits without a workspace, with one of the size the library names for the sizes as they
    are, with one of the size it uses and with a larger one; a smaller one is refused."""
    w = Workload("scratch", batch, seqlen, *dims, dtype="f32", init_std=0.5)
    i = make_inputs(w, seed=1, device="cuda")
    assert ssd.chunk_scan_segments(batch, seqlen, *dims, torch.float32) == 1

    def call(workspace):
        return ssd_chunk_scan(i["x"], i["dt"], i["A"], i["B"], i["C"], i["D"], chunk=dims[4], initial_states=i["init"], workspace=workspace)

    y, f = call(None)
    least, used = ssd.workspace_bytes(batch, seqlen, *dims), ssd.workspace_bytes(batch, seqlen, *dims, dtype=torch.float32)
    assert least <= used
    for size in (least, used, 4 * used):
        ws = torch.empty(size, dtype=torch.uint8, device="cuda")
        y2, f2 = call(ws)
        assert torch.equal(y, y2) and torch.equal(f, f2), size
        p = ssd.PreparedChunkScan(i["x"], i["dt"], i["A"], i["B"], i["C"], i["D"], chunk=dims[4], initial_states=i["init"], workspace=ws)
        y2, f2 = p()
        assert torch.equal(y, y2) and torch.equal(f, f2), size
    with pytest.raises(ssd.SsdError, match="workspace") as e:
        call(torch.empty(least - 256, dtype=torch.uint8, device="cuda"))
    assert e.value.code == 3


def test_state_passing_over_more_threads_than_one_dimension_of_a_launch():
    """2^31 state elements of one chunk each, and a few more: as many threads as a launch may not have along one dimension.  Without
    decay the state entering is the initial one and the final one the sum, one number per sequence."""
    B, H, P, N = 2 ** 15 + 3, 8, 64, 128
    number = torch.arange(B, device="cuda", dtype=torch.float32)
    S, init = (torch.empty(B, 1, H, P, N, device="cuda").copy_((f * number).view(B, 1, 1, 1, 1)) for f in (1.0, 0.5))
    prev, fin = ssd.state_passing(S, torch.zeros(B, H, 1, 4, 32, device="cuda"), init[:, 0], in_place=True)
    assert prev.data_ptr() == S.data_ptr()
    for got, f in ((prev, 0.5), (fin, 1.5)):
        rows = got.view(B, -1)
        assert torch.equal(rows.amax(1), f * number) and torch.equal(rows.amin(1), f * number)
