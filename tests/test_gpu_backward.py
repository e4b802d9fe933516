"""Backward pass of the scan through the C ABI against the float64 sequential adjoint
(oracle/ssd_backward_oracle.py, itself pinned by central differences of the forward oracle).

Parity rules, with tol = 1e-4 in float32 mode and 2e-2 in bf16 mode: max|out - ref| <= tol * rms(ref) for dx,
ddt, dB, dC and dinitial_states; the gradients stored in bf16 (dx, ddt, dB, dC) are allowed, on top of that, the
one rounding of the exact value that the output format itself costs (2^-8 |ref| per element), for the reason
given in _util.py for the forward's bf16 y.  dA and dD are sums over batch and time of terms of both signs
that largely cancel (with random dy, |dA| is some 1 % of the sum of the |terms|), so their error is measured on
the scale such a sum's rounding lives on: |out - ref| <= tol * (rms(ref) + 2-norm of the summed terms)."""
import numpy as np
import pytest
import torch

from oracle import ssd_backward_oracle as bwd
from oracle import ssd_oracle as orc
from trading_bot_0_amd import SsdError, ssd_chunk_scan, ssd_chunk_scan_backward
from trading_bot_0_amd.synthetic import Workload, make_inputs

from _util import TOL, np64, to_dev

pytestmark = pytest.mark.gpu


def check(out, ref, dtype, what, terms_norm=0.0):
    o = out.detach().float().cpu().numpy().astype(np.float64)
    rms = np.sqrt((ref ** 2).mean())
    allowed = TOL[dtype] * (rms + terms_norm)
    if out.dtype == torch.bfloat16:
        allowed = allowed + 2.0 ** -8 * np.abs(ref)
    worst = (np.abs(o - ref) / allowed).max()
    assert np.isfinite(worst) and worst <= 1.0, f"{what}: error is {worst:.3g} x the allowance (rms {rms:.3g})"


def run_case(w, seed, with_D=True, with_init=True, with_dfinal=True, chunk=None):
    cpu = make_inputs(w, seed=seed)
    if not with_init:
        cpu["init"] = None
    dev = to_dev(cpu)
    g = torch.Generator().manual_seed(seed + 100)
    dy = torch.randn(cpu["x"].shape, generator=g).to(w.torch_dtype)
    dfin = torch.randn(w.batch, w.nheads, w.headdim, w.dstate, generator=g) if with_dfinal else None
    D = cpu["D"] if with_D else None
    ref = bwd.ssd_backward_sequential(np64(cpu["x"]), np64(cpu["dt"]), np64(cpu["A"]), np64(cpu["B"]), np64(cpu["C"]),
                                      np64(D), np64(cpu["init"]), np64(dy), np64(dfin))
    Dd = dev["D"] if with_D else None
    q = chunk or w.chunk
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], Dd, dy.cuda(), chunk=q,
                                  initial_states=dev["init"], dfinal_states=None if dfin is None else dfin.cuda(),
                                  need_dinitial_states=True)
    torch.cuda.synchronize()
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(got[k_out], ref[k_ref], w.torch_dtype, f"{w.name} {k_out}")
    check(got["dA"], ref["dA"], w.torch_dtype, f"{w.name} dA", ref["dA_scale"])
    if with_D:
        check(got["dD"], ref["dD"], w.torch_dtype, f"{w.name} dD", ref["dD_scale"])
    else:
        assert got["dD"] is None
    return got, ref


SHAPES = [
    Workload("bwd_policy_like", 2, 300, 8, 32, 64, 1, 128, init_std=0.5),
    Workload("bwd_groups", 3, 77, 4, 16, 16, 2, 64, init_std=0.5),
    Workload("bwd_per_head_bc", 2, 256, 4, 64, 32, 4, 32, init_std=0.5),
    Workload("bwd_tiny_state", 2, 130, 2, 16, 64, 1, 64, init_std=0.5),
    Workload("bwd_three_heads_per_group", 2, 100, 6, 32, 32, 2, 64, init_std=0.5),   # group sums in their own kernel
    Workload("bwd_long_lookback_heads", 2, 200, 16, 64, 128, 2, 64, init_std=0.3),    # a 128-wide state: scanned in two parts
    Workload("bwd_wide_state_small_heads", 2, 150, 4, 32, 128, 1, 64, init_std=0.3),
]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("w", SHAPES, ids=lambda w: w.name)
def test_gradients_match_the_adjoint(w, dtype):
    run_case(w.with_dtype(dtype), seed=21)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("with_D,with_init,with_dfinal", [(False, False, False), (True, False, True), (False, True, False)])
def test_optional_operands(dtype, with_D, with_init, with_dfinal):
    w = Workload("bwd_optional", 2, 200, 8, 32, 64, 1, 64, dtype=dtype, init_std=0.5)
    run_case(w, seed=5, with_D=with_D, with_init=with_init, with_dfinal=with_dfinal)


@pytest.mark.parametrize("chunk", [32, 64, 128, 256])
def test_chunk_size_does_not_change_the_gradients(chunk):
    w = Workload("bwd_chunks", 2, 300, 8, 32, 64, 1, 128, dtype="f32", init_std=0.5)
    run_case(w, seed=8, chunk=chunk)


def test_plumbing_workload_gradients():
    from trading_bot_0_amd.synthetic import WORKLOADS
    run_case(WORKLOADS["plumbing_f32"], seed=0, with_init=False)


def test_strong_decay_and_heavy_tails():
    w = Workload("bwd_decay_extreme", 2, 384, 8, 32, 64, 1, 128, dtype="f32", a_log_range=(0.01, 64.0),
                 dt_law="mixture", x_law="student-t3")
    run_case(w, seed=3, with_init=False)
    run_case(w.with_dtype("bf16"), seed=3, with_init=False)


def test_directional_derivative_of_the_gpu_forward():
    """Independent of the oracle: the float32 GPU forward's change along a random direction equals the
    gradient's projection on it (central difference, step chosen for float32)."""
    w = Workload("bwd_fd", 2, 96, 4, 32, 64, 1, 32, dtype="f32", init_std=0.5)
    cpu = make_inputs(w, seed=2)
    dev = to_dev(cpu)
    g = torch.Generator().manual_seed(9)
    dy = torch.randn(cpu["x"].shape, generator=g).cuda()
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                  initial_states=dev["init"], need_dinitial_states=True)

    def loss(**kw):
        a = dict(x=dev["x"], dt=dev["dt"], A=dev["A"], B=dev["B"], C=dev["C"], D=dev["D"], init=dev["init"])
        a.update(kw)
        y, _ = ssd_chunk_scan(a["x"], a["dt"], a["A"], a["B"], a["C"], a["D"], chunk=w.chunk, initial_states=a["init"])
        return (y.double() * dy.double()).sum().item()

    for name, key, grad in (("x", "x", "dx"), ("B", "B", "dB"), ("C", "C", "dC"), ("dt", "dt", "ddt"), ("init", "init", "dinitial_states")):
        v = torch.randn(dev[key].shape, generator=g).cuda()
        if name == "dt":
            v = v * dev["dt"] * 0.5          # keep dt positive
        eps = 1e-2
        num = (loss(**{key: dev[key] + eps * v}) - loss(**{key: dev[key] - eps * v})) / (2 * eps)
        ana = (got[grad].double() * v.double()).sum().item()
        assert abs(num - ana) <= 2e-3 * max(1.0, abs(ana)), (name, num, ana)


def test_unsupported_shapes_are_refused():
    w = Workload("bwd_narrow_heads", 1, 64, 4, 8, 64, 1, 64, dtype="bf16")
    dev = to_dev(make_inputs(w, seed=0))
    with pytest.raises(SsdError) as e:
        ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], torch.zeros_like(dev["x"]), chunk=64)
    assert "headdim 16, 32 or 64" in str(e.value)
    w = Workload("bwd_ok", 1, 64, 2, 32, 64, 1, 64, dtype="bf16")
    dev = to_dev(make_inputs(w, seed=0))
    with pytest.raises(ValueError):
        ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], torch.zeros_like(dev["x"]), chunk=64,
                                dfinal_states=torch.zeros(1, 2, 32, 32, device="cuda"))


def test_full_size_policy_shape_against_batch_rows():
    """The benchmark shape (B=256, L=2048, bf16): the per-row gradients of two batch rows against the oracle;
    dA and dD, sums over the whole batch, through their additivity (the full batch equals its two halves added),
    and the per-row gradients of the halves bit for bit those of the full batch."""
    from trading_bot_0_amd.synthetic import WORKLOADS
    w = WORKLOADS["policy_bf16"]
    dev = make_inputs(w, seed=0, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(4)
    dy = torch.randn(dev["x"].shape, generator=g, device="cuda").to(torch.bfloat16)
    full = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                   need_dinitial_states=True)
    rows = [0, w.batch - 1]
    sub = lambda t: t[rows].contiguous()
    ref = bwd.ssd_backward_sequential(np64(sub(dev["x"])), np64(sub(dev["dt"])), np64(dev["A"]), np64(sub(dev["B"])),
                                      np64(sub(dev["C"])), np64(dev["D"]), None, np64(sub(dy)), None)
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(full[k_out][rows], ref[k_ref], torch.bfloat16, f"policy {k_out}")
    half = w.batch // 2
    parts = []
    for sl in (slice(0, half), slice(half, w.batch)):
        c = lambda t: t[sl].contiguous()
        parts.append(ssd_chunk_scan_backward(c(dev["x"]), c(dev["dt"]), dev["A"], c(dev["B"]), c(dev["C"]), dev["D"], c(dy),
                                             chunk=w.chunk))
    for k in ("dA", "dD"):
        both = parts[0][k].double() + parts[1][k].double()
        scale = full[k].double().abs().max().item()
        assert (full[k].double() - both).abs().max().item() <= 1e-5 * scale, k
    assert torch.equal(full["dx"][:half], parts[0]["dx"]) and torch.equal(full["dB"][half:], parts[1]["dB"])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("seqlen", [300, 77])
def test_gradients_with_restarts_inside_the_sequence(dtype, seqlen):
    w = Workload("bwd_reset", 4, seqlen, 8, 32, 64, 1, 128, dtype=dtype, init_std=0.7)
    cpu = make_inputs(w, seed=13)
    dev = to_dev(cpu)
    rng = np.random.default_rng(seqlen)
    m = (rng.random((w.batch, seqlen)) < 0.02).astype(np.uint8)
    m[0] = 0                                   # a row without restarts
    m[1, 0] = 1                                # discards the initial state: its gradient is zero
    for t in (31, 32, 63, 64, 65, 127, 128, seqlen - 1):   # chunk borders of the pass (64 steps) and the last step
        if t < seqlen:
            m[2, t] = 1
    m[3, 40:48] = 1                            # consecutive restarts
    g = torch.Generator().manual_seed(3)
    dy = torch.randn(cpu["x"].shape, generator=g).to(w.torch_dtype)
    dfin = torch.randn(w.batch, w.nheads, w.headdim, w.dstate, generator=g)
    ref = bwd.ssd_backward_sequential(np64(cpu["x"]), np64(cpu["dt"]), np64(cpu["A"]), np64(cpu["B"]), np64(cpu["C"]),
                                      np64(cpu["D"]), np64(cpu["init"]), np64(dy), np64(dfin), reset=m)
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy.cuda(), chunk=w.chunk,
                                  initial_states=dev["init"], dfinal_states=dfin.cuda(), need_dinitial_states=True,
                                  reset=torch.from_numpy(m).cuda())
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(got[k_out], ref[k_ref], w.torch_dtype, f"reset {k_out}")
    check(got["dA"], ref["dA"], w.torch_dtype, "reset dA", ref["dA_scale"])
    check(got["dD"], ref["dD"], w.torch_dtype, "reset dD", ref["dD_scale"])
    assert got["dinitial_states"][1].abs().max().item() == 0.0


@pytest.mark.parametrize("w", [
    Workload("bwd_sums_two_groups", 64, 150, 16, 32, 32, 2, 128, dtype="bf16", init_std=0.5),
    Workload("bwd_sums_ragged", 96, 129, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_sums_short", 100, 5, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_sums_slice_per_wave", 64, 150, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),  # too few groups for two
], ids=lambda w: w.name)
@pytest.mark.parametrize("with_D,with_init,with_dfinal", [(True, True, True), (False, False, False)])
def test_head_sums_taken_on_chip(w, with_D, with_init, with_dfinal):
    """Batches of eight-head groups large enough for the scans that add a group's heads themselves: every
    gradient of every row, with and without the optional operands, ragged last tiles, two groups."""
    run_case(w, seed=21, with_D=with_D, with_init=with_init, with_dfinal=with_dfinal)


@pytest.mark.parametrize("w", [
    Workload("bwd_far_anchors_wide", 192, 64 * 19 + 5, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),    # 20 tiles: runs of 8, 8, 4
    Workload("bwd_far_anchors_narrow", 192, 64 * 10 + 33, 8, 32, 32, 1, 64, dtype="bf16", init_std=0.5),  # 11 tiles: 8, 3
    Workload("bwd_far_anchors_whole_runs", 192, 64 * 16, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_far_anchors_strong_decay", 192, 64 * 12 + 1, 8, 32, 64, 1, 64, dtype="bf16", a_log_range=(0.01, 64.0),
             dt_law="mixture", x_law="student-t3"),
], ids=lambda w: w.name)
def test_decay_gradient_between_far_anchors(w):
    """Where the adjoint scan carries the row products, the two transposed scans' states meet only at every eighth
    tile boundary, and the decay gradient sums its per-step terms over runs of up to 512 steps: sequences of more than
    eight tiles, with a ragged last run and a ragged last tile, restarts on tile and run borders, an initial state and
    a gradient on the final state; both kinds of transposed scan (the one that keeps its tile states runs forward in
    time for a 64-wide state, backward for a 32-wide one).  Rows against the oracle; dA through additivity over the
    batch rows (a batch of three takes the general path, whose anchors stand at every tile)."""
    dev = make_inputs(w, seed=6, device="cuda")
    m = (np.random.default_rng(2).random((w.batch, w.seqlen)) < 0.004).astype(np.uint8)
    m[0] = 0
    for t in (63, 64, 511, 512, 513, 1023, 1024, w.seqlen - 1):   # tile and run borders
        if t < w.seqlen:
            m[1, t] = 1
    m[2, 0] = 1
    g = torch.Generator(device="cuda").manual_seed(4)
    dy = torch.randn(dev["x"].shape, generator=g, device="cuda").to(torch.bfloat16)
    dfin = torch.randn(w.batch, w.nheads, w.headdim, w.dstate, generator=g, device="cuda")
    reset = torch.from_numpy(m).cuda()
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                  initial_states=dev["init"], dfinal_states=dfin, need_dinitial_states=True, reset=reset)
    rows = [0, 1, 2]
    sub = lambda t: None if t is None else t[rows].contiguous()
    ref = bwd.ssd_backward_sequential(np64(sub(dev["x"])), np64(sub(dev["dt"])), np64(dev["A"]), np64(sub(dev["B"])),
                                      np64(sub(dev["C"])), np64(dev["D"]), np64(sub(dev["init"])), np64(sub(dy)),
                                      np64(sub(dfin)), reset=m[rows])
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(got[k_out][rows], ref[k_ref], torch.bfloat16, f"{w.name} {k_out}")
    # the same rows as a batch of their own: the general path.  ddt agrees to the bf16 rounding of either.
    small = ssd_chunk_scan_backward(sub(dev["x"]), sub(dev["dt"]), dev["A"], sub(dev["B"]), sub(dev["C"]), dev["D"], sub(dy),
                                    chunk=w.chunk, initial_states=sub(dev["init"]), dfinal_states=sub(dfin),
                                    need_dinitial_states=True, reset=reset[rows].contiguous())
    check(small["dA"], ref["dA"], torch.bfloat16, f"{w.name} dA (general path)", ref["dA_scale"])
    a, b_ = got["ddt"][rows].double(), small["ddt"].double()
    rms = b_.pow(2).mean().sqrt().item()
    assert ((a - b_).abs() <= 2.0 ** -7 * b_.abs() + 1e-3 * rms).all()
    # dA over the whole batch = the sum of dA over its halves (each half still takes the path under test)
    half = w.batch // 2
    total = torch.zeros_like(got["dA"], dtype=torch.float64)
    for i in range(2):
        sl = slice(i * half, (i + 1) * half)
        c = lambda t: None if t is None else t[sl].contiguous()
        part = ssd_chunk_scan_backward(c(dev["x"]), c(dev["dt"]), dev["A"], c(dev["B"]), c(dev["C"]), dev["D"], c(dy),
                                       chunk=w.chunk, initial_states=c(dev["init"]), dfinal_states=c(dfin), reset=c(reset))
        total += part["dA"].double()
        if i == 0:
            assert torch.equal(part["ddt"][rows], got["ddt"][rows])
    scale = got["dA"].double().abs().max().item()
    assert (got["dA"].double() - total).abs().max().item() <= 1e-5 * scale


@pytest.mark.parametrize("w", [
    Workload("bwd_segments_two_tiles", 2, 65, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),          # 2 segments of a tile
    Workload("bwd_segments_one_tile_each", 1, 64 * 6 + 1, 8, 32, 64, 1, 128, dtype="bf16", init_std=0.5),
    Workload("bwd_segments_ragged", 12, 64 * 23 + 31, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),  # the last is shorter
    Workload("bwd_segments_wide", 40, 64 * 13, 8, 32, 64, 1, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_segments_narrow_state", 3, 64 * 9 + 7, 8, 32, 32, 1, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_segments_three_groups", 2, 64 * 5 + 63, 24, 32, 64, 3, 64, dtype="bf16", init_std=0.5),
    Workload("bwd_segments_strong_decay", 4, 64 * 17 - 1, 8, 32, 64, 1, 64, dtype="bf16", a_log_range=(0.01, 64.0),
             dt_law="mixture", x_law="student-t3"),
], ids=lambda w: w.name)
@pytest.mark.parametrize("carried", [True, False])
def test_gradients_on_segments_of_the_sequence(w, carried):
    """Few sequences run on segments of several tiles, or one, that start from states of their own: restarts on every tile
    border around the segments', a row that restarts at once (whatever its initial state holds), with and without carried
    states, one to three groups of eight heads, both widths of the transposed scans."""
    dev = make_inputs(w, seed=8, device="cuda")
    m = (np.random.default_rng(3).random((w.batch, w.seqlen)) < 0.004).astype(np.uint8)
    m[0] = 0
    if w.batch > 1:
        m[1, 63::64] = 1
        m[1, 0] = 1
        m[-1, 64::64] = 1
    g = torch.Generator(device="cuda").manual_seed(5)
    dy = torch.randn(dev["x"].shape, generator=g, device="cuda").to(torch.bfloat16)
    dfin = torch.randn(w.batch, w.nheads, w.headdim, w.dstate, generator=g, device="cuda") if carried else None
    init = dev["init"] if carried else None
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                  initial_states=init, dfinal_states=dfin, need_dinitial_states=True,
                                  reset=torch.from_numpy(m).cuda())
    ref = bwd.ssd_backward_sequential(np64(dev["x"]), np64(dev["dt"]), np64(dev["A"]), np64(dev["B"]), np64(dev["C"]),
                                      np64(dev["D"]), np64(init), np64(dy), np64(dfin), reset=m)
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(got[k_out], ref[k_ref], torch.bfloat16, f"{w.name} {k_out}")
    check(got["dA"], ref["dA"], torch.bfloat16, f"{w.name} dA", ref["dA_scale"])
    check(got["dD"], ref["dD"], torch.bfloat16, f"{w.name} dD", ref["dD_scale"])


def test_restarts_on_the_one_pass_adjoint_scan():
    """Enough bf16 sequences for the adjoint recurrence to take the one-pass kernel: rows against the oracle."""
    w = Workload("bwd_reset_onepass", 96, 200, 8, 32, 64, 1, 128, dtype="bf16")
    dev = make_inputs(w, seed=2, device="cuda")
    m = (np.random.default_rng(1).random((w.batch, w.seqlen)) < 0.03).astype(np.uint8)
    m[5, 0] = 1
    m[5, 64] = 1
    g = torch.Generator(device="cuda").manual_seed(4)
    dy = torch.randn(dev["x"].shape, generator=g, device="cuda").to(torch.bfloat16)
    got = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                  need_dinitial_states=True, reset=torch.from_numpy(m).cuda())
    rows = [0, 5, 95]
    sub = lambda t: t[rows].contiguous()
    ref = bwd.ssd_backward_sequential(np64(sub(dev["x"])), np64(sub(dev["dt"])), np64(dev["A"]), np64(sub(dev["B"])),
                                      np64(sub(dev["C"])), np64(dev["D"]), None, np64(sub(dy)), None, reset=m[rows])
    for k_out, k_ref in (("dx", "dx"), ("ddt", "ddt"), ("dB", "dB"), ("dC", "dC"), ("dinitial_states", "dinit")):
        check(got[k_out][rows], ref[k_ref], torch.bfloat16, f"one-pass reset {k_out}")


@pytest.mark.parametrize("batch", [3, 96])
def test_backward_inside_a_captured_graph(batch):
    """The backward pass allocates nothing and synchronises nothing either, so a training step that holds it can be
    captured (trading_bots/src/torch/train/update.rs:206-330): the general path (3 sequences) and the path on the
    one-pass kernel's kinds (96).  Replays are interleaved with eager work, inputs change in place between them, and
    every replay is compared with an eager call on the same inputs."""
    w = Workload("bwd_graph", batch, 200, 8, 32, 64, 1, 128, dtype="bf16", init_std=0.3)
    dev = make_inputs(w, seed=5, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(9)
    dy = torch.randn(dev["x"].shape, generator=g, device="cuda").to(torch.bfloat16)
    call = lambda: ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                           initial_states=dev["init"], need_dinitial_states=True)
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = call()
    x_keep, dy_keep = dev["x"].clone(), dy.clone()
    for i in range(3):
        dev["x"].copy_(x_keep * 0.5 if i % 2 else x_keep)
        dy.copy_(dy_keep if i % 2 else dy_keep * 2)
        graph.replay()
        torch.cuda.synchronize()
        eager = call()
        torch.cuda.synchronize()
        for k in ("dx", "ddt", "dA", "dB", "dC", "dD", "dinitial_states"):
            assert torch.equal(captured[k], eager[k]), f"replay {i}: {k}"


def test_calls_from_several_threads_on_their_own_streams():
    """The library keeps no state between calls but a thread-local error string, so host threads may call it at the
    same time (the reference's tests run multi-threaded in one process, trading_bots/src/torch/test_rng.rs:1-40): four
    threads, each with its own stream, inputs and workspace, run forward and backward several times; every result
    equals the single-threaded one bit for bit."""
    import threading
    w = Workload("threads", 6, 257, 8, 32, 64, 1, 128, dtype="bf16", init_std=0.3)
    cases = []
    for seed in range(4):
        dev = make_inputs(w, seed=40 + seed, device="cuda")
        dy = torch.randn(dev["x"].shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(torch.bfloat16)
        y, fin = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=w.chunk, initial_states=dev["init"])
        grads = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                        initial_states=dev["init"], need_dinitial_states=True)
        cases.append((dev, dy, y, fin, grads))
    torch.cuda.synchronize()
    failures = []

    def worker(i):
        dev, dy, y_ref, fin_ref, g_ref = cases[i]
        stream = torch.cuda.Stream()
        try:
            with torch.cuda.stream(stream):
                for _ in range(5):
                    y, fin = ssd_chunk_scan(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], chunk=w.chunk,
                                            initial_states=dev["init"])
                    g = ssd_chunk_scan_backward(dev["x"], dev["dt"], dev["A"], dev["B"], dev["C"], dev["D"], dy, chunk=w.chunk,
                                                initial_states=dev["init"], need_dinitial_states=True)
                    stream.synchronize()
                    ok = torch.equal(y, y_ref) and torch.equal(fin, fin_ref) and all(
                        torch.equal(g[k], g_ref[k]) for k in ("dx", "ddt", "dA", "dB", "dC", "dD", "dinitial_states"))
                    if not ok:
                        failures.append(i)
        except Exception as e:  # noqa: BLE001 - reported below
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
