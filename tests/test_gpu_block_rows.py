"""The block's kernels for few rows at the lines of their dispatch."""
import pytest
import torch

from trading_bot_0_amd import block_post, block_post_proj, block_proj

pytestmark = pytest.mark.gpu

H, N, G = 8, 64, 1


def inputs(rows, di, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    y = torch.randn(1, rows, H, di // H, generator=g, device="cuda").to(torch.bfloat16)
    z = torch.randn(1, rows, 2 * di + 2 * G * N + H, generator=g, device="cuda").to(torch.bfloat16)
    nw = 1 + 0.2 * torch.randn(di, generator=g, device="cuda")
    w = (torch.randn(n, di, generator=g, device="cuda") / di ** 0.5).to(torch.bfloat16)
    return y, z, nw, w


@pytest.mark.parametrize("di,n", [(256, 256), (256, 72), (128, 200), (128, 8)])
def test_fused_out_projection_of_few_rows_is_the_one_of_many(di, n):
    """Workgroups of 32 rows (up to a round of them), of 64 (up to two) and the kernel of many rows give a row the same bits: slices
    of 40 000 rows, with last tiles that are whole, of one row and one short, against the whole."""
    y, z, nw, w = inputs(40000, di, n, di + n)
    whole = block_post_proj(y, z, nw, w, H, di // H, N, G)
    for rows in (1, 31, 32, 33, 600, 8191, 8192, 8193, 12000, 16385, 32767, 32768, 32769):
        for at in (0, 40000 - rows):
            part = block_post_proj(y[:, at:at + rows].contiguous(), z[:, at:at + rows].contiguous(), nw, w, H, di // H, N, G)
            assert torch.equal(part, whole[:, at:at + rows]), (rows, at)


def test_fused_out_projection_of_few_rows_next_to_the_two_stages():
    """Against float64 on the same inputs: no further off than the post stage and the projection one after the other."""
    y, z, nw, w = inputs(700, 256, 256, 3)
    v = y.double().view(1, 700, 256) * torch.nn.functional.silu(z[..., :256].double())
    exact = (v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-5) * nw.double()) @ w.double().t().contiguous()
    err = lambda o: ((o.double() - exact).norm() / exact.norm()).item()
    one, two = err(block_post_proj(y, z, nw, w, H, 32, N, G)), err(block_proj(block_post(y, z, nw, H, 32, N, G), w))
    assert one <= 1.02 * two, f"{one:.3e} against the two stages' {two:.3e}"


def test_fused_out_projection_writes_nothing_past_its_rows_and_columns():
    y, z, nw, w = inputs(45, 256, 72, 5)
    out = block_post_proj(y, z, nw, w, H, 32, N, G)
    big = torch.full((64, 256), 7.0, dtype=torch.bfloat16, device="cuda")
    from ctypes import byref, c_float

    from trading_bot_0_amd import ssd
    from trading_bot_0_amd.block import SsdBlockDims, _lib
    lib = _lib()
    ssd._check(lib, lib.ssd_block_post_proj_fwd(byref(SsdBlockDims(1, 45, H, 32, N, G, 4, 0)), ssd.SSD_DTYPE_BF16, y.data_ptr(),
                                                z.data_ptr(), nw.data_ptr(), c_float(1e-5), w.data_ptr(), 72, 256, big.data_ptr(),
                                                ssd._stream_ptr(y)))
    torch.cuda.synchronize()
    assert torch.equal(big[:45, :72], out[0]) and bool((big[45:] == 7).all()) and bool((big[:, 72:] == 7).all())


def block_inputs(B, L, dtype, seed, P=32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    C, E = H * P + 2 * G * N, 2 * H * P + 2 * G * N + H
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    z = rnd(B, L, E).to(dtype)
    reset = (torch.rand(B, L, generator=g, device="cuda") < 0.05).to(torch.uint8)
    return z, rnd(C, 4) / 2, rnd(C) * 0.1, rnd(H), reset, rnd


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L", [(40, 1111), (700, 33), (2000, 9), (6000, 3)])
def test_pre_stage_runs_of_four_and_of_eight(B, L, dtype):
    """Many rows walk runs of 8 timesteps, few of 4, with last runs of 1 to 3: single sequences, carried state and restarts among
    them, are bit for bit the batch's."""
    from trading_bot_0_amd import block_pre
    z, w, b, bias, reset, rnd = block_inputs(B, L, dtype, L)
    state = rnd(B, 3, w.shape[0]).to(dtype)
    whole = block_pre(z, w, b, bias, H, 32, N, G, conv_state=state, return_conv_state=True, reset=reset)
    for i in (0, 1, B // 2, B - 1):
        one = block_pre(z[i:i + 1].contiguous(), w, b, bias, H, 32, N, G, conv_state=state[i:i + 1].contiguous(),
                        return_conv_state=True, reset=reset[i:i + 1].contiguous())
        assert all(torch.equal(a, c[i:i + 1]) for a, c in zip(one, whole)), i


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L,restarts", [(5, 4111, False), (5, 4111, True), (700, 33, True), (1, 1, True), (1, 130, False), (9, 31, True)])
def test_pre_stage_backward_runs_of_eight_and_of_thirty_two(B, L, restarts, dtype):
    """Beyond 20 480 rows the conv's backward walks runs of 32 timesteps, below of 8: a batch's rows of dzxbcdt against those of its
    sequences alone, bit for bit, and the parameter gradients, float32 sums over B L terms in other orders, within 1e-5 of the
    terms' norm (the sequences' own sums added in float64)."""
    from trading_bot_0_amd.block import block_pre_bwd
    z, w, b, bias, reset, rnd = block_inputs(B, L, dtype, B + L)
    reset = reset if restarts else None
    dx, dB, dC, ddt = (rnd(*s).to(dtype) for s in ((B, L, H, 32), (B, L, G, N), (B, L, G, N), (B, L, H)))

    def run(i, j):
        part = lambda t: None if t is None else t[i:j].contiguous()
        dz = torch.zeros_like(part(z))
        out = block_pre_bwd(part(z), w, b, bias, part(dx), part(dB), part(dC), part(ddt), dz, H, 32, N, G, reset=part(reset))
        return dz, out[:3]

    dz, sums = run(0, B)
    each = [run(i, i + 1) for i in range(B if B < 20 else 20)]
    for i, (d, _) in enumerate(each):
        assert torch.equal(d, dz[i:i + 1]), i
    if B < 20:
        for k, s in enumerate(sums):
            ref = sum(e[1][k].double() for e in each)
            assert (s.double() - ref).norm() <= 1e-5 * (B * L) ** 0.5 * max(1.0, ref.norm().item() / (B * L) ** 0.5), k


@pytest.mark.parametrize("E,D", [(648, 256), (392, 128), (8, 8), (136, 72), (1024, 200), (2544, 16)])
@pytest.mark.parametrize("rows", [1, 31, 33, 64, 700, 8193, 20000])
def test_input_gradient_of_a_projection(rows, E, D):
    """a . w against float64, at the workgroups' sizes (32 x 128, 64 x 128, 64 x 256), features off the steps of 16 and columns off the
    blocks; a is the first columns of longer rows whose rest is not a number.  The bound is rounding alone: one of the result, and
    float32 sums of E terms."""
    from trading_bot_0_amd.block import block_dproj, turned_weight
    g = torch.Generator(device="cuda").manual_seed(rows + E)
    buf = torch.full((rows, (E + 63) // 64 * 64), float("nan"), dtype=torch.bfloat16, device="cuda")
    buf[:, :E] = torch.randn(rows, E, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(E, D, generator=g, device="cuda") / E ** 0.5).to(torch.bfloat16)
    out = block_dproj(buf[:, :E], turned_weight(w))
    ref, mag = buf[:, :E].double() @ w.double(), buf[:, :E].double().abs() @ w.double().abs()
    assert out.shape == (rows, D) and ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + E * 2.0 ** -24 * mag).all()
    assert torch.equal(block_dproj(buf[:, :E].contiguous(), turned_weight(w)), out)


@pytest.mark.parametrize("shape", [(256, 8, 32, 64, 1), (72, 8, 16, 16, 2), (128, 4, 40, 32, 1)])
def test_weights_converted_in_one_launch(shape):
    """The bf16 copies are torch's own rounding, the turned ones their transposes, padded with zeros; again after an update in place."""
    from trading_bot_0_amd import Mamba2Block
    from trading_bot_0_amd.block import turned_weight
    d_model, heads, P, ns, groups = shape
    blk = Mamba2Block(d_model, heads, P, ns, groups, seed=1)
    for _ in range(2):
        _, w_in, w_out, w_out_t, _, w_in_t = blk._converted(torch.bfloat16)
        assert torch.equal(w_in, blk.in_proj.to(torch.bfloat16)) and torch.equal(w_out, blk.out_proj.to(torch.bfloat16))
        assert torch.equal(w_out_t, w_out.t()) and torch.equal(w_in_t, turned_weight(w_in))
        blk.in_proj.mul_(1.5)
        blk.out_proj.add_(0.25)


@pytest.mark.parametrize("dims,B,L", [((256, 8, 32, 64, 1), 3, 77), ((256, 8, 32, 64, 1), 9, 2100), ((128, 8, 16, 16, 2), 2, 300),
                                      ((256, 16, 16, 32, 1), 1, 1), ((128, 8, 32, 64, 1), 2, 300), ((256, 8, 16, 16, 1), 3, 700),
                                      ((256, 8, 16, 16, 1), 4, 4096)])  # (d_model unlike nheads headdim: a launch per weight gradient)
@pytest.mark.parametrize("kind", ["plain", "reset", "state", "no D"])
def test_whole_passes_in_one_call_are_the_stages(dims, B, L, kind):
    """Forward (with what it keeps, or with a carried state) and backward as one call each against the same stages called one by
    one: the same kernels, so the same bits -- but for the two weight gradients, whose launch in common cuts the rows elsewhere: float32
    sums of up to B L terms in another order, within 1e-5 of their norm."""
    from trading_bot_0_amd import Mamba2Block
    blk = Mamba2Block(*dims, seed=2)
    blk.norm_w.add_(torch.randn(blk.norm_w.shape, device="cuda"), alpha=0.2)
    if kind == "no D":
        blk.D = None
    g = torch.Generator(device="cuda").manual_seed(L)
    u, dout = (torch.randn(B, L, dims[0], generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    reset = (torch.rand(B, L, generator=g, device="cuda") < 0.05) if kind == "reset" else None

    def passes():
        if kind != "state":
            out, ctx = blk.forward(u, reset=reset, save_for_backward=True)
            plain = blk.forward(u, reset=reset)
            assert torch.equal(out, plain)
            return {"out": out, **{k: v for k, v in ctx.items() if k != "u"}, **blk.backward(ctx, dout)}
        st = blk.new_state(B)
        first = blk.forward(u, state=st)
        second = blk.forward(u, state=st)   # continues the state in place
        return {"first": first, "second": second, "conv": st.conv, "ssm": st.ssm.state}

    one = passes()
    blk._one_call = lambda *a: False
    two = passes()
    assert one.keys() == two.keys()
    for k in one:
        if k in ("din_proj", "dout_proj"):
            assert (one[k].double() - two[k].double()).norm() <= 1e-5 * two[k].double().norm(), k
        else:
            assert (one[k] is None and two[k] is None) or torch.equal(one[k], two[k]), k


def test_whole_pass_captured_reads_the_parameters_at_replay():
    """A captured forward and backward, replayed after its input and A_log have been changed in place, with eager work in between,
    equal the eager calls bit for bit."""
    from trading_bot_0_amd import Mamba2Block
    blk = Mamba2Block(256, 8, 32, 64, seed=3)
    u, dout = (torch.randn(3, 200, 256, device="cuda").to(torch.bfloat16) for _ in range(2))

    def run():
        out, ctx = blk.forward(u, save_for_backward=True)
        return {"out": out, **blk.backward(ctx, dout)}

    run()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = run()
    for i in range(3):
        u.mul_(0.9)
        blk.A_log.add_(0.1)
        graph.replay()
        eager = run()
        torch.cuda.synchronize()
        for k in eager:
            assert torch.equal(res[k], eager[k]), (i, k)


def conv_backward_inputs(B, L):
    """Few channels (eight heads of 8, state 16, d_conv 2: 64 + 32 of x | B | C), so that many rows are cheap."""
    zeros = lambda *s: torch.zeros(*s, device="cuda")
    return (zeros(B, L, 168), zeros(96, 2), zeros(96), zeros(8), zeros(B, L, 8, 8), zeros(B, L, 1, 16), zeros(B, L, 1, 16),
            zeros(B, L, 8))


@pytest.mark.parametrize("B,L", [(128, 2048), (139, 2048), (3, 131072)])
def test_partial_sums_of_the_conv_backward_keep_float32_accuracy(B, L):
    """dconv_b over 1 024 workgroups' partial sums, as many as one launch adds, and over 1 112 and 1 536, which two launches do.  With
    every input zero the filter's output is zero and silu' one half, so a workgroup's partial sum is half of the one output gradient
    put into its 256 rows: 2^24 in the first sixteen, one in the others.  Adding those one by one behind a large one loses every one of
    them; no part may go through more than 24 additions, whose roundings are at most 2^-24 of the sum each."""
    from trading_bot_0_amd.block import block_pre_bwd
    z, w, b, bias, dx, dB, dC, ddt = conv_backward_inputs(B, L)
    parts = B * L // 256
    value = torch.ones(parts, device="cuda")
    value[:16] = 2.0 ** 24
    dx.view(parts, 256, 64)[:, 0, :] = 2 * value[:, None]
    db = block_pre_bwd(z, w, b, bias, dx, dB, dC, ddt, torch.zeros_like(z), 8, 8, 16, 1)[1]
    total = value.double().sum()
    assert ((db[:64].double() - total).abs() <= 24 * 2.0 ** -24 * total).all() and not bool(db[64:].any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L", [(140, 2001), (700, 33), (300, 1001)])
def test_parameter_gradients_of_the_conv_backward_over_many_rows(B, L, dtype):
    """dconv_w, dconv_b and ddt_bias against float64 autograd: 1 103 and 1 200 workgroups' partial sums (two launches, the second of
    shares that are not equal), and 175.  Bound: the roundings of 2^-24 in a term (8) and on its way through the sums, of the terms'
    absolute sum: a run of 32 steps, the eight runs of a workgroup, 24 additions of the workgroups; for dt the 12 rows of a thread, the 256
    threads of a workgroup and the same."""
    from trading_bot_0_amd.block import block_pre_bwd
    g = torch.Generator(device="cuda").manual_seed(B)
    rnd = lambda t, s=1.0: torch.randn(t.shape, generator=g, device="cuda") * s
    z, w, b, bias, dx, dB, dC, ddt = conv_backward_inputs(B, L)
    w, b, bias = rnd(w, 0.5), rnd(b, 0.1), rnd(bias)
    z, dx, dB, dC, ddt = (rnd(t).to(dtype) for t in (z, dx, dB, dC, ddt))
    dw, db, dbias = block_pre_bwd(z, w, b, bias, dx, dB, dC, ddt, torch.zeros_like(z), 8, 8, 16, 1)[:3]
    inp = z[..., 64:160].double()
    before = torch.nn.functional.pad(inp, (0, 0, 1, 0))[:, :-1]
    pre = b.double() + w[:, 0].double() * before + w[:, 1].double() * inp
    sg = torch.sigmoid(pre)
    d = torch.cat([t.reshape(B, L, -1) for t in (dx, dB, dC)], -1).double() * sg * (1 + pre * (1 - sg))
    dt_terms = ddt.double() * torch.sigmoid(z[..., 160:].double() + bias.double())
    for name, got, terms, roundings in (("dconv_w[0]", dw[:, 0], d * before, 72), ("dconv_w[1]", dw[:, 1], d * inp, 72),
                                        ("dconv_b", db, d, 72), ("ddt_bias", dbias, dt_terms, 300)):
        over = (got.double() - terms.sum((0, 1))).abs() / terms.abs().sum((0, 1)) * 2.0 ** 24
        assert bool((over <= roundings).all()), f"{name}: {over.max().item():.1f} roundings"


@pytest.mark.parametrize("rows", [8192, 60000])
def test_weight_gradient_loses_little_behind_a_large_product(rows):
    """One product of 2^24 and 2^-4 for every other row: sixteen of those make one, half a unit in the last place of the large one,
    and added to it one by one every such sum is lost.  A product goes through at most 16 additions in its run of 256 rows, one per
    run of its split (1 920 rows at 60 000: 8) and one per split (32), each with a rounding of at most 2^-24 of the sum."""
    from trading_bot_0_amd.block import block_wgrad
    a = torch.full((rows, 1024), 2.0 ** -4, dtype=torch.bfloat16, device="cuda")
    a[0] = 2.0 ** 24
    b = torch.ones(rows, 128, dtype=torch.bfloat16, device="cuda")
    total = 2.0 ** 24 + (rows - 1) * 2.0 ** -4
    assert bool(((block_wgrad(a, b).double() - total).abs() <= (16 + 8 + 32) * 2.0 ** -24 * total).all())
