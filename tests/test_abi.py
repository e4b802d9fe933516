"""The C-ABI library loads without a GPU, exports every symbol include/ssd_hip.h declares, and
rejects bad arguments with a code and a message before touching the device (the reference's
wrappers validate first and bail with a message, trading_bots/src/torch/fa4.rs:145-191)."""
import ctypes
import re
from ctypes import byref, c_size_t
from pathlib import Path

import pytest

from trading_bot_0_amd import ssd

REPO = Path(__file__).resolve().parent.parent
FAKE = 0x1000  # aligned, never dereferenced: validation fails before any launch


@pytest.fixture(scope="module")
def lib():
    return ssd.load_library()


def declared_symbols():
    text = (REPO / "include" / "ssd_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ssd_\w+)\s*\(", text)))


def test_header_symbols_are_exported(lib):
    names = declared_symbols()
    assert sorted(names) == sorted(ssd.EXPORTED_SYMBOLS)
    for n in names:
        assert getattr(lib, n) is not None


# ---- the Rust binding (bindings/rust/ssd.rs) against the header: there is no Rust toolchain here, so the extern
# block is checked as text: same functions, same number of parameters, same pointer constness, same pointee /
# integer kinds, same field lists of the three structs.

C_KINDS = {"void": "void", "float": "f32", "double": "f64", "char": "char", "uint8_t": "u8", "int": "int",
           "int64_t": "i64", "size_t": "usize", "ssd_dims": "dims", "ssd_step_dims": "step_dims",
           "ssd_block_dims": "block_dims"}
RUST_KINDS = {"c_void": "void", "f32": "f32", "f64": "f64", "c_char": "char", "u8": "u8", "c_int": "int", "i64": "i64",
              "usize": "usize", "SsdDims": "dims", "SsdStepDims": "step_dims", "SsdBlockDims": "block_dims"}


def c_type_kind(decl, with_name=True):
    """'const float *A' -> ('ptr_const', 'f32'); 'size_t workspace_bytes' -> ('value', 'usize')."""
    decl = decl.strip()
    if "*" in decl:
        base = decl[:decl.index("*")].split()
        const = "const" in base
        base = [t for t in base if t not in ("const", "struct")]
        assert len(base) == 1, decl
        return ("ptr_const" if const else "ptr_mut", C_KINDS[base[0]])
    toks = [t for t in decl.split() if t != "const"]
    if with_name:
        toks = toks[:-1]
    assert len(toks) == 1, decl
    return ("value", C_KINDS[toks[0]])


def rust_type_kind(ty):
    ty = ty.strip()
    m = re.fullmatch(r"\*(const|mut)\s+(\w+)", ty)
    if m:
        return ("ptr_const" if m.group(1) == "const" else "ptr_mut", RUST_KINDS[m.group(2)])
    return ("value", RUST_KINDS[ty])


def header_prototypes():
    text = (REPO / "include" / "ssd_hip.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    protos = {}
    for ret, name, args in re.findall(r"^\s*([\w\s\*]+?)\b(ssd_\w+)\s*\(([^)]*)\)\s*;", text, flags=re.M):
        params = [] if args.strip() in ("", "void") else [c_type_kind(a) for a in args.split(",")]
        protos[name] = (c_type_kind(ret, with_name=False), params)
    return protos


def rust_prototypes():
    text = (REPO / "bindings" / "rust" / "ssd.rs").read_text()
    text = re.sub(r"//[^\n]*", "", text)
    block = re.search(r'extern\s+"C"\s*\{(.*?)\n\}', text, flags=re.S).group(1)
    protos = {}
    for name, args, ret in re.findall(r"fn\s+(\w+)\s*\(([^)]*)\)\s*->\s*([^;]+);", block):
        params = []
        for a in args.split(","):
            if a.strip():
                params.append(rust_type_kind(a.split(":", 1)[1]))
        protos[name] = (rust_type_kind(ret), params)
    return protos


def test_rust_binding_matches_the_header():
    c, r = header_prototypes(), rust_prototypes()
    assert sorted(c) == sorted(ssd.EXPORTED_SYMBOLS)          # the parser sees every declaration
    assert sorted(r) == sorted(c), f"missing in ssd.rs: {sorted(set(c) - set(r))}, unknown: {sorted(set(r) - set(c))}"
    for name in c:
        assert r[name][0] == c[name][0], f"{name}: return type {r[name][0]} vs {c[name][0]}"
        assert len(r[name][1]) == len(c[name][1]), f"{name}: {len(r[name][1])} parameters in ssd.rs, {len(c[name][1])} in the header"
        for i, (a, b) in enumerate(zip(r[name][1], c[name][1])):
            assert a == b, f"{name}: parameter {i} is {a} in ssd.rs, {b} in the header"


def test_rust_wrappers_pass_the_callers_stream():
    """Every public wrapper that launches kernels takes a `stream: StreamHandle` and hands `stream_ptr(stream)` to the
    library as the last argument of its call; none passes a NULL stream of its own.  The getter the binding needs from
    the torch shim is declared with the shim's calling convention (a device index in, a raw handle out)."""
    text = re.sub(r"//[^\n]*", "", (REPO / "bindings" / "rust" / "ssd.rs").read_text())
    launching = {"ssd_chunk_scan": "ssd_chunk_scan_reset_fwd", "ssd_chunk_scan_noalloc": "ssd_chunk_scan_noalloc_fwd",
                 "ssd_step": "ssd_step_fwd", "ssd_steps": "ssd_steps_fwd", "ssd_chunk_scan_backward": "ssd_chunk_scan_bwd"}
    for wrapper, entry in launching.items():
        m = re.search(r"pub fn " + wrapper + r"\s*\(([^)]*)\)[^{]*\{(.*?)\n\}\n", text, flags=re.S)
        assert m, wrapper
        params, body = m.group(1), m.group(2)
        assert re.search(r"\bstream\s*:\s*StreamHandle\s*$", params.strip()), f"{wrapper} must end in stream: StreamHandle"
        call = re.search(entry + r"\s*\((.*?)\)\s*\}\)", body, flags=re.S)
        assert call, f"{wrapper} does not call {entry}"
        assert call.group(1).rstrip().endswith("stream_ptr(stream)"), f"{wrapper} must pass the caller's stream to {entry}"
    assert re.search(r"fn\s+stream_ptr\s*\(\s*stream\s*:\s*StreamHandle\s*\)\s*->\s*\*mut\s+c_void", text)
    assert re.search(r"pub type StreamHandle\s*=\s*Option<\*mut c_void>", text)
    assert re.search(r"pub fn at_cuda_current_stream\s*\(\s*device_index\s*:\s*i64\s*\)\s*->\s*\*mut c_void", text)
    # the patch for the shim that INTEGRATION.md gives declares the same function
    integ = (REPO / "INTEGRATION.md").read_text()
    assert "void *at_cuda_current_stream(int64_t device_index);" in integ


def test_rust_structs_match_the_header():
    htext = re.sub(r"/\*.*?\*/", "", (REPO / "include" / "ssd_hip.h").read_text(), flags=re.S)
    rtext = re.sub(r"//[^\n]*", "", (REPO / "bindings" / "rust" / "ssd.rs").read_text())
    for cname, rname in (("ssd_dims", "SsdDims"), ("ssd_step_dims", "SsdStepDims"), ("ssd_block_dims", "SsdBlockDims")):
        body = re.search(r"typedef struct[^{]*\{([^}]*)\}\s*" + cname + r"\s*;", htext, flags=re.S).group(1)
        cfields = []
        for stmt in body.split(";"):
            stmt = stmt.strip()
            if stmt:
                assert stmt.startswith("int64_t"), stmt
                cfields += [f.strip() for f in stmt[len("int64_t"):].split(",")]
        m = re.search(r"#\[repr\(C\)\]\s*(?:#\[[^\]]*\]\s*)*pub struct " + rname + r"\s*\{([^}]*)\}", rtext, flags=re.S)
        assert m, f"{rname} must be #[repr(C)]"
        rfields = re.findall(r"pub\s+(\w+)\s*:\s*i64", m.group(1))
        assert rfields == cfields, f"{rname}: {rfields} vs {cfields}"


def test_version_and_empty_error_slot(lib):
    assert lib.ssd_version() >= 100
    assert ssd.last_error(lib) is None


def dims(**kw):
    d = dict(batch=2, seqlen=256, nheads=4, headdim=32, dstate=64, ngroups=1, chunk=128)
    d.update(kw)
    return ssd.SsdDims(*[d[k] for k in ("batch", "seqlen", "nheads", "headdim", "dstate", "ngroups", "chunk")])


@pytest.mark.parametrize("layout", [dict(nheads=8, dstate=64), dict(nheads=8, dstate=32), dict(nheads=24, dstate=64, ngroups=3)])
def test_backward_workspace_of_few_sequences_holds_smaller_calls(lib, layout):
    """Where the backward pass runs on segments, what it asks for grows with the batch and with the length, although the number
    of segments does not: a workspace sized for the largest call of a program holds the others."""
    def need(batch, seqlen):
        out = c_size_t(0)
        d = ssd.SsdDims(batch, seqlen, layout["nheads"], 32, layout["dstate"], layout.get("ngroups", 1), 64)
        assert lib.ssd_chunk_scan_bwd_workspace_bytes(byref(d), 1, byref(out)) == 0
        return out.value

    most = 95 * 8 // layout["nheads"]
    lengths = (1, 64, 65, 129, 320, 512, 1000, 2048, 3000, 4096, 8191, 16384)
    sizes = [[need(batch, seqlen) for batch in range(1, most + 1)] for seqlen in lengths]
    assert all(a <= b for row in sizes for a, b in zip(row, row[1:])), "a larger batch asks for less"
    assert all(a <= b for col in zip(*sizes) for a, b in zip(col, col[1:])), "a longer sequence asks for less"


@pytest.mark.parametrize("layout", [(8, 32, 64, 1), (8, 16, 16, 1), (8, 32, 32, 2), (8, 32, 128, 1), (16, 16, 64, 2), (4, 32, 32, 1), (4, 64, 128, 1)])
@pytest.mark.parametrize("query", ["scan", "scan backward", "block forward", "block backward", "weight gradient"])
def test_workspace_of_the_largest_call_holds_the_others(query, layout):
    """What a query asks for grows with the batch and with the length, across every line at which the kernels behind it change."""
    from trading_bot_0_amd.block import SsdBlockDims, _lib
    lib = _lib()
    H, P, N, G = layout
    out = c_size_t(0)
    if query.startswith("block") and H % 8:
        pytest.skip("not the block's heads")

    def need(B, L):
        scan, block = ssd.SsdDims(B, L, H, P, N, G, 128), SsdBlockDims(B, L, H, P, N, G, 4, 0)
        rc = {"scan": lambda: lib.ssd_workspace_bytes(byref(scan), byref(out)),
              "scan backward": lambda: lib.ssd_chunk_scan_bwd_workspace_bytes(byref(scan), 1, byref(out)),
              "block forward": lambda: lib.ssd_block_forward_workspace_bytes(byref(block), 1, 256, 128, byref(out)),
              "block backward": lambda: lib.ssd_block_grad_workspace_bytes(byref(block), 1, 256, 128, byref(out)),
              "weight gradient": lambda: lib.ssd_block_wgrad_workspace_bytes(B * L, 2 * H * P + 2 * G * N + H // 8 * 8, 256, byref(out))}[query]()
        assert rc == 0, ssd.last_error(lib)
        return out.value

    for L in (1, 64, 300, 700, 2048, 4100):
        sizes = [need(B, L) for B in range(1, 420)]
        assert all(a <= b for a, b in zip(sizes, sizes[1:])), f"a larger batch of {L} steps asks for less"
    for B in (1, 8, 33, 60, 97, 200):
        sizes = [need(B, L) for L in range(1, 4200, 13)]
        assert all(a <= b for a, b in zip(sizes, sizes[1:])), f"longer sequences, {B} of them, ask for less"


def test_workspace_bytes_formula(lib):
    out = c_size_t(0)
    assert lib.ssd_workspace_bytes(byref(dims()), byref(out)) == 0
    B, H, nc, Q, P, N = 2, 4, 2, 128, 32, 64
    assert out.value == 4 * B * H * nc * Q * 4 + B * nc * H * P * N * 4
    # ragged seqlen rounds the chunk count up
    assert lib.ssd_workspace_bytes(byref(dims(seqlen=257)), byref(out)) == 0
    assert out.value == 4 * B * H * 3 * Q * 4 + B * 3 * H * P * N * 4


@pytest.mark.parametrize("kw,code,needle", [
    (dict(batch=0), 1, "positive"),
    (dict(seqlen=-5), 1, "positive"),
    (dict(nheads=6, ngroups=4), 1, "divisible"),
    (dict(dstate=48), 2, "dstate"),
    (dict(headdim=12), 2, "headdim"),
    (dict(headdim=128), 2, "headdim"),
    (dict(chunk=100), 2, "chunk"),
])
def test_bad_dims_are_rejected_with_message(lib, kw, code, needle):
    out = c_size_t(0)
    assert lib.ssd_workspace_bytes(byref(dims(**kw)), byref(out)) == code
    msg = ssd.last_error(lib)
    assert msg and needle in msg
    assert ssd.last_error(lib) is None  # fetching clears the slot


def test_float32_lds_limit(lib):
    d = dims(headdim=64, dstate=128, chunk=256)
    rc = lib.ssd_chunk_cumsum_fwd(byref(d), 0, FAKE, FAKE, FAKE, None)
    assert rc == 2 and "LDS" in ssd.last_error(lib)
    out = c_size_t(0)
    assert lib.ssd_workspace_bytes(byref(d), byref(out)) == 0  # fine in bf16


def test_null_misaligned_and_dtype(lib):
    d = dims()
    args = [FAKE] * 4 + [FAKE, None, None, FAKE, None, FAKE]  # x dt A B C D init y final ws
    assert lib.ssd_chunk_scan_fwd(byref(d), 1, None, *args[1:], 1 << 30, None) == 1
    assert "x must not be NULL" in ssd.last_error(lib)
    bad = list(args)
    bad[3] = FAKE + 2
    assert lib.ssd_chunk_scan_fwd(byref(d), 1, *bad, 1 << 30, None) == 1
    assert "16-byte aligned" in ssd.last_error(lib)
    assert lib.ssd_chunk_scan_fwd(byref(d), 7, *args, 1 << 30, None) == 1
    assert "dtype" in ssd.last_error(lib)
    assert lib.ssd_chunk_scan_fwd(byref(d), 1, *args, 16, None) == 3
    assert "workspace" in ssd.last_error(lib)
    assert lib.ssd_chunk_scan_fwd(None, 1, *args, 1 << 30, None) == 1
    sd = ssd.SsdStepDims(4, 8, 32, 64, 3)
    assert lib.ssd_step_fwd(byref(sd), 1, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, None, FAKE, None) == 1
    assert "divisible" in ssd.last_error(lib)
    sd = ssd.SsdStepDims(4, 8, 32, 64, 1)
    assert lib.ssd_step_fwd(byref(sd), 3, FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, None, FAKE, None) == 1
    assert "dtype" in ssd.last_error(lib)
    assert lib.ssd_step_fwd(byref(sd), 1, None, FAKE, FAKE, FAKE, FAKE, FAKE, None, FAKE, None) == 1
    assert "state must not be NULL" in ssd.last_error(lib)


def test_backward_rejects_null_dims(lib):
    out = c_size_t(0)
    assert lib.ssd_chunk_scan_bwd_workspace_bytes(None, 1, byref(out)) == 1
    assert "dims must not be NULL" in ssd.last_error(lib)
    args = [FAKE] * 5 + [None, None, None, FAKE, None] + [FAKE] * 5 + [None, None, FAKE]
    assert lib.ssd_chunk_scan_bwd(None, 1, *args, 1 << 30, None) == 1
    assert "dims must not be NULL" in ssd.last_error(lib)


def test_stage1_lds_bound_on_nheads(lib):
    """Stage 1 transposes a [chunk, nheads] tile of dt through LDS: (H*(Q+1)+Q)*4 bytes must fit 160 KiB."""
    out = c_size_t(0)
    ok = dims(nheads=152, chunk=256, headdim=32, dstate=32)       # 152*257*4 + 1024 = 157 280 bytes
    assert lib.ssd_workspace_bytes(byref(ok), byref(out)) == 0
    bad = dims(nheads=160, chunk=256, headdim=32, dstate=32)      # 165 504 bytes
    assert lib.ssd_workspace_bytes(byref(bad), byref(out)) == 2
    assert "stage 1" in ssd.last_error(lib)


def test_noalloc_entry_rejects_shapes_beyond_its_scratch(lib):
    """Validation happens before the device is touched: a staged shape whose workspace exceeds the static array
    is refused with the sizes in the message."""
    d = dims(batch=256, seqlen=2048, nheads=8, headdim=16, dstate=64, chunk=128)   # heads of 16: staged, 200 MB
    need = c_size_t(0)
    assert lib.ssd_workspace_bytes(byref(d), byref(need)) == 0 and need.value > (64 << 20)
    args = [FAKE] * 5 + [None, None, None, FAKE, None]   # x dt A B C D init reset y final
    assert lib.ssd_chunk_scan_noalloc_fwd(byref(d), 0, *args, None) == 3
    msg = ssd.last_error(lib)
    assert str(need.value) in msg and str(64 << 20) in msg
    assert lib.ssd_chunk_scan_noalloc_fwd(byref(d), 0, None, *args[1:], None) == 3   # (size is checked first)
    ssd.last_error(lib)
    assert lib.ssd_chunk_scan_noalloc_fwd(None, 1, *args, None) == 1
    assert "dims" in ssd.last_error(lib)


def test_error_slot_is_thread_local(lib):
    import threading
    out = c_size_t(0)
    assert lib.ssd_workspace_bytes(byref(dims(batch=0)), byref(out)) == 1
    seen = []
    t = threading.Thread(target=lambda: seen.append(ssd.last_error(lib)))
    t.start()
    t.join()
    assert seen == [None]
    assert "positive" in ssd.last_error(lib)


def test_host_wrappers_validate_before_calling():
    import torch
    x = torch.zeros(2, 64, 4, 32)
    with pytest.raises(ValueError, match="must be on the GPU"):
        ssd.ssd_chunk_scan(x, torch.zeros(2, 64, 4), torch.zeros(4), torch.zeros(2, 64, 1, 64),
                           torch.zeros(2, 64, 1, 64), chunk=32)
    with pytest.raises(ValueError, match="rank-4"):
        ssd.ssd_chunk_scan(x[0], torch.zeros(2, 64, 4), torch.zeros(4), torch.zeros(2, 64, 1, 64),
                           torch.zeros(2, 64, 1, 64), chunk=32)
    with pytest.raises(ValueError, match="float32 or bfloat16"):
        ssd.ssd_chunk_scan(x.half(), torch.zeros(2, 64, 4), torch.zeros(4), torch.zeros(2, 64, 1, 64),
                           torch.zeros(2, 64, 1, 64), chunk=32)
