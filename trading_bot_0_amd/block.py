"""A Mamba-2 block around the SSD scan: in-projection -> causal depthwise conv + SiLU on (x, B, C), softplus on
dt -> SSD scan -> gated RMSNorm -> out-projection.  It is the layer that would sit where the reference's
encoder block sits in `patch_trunk` (`trading_bots/src/torch/model/trading_model.rs:589-606`,
`trading_bots/src/torch/model/blocks/gqa.rs:82-109`), with the conv's streaming state carried next to the SSM
state the way the reference's `StreamState` carries its encoder memory (`trading_model.rs:56-75`).

Everything runs in libssd_hip -- the projections, the pre-scan and post-scan kernels and the weight gradients bound here, the
scan / step of `ssd.py` -- but the products its kernels do not take (float32, other widths and addresses, weight gradients of
many rows or wide; the gradient of the block's input), which are torch matmuls.
"""
from __future__ import annotations

import math
from ctypes import POINTER, Structure, byref, c_float, c_int, c_int64, c_size_t, c_void_p
from dataclasses import dataclass
from typing import Optional, Tuple

import torch

from . import ssd
from .stream_state import SsdStreamState


class SsdBlockDims(Structure):
    _fields_ = [(n, c_int64) for n in ("batch", "seqlen", "nheads", "headdim", "dstate", "ngroups", "d_conv", "zxbcdt_ld")]


_bound = False


def _lib():
    global _bound
    lib = ssd.load_library()
    if not _bound:
        P = c_void_p
        lib.ssd_block_pre_fwd.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, P, P, P, P, P, P, P, P]
        lib.ssd_block_post_fwd.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, c_float, P, P]
        lib.ssd_block_proj_fwd.argtypes = [c_int64, c_int64, c_int64, c_int64, c_int, P, P, P, P]
        lib.ssd_block_dproj.argtypes = [c_int64, c_int64, c_int64, c_int64, c_int64, c_int, P, P, P, P]
        lib.ssd_block_weights.argtypes = [c_int64, c_int64, c_int64, P, P, P, P, P, P, P]
        lib.ssd_block_wgrad_workspace_bytes.argtypes = [c_int64, c_int64, c_int64, POINTER(c_size_t)]
        lib.ssd_block_wgrad.argtypes = [c_int64, c_int64, c_int64, c_int64, c_int, P, P, P, P, c_size_t, P]
        lib.ssd_block_post_proj_fwd.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, c_float, P, c_int64, c_int64, P, P]
        lib.ssd_block_post_proj_fwd.restype = c_int
        lib.ssd_block_step_fwd.argtypes = [POINTER(SsdBlockDims), c_int, c_int64, P, P, P, P, P, P, P, P, c_float, P, P, P, P, P]
        lib.ssd_block_step_fwd.restype = c_int
        lib.ssd_block_pre_reset_fwd.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, P, P, P, P, P, P, P, P, P]
        lib.ssd_block_pre_reset_fwd.restype = c_int
        lib.ssd_block_bwd_workspace_bytes.argtypes = [POINTER(SsdBlockDims), c_int, POINTER(c_size_t)]
        lib.ssd_block_post_bwd.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, c_float, P, P, P, P, P, c_size_t, P]
        lib.ssd_block_post_bwd_yn.argtypes = [POINTER(SsdBlockDims), c_int, P, P, P, c_float, P, P, P, P, P, P, c_size_t, P]
        lib.ssd_block_pre_bwd.argtypes = [POINTER(SsdBlockDims), c_int] + [P] * 17 + [c_size_t, P]
        D, I = POINTER(SsdBlockDims), c_int64
        lib.ssd_block_forward_workspace_bytes.argtypes = lib.ssd_block_grad_workspace_bytes.argtypes = [D, c_int, I, I, POINTER(c_size_t)]
        lib.ssd_block_forward.argtypes = [D, c_int, I, I] + [P] * 8 + [c_float] + [P] * 14 + [c_size_t, P]
        lib.ssd_block_grad.argtypes = [D, c_int, I, I, P, P, I] + [P] * 7 + [c_float] + [P] * 20 + [c_size_t, P]
        for name in ("ssd_block_bwd_workspace_bytes", "ssd_block_post_bwd", "ssd_block_post_bwd_yn", "ssd_block_pre_bwd"):
            getattr(lib, name).restype = c_int
        lib.ssd_block_pre_fwd.restype = c_int
        lib.ssd_block_post_fwd.restype = c_int
        lib.ssd_block_proj_fwd.restype = c_int
        _bound = True
    return lib


def block_wgrad_supported(a: torch.Tensor, b: torch.Tensor) -> bool:
    """Whether `block_wgrad` takes these tensors (else the caller's BLAS does it)."""
    return (a.is_cuda and a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16 and b.shape[1] in (128, 256)
            and a.shape[1] % 8 == 0 and 0 < a.shape[1] <= 8192 and 0 < a.shape[0] < 2 ** 31 and a.stride(1) == 1
            and a.stride(0) % 8 == 0 and a.stride(0) >= a.shape[1] and a.data_ptr() % 16 == 0 and b.is_contiguous()
            and b.data_ptr() % 16 == 0)


def block_wgrad(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a^T b [E,D] in float32, summed over the rows of a [rows,E] (rows dense or evenly padded) and b [rows,D], bf16: the
    weight gradient of a projection (a = the gradient of its output, b = its input)."""
    lib = _lib()
    if a.dim() != 2 or b.dim() != 2 or a.shape[0] != b.shape[0] or a.device != b.device or not block_wgrad_supported(a, b):
        raise ValueError(f"block_wgrad does not take {tuple(a.shape)} {a.dtype} (strides {a.stride()}) and {tuple(b.shape)} {b.dtype}")
    rows, E, D = a.shape[0], a.shape[1], b.shape[1]
    need = c_size_t(0)
    ssd._check(lib, lib.ssd_block_wgrad_workspace_bytes(rows, E, D, byref(need)))
    ws = a.new_empty(need.value, dtype=torch.uint8) if need.value else None
    out = a.new_empty((E, D), dtype=torch.float32)
    ssd._check(lib, lib.ssd_block_wgrad(rows, E, D, a.stride(0), ssd.SSD_DTYPE_BF16, a.data_ptr(), b.data_ptr(), out.data_ptr(),
                                        ssd._ptr(ws), need.value, ssd._stream_ptr(a)))
    return out


def turned_weight(weight: torch.Tensor) -> torch.Tensor:
    """weight [a_features, out_features] as `block_dproj` takes it: transposed, a_features padded with zeros to a multiple of 16."""
    E, D = weight.shape
    t = weight.new_zeros((D, (E + 15) // 16 * 16))
    t[:, :E] = weight.t()
    return t


def block_dproj_supported(a: torch.Tensor, w_t: torch.Tensor) -> bool:
    """Whether `block_dproj` takes these tensors (else the caller's BLAS does it)."""
    return (a.is_cuda and a.dtype == torch.bfloat16 and w_t.dtype == torch.bfloat16 and a.shape[1] % 8 == 0 and 0 < a.shape[1] <= 2544
            and w_t.shape[0] % 8 == 0 and 0 < a.shape[0] < 2 ** 31 and a.stride(1) == 1 and a.stride(0) % 8 == 0
            and a.stride(0) >= a.shape[1] and a.data_ptr() % 16 == 0 and w_t.is_contiguous() and w_t.data_ptr() % 16 == 0)


def block_dproj(a: torch.Tensor, w_t: torch.Tensor) -> torch.Tensor:
    """a . w [rows, out_features] (bf16) for a [rows, a_features] (rows dense or evenly padded) and w_t = turned_weight(w): the
    gradient of a projection's input (a = the gradient of its output)."""
    lib = _lib()
    if a.dim() != 2 or w_t.dim() != 2 or w_t.shape[1] != (a.shape[1] + 15) // 16 * 16 or a.device != w_t.device \
            or not block_dproj_supported(a, w_t):
        raise ValueError(f"block_dproj does not take {tuple(a.shape)} {a.dtype} (strides {a.stride()}) and {tuple(w_t.shape)} {w_t.dtype}")
    out = a.new_empty((a.shape[0], w_t.shape[0]))
    ssd._check(lib, lib.ssd_block_dproj(a.shape[0], a.shape[1], w_t.shape[0], a.stride(0), w_t.shape[1], ssd.SSD_DTYPE_BF16,
                                        a.data_ptr(), w_t.data_ptr(), out.data_ptr(), ssd._stream_ptr(a)))
    return out


# rows and features up to which the library's kernel forms a projection's input gradient: 648 -> 256 in us, library / BLAS, 4 000 rows
# 8.1 / 9.5, 16 384 14.2 / 16.2, 24 000 26 / 21; 1 288 -> 256 at 800 rows 12.4 / 10.1 (and 4 / 20 of the host's time)
DPROJ_MAX_ROWS, DPROJ_MAX_FEATURES = 16384, 1024


def _wgrad_slab_limit(E: int, D: int) -> int:
    """The number of slabs from which the BLAS runs a weight gradient of E x D outputs at least as fast as `block_wgrad`: the more
    slabs the rows make the more of the chip its batched products fill, and the library's kernel reads b again for every 128
    of the E.  In us, library against BLAS, D 256: E 648, 32 slabs 173 / 258 (245 760 rows), 64 slabs 190 / 122 (262 144); E 392,
    16 slabs 57 / 79, 32 slabs 57 / 51 (131 072); E 128, 16 slabs 39 / 60, 32 slabs 39 / 35; E 1 160, 4 slabs 60 / 99 (49 156), 16 slabs
    300 / 279 (262 160) and E 1 288, 8 slabs 417 / 335; E 2 184, one slab 234 / 294 (72 829), 4 slabs 143 / 117; E 4 368, one 467 / 353.
    Both sides measured at E of 72 to 4 368, both D and 1 to 128 slabs."""
    if E > 896:
        return 8 if E <= 1792 else 2 if E <= 2304 else 0
    return 32 if 384 < E <= 512 or (E <= 128 and D == 256) else 64


def _wgrad_slabs(rows: int) -> int:
    """The equal slabs of 4 096 rows or more that a row count makes, a power of two."""
    slabs = 1
    while slabs < 128 and rows % (2 * slabs) == 0 and rows // (2 * slabs) >= 4096:
        slabs *= 2
    return slabs


def _weight_gradient(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a^T b in float32 for tall a [rows, E] (its rows may be a view into wider ones) and b [rows, D]: a sum over all
    rows of the batch and the sequence.  bf16 with D 128 or 256 runs on the library's kernel (72 828 rows, 648 x 256 outputs:
    59 us, the BLAS 151), except where the rows make enough slabs for the BLAS behind torch (`_wgrad_slab_limit`); there, and for
    everything else: as one GEMM the BLAS behind torch sees a contraction hundreds of thousands
    long against outputs a few hundred wide and runs it at a fifth of its rate, so the rows are cut into equal slabs,
    multiplied as one batched GEMM with float32 outputs, and the slabs' products added in order (measured on MI355X,
    524 288 rows: 648 x 256 outputs 1 333 -> 232 us, 256 x 256 outputs 1 059 -> 129 us; the float32 partial products also
    make the result more accurate than the single GEMM's bf16 output)."""
    rows = a.shape[0]
    slabs = _wgrad_slabs(rows)
    if slabs < _wgrad_slab_limit(a.shape[1], b.shape[1]) and block_wgrad_supported(a, b):
        return block_wgrad(a, b)
    if slabs == 1 or a.dtype == torch.float32:
        return torch.matmul(a.t(), b).float()
    a3 = a.unflatten(0, (slabs, rows // slabs))
    b3 = b.unflatten(0, (slabs, rows // slabs))
    return torch.bmm(a3.transpose(1, 2), b3, out_dtype=torch.float32).sum(0)


def in_proj_width(nheads, headdim, dstate, ngroups) -> int:
    return 2 * nheads * headdim + 2 * ngroups * dstate + nheads


def _row_stride(zxbcdt) -> int:
    """The row stride of zxbcdt [B,L,E]: dense, or the first E columns of a buffer with padded rows (what
    `block_proj(..., pad_rows=True)` returns)."""
    Bsz, L, E = zxbcdt.shape
    ld = zxbcdt.stride(1) if L > 1 else (zxbcdt.stride(0) if Bsz > 1 else E)
    if zxbcdt.data_ptr() % 16:
        raise ValueError("zxbcdt must be 16-byte aligned")
    if zxbcdt.is_contiguous():
        return E
    if zxbcdt.stride(2) != 1 or ld < E or (L > 1 and Bsz > 1 and zxbcdt.stride(0) != L * ld):
        raise ValueError(f"zxbcdt must be contiguous or have evenly padded rows, got strides {zxbcdt.stride()}")
    return ld


def block_pre(zxbcdt, conv_w, conv_b, dt_bias, nheads, headdim, dstate, ngroups, conv_state=None,
              return_conv_state=False, reset=None, conv_state_out=None):
    """zxbcdt [B,L,E] (rows dense or evenly padded) -> (x [B,L,H,P], Bm, Cm [B,L,G,N], dt [B,L,H][, conv state
    [B,d_conv-1,C]]).  `reset` [B,L] (uint8 or bool): a non-zero entry cuts the filter's history before that
    timestep.  `conv_state_out`: where to write the new conv state (may be `conv_state` itself for seqlen 1)."""
    lib = _lib()
    if zxbcdt.dim() != 3:
        raise ValueError(f"block input must be rank-3 [batch, seqlen, channels], got {tuple(zxbcdt.shape)}")
    Bsz, L, E = zxbcdt.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    C = H * P + 2 * G * N
    if E != in_proj_width(H, P, N, G):
        raise ValueError(f"block input must have {in_proj_width(H, P, N, G)} channels, got {E}")
    dtype = zxbcdt.dtype
    code = ssd._dtype_code(zxbcdt)
    if not zxbcdt.is_cuda:
        raise ValueError("zxbcdt must be a GPU tensor")
    ld = _row_stride(zxbcdt)
    if conv_w.dim() != 2 or conv_w.shape[0] != C:
        raise ValueError(f"conv_w must be [{C}, d_conv], got {tuple(conv_w.shape)}")
    d_conv = conv_w.shape[1]
    ssd._require(conv_w, "conv_w", (C, d_conv), torch.float32)
    ssd._require(conv_b, "conv_b", (C,), torch.float32)
    ssd._require(dt_bias, "dt_bias", (H,), torch.float32)
    if conv_state is not None:
        ssd._require(conv_state, "conv_state", (Bsz, d_conv - 1, C), dtype)
    x = zxbcdt.new_empty((Bsz, L, H, P))
    Bm = zxbcdt.new_empty((Bsz, L, G, N))
    Cm = zxbcdt.new_empty((Bsz, L, G, N))
    dt = zxbcdt.new_empty((Bsz, L, H))
    new_state = None
    if conv_state_out is not None:
        ssd._require(conv_state_out, "conv_state_out", (Bsz, d_conv - 1, C), dtype)
        new_state, return_conv_state = conv_state_out, True
    elif return_conv_state:
        new_state = zxbcdt.new_empty((Bsz, d_conv - 1, C))
    if reset is not None:
        if reset.dtype == torch.bool:
            reset = reset.view(torch.uint8)
        ssd._require(reset, "reset", (Bsz, L), torch.uint8)
    dims = SsdBlockDims(Bsz, L, H, P, N, G, d_conv, ld)
    ssd._check(lib, lib.ssd_block_pre_reset_fwd(byref(dims), code, zxbcdt.data_ptr(), conv_w.data_ptr(),
                                                conv_b.data_ptr(), dt_bias.data_ptr(), ssd._ptr(conv_state),
                                                ssd._ptr(new_state), ssd._ptr(reset), x.data_ptr(), Bm.data_ptr(),
                                                Cm.data_ptr(), dt.data_ptr(), ssd._stream_ptr(zxbcdt)))
    return (x, Bm, Cm, dt, new_state) if return_conv_state else (x, Bm, Cm, dt)


def block_post(y, zxbcdt, norm_w, nheads, headdim, dstate, ngroups, eps=1e-5):
    """out [B,L,H*P] = rmsnorm(y * silu(z)) * norm_w; y [B,L,H,P] in the activation dtype or float32."""
    lib = _lib()
    Bsz, L, E = zxbcdt.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    dtype = zxbcdt.dtype
    code = ssd._dtype_code(zxbcdt)
    if y.dtype != dtype:
        if not (dtype == torch.bfloat16 and y.dtype == torch.float32):
            raise ValueError(f"block y must be {dtype} (or float32 with bf16 activations), got {y.dtype}")
        code = ssd.SSD_DTYPE_BF16_Y32
    if not zxbcdt.is_cuda or E != in_proj_width(H, P, N, G):
        raise ValueError(f"zxbcdt must be a GPU tensor with {in_proj_width(H, P, N, G)} channels, got {tuple(zxbcdt.shape)}")
    ld = _row_stride(zxbcdt)
    ssd._require(y, "y", (Bsz, L, H, P), y.dtype)
    ssd._require(norm_w, "norm_w", (H * P,), torch.float32)
    out = torch.empty((Bsz, L, H * P), dtype=dtype, device=zxbcdt.device)
    dims = SsdBlockDims(Bsz, L, H, P, N, G, 4, ld)
    ssd._check(lib, lib.ssd_block_post_fwd(byref(dims), code, y.data_ptr(), zxbcdt.data_ptr(), norm_w.data_ptr(),
                                           c_float(eps), out.data_ptr(), ssd._stream_ptr(zxbcdt)))
    return out


def block_post_proj_supported(y: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether `block_post_proj` takes these tensors (else `block_post`, then the projection).  (The addresses: the kernels load 16
    bytes at a time, and a tensor that starts elsewhere in a flat buffer goes to the BLAS, which takes any.)"""
    return (y.is_cuda and y.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and weight.dim() == 2
            and weight.shape[1] in (128, 256) and weight.shape[0] % 8 == 0 and weight.shape[0] <= 256
            and (y.data_ptr() | weight.data_ptr()) % 16 == 0)


def block_post_proj(y, zxbcdt, norm_w, weight, nheads, headdim, dstate, ngroups, eps=1e-5):
    """out [B,L,out_features] = (rmsnorm(y * silu(z)) * norm_w) . weight^T as one kernel (bf16; weight
    [out_features, H*P]): `block_post` and the out-projection without the normalised rows going to memory between."""
    lib = _lib()
    Bsz, L, E = zxbcdt.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    if not zxbcdt.is_cuda or E != in_proj_width(H, P, N, G):
        raise ValueError(f"zxbcdt must be a GPU tensor with {in_proj_width(H, P, N, G)} channels, got {tuple(zxbcdt.shape)}")
    if zxbcdt.dtype != torch.bfloat16 or y.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("block_post_proj takes bfloat16 tensors")
    ld = _row_stride(zxbcdt)
    ssd._require(y, "y", (Bsz, L, H, P), torch.bfloat16)
    ssd._require(norm_w, "norm_w", (H * P,), torch.float32)
    if weight.dim() != 2 or weight.shape[1] != H * P or not weight.is_contiguous():
        raise ValueError(f"weight must be contiguous [out_features, {H * P}], got {tuple(weight.shape)}")
    out = zxbcdt.new_empty((Bsz, L, weight.shape[0]))
    dims = SsdBlockDims(Bsz, L, H, P, N, G, 4, ld)
    ssd._check(lib, lib.ssd_block_post_proj_fwd(byref(dims), ssd.SSD_DTYPE_BF16, y.data_ptr(), zxbcdt.data_ptr(),
                                                norm_w.data_ptr(), c_float(eps), weight.data_ptr(), weight.shape[0], 0,
                                                out.data_ptr(), ssd._stream_ptr(zxbcdt)))
    return out


# batches up to which the one-launch step (each workgroup reading both weight matrices whole) beats the stage kernels and the
# BLAS, in us with d_model 256, bf16 / float32, against those.  The overlapped kernel (64-wide state, at most 768 rows of w_in):
# eager 512 streams 21 / 24 against 92 / 92 (the host's issue of six launches), 1 024 40 / 48; replayed by `graphed_step` 512
# streams 25 / 28 against 36 / 41, 1 024 43 / 49 against 47 / 53.
FUSED_STEP_MAX_BATCH = 1024
# ... and the kernel for other shapes: one round of workgroups.  Replayed, 256 streams: state 32 21 / 24 against 35 / 88, state 128
# 30 / 32 against 43 / 100, two groups of 64 24 / 27 against 36 / 91; 384 streams 34 / 36 against 29 / 33, 47 / 50 against 41 / 46,
# 38 / 41 against 32 / 37; 1 024 65 / 70 against 38 / 43, 94 / 99 against 69 / 75, 77 / 82 against 49 / 55.  (Eager, where the
# stage kernels cost 92, it would win up to some 768; a step captured by the caller is not known to be one.)
FUSED_STEP_MAX_BATCH_OTHER = 256
# batches up to which a step that a caller captures keeps the A formed before (above, a captured step forms it at every replay)
STEP_CACHED_A_MAX_BATCH = 64


_STEP_DTYPES = (torch.bfloat16, torch.float32)


def _step_max_batch(d_model: int, nheads: int, headdim: int, dstate: int, ngroups: int) -> int:
    """The largest batch whose step is taken as one launch, by the kernel that the library runs for the shape (0: it takes none,
    or the launch's vectors, as it lays them out, do not fit the 64 KB of LDS that it asks for)."""
    d_inner, E = nheads * headdim, in_proj_width(nheads, headdim, dstate, ngroups)
    vectors = d_model + E + (E - d_inner - nheads) + (nheads + 3) // 4 * 4 + d_inner + 16
    if d_model not in (128, 256) or d_inner not in (128, 256) or dstate % 16 or 4 * vectors > 64 * 1024:
        return 0
    return FUSED_STEP_MAX_BATCH if dstate == 64 and E <= 768 else FUSED_STEP_MAX_BATCH_OTHER


def block_step_supported(u_t: torch.Tensor, d_inner: int, dstate: int) -> bool:
    """Whether `block_step` takes this step (else the stage kernels, one launch each)."""
    return (u_t.is_cuda and u_t.dtype in (torch.bfloat16, torch.float32) and u_t.dim() == 2
            and u_t.shape[1] in (128, 256) and d_inner in (128, 256) and dstate % 16 == 0 and u_t.data_ptr() % 16 == 0)


def block_step(u_t, w_in, conv_w, conv_b, dt_bias, A, D, norm_w, w_out, conv_state, ssm_state, nheads, headdim, dstate,
               ngroups, eps=1e-5, out=None):
    """One timestep of the whole block for every stream as one launch: u_t [B,d_model] -> out [B,d_model]; `conv_state`
    [B,d_conv-1,C] (activation dtype) and `ssm_state` [B,H,P,N] (float32) advance in place.  w_in [E,d_model] and
    w_out [d_model,H*P] in the activation dtype."""
    lib = _lib()
    Bsz, d_model = u_t.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    C = H * P + 2 * G * N
    E = in_proj_width(H, P, N, G)
    dtype = u_t.dtype
    code = ssd._dtype_code(u_t)
    d_conv = conv_w.shape[1]
    ssd._require(u_t, "u_t", (Bsz, d_model), dtype)
    ssd._require(w_in, "w_in", (E, d_model), dtype)
    ssd._require(w_out, "w_out", (d_model, H * P), dtype)
    ssd._require(conv_w, "conv_w", (C, d_conv), torch.float32)
    ssd._require(conv_b, "conv_b", (C,), torch.float32)
    ssd._require(dt_bias, "dt_bias", (H,), torch.float32)
    ssd._require(A, "A", (H,), torch.float32)
    if D is not None:
        ssd._require(D, "D", (H,), torch.float32)
    ssd._require(norm_w, "norm_w", (H * P,), torch.float32)
    ssd._require(conv_state, "conv_state", (Bsz, d_conv - 1, C), dtype)
    ssd._require(ssm_state, "ssm_state", (Bsz, H, P, N), torch.float32)
    if out is None:
        out = u_t.new_empty((Bsz, d_model))
    else:
        ssd._require(out, "out", (Bsz, d_model), dtype)
    dims = SsdBlockDims(Bsz, 1, H, P, N, G, d_conv, 0)
    ssd._check(lib, lib.ssd_block_step_fwd(byref(dims), code, d_model, u_t.data_ptr(), w_in.data_ptr(), conv_w.data_ptr(),
                                           conv_b.data_ptr(), dt_bias.data_ptr(), A.data_ptr(), ssd._ptr(D),
                                           norm_w.data_ptr(), c_float(eps), w_out.data_ptr(), conv_state.data_ptr(),
                                           ssm_state.data_ptr(), out.data_ptr(), ssd._stream_ptr(u_t)))
    return out


def block_bwd_workspace(batch, seqlen, nheads, headdim, dstate, ngroups, d_conv=4, dtype=torch.bfloat16, device="cuda"):
    """Scratch for the partial sums of block_post_bwd / block_pre_bwd (one buffer serves both calls of a pass)."""
    lib = _lib()
    need = c_size_t(0)
    dims = SsdBlockDims(batch, seqlen, nheads, headdim, dstate, ngroups, d_conv, 0)
    code = ssd.SSD_DTYPE_F32 if dtype == torch.float32 else ssd.SSD_DTYPE_BF16
    ssd._check(lib, lib.ssd_block_bwd_workspace_bytes(byref(dims), code, byref(need)))
    return torch.empty(need.value, dtype=torch.uint8, device=device)


def block_post_bwd(y, zxbcdt, norm_w, dout, dzxbcdt, nheads, headdim, dstate, ngroups, eps=1e-5, workspace=None,
                   d_conv=4, yn_out=None):
    """Gradients of block_post: returns (dy [B,L,H,P], dnorm_w [H*P]) and writes dz into the z channels of dzxbcdt
    (a tensor laid out like zxbcdt, same row stride).  `d_conv` is the block's filter length: the library sizes the
    scratch both backward calls of a pass share from it, so it must be the one `workspace` was sized with.
    With `yn_out` [B,L,H*P] (zxbcdt's dtype) the call also writes the forward's normalised rows into it, bit for bit
    what `block_post` returns (for a forward that ran `block_post_proj` and kept none)."""
    lib = _lib()
    Bsz, L, E = zxbcdt.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    dtype = zxbcdt.dtype
    code = ssd._dtype_code(zxbcdt)
    if y.dtype != dtype:
        if not (dtype == torch.bfloat16 and y.dtype == torch.float32):
            raise ValueError(f"block y must be {dtype} (or float32 with bf16 activations), got {y.dtype}")
        code = ssd.SSD_DTYPE_BF16_Y32
    ld = _row_stride(zxbcdt)
    if tuple(dzxbcdt.shape) != (Bsz, L, E) or dzxbcdt.dtype != dtype or _row_stride(dzxbcdt) != ld:
        raise ValueError("dzxbcdt must have zxbcdt's shape, dtype and row stride")
    ssd._require(y, "y", (Bsz, L, H, P), y.dtype)
    ssd._require(dout, "dout", (Bsz, L, H * P), dtype)
    ssd._require(norm_w, "norm_w", (H * P,), torch.float32)
    dy = zxbcdt.new_empty((Bsz, L, H, P))
    dnorm_w = zxbcdt.new_empty(H * P, dtype=torch.float32)
    if workspace is None:
        workspace = block_bwd_workspace(Bsz, L, H, P, N, G, d_conv, dtype, zxbcdt.device)
    dims = SsdBlockDims(Bsz, L, H, P, N, G, d_conv, ld)
    if yn_out is not None:
        ssd._require(yn_out, "yn_out", (Bsz, L, H * P), dtype)
    ssd._check(lib, lib.ssd_block_post_bwd_yn(byref(dims), code, y.data_ptr(), zxbcdt.data_ptr(), norm_w.data_ptr(), c_float(eps),
                                              dout.data_ptr(), dy.data_ptr(), dzxbcdt.data_ptr(), dnorm_w.data_ptr(),
                                              None if yn_out is None else yn_out.data_ptr(),
                                              workspace.data_ptr(), workspace.numel(), ssd._stream_ptr(zxbcdt)))
    return dy, dnorm_w


def block_pre_bwd(zxbcdt, conv_w, conv_b, dt_bias, dx, dB, dC, ddt, dzxbcdt, nheads, headdim, dstate, ngroups,
                  conv_state=None, reset=None, dconv_state_out=None, need_dconv_state=False, workspace=None):
    """Gradients of block_pre: writes the x | B | C | dt channels of dzxbcdt and returns (dconv_w [C,d_conv],
    dconv_b [C], ddt_bias [H], dconv_state [B,d_conv-1,C] or None)."""
    lib = _lib()
    Bsz, L, E = zxbcdt.shape
    H, P, N, G = nheads, headdim, dstate, ngroups
    C = H * P + 2 * G * N
    dtype = zxbcdt.dtype
    code = ssd._dtype_code(zxbcdt)
    ld = _row_stride(zxbcdt)
    d_conv = conv_w.shape[1]
    if tuple(dzxbcdt.shape) != (Bsz, L, E) or dzxbcdt.dtype != dtype or _row_stride(dzxbcdt) != ld:
        raise ValueError("dzxbcdt must have zxbcdt's shape, dtype and row stride")
    ssd._require(conv_w, "conv_w", (C, d_conv), torch.float32)
    ssd._require(conv_b, "conv_b", (C,), torch.float32)
    ssd._require(dt_bias, "dt_bias", (H,), torch.float32)
    ssd._require(dx, "dx", (Bsz, L, H, P), dtype)
    ssd._require(dB, "dB", (Bsz, L, G, N), dtype)
    ssd._require(dC, "dC", (Bsz, L, G, N), dtype)
    ssd._require(ddt, "ddt", (Bsz, L, H), dtype)
    for name, t in (("conv_state", conv_state), ("dconv_state_out", dconv_state_out)):
        if t is not None:
            ssd._require(t, name, (Bsz, d_conv - 1, C), dtype)
    if reset is not None:
        if reset.dtype == torch.bool:
            reset = reset.view(torch.uint8)
        ssd._require(reset, "reset", (Bsz, L), torch.uint8)
    dconv_w = zxbcdt.new_empty((C, d_conv), dtype=torch.float32)
    dconv_b = zxbcdt.new_empty(C, dtype=torch.float32)
    ddt_bias = zxbcdt.new_empty(H, dtype=torch.float32)
    dstate = zxbcdt.new_empty((Bsz, d_conv - 1, C)) if need_dconv_state else None
    if workspace is None:
        workspace = block_bwd_workspace(Bsz, L, H, P, N, G, d_conv, dtype, zxbcdt.device)
    dims = SsdBlockDims(Bsz, L, H, P, N, G, d_conv, ld)
    ssd._check(lib, lib.ssd_block_pre_bwd(byref(dims), code, zxbcdt.data_ptr(), conv_w.data_ptr(), conv_b.data_ptr(),
                                          dt_bias.data_ptr(), ssd._ptr(conv_state), ssd._ptr(reset), dx.data_ptr(),
                                          dB.data_ptr(), dC.data_ptr(), ddt.data_ptr(), ssd._ptr(dconv_state_out),
                                          dzxbcdt.data_ptr(), dconv_w.data_ptr(), dconv_b.data_ptr(), ddt_bias.data_ptr(),
                                          ssd._ptr(dstate), workspace.data_ptr(), workspace.numel(),
                                          ssd._stream_ptr(zxbcdt)))
    return dconv_w, dconv_b, ddt_bias, dstate


def block_proj_supported(u: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether `block_proj` takes this product (else the caller's BLAS does it)."""
    return (u.is_cuda and u.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and u.shape[-1] in (128, 256)
            and weight.shape[0] % 8 == 0 and u.numel() > 0 and (u.data_ptr() | weight.data_ptr()) % 16 == 0)


def block_proj(u: torch.Tensor, weight: torch.Tensor, pad_rows: bool = False) -> torch.Tensor:
    """u [..., in_features] (bf16) times weight [out_features, in_features]^T -> [..., out_features] (bf16), float32
    accumulation: the block's in- and out-projection as one memory-bound kernel.  With pad_rows the result is the
    first out_features columns of a buffer whose rows are a multiple of 128 bytes apart (a non-contiguous view that
    `block_pre` and `block_post` take): every line the kernel writes is then a whole one."""
    lib = _lib()
    if u.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError(f"block_proj takes bfloat16 tensors, got {u.dtype} and {weight.dtype}")
    if weight.dim() != 2 or u.shape[-1] != weight.shape[1]:
        raise ValueError(f"block_proj: u [..., {u.shape[-1]}] does not match weight {tuple(weight.shape)}")
    if not u.is_contiguous() or not weight.is_contiguous():
        raise ValueError("block_proj takes contiguous tensors")
    rows = u.numel() // u.shape[-1]
    width = weight.shape[0]
    ld = (width + 63) // 64 * 64 if pad_rows else width
    out = u.new_empty(u.shape[:-1] + (ld,))
    ssd._check(lib, lib.ssd_block_proj_fwd(rows, u.shape[-1], width, ld, ssd.SSD_DTYPE_BF16, u.data_ptr(),
                                           weight.data_ptr(), out.data_ptr(), ssd._stream_ptr(u)))
    return out[..., :width] if ld != width else out


@dataclass
class Mamba2StreamState:
    """Streaming memory of one block: the conv's last d_conv-1 inputs and the SSM state."""
    conv: torch.Tensor          # [B, d_conv-1, H*P + 2*G*N], activation dtype
    ssm: SsdStreamState         # [B, H, P, N] float32

    def reset(self) -> None:
        self.conv.zero_()
        self.ssm.reset()

    def reset_rows(self, rows: torch.Tensor) -> None:
        if rows.dtype == torch.bool:
            self.conv.mul_((~rows).to(self.conv.dtype).view(-1, 1, 1))
        else:
            self.conv.index_fill_(0, rows, 0.0)
        self.ssm.reset_rows(rows)


class Mamba2Block:
    """Parameters and forward of one block.  Parameters are float32 masters; the projections run in the
    activation dtype of the input (bf16 on the GPU, as the reference policy runs,
    `trading_bots/src/torch/model/trading_model.rs:140-146`)."""

    def __init__(self, d_model, nheads, headdim, dstate, ngroups=1, d_conv=4, chunk=128, eps=1e-5, device="cuda",
                 seed=0):
        self.d_model, self.H, self.P, self.N, self.G = d_model, nheads, headdim, dstate, ngroups
        self.d_conv, self.chunk, self.eps = d_conv, chunk, eps
        self.d_inner = nheads * headdim
        self.conv_dim = self.d_inner + 2 * ngroups * dstate
        self._step_limit = _step_max_batch(d_model, nheads, headdim, dstate, ngroups)
        E = in_proj_width(nheads, headdim, dstate, ngroups)
        g = torch.Generator(device="cpu")
        g.manual_seed(seed)

        def rnd(*shape, scale=1.0):
            return (torch.randn(*shape, generator=g) * scale).to(device)

        self.in_proj = rnd(E, d_model, scale=1.0 / math.sqrt(d_model))
        self.conv_w = rnd(self.conv_dim, d_conv, scale=1.0 / math.sqrt(d_conv))
        self.conv_b = rnd(self.conv_dim, scale=0.1)
        # dt after softplus spread over [1e-3, 1e-1] (log-uniform), as Mamba-2 initialises it
        dt0 = torch.exp(torch.rand(nheads, generator=g) * (math.log(0.1) - math.log(1e-3)) + math.log(1e-3))
        self.dt_bias = (dt0 + torch.log(-torch.expm1(-dt0))).to(device)
        self.A_log = torch.log(torch.rand(nheads, generator=g) * 15.0 + 1.0).to(device)
        self.D = torch.ones(nheads, device=device)
        self.norm_w = torch.ones(self.d_inner, device=device)
        self.out_proj = rnd(d_model, self.d_inner, scale=1.0 / math.sqrt(self.d_inner))

    @property
    def A(self) -> torch.Tensor:
        return -torch.exp(self.A_log)

    def new_state(self, batch, dtype=torch.bfloat16) -> Mamba2StreamState:
        conv = torch.zeros((batch, self.d_conv - 1, self.conv_dim), dtype=dtype, device=self.in_proj.device)
        return Mamba2StreamState(conv, SsdStreamState.build(batch, self.H, self.P, self.N, device=self.in_proj.device))

    def forward(self, u: torch.Tensor, state: Optional[Mamba2StreamState] = None,
                reset: Optional[torch.Tensor] = None, save_for_backward: bool = False):
        """u [B,L,d_model] -> [B,L,d_model].  With `state`, continues from it and leaves it at the end of the
        window (a prefix scan; then `step` per bar).  `reset` [B,L]: episode boundaries inside the window -- a
        non-zero entry restarts both the SSM state and the conv's history before that timestep, exactly what
        `Mamba2StreamState.reset_rows` does between two steps of a stream.  With `save_for_backward` (windows
        without a carried state) returns (out, ctx) for `backward`."""
        if u.dim() != 3 or u.shape[2] != self.d_model:
            raise ValueError(f"block input must be [batch, seqlen, {self.d_model}], got {tuple(u.shape)}")
        if reset is not None and state is not None:
            raise ValueError("restarts inside the window and a carried conv state cannot be combined")
        if save_for_backward and state is not None:
            raise ValueError("backward through a window that continues a carried state is not supported")
        weights = self._converted(u.dtype)
        if self._one_call(u, weights):
            return self._forward_in_one_call(u, weights, state, reset, save_for_backward)
        zxbcdt = self._project(u, self._weights(u.dtype)[0], pad_rows=True)  # internal to the block: rows of whole lines
        if state is None:
            x, Bm, Cm, dt = block_pre(zxbcdt, self.conv_w, self.conv_b, self.dt_bias, self.H, self.P, self.N, self.G,
                                      reset=reset)
            y, _ = ssd.ssd_chunk_scan(x, dt, self.A, Bm, Cm, self.D, chunk=self.chunk, return_final_states=False,
                                      reset=reset)
        else:
            x, Bm, Cm, dt, conv = block_pre(zxbcdt, self.conv_w, self.conv_b, self.dt_bias, self.H, self.P, self.N,
                                            self.G, conv_state=state.conv, return_conv_state=True)
            state.conv = conv
            y = state.ssm.init_from_prefix(x, dt, self.A, Bm, Cm, self.D, chunk=self.chunk)
        w_out = self._weights(u.dtype)[1]
        if block_post_proj_supported(y, w_out):
            # gate, norm and out-projection as one kernel: the normalised rows never reach memory (the backward pass
            # needs them for one weight gradient only, and has its post stage write them on the way: yn=None).  256 -> 256 in us, one
            # kernel / two: 512 rows 6.8 / 7.1, 8 191 rows 7.5 / 11.0
            out = block_post_proj(y, zxbcdt, self.norm_w, w_out, self.H, self.P, self.N, self.G, self.eps)
            yn = None
        else:
            yn = block_post(y, zxbcdt, self.norm_w, self.H, self.P, self.N, self.G, self.eps)
            out = self._project(yn, w_out)
        if save_for_backward:
            return out, dict(u=u, zxbcdt=zxbcdt, x=x, Bm=Bm, Cm=Cm, dt=dt, y=y, yn=yn, reset=reset)
        return out

    def _one_call(self, u: torch.Tensor, weights) -> bool:
        """Whether the library runs the whole pass as one call (else the stages one by one): what each of its kernels asks for."""
        return (u.dtype == torch.bfloat16 and self.d_inner in (128, 256) and self.d_model in (128, 256)
                and weights[1].shape == (in_proj_width(self.H, self.P, self.N, self.G), self.d_model)
                and weights[2].shape == (self.d_model, self.d_inner) and u.device == weights[1].device == weights[2].device
                and block_proj_supported(u, weights[1]) and weights[2].data_ptr() % 16 == 0
                and self.A_log.dtype == torch.float32 and self.A_log.is_contiguous() and self.A_log.data_ptr() % 16 == 0)

    def _parameters_checked(self):
        """The float32 parameters between the projections, looked at as the stages do; D or None."""
        for name, t, shape in (("conv_w", self.conv_w, (self.conv_dim, self.d_conv)), ("conv_b", self.conv_b, (self.conv_dim,)),
                               ("dt_bias", self.dt_bias, (self.H,)), ("A_log", self.A_log, (self.H,)),
                               ("norm_w", self.norm_w, (self.d_inner,))):
            ssd._require(t, name, shape, torch.float32)
        if self.D is not None:
            ssd._require(self.D, "D", (self.H,), torch.float32)

    def _forward_in_one_call(self, u, weights, state, reset, save_for_backward):
        """`forward` as one call of the library: seven launches at a few rows, for which the stages' calls took the host longer than
        the GPU (4 x 4 096: 85 us of the host, 71 of the GPU)."""
        lib = _lib()
        Bsz, L, _ = u.shape
        H, P, N, G = self.H, self.P, self.N, self.G
        self._parameters_checked()
        u_in, u = u, u.contiguous()
        E = in_proj_width(H, P, N, G)
        ld = (E + 63) // 64 * 64    # rows of whole lines: internal to the block
        dims = SsdBlockDims(Bsz, L, H, P, N, G, self.d_conv, ld)
        conv = conv_out = init = final = None
        if state is not None:
            ssd._require(state.conv, "conv_state", (Bsz, self.d_conv - 1, self.conv_dim), u.dtype)
            if state.ssm.batch != Bsz:
                raise ValueError(f"stream state batch size mismatch: state has {state.ssm.batch}, input has {Bsz}")
            final = state.ssm.state
            ssd._require(final, "final_out", (Bsz, H, P, N), torch.float32)
            if state.ssm.initialized:
                init = final
            conv, conv_out = state.conv, torch.empty_like(state.conv)
        if reset is not None:
            if reset.dtype == torch.bool:
                reset = reset.view(torch.uint8)
            ssd._require(reset, "reset", (Bsz, L), torch.uint8)
        need = c_size_t(0)
        ssd._check(lib, lib.ssd_block_forward_workspace_bytes(byref(dims), ssd.SSD_DTYPE_BF16, self.d_model, self.chunk, byref(need)))
        rows, DI, GN = Bsz * L, self.d_inner, G * N
        out = u.new_empty((Bsz, L, self.d_model))
        if save_for_backward:
            buf = u.new_empty((Bsz, L, ld))
            x, Bm, Cm, dt, y = (u.new_empty((Bsz, L) + s) for s in ((H, P), (G, N), (G, N), (H,), (H, P)))
            ws = u.new_empty(need.value, dtype=torch.uint8)
            inner = [t.data_ptr() for t in (buf, x, Bm, Cm, dt, y, ws)]
        else:   # one buffer for all that is not kept
            sizes = [2 * rows * ld, 2 * rows * DI, 2 * rows * GN, 2 * rows * GN, 2 * rows * H, 2 * rows * DI]
            at, inner = 0, []
            for n in sizes:
                inner.append(at)
                at += (n + 255) // 256 * 256
            ws = u.new_empty(at + need.value, dtype=torch.uint8)
            base = ws.data_ptr()
            inner = [base + i for i in inner] + [base + at]
        ssd._check(lib, lib.ssd_block_forward(
            byref(dims), ssd.SSD_DTYPE_BF16, self.d_model, self.chunk, u.data_ptr(), weights[1].data_ptr(), self.conv_w.data_ptr(),
            self.conv_b.data_ptr(), self.dt_bias.data_ptr(), self.A_log.data_ptr(), ssd._ptr(self.D), self.norm_w.data_ptr(), self.eps,
            weights[2].data_ptr(), ssd._ptr(reset), ssd._ptr(conv), ssd._ptr(conv_out), ssd._ptr(init), ssd._ptr(final), *inner[:6],
            out.data_ptr(), inner[6], need.value, ssd._stream_ptr(u)))
        if state is not None:
            state.conv = conv_out
            state.ssm.initialized = True
        if save_for_backward:
            zxbcdt = buf[..., :E] if ld != E else buf
            return out, dict(u=u_in, zxbcdt=zxbcdt, x=x, Bm=Bm, Cm=Cm, dt=dt, y=y, yn=None, reset=reset)
        return out

    def _backward_in_one_call(self, ctx, dout, weights):
        """`backward` as one call of the library, where its kernels take both projections' weight gradients (None otherwise)."""
        u, zxbcdt, y, reset, x, Bm, Cm, dt = (ctx[k] for k in ("u", "zxbcdt", "y", "reset", "x", "Bm", "Cm", "dt"))
        Bsz, L, _ = u.shape
        H, P, N, G = self.H, self.P, self.N, self.G
        rows, E, DI, DM = Bsz * L, in_proj_width(H, P, N, G), self.d_inner, self.d_model
        slabs = _wgrad_slabs(rows)
        if (ctx["yn"] is not None or not self._one_call(u, weights) or not u.is_contiguous() or dout.dtype != u.dtype
                or tuple(dout.shape) != (Bsz, L, DM) or dout.device != u.device or not dout.is_contiguous() or dout.data_ptr() % 16
                or slabs >= _wgrad_slab_limit(E, DM) or slabs >= _wgrad_slab_limit(DM, DI) or E > 8192 or weights[5] is None):
            return None
        lib = _lib()
        self._parameters_checked()
        if tuple(zxbcdt.shape) != (Bsz, L, E) or zxbcdt.dtype != u.dtype or not zxbcdt.is_cuda:
            return None
        ld = _row_stride(zxbcdt)
        for name, t, shape in (("x", x, (Bsz, L, H, P)), ("B", Bm, (Bsz, L, G, N)), ("C", Cm, (Bsz, L, G, N)), ("dt", dt, (Bsz, L, H)),
                               ("y", y, (Bsz, L, H, P))):
            ssd._require(t, name, shape, u.dtype)
        if reset is not None:
            if reset.dtype == torch.bool:
                reset = reset.view(torch.uint8)
            ssd._require(reset, "reset", (Bsz, L), torch.uint8)
        dims = SsdBlockDims(Bsz, L, H, P, N, G, self.d_conv, ld)
        need = c_size_t(0)
        ssd._check(lib, lib.ssd_block_grad_workspace_bytes(byref(dims), ssd.SSD_DTYPE_BF16, DM, self.chunk, byref(need)))
        ws = u.new_empty(need.value, dtype=torch.uint8)
        dbuf = u.new_empty((Bsz, L, ld))
        f32 = lambda *shape: u.new_empty(shape, dtype=torch.float32)
        own_du = rows <= DPROJ_MAX_ROWS and E <= DPROJ_MAX_FEATURES
        g = dict(du=u.new_empty((Bsz, L, DM)) if own_du else None, din_proj=f32(E, DM), dconv_w=f32(self.conv_dim, self.d_conv),
                 dconv_b=f32(self.conv_dim), ddt_bias=f32(H), dA=f32(H), dA_log=f32(H), dD=None if self.D is None else f32(H),
                 dnorm_w=f32(DI), dout_proj=f32(DM, DI))
        ssd._check(lib, lib.ssd_block_grad(
            byref(dims), ssd.SSD_DTYPE_BF16, DM, self.chunk, u.data_ptr(), weights[5].data_ptr(), weights[5].shape[1],
            weights[3].data_ptr(), self.conv_w.data_ptr(), self.conv_b.data_ptr(), self.dt_bias.data_ptr(), self.A_log.data_ptr(),
            ssd._ptr(self.D), self.norm_w.data_ptr(), self.eps, ssd._ptr(reset), zxbcdt.data_ptr(), x.data_ptr(), Bm.data_ptr(),
            Cm.data_ptr(), dt.data_ptr(), y.data_ptr(), dout.data_ptr(), *[ssd._ptr(t) for t in g.values()], dbuf.data_ptr(),
            ws.data_ptr(), need.value, ssd._stream_ptr(u)))
        if not own_du:
            g["du"] = torch.matmul(dbuf.view(rows, ld)[:, :E], weights[1]).view(Bsz, L, DM)
        return g

    def backward(self, ctx: dict, dout: torch.Tensor) -> dict:
        """Gradients of sum(out * dout) with respect to the input and every parameter, from the tensors `forward`
        kept: two products per projection, the library's post, scan and pre backward kernels between them.
        Returns du [B,L,d_model] and float32 din_proj, dconv_w, dconv_b, ddt_bias, dA, dA_log, dD, dnorm_w, dout_proj."""
        u, zxbcdt, y, yn, reset = ctx["u"], ctx["zxbcdt"], ctx["y"], ctx["yn"], ctx["reset"]
        x, Bm, Cm, dt = ctx["x"], ctx["Bm"], ctx["Cm"], ctx["dt"]
        Bsz, L, _ = u.shape
        act = u.dtype
        E = in_proj_width(self.H, self.P, self.N, self.G)
        weights = self._converted(act)
        grads = self._backward_in_one_call(ctx, dout, weights)
        if grads is not None:
            return grads
        w_in = weights[1]
        A = self.A
        dout2 = dout.reshape(Bsz * L, self.d_model)
        dyn = self._project(dout2, self._out_proj_transposed(act)).view(Bsz, L, self.d_inner)
        # (a forward that ran gate, norm and out-projection as one kernel kept no normalised rows: post_bwd writes them)
        yn_new = None if yn is not None else torch.empty((Bsz, L, self.d_inner), dtype=act, device=u.device)
        # the gradient of zxbcdt, with zxbcdt's own (padded) row stride
        ld = _row_stride(zxbcdt)
        dbuf = torch.empty((Bsz, L, ld), dtype=act, device=u.device)
        dzx = dbuf[..., :E] if ld != E else dbuf
        ws = block_bwd_workspace(Bsz, L, self.H, self.P, self.N, self.G, self.d_conv, act, u.device)
        dy, dnorm_w = block_post_bwd(y, zxbcdt, self.norm_w, dyn, dzx, self.H, self.P, self.N, self.G, self.eps, workspace=ws,
                                     d_conv=self.d_conv, yn_out=yn_new)
        dout_proj = _weight_gradient(dout2, (yn if yn is not None else yn_new).reshape(Bsz * L, self.d_inner))
        g = ssd.ssd_chunk_scan_backward(x, dt, A, Bm, Cm, self.D, dy, chunk=self.chunk, reset=reset)
        dconv_w, dconv_b, ddt_bias, _ = block_pre_bwd(zxbcdt, self.conv_w, self.conv_b, self.dt_bias, g["dx"], g["dB"],
                                                      g["dC"], g["ddt"], dzx, self.H, self.P, self.N, self.G, reset=reset,
                                                      workspace=ws)
        dz2 = dbuf.view(Bsz * L, ld)[:, :E]
        w_in_t = self._converted(act)[5]
        if Bsz * L <= DPROJ_MAX_ROWS and E <= DPROJ_MAX_FEATURES and w_in_t is not None and block_dproj_supported(dz2, w_in_t):
            du = block_dproj(dz2, w_in_t).view(Bsz, L, self.d_model)
        else:
            du = torch.matmul(dz2, w_in).view(Bsz, L, self.d_model)
        din_proj = _weight_gradient(dz2, u.reshape(Bsz * L, self.d_model))
        return dict(du=du, din_proj=din_proj, dconv_w=dconv_w, dconv_b=dconv_b, ddt_bias=ddt_bias, dA=g["dA"],
                    dA_log=g["dA"] * A, dD=g["dD"], dnorm_w=dnorm_w, dout_proj=dout_proj)

    def _project(self, u: torch.Tensor, weight: torch.Tensor, pad_rows: bool = False) -> torch.Tensor:
        """u . weight^T in the activation dtype: the library's kernel where it takes the shape (bf16, in_features 128
        or 256), else the BLAS behind torch.  In us of the GPU, library against BLAS: 256 -> 648 at 512 rows 6.4 / 4.7, 2 048 rows
        6.5 / 6.7, 16 383 rows 14.6 / 24.2; 256 -> 256 at 512 rows 6.1 / 4.2, 8 192 rows 6.7 / 6.5, 16 383 rows 7.6 / 7.8; and of the
        host's time to issue it 8 against 19, which is what counts at few rows unless the caller replays a graph."""
        w = weight.to(u.dtype).contiguous()
        u = u.contiguous()
        if block_proj_supported(u, w):
            return block_proj(u, w, pad_rows=pad_rows)
        return torch.matmul(u, w.t()).contiguous()

    def _converted(self, dtype: torch.dtype):
        """(key, in_proj, out_proj, out_proj^T, step limit, in_proj turned as `block_dproj` takes it) in the activation dtype, converted
        once per dtype (and again when a master copy has been modified in place)."""
        key = (dtype, self.in_proj._version, self.out_proj._version, self.in_proj.data_ptr(), self.out_proj.data_ptr())
        cached = getattr(self, "_weights_cache", None)
        if cached is None or cached[0] != key:
            w_in, w_out, w_out_t, w_in_t = self._convert(dtype)
            # (with them: the batch up to which a step is one launch, whose kernel reads both 16 bytes at a time)
            limit = self._step_limit if dtype in _STEP_DTYPES and (w_in.data_ptr() | w_out.data_ptr()) % 16 == 0 else 0
            cached = (key, w_in, w_out, w_out_t, limit, w_in_t)
            self._weights_cache = cached
        return cached

    def _convert(self, dtype: torch.dtype):
        """in_proj, out_proj, out_proj^T and in_proj turned (bf16 only, else None) in `dtype`: one launch where the masters are float32
        and bf16 is asked for, as after every update of the weights."""
        wi, wo = self.in_proj, self.out_proj
        if (dtype == torch.bfloat16 and wi.is_cuda and wo.device == wi.device and wi.dtype == wo.dtype == torch.float32
                and wi.is_contiguous() and wo.is_contiguous() and wi.dim() == wo.dim() == 2 and wi.shape[1] == wo.shape[0]
                and wi.numel() and wo.numel() and (wi.data_ptr() | wo.data_ptr()) % 16 == 0):
            lib = _lib()
            (E, D), DI = wi.shape, wo.shape[1]
            new = lambda *shape: wi.new_empty(shape, dtype=dtype)
            w_in, w_out, w_out_t, w_in_t = new(E, D), new(D, DI), new(DI, D), new(D, (E + 15) // 16 * 16)
            ssd._check(lib, lib.ssd_block_weights(E, D, DI, wi.data_ptr(), wo.data_ptr(), w_in.data_ptr(), w_in_t.data_ptr(),
                                                  w_out.data_ptr(), w_out_t.data_ptr(), ssd._stream_ptr(wi)))
            return w_in, w_out, w_out_t, w_in_t
        w_in, w_out = wi.to(dtype).contiguous(), wo.to(dtype).contiguous()
        return w_in, w_out, w_out.t().contiguous(), turned_weight(w_in) if dtype == torch.bfloat16 else None

    def _weights(self, dtype: torch.dtype):
        """The two projection matrices in the activation dtype."""
        return self._converted(dtype)[1:3]

    def _out_proj_transposed(self, dtype: torch.dtype) -> torch.Tensor:
        """out_proj^T [d_inner, d_model] in the activation dtype (the backward's dyn = dout . out_proj is then a
        product of the forward's form, which the library's projection kernel takes), cached with the others."""
        return self._converted(dtype)[3]

    def _A_cached(self) -> torch.Tensor:
        """-exp(A_log), computed once per version of A_log (a launch of its own otherwise, per step)."""
        key = (self.A_log._version, self.A_log.data_ptr())
        cached = getattr(self, "_A_cache", None)
        if cached is None or cached[0] != key:
            cached = (key, -torch.exp(self.A_log))
            self._A_cache = cached
        return cached[1]

    def step(self, u_t: torch.Tensor, state: Mamba2StreamState, fused: Optional[bool] = None) -> torch.Tensor:
        """One timestep for every stream: u_t [B,d_model] -> [B,d_model]; advances `state` in place.  `fused`: run the
        step as one launch (default: where the fused kernel takes the shape, up to 1 024 or 256 streams) or as the stage kernels
        with the projections on the BLAS behind torch."""
        if u_t.dim() != 2 or u_t.shape[1] != self.d_model:
            raise ValueError(f"block step input must be [batch, {self.d_model}], got {tuple(u_t.shape)}")
        batch = u_t.shape[0]
        _, w_in, w_out, _, limit, _ = self._converted(u_t.dtype)
        if fused is None:
            fused = batch <= limit and u_t.is_cuda and u_t.data_ptr() % 16 == 0
        if fused:   # the whole step as one launch: what a step costs at a few streams is issuing its launches
            # (a captured step of more streams forms A at every replay, as one of stage kernels does)
            fresh = batch > STEP_CACHED_A_MAX_BATCH and torch.cuda.is_current_stream_capturing()
            out = block_step(u_t.contiguous(), w_in, self.conv_w, self.conv_b, self.dt_bias, self.A if fresh else self._A_cached(),
                             self.D, self.norm_w, w_out, state.conv, state.ssm.state, self.H, self.P, self.N, self.G, self.eps)
            state.ssm.initialized = True    # as `SsdStreamState.step` leaves it
            return out
        zxbcdt = torch.matmul(u_t, w_in.t()).unsqueeze(1).contiguous()
        x, Bm, Cm, dt, _ = block_pre(zxbcdt, self.conv_w, self.conv_b, self.dt_bias, self.H, self.P, self.N,
                                     self.G, conv_state=state.conv, conv_state_out=state.conv)  # in place
        y = state.ssm.step(x[:, 0], dt[:, 0], self.A, Bm[:, 0], Cm[:, 0], self.D)
        yn = block_post(y.unsqueeze(1), zxbcdt, self.norm_w, self.H, self.P, self.N, self.G, self.eps)
        return torch.matmul(yn[:, 0], w_out.t())

    def graphed_step(self, state: Mamba2StreamState, dtype: torch.dtype = torch.bfloat16) -> "GraphedBlockStep":
        """`step` for `state`'s streams captured once in a HIP graph and replayed per bar: at a few streams a step
        is five launches of a few microseconds each and the host's time to issue them is what a step costs (the
        reference captures its launch-bound loops the same way, trading_bots/src/torch/cuda/graph.rs)."""
        return GraphedBlockStep(self, state, dtype)



class GraphedBlockStep:
    """A captured `Mamba2Block.step` over fixed buffers.  Calling it copies the bar's input into the captured input
    buffer, replays the graph and returns the captured output buffer (overwritten by the next call).  The state it
    was built for advances in place, as with `step`; the block's parameters are read at replay time, except the
    projection matrices, whose activation-dtype copies are made at capture.  (A = -exp(A_log) of a step captured as one launch is
    a buffer of the graph's own, filled again when A_log has been modified.)"""

    def __init__(self, block: Mamba2Block, state: Mamba2StreamState, dtype: torch.dtype):
        batch = state.conv.shape[0]
        dev = state.conv.device
        self.u = torch.zeros((batch, block.d_model), dtype=dtype, device=dev)
        # what the warm-up steps below do to the state is undone afterwards
        conv_keep, ssm_keep = state.conv.clone(), state.ssm.state.clone()
        self.block, self.A = block, None
        self.weights = block._weights(dtype)    # (kept: the graph reads these copies, whatever becomes of the block's)

        def step():
            if self.A is None:
                return block.step(self.u, state, fused=False)
            state.ssm.initialized = True
            return block_step(self.u, self.weights[0], block.conv_w, block.conv_b, block.dt_bias, self.A, block.D, block.norm_w,
                              self.weights[1], state.conv, state.ssm.state, block.H, block.P, block.N, block.G, block.eps)

        if batch <= block._converted(dtype)[4] and block_step_supported(self.u, block.d_inner, block.N):
            self.A, self.A_key = block.A, (block.A_log._version, block.A_log.data_ptr())
        side = torch.cuda.Stream(device=dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            for _ in range(2):  # library handles, kernel modules and the weights' copies exist before the capture
                step()
        torch.cuda.current_stream(dev).wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = step()
        state.conv.copy_(conv_keep)
        state.ssm.state.copy_(ssm_keep)

    def __call__(self, u_t: torch.Tensor) -> torch.Tensor:
        self.u.copy_(u_t)
        if self.A is not None:
            key = (self.block.A_log._version, self.block.A_log.data_ptr())
            if key != self.A_key:
                self.A.copy_(self.block.A)
                self.A_key = key
        self.graph.replay()
        return self.out
