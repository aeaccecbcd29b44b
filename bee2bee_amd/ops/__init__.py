"""Op dispatch: hand-written CDNA4 HIP kernels on GPU, fp32 torch reference
on CPU.

Policy: when the tensors live on a GPU the HIP extension `_bee2bee_hip` is
REQUIRED — a missing/failed extension raises immediately rather than silently
falling back to eager PyTorch. The torch reference path (ops/reference.py) runs
only for CPU tensors (tests and GPU-less plumbing runs).

Kernels (ops/csrc/): fused (add+)RMSNorm, RoPE, paged KV store, paged GQA
decode attention, MFMA flash prefill attention, SwiGLU, top-k gating, grouped
expert GEMM, projections with what stands around them. Other projection GEMMs go
through hipBLASLt via torch.nn.functional.linear.

Which projections are whose is measured: decode steps of a few rows (one to six in
small stacks, two in deep ones: `stack_rows`) are one launch of decode_stack.hip;
else up to 16 rows (`few_rows`; logits: `head_rows`) the
kernels of linear_rows.hip, one launch for norm, product and what follows; 17 to 256
rows, of wide stacks fewer (`mid_rows`, `mid_shape`, `mid_gated`) linear_mid.hip,
split over K or activated; more rows linear_wide.hip where `wide_plan` says so:
all gated ones, and others where its times are below the library's. The grouped
kernel
driven as a single-segment GEMM loses to the library on all shapes
(scripts/bench_skinny.py: N/64 workgroups starve the chip); it stays for experts
because the E-way grid and the device-side segment offsets are what the library
cannot express.
"""
from __future__ import annotations

import os
from typing import Optional, Tuple

import torch

from . import reference

_hip = None
_hip_err: Optional[str] = None


def _load_hip():
    global _hip, _hip_err
    if _hip is not None or _hip_err is not None:
        return _hip
    try:
        import importlib

        _hip = importlib.import_module("bee2bee_amd.ops._bee2bee_hip")
    except Exception as e:  # noqa: BLE001
        _hip_err = str(e)
        _hip = None
    return _hip


def hip_available() -> bool:
    return _load_hip() is not None


def require_hip():
    """The GPU path: returns the extension module or raises loudly."""
    mod = _load_hip()
    if mod is None:
        raise RuntimeError(
            "bee2bee_amd HIP extension (_bee2bee_hip) is not built/loadable "
            f"but a GPU tensor was passed. Build it with `python setup.py "
            f"build_ext --inplace` (PYTORCH_ROCM_ARCH=gfx950). Import error: {_hip_err}"
        )
    return mod


def _use_hip(t: torch.Tensor) -> bool:
    if not t.is_cuda:
        return False
    if os.environ.get("BEE2BEE_FORCE_REFERENCE") == "1":
        return False
    return True


# --------------------------------------------------------------------- ops


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if _use_hip(x):
        return require_hip().rmsnorm(x, weight, eps)
    return reference.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float
) -> Tuple[torch.Tensor, torch.Tensor]:
    """residual += x (in fp32 semantics); y = rmsnorm(residual) * weight.
    Returns (y, new_residual). The HIP kernel fuses both passes in one HBM
    round-trip (memory-bound op — G13/B.Elementwise)."""
    if _use_hip(x):
        return require_hip().fused_add_rmsnorm(x, residual, weight, eps)
    return reference.fused_add_rmsnorm(x, residual, weight, eps)


rope_tables = reference.rope_tables


def rope_inplace(
    q: torch.Tensor,
    k: torch.Tensor,
    positions: torch.Tensor,
    cos: torch.Tensor,
    sin: torch.Tensor,
) -> None:
    if _use_hip(q):
        require_hip().rope_inplace(q, k, positions, cos, sin)
        return
    reference.rope_inplace(q, k, positions, cos, sin)


def kv_cache_store(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
) -> None:
    if _use_hip(k):
        require_hip().kv_cache_store(k, v, k_cache, v_cache, slot_mapping)
        return
    reference.kv_cache_store(k, v, k_cache, v_cache, slot_mapping)


def attn_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: float,
    order: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """order: decode_plan's, in which the contexts are read."""
    if _use_hip(q):
        return require_hip().attn_decode(
            q, k_cache, v_cache, block_table, seq_lens, scale, order
        )
    return reference.attn_decode(q, k_cache, v_cache, block_table, seq_lens, scale)


def attn_decode_lse(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    scale: float,
):
    """attn_decode that ALSO returns the per-(seq, q-head) flash merge
    state (m, l) — what context-parallel ranks exchange (parallel/cp.py)."""
    if _use_hip(q):
        out, ml = require_hip().attn_decode_lse(
            q, k_cache, v_cache, block_table, seq_lens, scale
        )
        return out, ml
    return reference.attn_decode_lse(
        q, k_cache, v_cache, block_table, seq_lens, scale)


def attn_prefill(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    cu_seqlens: torch.Tensor,
    max_seqlen: int,
    scale: float,
    causal: bool = True,
) -> torch.Tensor:
    if _use_hip(q):
        return require_hip().attn_prefill(
            q, k, v, cu_seqlens, max_seqlen, scale, causal
        )
    return reference.attn_prefill(q, k, v, cu_seqlens, max_seqlen, scale, causal)


def attn_prefill_paged(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_table: torch.Tensor,
    seq_lens: torch.Tensor,
    cu_q: torch.Tensor,
    max_qlen: int,
    scale: float,
) -> torch.Tensor:
    """Chunked prefill: packed query chunks (cu_q) attend to the full paged
    history (seq_lens includes the chunk; its K/V are already stored)."""
    if _use_hip(q):
        return require_hip().attn_prefill_paged(
            q, k_cache, v_cache, block_table, seq_lens, cu_q, max_qlen, scale
        )
    query_lens = cu_q[1:] - cu_q[:-1]
    return reference.attn_decode_with_history(
        q, k_cache, v_cache, block_table, seq_lens, query_lens, scale
    )


def layernorm(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor,
              eps: float) -> torch.Tensor:
    if _use_hip(x):
        return require_hip().layernorm(x, weight, bias, eps)
    return reference.layernorm(x, weight, bias, eps)


def fused_add_layernorm(x, residual, weight, bias, eps: float):
    if _use_hip(x):
        return tuple(require_hip().fused_add_layernorm(
            x, residual, weight, bias, eps))
    return reference.fused_add_layernorm(x, residual, weight, bias, eps)


def gelu(x: torch.Tensor) -> torch.Tensor:
    if _use_hip(x):
        return require_hip().gelu(x)
    return reference.gelu(x)


def swiglu(gate_up: torch.Tensor) -> torch.Tensor:
    if _use_hip(gate_up):
        return require_hip().swiglu(gate_up)
    return reference.swiglu(gate_up)


# ---------------------------------------------------- steps of a few rows
# One launch a projection, with the norm before it and what follows it folded
# in. norm: (weight, bias or None, eps) - with a bias layer norm, without RMS
# norm - or (squares, eps): RMS norm of rows that rows_linear's `then` made.

ROWS_MAX = 16


def few_rows(x: torch.Tensor) -> bool:
    """Steps that the few-row projections take: 1 to ROWS_MAX contiguous,
    16-byte aligned bf16 rows on the GPU."""
    return (x.dim() == 2 and 1 <= x.shape[0] <= ROWS_MAX and _use_hip(x)
            and x.dtype is torch.bfloat16 and x.is_contiguous()
            and x.data_ptr() % 16 == 0)


def head_rows(x: torch.Tensor, layer_norm: bool) -> bool:
    """Few rows whose logits are rows_linear's, where mid_head does not take
    them; the others' are a norm and the library's. Measured (us, rows_linear /
    norm and library): 128256 columns of 8192 359 / 374 at 8 rows, 376 / 365 at
    12, 402 / 364 at 16, 152064 459 / 464 at 12. A layer norm's mean and deviation are taken by each of the hundreds of
    workgroups: 50257 of 768 22.0 / 21.8 at 1 row, 22.8 / 22.1 at 4 (a launch
    less for the host: 20 us of a step that is not captured), 25 / 22.5 at 8, 30
    / 23 at 16."""
    if layer_norm:
        return few_rows(x) and x.shape[0] <= 4
    return few_rows(x) and (x.shape[0] <= 12 or x.shape[1] < 8192)


_ACTS = {None: 0, "swiglu": 1, "gelu": 2}


def _norm_args(norm):
    """weight, bias, squares, eps of the bindings."""
    if norm is None:
        return None, None, None, 0.0
    if len(norm) == 2:
        return None, None, norm[0], norm[1]
    return norm[0], norm[1], None, norm[2]


def rows_linear(x, w, bias=None, resid=None, norm=None, act=None,
                keep32=False, then=None):
    """act(norm(x) w^T + bias) + resid. act: None, "gelu" (tanh form), or
    "swiglu" (w holds the gate's rows, then the values'; no bias). x of a layer
    norm, and resid, may be fp32. Without act: keep32 leaves the result in
    fp32; `then`, the weight of the RMS norm that reads it, adds what that
    norm's projection takes: -> (result, result * then, sums of squares of 8
    columns each)."""
    if _use_hip(x):
        nw, nb, squares, eps = _norm_args(norm)
        if then is None:
            return require_hip().rows_linear(x, w, bias, resid, nw, nb,
                                             squares, eps, _ACTS[act], keep32)
        return require_hip().rows_sum(x, w, bias, resid, nw, nb, squares, eps,
                                      keep32, then)
    return reference.rows_linear(x, w, bias, resid, norm, act, keep32, then)


def rows_qkv(x, w, bias, norm, n_heads: int, positions, cos, sin, k_cache,
             v_cache, slot_mapping):
    """norm(x) w^T + bias split into q|k|v; q and k rotated (positions None:
    not), k and v stored into their pages. -> q [T, n_heads, hd]."""
    if _use_hip(x):
        return require_hip().rows_qkv(x, w, bias, *_norm_args(norm), n_heads,
                                      positions, cos, sin, k_cache, v_cache,
                                      slot_mapping)
    return reference.rows_qkv(x, w, bias, norm, n_heads, positions, cos, sin,
                              k_cache, v_cache, slot_mapping)


def stack_rows(spec) -> int:
    """Most rows of a decode step whose layers decode_stack takes, 0 for stacks
    that it does not: dense ones with sizes of whole steps of 64, heads of 64 or
    128, a layer norm of up to 1024 columns, and as many rows as fit into a CU's
    LDS."""
    return require_hip().stack_rows(
        spec.hidden_size, spec.n_heads, spec.n_kv_heads, spec.head_dim,
        spec.intermediate_size, spec.norm_type == "layernorm")


def decode_stack(x, layers, pages, n_heads: int, act: str, eps: float,
                 scale: float, positions, cos, sin, slot_mapping, block_table,
                 seq_lens, workgroups: int = 256, status=None,
                 patience: int = 1 << 22, absent: int = 0):
    """Decoder layers of one token of each of x's rows [M, H], on the GPU:
    q|k|v (rotated where positions and cos are given) with its page store,
    attention against the pages, output, feed-forward. layers: their weights;
    pages: their (keys, values); slot_mapping None: decode_slots'. workgroups:
    fewer than 256 compute the same, and up to 256 more find their share taken.
    status: a pinned int32 on the host, which is
    1 after a launch whose workgroups gave up a wait for each other, after
    `patience` polls in which none got on: its result is not valid then, and what
    depends on words that did not come is in no page. absent: so many of the 256
    shares are marked as taken, though nobody takes them, so that such a wait
    ends."""
    return require_hip().decode_stack(
        x, [[w.wqkv, w.wo, w.w_gate_up, w.w_down, w.wqkv_bias, w.wo_bias,
             w.w_gate_up_bias, w.w_down_bias, w.attn_norm, w.mlp_norm,
             w.attn_norm_bias, w.mlp_norm_bias, *kv]
            for w, kv in zip(layers, pages)],
        n_heads, act == "gelu", eps, scale, positions, cos, sin, slot_mapping,
        block_table, seq_lens, workgroups, status, patience, absent)


# Steps of some tens of rows: projections as fp32 parts over their inner
# dimension, which the next kernel sums, or as activated bf16 rows.

MID_MAX = 128
DEEP_MAX = 256
DEEP_SIZE = 9_000_000


def mid_rows(x: torch.Tensor) -> bool:
    """Steps of ROWS_MAX + 1 to MID_MAX contiguous bf16 rows on the GPU."""
    return (x.dim() == 2 and ROWS_MAX < x.shape[0] <= MID_MAX and _use_hip(x)
            and x.dtype is torch.bfloat16 and x.is_contiguous())


def ring_rows(x: torch.Tensor) -> bool:
    """Rows that mid_rows_linear takes: 1 to DEEP_MAX contiguous bf16 rows on the
    GPU."""
    return (x.dim() == 2 and 1 <= x.shape[0] <= DEEP_MAX and _use_hip(x)
            and x.dtype is torch.bfloat16 and x.is_contiguous())


def mid_shape(rows: int, width: int, depth: int) -> bool:
    """Projections that mid_linear takes: all up to MID_MAX rows, above it those
    that outweigh their parts, and of at most 4M weights all up to 160 rows and
    deep ones: the library is up to 2 us ahead on these, but its launches cost the
    host 20 us and not 6, which is what a step of such a stack takes if it is not
    captured (six layers of 768, prompts of 140 / 200 / 256 tokens 490 / 685 / 685
    us, with the library's 770; captured, 332 / 355 / 358 and 329 / 347 / 345).
    Measured with the kernel that reads them
    (us, the library's in brackets): at 128 / 160 / 224 rows 6144x4096 25.1 (30.4)
    / 26.4 (33.2) / 30.3 (42.5), 5120x3072 21.7 (25.5) / 23.4 (28.4) / 26.9
    (34.7), 4608x3584 22.2 (27.6) / 23.5 (29.6) / 26.9 (37.6), 3072x3072 15.8
    (23.7) / 17.7 (20.1) / 20.8 (21.5), 3072x2048 13.9 (15.7) / 15.4 (13.0) / 18.4
    (15.0), 2048x2048 12.0 (11.5) / 13.5 (12.1) at 160, 768x3072 10.6 (10.4) /
    11.8 (10.7) / 13.6 (11.7)."""
    if width * depth <= 4 << 20 and (rows <= 160 or 2 * depth >= 7 * width):
        return True
    return rows <= MID_MAX or width * depth >= (
        16_000_000 if width > depth else DEEP_SIZE)


def mid_gated(rows: int, width: int, depth: int) -> bool:
    """Gated projections that mid_rows_linear takes (width: of one half). What
    ends it are the input rows, which each CU draws beside its share of the
    weights; wide_linear takes the others. Measured beside the library's product
    and swiglu (us): 2x14336x4096
    36.9 (56.7) at 24 rows, 49.8 (57.8) at 128, 63 (69.6) at 200, 72.5 (71.6) at
    256; 2x18944x3584 45.3 (56.8), 57.7 (71.6), 61 (75.5) at 160, 107 (83) at
    200; 2x8192x2048 14.1 (20.8), 21.7 (23.9), 25 (30.6) at 192, 29 (33) at 256;
    2x5504x2048 13.0 (18.8), 18.5 (21.6), 23.5 (28.6) at 192, 27.9 (30.7) at 256;
    2x2048x768 6.9 (9.4), 9.7 (10.4), 11.9 (10.3). Beside wide_linear at 160 / 192 /
    224 rows: 2x5504x2048 20.4 (27.4) / 22.9 (28.9) / 25.5 (30.2), 2x9216x1408 22.1
    (26.8) / 23.9 (22.6) / 25.8 (23.7), 2x12288x1024 19.0 (20.4) / 21.1 (18.3) / 23.2
    (18.9), 2x16384x768 18.4 (17.6) / 20.5 (17.3) / 22.6 (17.6). More than 12 tiles of 8 columns a CU go
    in rounds, each with a start of its own: 2x27648x5120 96 (100), 107 (105) at
    48, 134 (123) at 128, but 2x28672x8192 141 (181), 153 (186), 194 (211)."""
    tiles = -(-width // 2048)           # of 8 columns, a CU
    if width * depth >= 1 << 30:        # the kernel's offsets are of 32 bits
        return False
    if tiles > 12:
        return rows <= (MID_MAX if depth >= 8192 else 32)
    if rows <= MID_MAX:
        return True
    if tiles > 8:
        return rows <= 160
    if width * depth < 11_000_000:
        return False
    if tiles > 4 and width * depth < 16_000_000:
        return rows <= 160 and depth >= 1024
    return rows <= (256 if tiles <= 4 else 224)


def mid_gelu(rows: int, width: int, depth: int) -> bool:
    """Projections with bias and gelu that mid_rows_linear takes: 3072x768 7.7 us
    at 24 rows, 9.8 at 64 (library 9.8, 10.1), 8192x2048 12.3, 15.9 (15.9, 16.4),
    20480x5120 45, 53 (45, 51)."""
    return rows <= 64 and width <= 8192


def mid_head(rows: int, width: int, depth: int) -> bool:
    """Logits that mid_rows_linear takes. Groups of 8 tiles of 16 columns, a
    CU's one after the other: where the last round leaves more than a twentieth
    of the chip idle (152064 columns) the library is ahead above 64 rows, and of
    the largest heads wide_linear from 129 rows on; above 160 rows it is also where
    rounds are short (few steps of K) or have fewer than 8 tiles for the waves that
    take two each. Beside the library's product,
    and wide_linear's where there is one (us): 128256x4096 159 (193) at 24 rows,
    188 (218) at 80, 214 (239, 210) at 128, 224 (251, 216) at 160; 32000x4096 41
    (63), 45 (66), 52 (68), 57 (69), 65 (78) at 200, 73 (79) at 256; 128256x2048
    82 (121), 102 (129), 120 (134), 129 (141, 137), 143 (178, 144); 152064x3584
    176 (242), 220 (213), 249 (245, 241); of rows of 768 17.0 (18.6), 22.6
    (20.8). At 160 / 192 / 224 / 256 rows: 65536x8192 190 (211, 204) / 209 (212, 205);
    64000x4096 110 (136, 131) at 161, 112 (138, 133); 28672x4096 53 (56) / 56 (60) / 60
    (64) / 67 (67); 32000x2048 33 (39) / 34 (39) / 37 (40) / 42 (40); 32000x1024 22 (21)
    / 22 (22) / 25 (23) / 27 (24); 65536x2048 67 (77) at 161, 67 (77) / 73 (78) / 80 (78);
    57344x2048 59 (59) / 64 (59) / 68 (62) / 73 (60), 49152x2048 57 (56) at 161, 60 (55)
    / 65 (57) / 75 (56); 65536x1536 54 (54) / 55 (48) / 59 (50) / 65 (52). Few rows (one launch of rows_linear in brackets; a norm takes 2.5
    us): 1 / 16 rows 128256x4096 155 (178) / 157 (188), 152064x3584 163 (182) /
    167 (204), 128256x2048 78 (93) / 80 (101); of rows of 8192 1 / 8 / 12 rows
    128256 370 (363) / 371 (359) / 370 (376), 152064 454 (427) / 458 (438) / 454
    (459)."""
    if rows <= ROWS_MAX and width * depth < 100_000_000:
        return False
    if rows <= 8 and depth >= 8192:
        return False
    tiles = -(-width // 16)
    rounds = -(-tiles // 2048)
    full = 256 * rounds * -(-tiles // (256 * rounds))
    if width % 4 or rows > DEEP_MAX or (depth < 1024 and rows > 48):
        return False
    if rows > MID_MAX and depth < 8192 and width * depth > 280_000_000:
        return False
    if rows > 160:
        each = full // (256 * rounds)
        if width * depth > (280_000_000 if rows <= 192 else 150_000_000):
            return False
        if rounds > 1 and not (rows <= 192 and each == 8 and depth >= 2048):
            return False
        if depth < 1536 or (rows > 224 and (depth < 4096 or each < 7)):
            return False
    return rows <= 64 or tiles * 20 >= full * 19


def deep_rows(x: torch.Tensor) -> bool:
    """Steps of MID_MAX + 1 to DEEP_MAX contiguous bf16 rows on the GPU."""
    return (x.dim() == 2 and MID_MAX < x.shape[0] <= DEEP_MAX and _use_hip(x)
            and x.dtype is torch.bfloat16 and x.is_contiguous())


def wide_rows(x: torch.Tensor) -> bool:
    """Steps of more than DEEP_MAX contiguous bf16 rows on the GPU."""
    return (x.dim() == 2 and x.shape[0] > DEEP_MAX and _use_hip(x)
            and x.dtype is torch.bfloat16 and x.is_contiguous())


_FORMS = {"rows": 0, "gated": 1, "parts": 2}


def wide_plan(rows: int, width: int, depth: int, form: str) -> int:
    """How wide_linear takes a projection on the GPU; 0: it is left to the
    library. form: "rows", "gated" (width: of one half) or "parts", whose reader
    sums parts or takes rows."""
    return require_hip().wide_plan(rows, width, depth, _FORMS[form])


def wide_linear(x, w, plan: int, act=None):
    """x w^T in bf16, or as parts [S, T, N] fp32 where the plan has several; act
    "swiglu" as in rows_linear."""
    if _use_hip(x):
        return require_hip().wide_linear(x, w, plan, act == "swiglu")
    if plan // 8 % 16 > 1:
        return reference.mid_linear(x, w)
    return reference.rows_linear(x, w, act=act)


def mid_linear(x, w):
    """Parts [S, T, N] fp32 whose sum over S is x w^T."""
    if _use_hip(x):
        return require_hip().mid_linear(x, w)
    return reference.mid_linear(x, w)


def mid_rows_linear(x, w, bias=None, act=None):
    """act(x w^T + bias) of up to DEEP_MAX rows; act as in rows_linear (swiglu:
    no bias)."""
    if _use_hip(x):
        return require_hip().mid_rows_linear(x, w, bias, _ACTS[act])
    return reference.rows_linear(x, w, bias, act=act)


def add_norm_parts(part, bias, resid, norm=None, dtype=None):
    """-> (norm(resid + parts + bias) or None without a norm, that sum in dtype,
    resid's by default). bf16 or fp32."""
    dtype = dtype or resid.dtype
    if _use_hip(part):
        nw, nb, eps = norm or (None, None, 0.0)
        return require_hip().add_norm_parts(part, bias, resid, nw, nb, eps,
                                            dtype is torch.float32)
    return reference.add_norm_parts(part, bias, resid, norm, dtype)


def rope_store_qkv(qkv, bias, n_heads: int, positions, cos, sin, k_cache,
                   v_cache, slot_mapping):
    """qkv: rows [T, N] (changed in place) or parts [S, T, N]. Bias added, q
    and k rotated (positions None: not), k and v stored into their pages. ->
    [T, N]."""
    if _use_hip(qkv):
        return require_hip().rope_store_qkv(qkv, bias, n_heads, positions,
                                            cos, sin, k_cache, v_cache,
                                            slot_mapping)
    return reference.rope_store_qkv(qkv, bias, n_heads, positions, cos, sin,
                                    k_cache, v_cache, slot_mapping)


def decode_slots(block_table, positions, block_size: int):
    """slot[b] = block_table[b][pos // bs] * bs + pos % bs."""
    if (_use_hip(positions) and positions.dtype is torch.int32
            and block_table.dtype is torch.int32 and positions.dim() == 1
            and positions.is_contiguous() and block_table.stride(1) == 1):
        return require_hip().decode_slots(block_table, positions, block_size)
    return reference.decode_slots(block_table, positions, block_size)


def decode_plan(block_table, positions, block_size: int, seq_lens,
                kv_heads: int):
    """-> (decode_slots, the rows' numbers by length, longest first, which
    attn_decode takes, or None). Workgroups that start last should be short ones:
    us of attention, as the rows stand / in that order, bf16, 8 key heads of size
    128, of 250 to 2000 tokens, 16 sequences 19.6 / 19.7, 24 28.3 / 28.4 (fp8 19.5 /
    18.7), 48 50.8 / 45.1, 128 104 / 96, of 375 to 3000 200 229 / 215 (fp8 121 /
    114), of 137 to 1100 400 167 / 160 (fp8 90 / 94), 1536 604 / 617: many workgroups
    even out by themselves, and neighbours of one length hold each other up. The
    order is found in 0.3 us more than the slots alone up to 24 rows, 1.3 at 100, 2.2
    at 200, 21 at 2048."""
    if (80 <= positions.numel() * kv_heads <= 2048 and _use_hip(positions)
            and all(t.dtype is torch.int32 for t in (block_table, positions,
                                                     seq_lens))
            and positions.dim() == 1 and seq_lens.dim() == 1
            and positions.is_contiguous() and seq_lens.is_contiguous()
            and block_table.stride(1) == 1
            and seq_lens.shape[0] >= positions.shape[0]):
        return require_hip().decode_plan(block_table, positions, block_size,
                                         seq_lens)
    return decode_slots(block_table, positions, block_size), None


def embed_positions(ids, table, positions, pos_table):
    """table[ids] + pos_table[positions]."""
    if (_use_hip(table) and table.dtype is torch.bfloat16
            and ids.dtype is torch.int64 and positions.dtype is torch.int32
            and ids.dim() == 1 and ids.is_contiguous()
            and positions.shape == ids.shape and positions.is_contiguous()
            and pos_table.dtype is table.dtype and table.shape[1] % 8 == 0):
        return require_hip().embed_positions(ids, table, positions, pos_table)
    return reference.embed_positions(ids, table, positions, pos_table)


def moe_topk_gate(logits: torch.Tensor, top_k: int):
    # gating math is tiny ([T, E]); torch ops are fine on both devices
    return reference.moe_topk_gate(logits, top_k)


def grouped_gemm(
    x: torch.Tensor, w: torch.Tensor, offsets: torch.Tensor
) -> torch.Tensor:
    """Per-expert segment GEMM out[seg_e] = x[seg_e] @ w[e].T — the MoE
    expert projection (segment sizes stay on device; graph-capturable)."""
    if _use_hip(x):
        return require_hip().grouped_gemm(x, w, offsets)
    return reference.grouped_gemm(x, w, offsets)


# ------------------------------------------------------------ hybrid stacks
# Mechanisms of the hybrid (latent-attention / linear-attention) layers.
# Batch conventions: see ops/reference.py. Unlike the dense-transformer ops
# above, these kernels are instantiated for bf16 AND fp32 activations; what
# the designs compute in 32-bit (residual, norms, scores, recurrent state)
# is fp32 in both.


def scalar_rmsnorm(x, gain: float, eps: float, out_dtype):
    if _use_hip(x):
        return require_hip().scalar_rmsnorm(x, float(gain), eps, out_dtype)
    return reference.scalar_rmsnorm(x, gain, eps, out_dtype)


def add_scalar_rmsnorm(resid, y, post_gain: float, pre_gain, eps: float,
                       out_dtype, y2=None):
    """resid(fp32) += norm(y [+ y2])*post_gain in place; ->
    norm(resid)*pre_gain (None when pre_gain is None). One fused pass on
    GPU; y2 (e.g. a shared expert's output) is summed to y in fp32."""
    if _use_hip(resid):
        return require_hip().add_scalar_rmsnorm(
            resid, y, y2, float(post_gain),
            None if pre_gain is None else float(pre_gain), eps, out_dtype)
    return reference.add_scalar_rmsnorm(resid, y, post_gain, pre_gain, eps,
                                        out_dtype, y2=y2)


def canon_conv(h, w, state, state_slots, cu_seqlens, seq_idx, positions):
    if _use_hip(h):
        return require_hip().canon_conv(h, w, state, state_slots, cu_seqlens,
                                        seq_idx, positions)
    return reference.canon_conv(h, w, state, state_slots, cu_seqlens, seq_idx,
                                positions)


def latent_rope_store(q_rot, kv, kv_norm, eps: float, kv_rank: int,
                      rope_dims: int, positions, cos, sin, cache,
                      slot_mapping, interleaved: bool = False) -> None:
    if _use_hip(kv):
        require_hip().latent_rope_store(q_rot, kv, kv_norm, eps, kv_rank,
                                        rope_dims, positions, cos, sin, cache,
                                        slot_mapping, interleaved)
        return
    reference.latent_rope_store(q_rot, kv, kv_norm, eps, kv_rank, rope_dims,
                                positions, cos, sin, cache, slot_mapping,
                                interleaved)


def latent_attn(q_abs, q_rot, gate, cache, block_table, positions, seq_idx,
                cu_seqlens, window: int, scale: float, max_qlen: int = 0,
                sink=None):
    """max_qlen: longest chunk in the batch (host int); 1 selects the
    decode kernel, larger the query-tiled prefill kernel. window 0: every
    earlier position; sink fp32 [heads]: a logit per head in the softmax
    denominator; gate None: no output gate."""
    if _use_hip(q_abs):
        return require_hip().latent_attn(q_abs, q_rot, gate, cache,
                                         block_table, positions, seq_idx,
                                         cu_seqlens, window, scale, max_qlen,
                                         sink)
    return reference.latent_attn(q_abs, q_rot, gate, cache, block_table,
                                 positions, seq_idx, cu_seqlens, window, scale,
                                 sink)


def lightning_attn(q, k, v, decay, state, state_slots, cu_seqlens, positions,
                   max_qlen: int = 0):
    if _use_hip(q):
        return require_hip().lightning_attn(q, k, v, decay, state,
                                            state_slots, cu_seqlens,
                                            positions, max_qlen)
    return reference.lightning_attn(q, k, v, decay, state, state_slots,
                                    cu_seqlens, positions)


def gated_rmsnorm(x, w, gate, eps: float, out_dtype):
    if _use_hip(x):
        return require_hip().gated_rmsnorm(x, w, gate, eps, out_dtype)
    return reference.gated_rmsnorm(x, w, gate, eps, out_dtype)


def clamped_glu(gate_up, limit: float, alpha: float):
    if _use_hip(gate_up):
        return require_hip().clamped_glu(gate_up, float(limit), float(alpha))
    return reference.clamped_glu(gate_up, limit, alpha)


# ---------------------------------------------- parallel-form hybrid stacks
# (ops/reference.py documents shapes). Ops with an `out` argument write a
# strided column slice of a wider activation buffer in place.

rope_tables_f64 = reference.rope_tables_f64


def rmsnorm_f32(x, w, eps: float, out_dtype):
    if _use_hip(x):
        return require_hip().add_rmsnorm_f32(x, None, w, eps, out_dtype, False)
    return reference.rmsnorm_f32(x, w, eps, out_dtype)


def add_rmsnorm_f32(resid, y, w, eps: float, out_dtype):
    """resid(fp32) += y in place; -> unit(resid) * w (None when w is None)."""
    if _use_hip(resid):
        return require_hip().add_rmsnorm_f32(resid, y, w, eps, out_dtype, True)
    return reference.add_rmsnorm_f32(resid, y, w, eps, out_dtype)


def relu2(x, out) -> None:
    if _use_hip(x):
        require_hip().relu2(x, out)
        return
    reference.relu2(x, out)


def qk_norm_rope_store(q, k, q_norm, k_norm, eps: float, rope_dims: int,
                       positions, cos, sin, q_mult, k_cache, v_cache,
                       slot_mapping, v=None) -> None:
    """v None: the values are the keys as projected."""
    if _use_hip(q):
        require_hip().qk_norm_rope_store(q, k, q_norm, k_norm, eps, rope_dims,
                                         positions, cos, sin, q_mult, k_cache,
                                         v_cache, slot_mapping, v)
        return
    reference.qk_norm_rope_store(q, k, q_norm, k_norm, eps, rope_dims,
                                 positions, cos, sin, q_mult, k_cache,
                                 v_cache, slot_mapping, v)


def sink_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
              cu_seqlens, sink, window: int, out, out_scale: float,
              max_qlen: int = 0) -> None:
    if _use_hip(q):
        require_hip().sink_attn(q, k_cache, v_cache, block_table, positions,
                                seq_idx, cu_seqlens, sink, window, out,
                                float(out_scale), max_qlen)
        return
    reference.sink_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
                        cu_seqlens, sink, window, out, out_scale)


def short_conv(x, w, state, state_slots, cu_seqlens, seq_idx, positions,
               silu: bool = True, bias=None, out_dtype=torch.float32):
    if _use_hip(x):
        return require_hip().short_conv(x, w, state, state_slots, cu_seqlens,
                                        seq_idx, positions, silu, bias,
                                        out_dtype)
    return reference.short_conv(x, w, state, state_slots, cu_seqlens, seq_idx,
                                positions, silu, bias, out_dtype)


def delta_gates(qk, n_qk_heads: int, dim: int, b, a, dt_bias, rate,
                channel_decay: bool):
    if _use_hip(qk):
        return tuple(require_hip().delta_gates(qk, n_qk_heads, dim, b, a,
                                               dt_bias, rate, channel_decay))
    return reference.delta_gates(qk, n_qk_heads, dim, b, a, dt_bias, rate,
                                 channel_decay)


def delta_rule(q, k, v, beta, g, state, state_slots, cu_seqlens, positions):
    if _use_hip(q):
        return require_hip().delta_rule(q, k, v, beta, g, state, state_slots,
                                        cu_seqlens, positions)
    return reference.delta_rule(q, k, v, beta, g, state, state_slots,
                                cu_seqlens, positions)


def head_gated_norm(o, w, gate, gate_act: str, eps: float, out,
                    out_scale: float) -> None:
    if _use_hip(o):
        require_hip().head_gated_norm(o, w, gate, gate_act == "sigmoid", eps,
                                      out, float(out_scale))
        return
    reference.head_gated_norm(o, w, gate, gate_act, eps, out, out_scale)


def retention_attn(q, k, v, decay, rope_dims: int, cos, sin, k_scale: float,
                   state, state_slots, cu_seqlens, positions,
                   max_qlen: int = 0):
    if _use_hip(q):
        return require_hip().retention_attn(q, k, v, decay, rope_dims, cos,
                                            sin, float(k_scale), state,
                                            state_slots, cu_seqlens,
                                            positions, max_qlen)
    return reference.retention_attn(q, k, v, decay, rope_dims, cos, sin,
                                    k_scale, state, state_slots, cu_seqlens,
                                    positions)


# ----------------------------------------------- weighted-sandwich stacks
# (ops/reference.py documents shapes and formulas)

rope_tables_scaled = reference.rope_tables_scaled


def add_group_rmsnorm(resid, y, w_post, step, w_pre, groups: int, eps: float,
                      out_dtype):
    """resid(fp32) += group_norm(y) * w_post [+ step] in place; ->
    group_norm(resid) * w_pre (None when w_pre is None). y None: only the
    step and the norm. One pass over HBM per operand on the GPU."""
    if _use_hip(resid):
        return require_hip().add_group_rmsnorm(resid, y, w_post, step, w_pre,
                                               groups, eps, out_dtype)
    return reference.add_group_rmsnorm(resid, y, w_post, step, w_pre, groups,
                                       eps, out_dtype)


def rope_unit_store(q, k, v, eps: float, rope_dims: int, positions, cos, sin,
                    q_mult: float, k_cache, v_cache, slot_mapping) -> None:
    if _use_hip(q):
        require_hip().rope_unit_store(q, k, v, eps, rope_dims, positions, cos,
                                      sin, float(q_mult), k_cache, v_cache,
                                      slot_mapping)
        return
    reference.rope_unit_store(q, k, v, eps, rope_dims, positions, cos, sin,
                              q_mult, k_cache, v_cache, slot_mapping)


def talk_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
              cu_seqlens, talk, gate, window: int, out,
              max_qlen: int = 0, path: str = "auto") -> None:
    """max_qlen: longest chunk of the step (host int); with bf16 pages, a
    matrix-core head size and a chunk of at least 16 rows the step takes
    the query-tiled kernel. path (GPU only): "auto", or force "scored"
    (scores written once, heads mixed before the values are read) or
    "cross" (every head's weights against every value head, mixed after)."""
    if _use_hip(q):
        require_hip().talk_attn(q, k_cache, v_cache, block_table, positions,
                                seq_idx, cu_seqlens, talk, gate, window, out,
                                max_qlen,
                                {"auto": 0, "scored": 1, "cross": 2}[path])
        return
    reference.talk_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
                        cu_seqlens, talk, gate, window, out)


def polynorm(z, coef, eps: float, out_dtype):
    if _use_hip(z):
        return require_hip().polynorm(z, coef, eps, out_dtype)
    return reference.polynorm(z, coef, eps, out_dtype)


def silu_glu(gate_up):
    if _use_hip(gate_up):
        return require_hip().silu_glu(gate_up)
    return reference.silu_glu(gate_up)


def group_topk_gate(logits, top_k: int, n_groups: int, keep_groups: int,
                    score: str = "softmax", group_top: int = 1,
                    choice_bias=None, renorm: bool = False,
                    route_scale: float = 1.0):
    """One kernel on the GPU (a thread per token, scores in LDS) while the
    experts of a workgroup's tokens fit; torch ops otherwise and on the
    CPU."""
    E = logits.shape[1]
    if _use_hip(logits) and (E + n_groups) * 256 <= 64 * 1024:
        w, idx = require_hip().group_topk_gate(
            logits.float().contiguous(), top_k, n_groups, keep_groups,
            score == "sigmoid", group_top, choice_bias, renorm,
            float(route_scale))
        return w, idx
    return reference.group_topk_gate(logits, top_k, n_groups, keep_groups,
                                     score, group_top, choice_bias, renorm,
                                     route_scale)


# ------------------------------------------- gated parallel-form stacks
# (ops/reference.py documents shapes and formulas)

rope_freq_tables = reference.rope_freq_tables


def rope_store(q, k, v, q_out, rope_dims: int, interleaved: bool, positions,
               cos, sin, q_mult: float, k_cache, v_cache,
               slot_mapping) -> None:
    if _use_hip(q_out):
        require_hip().rope_store(q, k, v, q_out, rope_dims, interleaved,
                                 positions, cos, sin, float(q_mult), k_cache,
                                 v_cache, slot_mapping)
        return
    reference.rope_store(q, k, v, q_out, rope_dims, interleaved, positions,
                         cos, sin, q_mult, k_cache, v_cache, slot_mapping)


def gqa_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
             cu_seqlens, softcap: float, talk, sink, head_gate, window: int,
             out, max_qlen: int = 0, dist=None, out_scale: float = 1.0,
             keep_first: int = 0) -> None:
    """max_qlen: longest chunk of the step (host int). dist fp32 [2, H]: a
    logarithmic distance bias on the scores; keep_first: the sequence's
    first positions stay visible past the window; out_scale multiplies the
    result (none of the three together with a cap or a score mix). Without
    a cap and a
    score mix the step runs on the sink-attention kernels; with them, on
    the score-mixing kernels. Both take bf16 prompt portions with head size
    64/128 to the matrix cores."""
    if _use_hip(q):
        if talk is None and not softcap:
            require_hip().sink_attn(q, k_cache, v_cache, block_table,
                                    positions, seq_idx, cu_seqlens, sink,
                                    window, out, float(out_scale), max_qlen,
                                    head_gate, dist, keep_first)
        else:
            if dist is not None or keep_first or out_scale != 1.0:
                raise ValueError("a distance bias, kept first tokens and an "
                                 "output scale do not combine with a score "
                                 "cap or mix")
            if talk is None:    # a cap alone: mix with the identity
                talk = torch.eye(q.shape[1], dtype=torch.float32,
                                 device=q.device)
            require_hip().mixed_score_attn(q, k_cache, v_cache, block_table,
                                           positions, seq_idx, cu_seqlens,
                                           float(softcap), talk, sink,
                                           head_gate, window, out, max_qlen)
        return
    reference.gqa_attn(q, k_cache, v_cache, block_table, positions, seq_idx,
                       cu_seqlens, softcap, talk, sink, head_gate, window, out,
                       dist, out_scale, keep_first)


def min_gru(z, x, g, state, state_slots, cu_seqlens, positions, out,
            max_qlen: int = 0) -> None:
    if _use_hip(z):
        require_hip().min_gru(z, x, g, state, state_slots, cu_seqlens,
                              positions, out, max_qlen)
        return
    reference.min_gru(z, x, g, state, state_slots, cu_seqlens, positions, out)


def pair_rmsnorm_mean(a, wa, b, wb, eps: float, out_dtype):
    if _use_hip(a):
        return require_hip().pair_rmsnorm_mean(a, wa, b, wb, eps, out_dtype)
    return reference.pair_rmsnorm_mean(a, wa, b, wb, eps, out_dtype)


def slice_rmsnorm(x, w, eps: float):
    if _use_hip(x):
        return require_hip().slice_rmsnorm(x, w, eps)
    return reference.slice_rmsnorm(x, w, eps)


def gated_add_rmsnorm(resid, y1, g1, y2, g2, extra, w, eps: float,
                      out_dtype):
    """resid(fp32) += sigmoid(g1) y1 [+ sigmoid(g2) y2] [+ extra] in place;
    -> unit(resid) * w (None when w is None). One pass on the GPU."""
    if _use_hip(resid):
        return require_hip().gated_add_rmsnorm(resid, y1, g1, y2, g2, extra,
                                               w, eps, out_dtype)
    return reference.gated_add_rmsnorm(resid, y1, g1, y2, g2, extra, w, eps,
                                       out_dtype)


def gelu_erf(x):
    if _use_hip(x):
        return require_hip().gelu_erf(x)
    return reference.gelu_erf(x)


# --------------------------------------------------- dynamic-tanh stacks
# (ops/reference.py documents shapes and formulas)


def add_tanh_norm(resid, y, post, pre, out_dtype):
    """resid(fp32) += tanh(a y) w + b in place (post = (a, w, b), when y is
    given); -> the same form of resid with pre (None when pre is None). One
    element-wise pass on the GPU."""
    if _use_hip(resid):
        pa, pw, pb = post if post is not None else (0.0, None, None)
        na, nw, nb = pre if pre is not None else (0.0, None, None)
        return require_hip().add_tanh_norm(resid, y, pa, pw, pb, na, nw, nb,
                                           out_dtype)
    return reference.add_tanh_norm(resid, y, post, pre, out_dtype)


def proj_norm_store(q, k, v, q_norm, k_norm, v_unit: bool, eps: float,
                    q_mult: float, k_cache, v_cache, slot_mapping) -> None:
    if _use_hip(q):
        require_hip().proj_norm_store(q, k, v, q_norm, k_norm, v_unit, eps,
                                      float(q_mult), k_cache, v_cache,
                                      slot_mapping)
        return
    reference.proj_norm_store(q, k, v, q_norm, k_norm, v_unit, eps, q_mult,
                              k_cache, v_cache, slot_mapping)


# --------------------------------------------- scaled parallel-form stacks
# (ops/reference.py documents shapes and formulas)

_inv_freq = {}


def embed_sinusoid(ids, table, scale: float, positions):
    """fp32 rows table[id] * scale + the position's sin/cos vector."""
    W = table.shape[1]
    key = (W, table.device)
    f = _inv_freq.get(key)
    if f is None:
        f = _inv_freq[key] = reference.sinusoid_freqs(W, table.device)
    if _use_hip(table):
        return require_hip().embed_sinusoid(ids, table, float(scale),
                                            positions, f)
    return reference.embed_sinusoid(ids, table, scale, positions, f)


def add_norm_pair(resid, y, w_post, wa, wb, eps: float, out_dtype):
    """resid(fp32) += unit(y) * w_post in place (when y is given); -> (unit(
    resid) * wa, unit(resid) * wb), None for a weight that is None. One pass
    on the GPU."""
    if _use_hip(resid):
        return tuple(require_hip().add_norm_pair(resid, y, w_post, wa, wb,
                                                 eps, out_dtype))
    return reference.add_norm_pair(resid, y, w_post, wa, wb, eps, out_dtype)


def scaled_add(resid, y1, s1, y2, s2, y3, out_dtype):
    """resid(fp32) += s1 * y1 [+ s2 * (y2 [+ y3])] in place; -> resid in
    out_dtype (resid itself when that is fp32)."""
    if _use_hip(resid):
        return require_hip().scaled_add(resid, y1, s1, y2, s2, y3, out_dtype)
    return reference.scaled_add(resid, y1, s1, y2, s2, y3, out_dtype)


def side_gate(g, table, offset: int, ids):
    """gelu_tanh(g) * table[ids, offset : offset + width of g]."""
    if _use_hip(g):
        return require_hip().side_gate(g, table, offset, ids)
    return reference.side_gate(g, table, offset, ids)


def packed_attn_covers(dtype, dim: int, vdim: int) -> bool:
    """Shapes the packed-key prompt attention has a kernel for."""
    return (dtype is torch.bfloat16 and dim == vdim and dim in (64, 128)
            and hip_available())


def packed_attn(q, k, v, cu_seqlens, scale: float, window: int, gate,
                max_qlen: int):
    """Whole prompts: every chunk starts at position 0 and attends to itself
    only, so keys and values come packed instead of from pages."""
    if _use_hip(q):
        return require_hip().packed_attn(q, k, v, cu_seqlens, float(scale),
                                         window, gate, max_qlen)
    return reference.packed_attn(q, k, v, cu_seqlens, scale, window, gate)


def ssd_scan(xbc, dt, dt_bias, rate, skip, groups: int, state, state_slots,
             cu_seqlens, positions, max_qlen: int = 0):
    """max_qlen: longest chunk of the step (host int); long chunks take the
    chunk-parallel kernels, short ones and decode rows the token-serial
    one."""
    if _use_hip(xbc):
        return require_hip().ssd_scan(xbc, dt, dt_bias, rate, skip, groups,
                                      state, state_slots, cu_seqlens,
                                      positions, max_qlen)
    return reference.ssd_scan(xbc, dt, dt_bias, rate, skip, groups, state,
                              state_slots, cu_seqlens, positions)


def gated_group_norm(y, z, w, groups: int, eps: float, out,
                     out_scale: float) -> None:
    if _use_hip(y):
        require_hip().gated_group_norm(y, z, w, groups, eps, out,
                                       float(out_scale))
        return
    reference.gated_group_norm(y, z, w, groups, eps, out, out_scale)


# ------------------------------------------------------- routed experts


def routed_relu2(z, weights, idx, n_experts: int, ff: int):
    if _use_hip(z):
        return require_hip().routed_relu2(z, weights, idx, n_experts, ff)
    return reference.routed_relu2(z, weights, idx, n_experts, ff)


def routed_silu_glu(gu, weights, idx):
    if _use_hip(gu):
        return require_hip().routed_silu_glu(gu, weights, idx)
    return reference.routed_silu_glu(gu, weights, idx)


def moe_sort(idx, n_experts: int):
    """(token, choice) pairs in expert order: -> pos [T, k] (row of each
    pair), tok [T * k] (token of each row), offs [E + 1], int32."""
    if _use_hip(idx):
        return tuple(require_hip().moe_sort(idx, n_experts))
    return reference.moe_sort(idx, n_experts)


def moe_combine(y, pos, weights):
    """out[t] = sum_j weights[t, j] * y[pos[t, j]], summed in fp32."""
    if _use_hip(y):
        return require_hip().moe_combine(y, pos, weights)
    return reference.moe_combine(y, pos, weights)
