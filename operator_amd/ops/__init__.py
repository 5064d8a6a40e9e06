"""Device ops of the explanation model and the log scanner.

GPU tensors always go to the hand-written gfx950 kernels in ``operator_amd._C``
(loading fails loudly if the extension is missing); CPU tensors use the fp32
reference implementations in :mod:`operator_amd.ops.reference`.
"""
from __future__ import annotations

import functools
import json
import os

import torch
import torch.nn.functional as F

from . import reference
from ._native import kernels, native_available, patterns

__all__ = [
    "rmsnorm", "silu_mul", "embedding", "rope_kv", "attn_prefill", "attn_decode", "attn_decode_rope", "sample",
    "kernels", "patterns", "native_available", "reference", "prefill_work_list", "prefill_block_q", "prefill_variant", "decode_splits",
    "decode_workspace", "linear", "gemm_splits", "gemm_plan", "gate_up_silu", "interleave_gate_up",
    "quantize_fp8", "rmsnorm_fp8", "silu_quantize_fp8", "linear_fp8", "fp8_plan", "SplitK", "linear_tile", "tile_ok", "BLAS_CALLS",
    "linear_f32", "decoder",
]

# never split a sequence into pieces shorter than this / split only while B x Hkv
# decode-attention workgroups < this (env overrides for tuning runs)
DECODE_MIN_SPLIT_TOKENS = int(os.environ.get("OAMD_DECODE_MIN_SPLIT", "256"))
# one workgroup per CU: the best split count at every measured (B, group, ctx) of
# profiles/attn_decode_splits_sweep_r5.jsonl lands at B x Hkv x splits ~ 256
DECODE_TARGET_BLOCKS = int(os.environ.get("OAMD_DECODE_TARGET_BLOCKS", "256"))
# attn_decode schedule bits (csrc/kernels/attn_decode.hip): 2 = NT 2 (two 16-token tiles per wave),
# 4 = one kv-head across all sequences first (else a sequence's kv-heads back to back)
DECODE_ATTN_VARIANT = int(os.environ.get("OAMD_DECODE_ATTN_VARIANT", "0"))


class SplitK:
    """A product left as S fp32 split-K slabs [S, M, N], of a decode batch or of prompts of up to 4096 rows (a bias is in
    the first slab); the consumer (a norm, rope_kv, a head or stream kernel, the fp8 SwiGLU) sums them, so the GEMM's
    separate reduction pass disappears. ``linear(defer_reduce=True)`` returns one where it cuts K, else a tensor."""

    __slots__ = ("p", "S", "shape", "device", "dtype", "is_cuda")

    def __init__(self, p: torch.Tensor, S: int, M: int, N: int):
        self.p, self.S, self.shape = p, S, (M, N)
        self.device, self.dtype, self.is_cuda = p.device, torch.bfloat16, True

    def materialize(self) -> torch.Tensor:
        M, N = self.shape
        return self.p[: self.S * M * N].view(self.S, M, N).sum(0).to(torch.bfloat16)


class Normed:
    """rmsnorm(t (+ residual)) that the projection it is for computes itself (``norm_into``); ``sum`` takes t + residual."""

    __slots__ = ("t", "w", "eps", "residual", "blocks", "sum", "shape", "is_cuda")

    def __init__(self, t, w: torch.Tensor, eps: float, residual: torch.Tensor | None, blocks: int):
        self.t, self.w, self.eps, self.residual, self.blocks = t, w, eps, residual, blocks
        self.sum = None if residual is None else torch.empty_like(residual)
        self.shape, self.is_cuda = t.shape, True

    def into(self, wt: torch.Tensor, y: torch.Tensor | None, p: torch.Tensor | None, act: int = 0) -> None:
        x, S = (self.t.p, self.t.S) if isinstance(self.t, SplitK) else (self.t, 0)
        kernels().gemm_rows_norm(x, S, self.residual, self.sum, self.w, self.eps, wt, y, p, act, self.blocks)


def norm_into(t, w: torch.Tensor, eps: float, residual: torch.Tensor | None, wt: torch.Tensor, glu: bool = False) -> Normed | None:
    """rmsnorm(t (+ residual)) of a few decode rows for the projection ``wt`` (``glu``: gate_up_silu of 64-row blocks) as a part of that
    projection's kernel, or None where it is a kernel of its own. The residual stream goes on in the result's ``sum``."""
    if not (t.is_cuda and t.dtype == torch.bfloat16 and wt.dtype == torch.bfloat16 and wt.is_contiguous() and len(t.shape) == 2
            and (t.S <= 8 if isinstance(t, SplitK) else t.is_contiguous()) and (residual is None or residual.is_contiguous())):
        return None
    (M, K), N = t.shape, wt.shape[0]
    blocks = _norm_blocks(M, N, K, glu)
    return None if blocks is None else Normed(t, w, eps, residual, blocks)


def rmsnorm(x, w: torch.Tensor, eps: float, residual: torch.Tensor | None = None,
            out: torch.Tensor | None = None) -> torch.Tensor:
    """RMSNorm; if ``residual`` is given it is updated in place to x + residual first.
    ``x`` may be a :class:`SplitK` (slabs summed inside the kernel)."""
    if isinstance(x, SplitK):
        M, N = x.shape
        y = out if out is not None else torch.empty(M, N, dtype=torch.bfloat16, device=x.device)
        kernels().rmsnorm(y, residual, w, y, eps, x.p, x.S)  # y doubles as the shape carrier
        return y
    if not x.is_cuda:
        y, r = reference.rmsnorm(x, w, eps, residual)
        if residual is not None:
            residual.copy_(r)
        if out is not None:
            out.copy_(y)
            return out
        return y
    y = out if out is not None else torch.empty_like(x)
    kernels().rmsnorm(x, residual, w, y, eps)
    return y


def rmsnorm_fp8(x, w: torch.Tensor, eps: float, residual: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """quantize_fp8(rmsnorm(x, ...)) — on the GPU one kernel, the input of an fp8 projection."""
    slabs = isinstance(x, SplitK)
    if not slabs and not x.is_cuda:
        return quantize_fp8(rmsnorm(x, w, eps, residual=residual))
    q = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    sx = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
    kernels().rmsnorm_fp8(None if slabs else x, residual, w, q, sx, eps, *((x.p, x.S) if slabs else ()))
    return q, sx


# activation of a gated feed-forward (common.h Glu): act(gate) * up
SILU, GELU_TANH = 1, 2


def silu_mul(gu: torch.Tensor, out: torch.Tensor | None = None, block: int | None = None, act: int = SILU) -> torch.Tensor:
    """act(gate) * up for gate|up interleaved in ``block``-feature blocks (None: [gate | up])."""
    if not gu.is_cuda:
        r = reference.silu_mul(gu, block, act == GELU_TANH)
        if out is not None:
            out.copy_(r)
            return out
        return r
    inter = gu.shape[1] // 2
    o = out if out is not None else torch.empty(gu.shape[0], inter, dtype=gu.dtype, device=gu.device)
    kernels().silu_mul(gu, o, block or 0, act)
    return o


GU_BLOCK = 64  # gate|up weight rows interleaved in 64-feature blocks (fused SwiGLU epilogue)


def interleave_gate_up(g: torch.Tensor, u: torch.Tensor, block: int = GU_BLOCK) -> torch.Tensor:
    """[g; u] rows -> blocks of ``block`` gate rows followed by the same features' up rows."""
    inter, H = g.shape
    return torch.stack([g.reshape(inter // block, block, H), u.reshape(inter // block, block, H)], 1).reshape(
        2 * inter, H).contiguous()


def _gu_splits(M: int, N: int, K: int, bm: int = 0) -> int:
    """K slices of a narrow gate|up decode GEMM: one block per tile leaves most CUs
    idle below 96 tiles, and the extra SwiGLU pass over the slabs is worth it."""
    tiles = N // 128 * (M // (bm or row_tile(M)))
    S = 1
    while tiles * S < 96 and S < 8 and K // 64 >= 4 * S:
        S *= 2
    return S


def gate_up_plan(M: int, N: int):
    """Kernel of a gate|up decode bucket of 64 to 256 rows without a measured entry: row tile of gemm_decode, "pp256"
    (gemm_pp) or None (gemm_mid). A workgroup takes in about 45 bytes per ns of both operands, so the
    smallest tile that still leaves one workgroup per CU wins (256 rows of 16384 x 2048: two 128-row tiles 28 us,
    one of 256 38; 128 rows of it: 64-row tiles 22 us, 128 25; of 28672 x 4096 128-row tiles 58, gemm_pp's 61), then the one whose
    workgroups come in one round (128 rows of 57344 x 8192: gemm_mid's 224 units 179 us, gemm_pp 217). 256 rows stay on gemm_pp: gemm_mid's W
    tile goes to two CUs (28672 x 4096 by itself 70 us against 78, but 12 us behind within a decode step)."""
    tiles = N // 128
    if M == 64:
        return 64
    if M == 128:
        return 64 if 2 * tiles <= CUS else 128 if tiles <= CUS else None
    if M == 256:
        return 128 if 2 * tiles <= CUS else "pp256"
    return 64 if M // 64 * tiles <= CUS else None


# stages of gemm_decode's gated tiles of other widths, by (rows, columns)
_GU_TILES = {(64, 64): 4, (128, 64): 4, (256, 64): 4, (64, 160): 4, (128, 160): 3, (256, 160): 3}


@functools.lru_cache(maxsize=4096)
def gate_up_tile(M: int, N: int, K: int) -> tuple[int, int, int] | None:
    """(rows, columns, stages) of a gated decode tile of 64 or 160 columns, or None for gate_up_plan's of 128. What a workgroup takes
    in sets its time, so the best width is the one whose workgroups are one round of the CUs, none of them idle (us): 64 rows of 16384 x 2048 in 128 tiles of 128
    columns 20.5, in 256 of 64 16.7; of 37888 x 3584 in 296 of 128 62, 237 of 160 44; 128 rows of it (gemm_mid) 67 and 50, 256 rows (gemm_pp) 112 and
    75; 256 rows of 8192 x 4096 43 and, in 128 x 64, 32. Taken where rounds times rows and columns are a tenth less; the smallest differences
    that were timed gained 8 %. Fewer than 96 tiles are cut along K (_gu_splits), which for longer rows is as fast (64 rows of 8192 x
    4096 25.1 and 25.3); 192 rows, no bucket's, have their 64-row tiles."""
    cost = lambda bm, bn: -(-(M // bm * -(-N // bn)) // CUS) * (bm + bn)  # noqa: E731
    now = gate_up_plan(M, N)
    if (M == 192 and now is None) or (isinstance(now, int) and _gu_splits(M, N, K, now) > 1 and K > 2048):
        return None
    tiles = [t for t in _GU_TILES if M % t[0] == 0 and 96 <= M // t[0] * -(-N // t[1]) <= CUS]
    best = min(tiles, key=lambda t: (cost(*t), t), default=None)
    if best is None or cost(*best) >= 0.9 * (cost(now, 128) if isinstance(now, int) else cost(256, 128) if now else cost(128, 256)):
        return None
    return *best, _GU_TILES[best]


def gate_up_silu(x: torch.Tensor, wgu: torch.Tensor, block: int | None, act: int = SILU, prompt: bool = False) -> torch.Tensor:
    """act(x Wg^T) * (x Wu^T) from the interleaved gate|up weight (``act``: SILU or GELU_TANH). Decode
    buckets run one fused gfx950 kernel (GEMM + gated epilogue, no [M, 2I] intermediate);
    other shapes run the GEMM then the silu_mul kernel. ``prompt``: as for ``linear``."""
    M, K = x.shape
    N = wgu.shape[0]
    if isinstance(x, Normed):
        y = torch.empty(M, N // 2, dtype=wgu.dtype, device=wgu.device)
        x.into(wgu, y, None, act)
        return y
    if x.is_cuda and block == 64 and f32_ok(x, wgu):
        return linear_f32(x, wgu, glu=act, prompt=prompt)
    if (x.is_cuda and block == 64 and x.dtype == torch.bfloat16 and M <= SKINNY_MAX_M and N % 128 == 0
            and K % 128 == 0 and x.is_contiguous() and wgu.is_contiguous()
            and skinny_plan(M, N, K) is not None and _gemm_table_get().get(("silu", M, N, K)) != "blas"):
        y = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
        plan = rows_plan(M, N, K, True)
        if plan is None:
            kernels().gemm_skinny(x, wgu, y, None, 1, act)
        else:
            kernels().gemm_skinny(x, wgu, y, None, 1, act, plan[1])
        return y
    if (x.is_cuda and block == 64 and x.dtype == torch.bfloat16 and M % 64 == 0 and M <= 256 and N % 128 == 0
            and K % 64 == 0 and x.is_contiguous() and wgu.is_contiguous()):
        t = _gemm_table_get().get(("silu", M, N, K))
        if t is None and (tile := gate_up_tile(M, N, K)) is not None:
            y = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
            kernels().gemm_decode(x, wgu, y, None, 1, tile[1], tile[0], act, False, tile[2])
            return y
        bm = gate_up_plan(M, N) if t is None else t if isinstance(t, str) else t[0]
        if t is None and bm is None:
            return linear_tile(x, wgu, glu=act, prompt=prompt)
        if isinstance(bm, str) and bm.startswith("pp"):   # ping-pong kernel, nt weight loads (bm 128 / 256)
            y = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
            bm = int(bm[2:])
            ws, fl = _pp_sk_workspace(x.device, N // 128) if (bm == 256 and PP_STREAM_K) else (None, None)
            kernels().gemm_pp(x, wgu, y, None, 1, bm, act, True, False, ws, fl)
            return y
        if t is None and (S := _gu_splits(M, N, K, bm)) > 1:   # too few column tiles to fill the GPU: split K
            y = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
            slabs = torch.empty(S * M * N, dtype=torch.float32, device=x.device)
            kernels().gemm_decode(x, wgu, None, slabs, S, 128, bm, False, False, 3)
            kernels().splitk_silu(slabs, y, S, act)
            return y
        if t != "blas":
            # one workgroup per CU: a fourth stage (28672 x 4096: 64 rows 41 us on three, 38, 128 rows 53.5 and 51); two keep theirs in LDS on three
            ns = t[1] if t and len(t) > 1 else 4 if bm <= 128 and M // bm * (N // 128) <= CUS else 3
            y = torch.empty(M, N // 2, dtype=x.dtype, device=x.device)
            kernels().gemm_decode(x, wgu, y, None, 1, 128, bm, act, False, ns)
            return y
    if block == 64 and tile_ok(x, wgu) and N % 128 == 0:
        return linear_tile(x, wgu, glu=act, prompt=prompt)   # prefill: gating fused into the tile epilogue
    return silu_mul(linear(x, wgu, prompt=prompt), block=block, act=act)


# Stream-K form of the 256-row gate|up+SwiGLU decode GEMM (csrc/kernels/gemm_pp.hip SK): one block per
# CU over the flattened (tile, K-step) stream instead of one block per 128-feature tile (224 of 256 CUs
# busy at the 8B shape). OAMD_PP_STREAM_K=1 turns it on (A/B runs).
PP_STREAM_K = os.environ.get("OAMD_PP_STREAM_K", "0") == "1"
_PP_SK_WS: dict = {}


def _pp_sk_workspace(device, tiles: int):
    """(fp32 partials, zeroed int flags) for the stream-K gate|up kernel, one pair per (device,
    tile count), kept for the life of the process: captured decode graphs hold the pointers, and the
    kernel leaves the flags zero. A stream runs one such GEMM at a time (the engine's decode stream)."""
    key = (str(device), tiles)
    ws = _PP_SK_WS.get(key)
    if ws is None:
        ws = (torch.empty(tiles * 32768, dtype=torch.float32, device=device),
              torch.zeros(tiles, dtype=torch.int32, device=device))
        _PP_SK_WS[key] = ws
    return ws


def embedding(ids: torch.Tensor, table: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    if not ids.is_cuda:
        r = reference.embedding(ids, table)
        if out is not None:
            out.copy_(r)
            return out
        return r
    o = out if out is not None else torch.empty(ids.numel(), table.shape[1], dtype=table.dtype, device=ids.device)
    kernels().embedding(ids, table, o)
    return o


def rope_kv(qkv: torch.Tensor, pos: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, Hq: int, Hkv: int,
            k_cache: torch.Tensor | None = None, v_cache: torch.Tensor | None = None,
            slots: torch.Tensor | None = None, want_kv: bool = True,
            q_out: torch.Tensor | None = None, bias: torch.Tensor | None = None,
            k_scale: float = 1.0, v_scale: float = 1.0):
    """Rotate q/k of the packed qkv rows and scatter k/v into the paged cache.
    ``bias`` [(Hq + 2 Hkv) D] is added to the projection first (Qwen2); with split-K
    slabs it is added before the single bf16 rounding. An e4m3fn cache stores
    x / k_scale, x / v_scale.

    Returns (q [T,Hq,D], k [T,Hkv,D] | None, v [T,Hkv,D] | None).
    """
    if isinstance(qkv, SplitK):
        T = qkv.shape[0]
        D = cos.shape[1] * 2
        dev = qkv.device
        q = q_out if q_out is not None else torch.empty(T, Hq, D, dtype=torch.bfloat16, device=dev)
        k = torch.empty(T, Hkv, D, dtype=torch.bfloat16, device=dev) if want_kv else None
        v = torch.empty(T, Hkv, D, dtype=torch.bfloat16, device=dev) if want_kv else None
        kernels().rope_kv(q, pos, cos, sin, Hq, Hkv, q, k, v, k_cache, v_cache, slots, qkv.p, qkv.S, bias,
                          k_scale, v_scale)
        return q, k, v
    if not qkv.is_cuda:
        if bias is not None:
            qkv = (qkv.float() + bias.float()).to(qkv.dtype)
        q, k, v = reference.rope_kv(qkv, pos, cos, sin, Hq, Hkv, k_cache, v_cache, slots, k_scale, v_scale)
        if q_out is not None:
            q_out.copy_(q.reshape(q_out.shape))
            q = q_out
        return q, (k if want_kv else None), (v if want_kv else None)
    T = qkv.shape[0]
    D = cos.shape[1] * 2
    q = q_out if q_out is not None else torch.empty(T, Hq, D, dtype=qkv.dtype, device=qkv.device)
    k = torch.empty(T, Hkv, D, dtype=qkv.dtype, device=qkv.device) if want_kv else None
    v = torch.empty(T, Hkv, D, dtype=qkv.dtype, device=qkv.device) if want_kv else None
    kernels().rope_kv(qkv, pos, cos, sin, Hq, Hkv, q, k, v, k_cache, v_cache, slots, None, 1, bias, k_scale, v_scale)
    return q, k, v


# v3 schedule options (csrc/kernels/attn_prefill.hip OPT bits): l = K/V loads after the
# S MFMAs, r = deferred rescale, d = two LDS tile buffers (one barrier per tile)
_PREFILL_VARIANTS = {"v1": 1, "v2": 2, "v3": 3, "v4": 4}


def prefill_variant(Hq: int, Hkv: int) -> int:
    """attn_prefill kernel variant: 1 = per-query-head (any G), 2 = GQA-grouped 16-row waves
    (G = Hq / Hkv in 1, 2, 4, 8), 3 = GQA-grouped swapped-operand 32x32 MFMA waves in 8-wave
    workgroups (G <= 8), 4 = the same waves in 4-wave workgroups, two per CU (G <= 4;
    profiles/prefill_attn_v3_vs_v4.jsonl: 6-9 % faster at 16x1024 and mixed lengths, equal at
    4x4096). Default: v4 where G <= 4, else v3. OAMD_PREFILL_ATTN=v1|v2|v3|v4 overrides it; a
    grouped variant that cannot take G falls back to v3, then v1."""
    G = Hq // Hkv if Hkv and Hq % Hkv == 0 else 0
    want = _PREFILL_VARIANTS.get(os.environ.get("OAMD_PREFILL_ATTN", ""), 4 if 1 <= G <= 4 else 3)
    if want == 2 and G not in (1, 2, 4, 8):
        want = 3
    if want == 4 and G > 4:
        want = 3
    return want if 1 <= G <= 8 else 1


def prefill_block_q(Hq: int, Hkv: int, variant: int | None = None) -> int:
    """Query rows per attn_prefill work item: 64 (v1), 16 x (8 / G) (v2), 32 x (8 / G) (v3),
    32 x (4 / G) (v4)."""
    v = prefill_variant(Hq, Hkv) if variant is None else variant
    if v == 1:
        return 64
    G = Hq // Hkv
    return (16 if v == 2 else 32) * ((4 if v == 4 else 8) // G)


def prefill_work_list(seq_lens: list[int], block_q: int = 64) -> tuple[list[int], list[int]]:
    """(work_seq, work_q0) for attn_prefill: one item per ``block_q``-row query block; longest first."""
    items = []
    for s, L in enumerate(seq_lens):
        for q0 in range(0, L, block_q):
            items.append((q0, s))
    items.sort(key=lambda t: -t[0])  # heavy (late, long-causal) blocks first
    return [s for _, s in items], [q0 for q0, _ in items]


def attn_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, seq_lens: list[int], scale: float,
                 out: torch.Tensor | None = None, work: tuple[torch.Tensor, torch.Tensor, torch.Tensor] | None = None,
                 prefix: tuple | None = None):
    """Causal attention over packed sequences (q [T,Hq,D], k/v [T,Hkv,D]).

    ``prefix`` = (pk, pv, seq_pfx, pfx_lens): a shared prompt prefix (LLMEngine prefix
    sharing) whose cached K/V rows pk / pv [P, Hkv, D] come before sequence s's own keys
    for its first pfx_lens[s] keys (<= P); the own query rows sit at
    positions pfx_lens[s] + row and see every prefix key. seq_pfx: the same lengths as an
    int32 device tensor (GPU), pfx_lens: as a host list (CPU reference; may be None on
    the GPU)."""
    cu = [0]
    for L in seq_lens:
        cu.append(cu[-1] + int(L))
    if not q.is_cuda:
        r = reference.attn_prefill(q, k, v, cu, scale,
                                   prefix=None if prefix is None else (prefix[0], prefix[1], prefix[3]))
        if out is not None:
            out.copy_(r)
            return out
        return r
    o = out if out is not None else torch.empty_like(q)
    if work is None:
        var = prefill_variant(q.shape[1], k.shape[1])
        ws, wq = prefill_work_list([int(x) for x in seq_lens], prefill_block_q(q.shape[1], k.shape[1], var))
        dev = q.device
        work = (torch.tensor(cu, dtype=torch.int32, device=dev), torch.tensor(ws, dtype=torch.int32, device=dev),
                torch.tensor(wq, dtype=torch.int32, device=dev), var)
    # work = (cu_seqlens, work_seq, work_q0, variant); the work list must be cut at that variant's block_q
    var = work[3] if len(work) > 3 else 1
    if prefix is not None:
        if var not in (3, 4):
            raise ValueError("a shared prefix needs attn_prefill variant 3 or 4")
        kernels().attn_prefill(q, k, v, o, work[0], work[1], work[2], scale, var, prefix[0], prefix[1], prefix[2])
    else:
        kernels().attn_prefill(q, k, v, o, work[0], work[1], work[2], scale, var)
    return o


GEMM_DECODE_M = (64, 128, 256)  # decode buckets the gfx950 gemm_decode kernel is tuned for
_GEMM_TABLE_PATH = os.environ.get("OAMD_GEMM_TABLE") or os.path.join(os.path.dirname(os.path.abspath(__file__)),
                                                                     "gemm_tuned.json")
_gemm_table: dict | None = None


def _gemm_table_get() -> dict:
    """Measured best (bm, bn, splits) per decode GEMM shape on MI355X, written by
    ``tools/bench_gemm.py --write-table`` ("blas" = hipBLASLt wins that shape)."""
    global _gemm_table
    if _gemm_table is None:
        try:
            with open(_GEMM_TABLE_PATH) as f:
                _gemm_table = {tuple(x if x in ("silu", "skinny") else int(x) for x in k.split(",")): v
                               for k, v in json.load(f).items()}
        except (OSError, ValueError):
            _gemm_table = {}
    return _gemm_table


def row_tile(M: int) -> int:
    """Largest gemm_decode row tile (256, 128, 64) dividing M (M % 64 == 0): a bucket of
    192 rows runs three 64-row tiles, not one 192-row tile the kernel has no variant for."""
    return next(b for b in (256, 128, 64) if M % b == 0)


LM_HEAD_MIN_N = 32768


def _measured_blas(M: int, N: int, K: int) -> bool:
    """The tuned table measured hipBLASLt fastest for this decode-bucket shape (small-M
    GEMMs that neither the decode kernels nor the 256-row tile kernel win)."""
    if N >= LM_HEAD_MIN_N:   # vocabulary projections never do (gemm_skinny, gemm_mid, gemm_decode or gemm_tile)
        return False
    t = _gemm_table_get()
    return t.get(("skinny", M, N, K) if M <= SKINNY_MAX_M else (M, N, K)) == "blas"


def gemm_splits(M: int, N: int, K: int) -> int:
    """K slices (1, 2, 4 or 8) that bring gemm_decode's 64-column tiles to one block per CU, for callers that pass
    ``linear`` their own ``splits``; its own plans are gemm_plan's."""
    best = 1
    for S in (1, 2, 4, 8):
        if K % (64 * S):
            break
        best = S
        if N // 64 * S >= CUS:
            break
    return best


def gemm_plan(M: int, N: int, K: int, defer: bool = True):
    """(bm, bn, splits, stages) for the gfx950 gemm_decode kernel, or None for the tile kernels (or hipBLASLt).
    ``defer``: the consumer sums the K slices."""
    if M % 64 or N % 64 or K % 64 or M > 256:
        return None
    t = _gemm_table_get().get((M, N, K))
    if t in ("blas", "tile"):   # hipBLASLt / the 256x256-tile kernel (linear decides which)
        return None
    if t is not None:
        return tuple(t)   # (bm, bn, S[, stages]) for gemm_decode
    if N >= LM_HEAD_MIN_N:
        return _vocab_plan(M, N, K)
    return _decode_plan(M, N, K, defer)


def _slab_us(S: int, M: int, N: int, defer: bool) -> float:
    """Writing and reading S fp32 slabs, and the reduce pass where the consumer does not sum them."""
    return 0.0 if S == 1 else S * M * N * 1.8e-6 + (0 if defer else 6)


@functools.lru_cache(maxsize=4096)
def _decode_tiles(M: int, N: int, K: int, defer: bool):
    """(estimate in us, (rows, columns, K slices, stages)) of a decode bucket's projection on gemm_decode. A CU takes in 40 to 47 bytes per ns through LDS-DMA
    whatever the tile, so a workgroup's time is its K steps times its (rows + columns) of 128 bytes, and the best
    plan has the fewest such bytes at one workgroup per CU: 64 rows of 5120 x 14336 in 64 x 128 tiles and 5
    slices 29 us (64 x 64 tiles, 4 slices: 42), 256 rows of 3584 x 3584 in 128 x 128 tiles 14 (256 x 64: 19), 64
    rows of 2048 x 2048 in 64 x 64 tiles 4.6."""
    best = None
    for bm in (64, 128, 256):
        for bn in (64, 128):
            if M % bm or N % bn:
                continue
            tiles = M // bm * (N // bn)
            for S in range(1, max(1, min(16, K // 128, CUS // tiles)) + 1):
                t = 4 + -(-tiles * S // CUS) * -(-(K // 64) // S) * (bm + bn) * 128 / 45e3 + _slab_us(S, M, N, defer)
                cost = (max(t, 2e-6 * N * K / 5.8), t)
                if best is None or cost < best[0]:
                    best = cost, (bm, bn, S, 4 if bm + bn <= 320 else 3)
    return best[0][0], best[1]


def _decode_plan(M: int, N: int, K: int, defer: bool):
    """_decode_tiles' plan, or None for gemm_mid, whose loop is a little faster but starts later (256 rows of
    8192 x 8192: 42 us against 46 and, in 256 x 64 tiles, 61)."""
    cost, plan = _decode_tiles(M, N, K, defer)
    S = mid_plan(M, N, K, defer)
    return None if S is not None and _mid_cost(M, N, K, S, defer) < cost else plan


def _vocab_plan(M: int, N: int, K: int):
    """Decode-bucket vocabulary projection: one row tile of all rows against 128-column tiles, so that the weights
    are read once (256 rows of 32768 x 4096: 73 us, 102 on 64 columns; 128 rows 59 and 62). A 128256-row
    vocabulary at 256 rows is the tile kernel's (253 us against 289), one of 8192 columns too past 64 rows (128 rows 418 against
    447, 256 rows 449 against 617; 64 rows 374 against 334, on tiles whose K steps go round: more columns that are no multiple of 2048 stay); rows that are not one tile would read the weights again. Both lines lie between
    sizes that were timed: 32000 to 152064 rows of 2048 to 8192 columns, 64 to 256 rows, none of them slower than on 64 columns
    (152064 x 3584: 64 rows 192 us against 223, 256 rows 306 against 430; profiles/plans_before_after.txt)."""
    if row_tile(M) != M or (K >= 8192 and (M > 64 or K % 2048)) or (M == 256 and N >= 2 * LM_HEAD_MIN_N) or N % 128:
        return None
    return (M, 128, 1, 3)


@functools.lru_cache(maxsize=4096)
def vocab_rows_plan(M: int, N: int, K: int):
    """gemm_decode's plan for the vocabulary of 9 to 127 rows (as many prompts' first tokens), or None: a part of the one row tile that a decode bucket
    has, whose K steps start apart. It streams the weights at 5.2 to 6.4 TB/s, gemm_mid's and gemm_skinny's tiles at 4.1 to 5.3 (9 to 63 rows, us): 128256 x 4096
    222 to 232 and 175, x 2048 118 to 123 and 101, x 8192 370 and 333, 152064 x 3584 207 to 216 and 198, 32768 x 4096 71 to 75 and 43, 32000 x 2048 30 to 37 and
    25. Fewer columns leave CUs without a tile (16128 x 4096 31 and 39). Of 65 to 127 rows a vocabulary of one or two rounds gains (32768 x
    4096 76 to 83 and 56, 32000 x 2048 38 and 32), a larger one does not (128256 x 2048 123 to 131 and 127, 152064 x 3584 216 to 233 and 245)."""
    if not ROWS_MAX_M < M < 128 or M == 64 or 10 * (N // 128) < 9 * CUS or N % 128 or K % 64 or (M > 64 and N >= 2 * LM_HEAD_MIN_N):
        return None
    plan = gemm_plan(64 if M < 64 else 128, N, K, False)
    return plan if plan is not None and plan[0] >= M and plan[2] == 1 else None


SKINNY_MAX_M = 32
F32_ROWS_MAX_M = 16


def skinny_plan(M: int, N: int, K: int) -> int | None:
    """Split-K count for the gfx950 gemm_skinny kernel (M <= 32 decode buckets; products that rows_plan takes have its slices), or
    None for hipBLASLt: tuned table entry ``skinny,M,N,K`` if present, else split K until
    the 16-row tiles give >= 512 blocks (K permitting)."""
    if M > SKINNY_MAX_M or N % 16 or K % 128 or os.environ.get("OAMD_SKINNY", "1") == "0":
        return None
    t = _gemm_table_get().get(("skinny", M, N, K))
    if t == "blas":
        return None
    if t is not None:
        return int(t)
    S = 1
    while (N // 16) * S < 512 and S < 8 and K % (128 * S * 2) == 0:
        S *= 2
    return S


ROWS_MAX_M = 8


def _skinny_rounds_full(N: int, K: int, glu: bool) -> bool:
    """Where gemm_skinny is faster than gemm_rows for five to eight short rows: in one slice, and its last round of 8192 rows of W is full or nearly
    (8 rows on gemm_rows and on gemm_skinny, us: 16384 x 1536 15.5 and 14.1, 14464 x 1536 14.5 and 13.4, 14336 12.9 and 13.2, 24448 21.2 and 19.9; 7168 x
    1536 gated 8.3 and 8.1, in two slices of gemm_skinny 8.1 and 10.1; 16256 x 2304 21.1 and 19.4, 14464 19.5 and 18.9, 20480 25.5 and 25.6; 16256 x 2176
    gated 22.0 and 18.9; 8192 x 2048 9.5 and 9.2, 16256 15.6 and 15.9; 16384 x 1792 15.9 and 16.5, x 2560 22.0 and 23.6. At 1664 columns it is one of 5 and 6 gated
    rows, 16256 5 %; at 2432 one of 8064 and 16256 rows of W, 6 %, not of 14464 and 24448. Gated 5 rows of 98304 x 1536 73.7 and 67.8)."""
    lacks = -N % 8192
    if not (glu or N >= 8192 or K % 256):   # gemm_skinny in slices
        return False
    if K <= 1536 or 2048 < K < 2432 or (K == 2048 and N <= 8192) or (K == 1664 and glu and N > 8192):
        full = lacks < 2048
    else:
        full = (K == 1664 or 2048 < K < 2560) and lacks < (256 if K > 2048 and N <= 16384 else 1)
    return full or (glu and K <= 1664 and N > LM_HEAD_MIN_N)


def _rows_in_step(N: int, K: int, B: int, glu: bool) -> bool:
    """Whether gemm_rows' workgroups start at rows of W that are served from the same memory channels: 512 KiB or 1 MiB apart but for a 128th (of gate | up
    a 64th). One row on 256 workgroups and on 768, us: 16256 x 4096 (63.5 rows, 508 KiB) 31.0 and 23.4, 16512 31.9 and 23.5, 16384 21.9 and 23.2, 16224 24.8 and 23.1; 8128 x
    8192 (508) 31.5 and 23.0, 11008 x 6144 (516) 31.5 and 22.4, 18864 x 3584 (516) 31.6 and 23.0; 9440 x 14336 (1032) 54.8 and 43.6; gated 16128 x 8192 (1008) 63.3
    and 42.4, 16640 x 4096 (520) 26.4 and 23.5."""
    apart = 2 * K * N / (B << 19)
    return any(abs(abs(apart / m - 1) - (2 if glu else 1) / 128) < 0.35 / 128 for m in (1, 2))


@functools.lru_cache(maxsize=4096)
def rows_plan(M: int, N: int, K: int, glu: bool = False) -> tuple[int, int] | None:
    """(K slices, workgroups) of one to eight rows on the row-streaming kernel (gemm_rows.hip), or None for gemm_skinny: shorter rows, which
    leave lanes idle, and products of a few us, where the sums over lanes weigh (M > 4: 2048 x 2048 5.1 us against 4.8, 4096 x 4096 9.0 and 9.7;
    else 1072 x 2048 3.8 and 3.6, 2048 x 1536 3.7 and 4.3).

    One slice where the rows of X fit in registers. One workgroup per CU for most products (4096 x 14336 19.4 us, 20.6 on two per CU, 22.1 on
    four), three or four, whichever comes out more even, for those that take 30 us (28672 x 4096 gated 37.1 on one, 36.2 on four); rows of
    up to 2048 columns in one pass of eight rows a workgroup (32000 x 2048 22.3 on one per CU, 20.4 so), but not on one and a half per CU (3072 x
    2048: 384 workgroups 4.6, 192 of sixteen rows 4.4).

    Five rows and more keep the vector units busy a whole piece of 2048 columns (512 a wave) at a time, so that short rows that leave one part empty are no
    longer bound by the stream (weights that no cache holds, 8 rows): vocabularies of 128256 x 1536 96 us and 72 on gemm_mid, x 2304 129 and 101,
    61440 x 2560 63 and 57, but 34432 x 2560 40 and 44, 128256 x 2048 102 and 112, x 3072 137 and 135; and where gemm_skinny's tiles come in full
    rounds (_skinny_rounds_full)."""
    if M > ROWS_MAX_M or K % 128 or K < 1536 or N % (128 if glu else 16) or N * K < (2.5e6 if M <= 4 else 8.5e6):
        return None
    if M > 4 and not glu and K < 2816 and K % 2048 and (K <= 2304 or N >= 48 << 10) and _mid_beats_skinny(M, N, K, False):
        return None
    if M > 4 and _skinny_rounds_full(N, K, glu):
        return None
    mt = 1 << (M - 1).bit_length()
    pieces = lambda s: -(-K // (2048 * s))  # noqa: E731 -- 512 columns a wave and piece
    S = next((s for s in ((1,) if glu else (1, 2, 4, 8)) if K % (128 * s) == 0 and pieces(s) <= 8 and mt * pieces(s) <= 32), None)
    if S is None:
        return None
    units = N // 2 if glu else N
    if pieces(S) == 1:
        B = N // 8 if N // 8 <= CUS or N // 8 >= 2 * CUS else N // 16
    else:
        counts = (CUS, 3 * CUS) if N * K < 9e7 or units < 48 * CUS else sorted((3 * CUS, 4 * CUS), key=lambda b: (-(-units // b) * b, -b))
        B = next((b for b in counts if not _rows_in_step(N, K, b, glu)), counts[0])
    while (-(-units // B) * (2 if glu else 1) + 8) * mt * 64 > 48 << 10:   # the workgroup's sums in LDS
        B *= 2
    return S, B


def _norm_blocks(M: int, N: int, K: int, glu: bool) -> int | None:
    """Workgroups of a product of gemm_rows that normalises its rows itself, or None where rmsnorm in front of it is faster. Every workgroup does it
    again, so many small ones are for a row or two only (us with rmsnorm and without: 28672 x 4096 gated of one row on 1024 41.0 and 38.2, of four 40.5
    and 40.7), none at all for short rows (16384 x 2048 gated, one row: 2048 workgroups 15.0 and 16.4, 256 14.3; 151936 x 1536 on 1024 71.8 and
    73.0), one per CU for up to four rows (6144 x 4096: 13.4 and 10.7, four rows 14.1 and 13.1). Eight pieces of rows (a power of
    two) and 512 columns are what a wave's registers hold."""
    plan = rows_plan(M, N, K, glu) if M <= 4 else None
    if plan is None or plan[0] != 1 or (1 << (M - 1).bit_length()) * -(-K // 2048) > 8:
        return None
    if skinny_plan(M, N, K) is None or (_gemm_table_get().get(("silu", M, N, K)) == "blas" if glu else _measured_blas(M, N, K)):
        return None   # hipBLASLt's, by OAMD_SKINNY=0 or a measured entry
    B = plan[1] if plan[1] <= 4 * CUS else CUS
    return None if (B < plan[1] and N * K >= 5e7) or (M > 2 and plan[1] > CUS) or (-(-(N // 2 if glu else N) // B) * (2 if glu else 1) + 8) * (1 << (M - 1).bit_length()) * 64 > 48 << 10 else B


def _mid_beats_skinny(M: int, N: int, K: int, defer: bool) -> bool:
    """gemm_skinny streams the weights once per call but pays for every row (a 128256 x 4096 vocabulary: 191 us at
    1 row, 222 at 8, 300 at 32; 4096 x 14336 26, 27 and 38: 2 % of the one-row time per row, 4 where its tiles do not come in
    whole rounds, which is what the estimate takes); gemm_mid's 128-row tile costs the same at any of them (217 us; 25).
    A few rows of a projection stay: the consumer of up to 16 slabs waits longer than is gained (16 rows of 4096 x 14336: 30
    against 25 before the slabs are read). So do shapes with a measured entry.

    Few rows stream the weights at 5.3 to 5.8 TB/s, rows of 2048 or 4096 columns (a power of two: neighbouring rows
    share memory channels) at 4.1 to 4.8: vocabularies of 32768 x 4096, 5 rows 55 us against 66, of 128256 x 3072 176
    against 135. A consumer that sums up to 16 slabs of a few rows waits for them in turn, 2 us (5): 24 rows of
    2560 x 2048 with the norm behind them 11.5 us against 13.8, 17 of 4096 x 4096 16.1 against 17.9."""
    if M <= (4 if N >= LM_HEAD_MIN_N else 16) or ("skinny", M, N, K) in _gemm_table_get():
        return False
    return _mid_few_rows(M, N, K, defer)


@functools.lru_cache(maxsize=4096)
def _mid_few_rows(M: int, N: int, K: int, defer: bool) -> bool:
    """The estimates of _mid_beats_skinny."""
    S = mid_plan(M, N, K, defer)
    if S is None:
        return False
    shared = K & (K - 1) == 0 and K <= 4096
    mid = _mid_cost(M, N, K, S, defer)
    if N >= LM_HEAD_MIN_N:
        mid = max(mid, 6 + 2e-6 * N * K / (4.2 if shared else 5.2))
    elif defer and S > 1:
        mid += 5 if shared else 2
    return mid < (3 + 2e-6 * N * K / 5.4) * (1 + 0.04 * M)


# Every GPU GEMM of the model runs on the hand-written gfx950 kernels: prompts on gemm_mid or gemm_tile (csrc/kernels/gemm_tile.hip),
# whichever has the tiles that fit (tile_rows, prompt_tile), in K slices (mid_plan) on gemm_mid, decode buckets on
# gemm_pp / gemm_tn / gemm_mid / gemm_skinny / gemm_rows, the lm_head on whichever of them its rows call for (_mid_beats_skinny,
# _vocab_plan, mid_plan), fp8 on gemm_fp8 and, past 64 rows, gemm_fp8_tile, fp32 on gemm_f32 in one of its two forms (f32_split_slices). hipBLASLt is reached
# only by shapes none of them takes (K % 64 != 0, N % 16 != 0, non-bf16), counted in BLAS_CALLS.
# OAMD_PREFILL_BLAS=1 routes the plain prefill projections (QKV, O, down) to hipBLASLt instead, for
# A/B runs against the vendor library (profiles/gemm_tile_p5_vs_hipblaslt_r6.jsonl).
PREFILL_BLAS = os.environ.get("OAMD_PREFILL_BLAS", "0") == "1"
BLAS_CALLS = {"n": 0}   # GPU GEMMs that FELL BACK to hipBLASLt (tests assert it stays 0 on model shapes)
BLAS_PLANNED = {"n": 0}   # plain prefill projections run on hipBLASLt by design (PREFILL_BLAS)


def _blas(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None, bias: torch.Tensor | None,
          planned: bool = False):
    if x.is_cuda and planned:
        BLAS_PLANNED["n"] += 1
    elif x.is_cuda:
        BLAS_CALLS["n"] += 1
        if os.environ.get("OAMD_FORBID_BLAS") == "1":
            raise RuntimeError(f"hipBLASLt fallback for x {tuple(x.shape)} {x.dtype}, w {tuple(w.shape)} "
                               "(OAMD_FORBID_BLAS=1)")
    if out is not None:
        return F.linear(x, w, bias, out=out) if bias is None else out.copy_(F.linear(x, w, bias))
    return F.linear(x, w, bias)


def tile_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Shapes the 256x256-tile gfx950 GEMM (gemm_tile) takes: bf16, K % 64, N % 16."""
    return (x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2
            and x.is_contiguous() and w.is_contiguous() and x.shape[1] % 64 == 0 and w.shape[0] % 16 == 0
            and x.shape[0] >= 1)


def tile_out_ok(out: torch.Tensor | None) -> bool:
    """An explicit output gemm_tile can write: unit column stride, a row stride that is a
    multiple of 4 elements and an 8-byte-aligned base (its epilogue stores 4 bf16 at once);
    anything else falls back instead of tripping the binding's TORCH_CHECK."""
    return out is None or (out.dim() == 2 and out.stride(1) == 1 and out.stride(0) % 4 == 0
                           and out.data_ptr() % 8 == 0 and out.dtype == torch.bfloat16)


# Costs, in us, of the two bf16 tile kernels on one MI355X with weights that stream from HBM (measured on
# 48 to 6144 rows of 2048 to 28672 x 2048 to 14336 weights): a step is one 64-column piece of K on every
# busy CU, dearer with the whole chip busy (clock, L2) and where no two workgroups share a weight panel. The plans are for
# the whole card's CUs; on a part of one the kernels' grids adapt, and the plans cost speed only.
CUS = 256


def _tile_cost(M: int, N: int, K: int) -> float:
    """gemm_tile: 256 x 256 tiles over the whole K, one workgroup per CU."""
    units = -(-M // 256) * -(-N // 256)
    return max(3 + -(-units // CUS) * (K // 64) * (1.25 + 0.2 * min(1.0, units / CUS)), 2e-6 * N * K / 4.6)


def _mid_cost(M: int, N: int, K: int, S: int, defer: bool) -> float:
    """gemm_mid: 128 x 256 tiles, K in S slices whose slabs are written, then read by a reduce pass or (``defer``) by
    the consumer."""
    mt = -(-M // 128)
    units = mt * -(-N // 256) * S
    rounds = -(-units // CUS)
    step = 0.7 + (0.15 if M > 256 else 0.3) * min(1.0, units / CUS)   # few rows: the weights come from HBM
    t = (4 if M > 256 else 6) + rounds * -(-(K // 64) // S) * step + 3 * (rounds - 1)   # a tile's stores between rounds
    return max(t + _slab_us(S, M, N, defer), 2e-6 * N * K / 4.9)


@functools.lru_cache(maxsize=4096)
def mid_plan(M: int, N: int, K: int, defer: bool, slices: bool = True, prompt: bool = False) -> int | None:
    """K slices for gemm_mid (1: none), or None where the 256-row tiles are cheaper. One prompt of a few hundred
    tokens has fewer 256-row tiles than the GPU has CUs: smaller tiles and K slices fill it (885 rows: 4096 x 14336
    103 us against 297, 6144 x 4096 56 against 89); once every CU has a 256-row tile, that tile's fewer operand
    bytes per product win (4096 rows of 4096 x 14336: 325 us against 371).

    Above 256 rows, and from 33 rows of a ``prompt`` on, the plan is the next multiple of 512's: a prefill graph pads its
    batch to such a size, and a prompt's numbers are the same padded or not (100 rows of 4096 x 14336 with the norm behind them: 58 us in the four slices of 512 rows, 36 in fourteen, 285 on
    the 256-row tiles). From LM_HEAD_MIN_N features on, where 512 rows run on the 256-row tiles, a prompt is not sliced. Past
    4096 rows the graphs' sizes are coarser and little is left to gain. Prompts of up to 32, and of 64, 128, 192 or 256
    rows run on a decode kernel when they are not padded."""
    prompt = prompt and M > SKINNY_MAX_M
    if M > 256 or (prompt and N < LM_HEAD_MIN_N):
        M = -(-M // 512) * 512
    if M < 1 or M > 4096 or K < 128 or (M > 128 and N >= LM_HEAD_MIN_N):   # 256 rows of a vocabulary: 282 us against 253
        return None
    tiles = -(-M // 128) * -(-N // 256)
    most = 1 if not slices or (prompt and N >= LM_HEAD_MIN_N) else min(16, K // 128, 2 * CUS // tiles)
    cost, S = min((_mid_cost(M, N, K, s, defer), s) for s in range(1, max(1, most) + 1))
    return S if cost < _tile_cost(M, N, K) else None


# us of a 64-column piece of K on a CU, and what it takes more with every CU busy (power, L2): gemm_mid's tiles of 96, 128
# and 160 rows, gemm_tile's of 192, 224 and 256 (fitted to those products)
_ROW_STEP = {96: (0.68, 0.02), 128: (0.70, 0.14), 160: (0.68, 0.32), 192: (0.78, 0.40), 224: (0.90, 0.44), 256: (1.03, 0.48)}


def _rows_us(rows: int, M: int, N: int, K: int, S: int) -> float:
    units = -(-M // rows) * -(-N // 256) * S
    full, last = divmod(units, CUS)
    one, busy = _ROW_STEP[rows]
    rounds = full * (one + busy) + (one + busy * last / CUS if last else 0)
    return -(-(K // 64) // S) * rounds + 5 + 3 * ((units - 1) // CUS)   # a tile's stores between rounds


@functools.lru_cache(maxsize=4096)
def tile_rows(M: int, N: int, K: int, S: int = 1) -> int:
    """Rows of the tiles (256 columns wide) of a prompt's product in S slices of K: 96, 128 or 160 (gemm_mid) or, in one
    slice, 192, 224 or 256 (gemm_tile). All sum a K slice in the same order, so the bits are the same and the rows are free: those whose
    rounds of one workgroup per CU take least. Fewer rows fill the CUs (885 rows of 6144 x 4096: 168 tiles of
    128 rows 55 us, 240 of 96 49), more rows save a round (300 rows of 28672 x 4096: 336 tiles of 128 rows 110 us, 224 of 160 68,
    224 of 256 95; 1500 rows of 6144 x 4096: 93, 62 and 90; 885 rows of 28672 x 4096: 196 us on 160 rows, 182 on 224, 199 on 256;
    380 rows of it 120 on 128, 82 on 192, 106 on 256) and per product take in fewer bytes (4096 rows of 4096 x
    14336: 362, 421 and 317). Over 506 products of 27 shapes, 129 to 28208 rows, the estimate's choices take 0.3 % more than
    the best ones. Up to 128 rows are one tile."""
    if M <= 128:
        return 128
    return min((_rows_us(r, M, N, K, S), r) for r in ((96, 128, 160) if S > 1 else _ROW_STEP))[1]


# us of a prompt's tiles by (rows, columns): to start and to store, a 64-column piece of K on a CU, what it takes more with every CU busy, between
# rounds. Fitted to 504 products of 25 shapes, 33 to 2000 rows, in their plans' slices, weights from HBM; 192 to 256 rows by 128 columns to 266 of 14, 140 to
# 3000 rows, and 1 us to start added, without which two products of some 20 us were 2 and 5 % slower
_MID_US = {(64, 64): (4.13, 0.186, 0.078, 0.4), (128, 64): (4.55, 0.221, 0.158, 1.2), (64, 128): (4.8, 0.376, 0.049, 0.4),
           (96, 128): (5.64, 0.404, 0.048, 1.3), (128, 128): (5.64, 0.404, 0.175, 2.4), (160, 128): (7.22, 0.439, 0.111, 3.1),
           (192, 128): (7.51, 0.463, 0.210, 3.0), (224, 128): (7.82, 0.469, 0.291, 2.0), (256, 128): (8.41, 0.482, 0.353, 2.4),
           (64, 256): (4.75, 0.684, 0.060, 1.4), (96, 256): (6.46, 0.679, 0.106, 2.0), (128, 256): (7.07, 0.697, 0.210, 2.3),
           (160, 256): (9.97, 0.683, 0.211, 6.2), (192, 256): (10.32, 0.696, 0.317, 10.5), (224, 256): (11.09, 0.789, 0.363, 12.0),
           (256, 256): (11.87, 0.899, 0.394, 12.0)}
NARROW_MAX_M = 4096


def _mid_us(rows: int, cols: int, M: int, N: int, K: int, S: int) -> float:
    start, one, busy, between = _MID_US[rows, cols]
    units = -(-M // rows) * -(-N // cols) * S
    full, last = divmod(units, CUS)
    rounds = full * (one + busy) + (one + busy * last / CUS if last else 0)
    return start + -(-(K // 64) // S) * rounds + between * ((units - 1) // CUS)


@functools.lru_cache(maxsize=4096)
def prompt_tile(M: int, N: int, K: int, S: int = 1, glu: int = 0) -> tuple[int, int]:
    """(rows, columns) of the tiles of a prompt's product in S slices of K: tile_rows' by 256 columns, or gemm_mid's of 64 or 128 columns
    where those are estimated 7 % faster. Few rows in few slices leave most CUs without a tile of 256 columns (100 rows, us: 6144 x 4096 in two
    slices 48 workgroups 31, 192 of 128 x 64 18; 4096 x 14336 in four 64 workgroups 55, 256 29; 28672 x 4096 gated 112 workgroups 65, 224 of 128 x 128
    56; 40 rows of 16384 x 2048 gated 27 and, in 64 x 128 tiles, 20); 200 rows of 4096 x 14336 48 on 96 x 256, 37 on 160 x 128. The sums, and so the bits, are
    the same for all. 333 of those 504 products take narrow tiles, 0.68 of the time of the others on average, and 16 of 84 more of 1600 to 3800 rows (2300 of
    2048 x 8192 89 us on 96 x 256, 70 on 160 x 128); none was slower. Tiles of 192 to 256 rows by 128 columns take in the fewest bytes for what they compute where the wide
    ones' rounds do not come out: 43 of 266 more have them, 2 to 16 % faster (885 rows of 4096 x 14336 101 us on 128 x 256, 96 on 224 x 128; 1200 of 4608 x 3584 47
    and, on 192 x 128, 40), none slower by more than the 1.5 % that two runs differ by. A gated product's
    narrowest tile is the 128 rows of W that hold 64 gates and what they multiply."""
    first = tile_rows(M, N, K, S), 256
    if M > NARROW_MAX_M:
        return first
    us, tile = min((_mid_us(*t, M, N, K, S), t) for t in _MID_US
                   if (t[1] < 256 or t[0] == 64) and (t[1] > 64 or not glu or S > 1))
    return tile if us < 0.93 * _mid_us(*first, M, N, K, S) else first


def loose_tiles(M: int, N: int, K: int) -> bool:
    """One row tile of a vocabulary whose rows are a power of two apart: gemm_tile's schedule of a workgroup per tile (h4), whose workgroups
    drift apart. In the persistent one all CUs walk their weight rows in step, and rows 8 or 16 KiB apart share memory channels:
    128256 x 4096 253 us against 290 at 256 rows (285 and 293 within a decode step), 258 and 272 at 192, 258 and 259 at 129; 128256 x 8192 485 and 506 at 256, but 471 and
    450 at 192. Rows of 3072 or 3584 columns (152064 x 3584: 319 and 304) and vocabularies of one round (32768 x 4096: 106 and 95) are not
    slowed. The bits are the same."""
    return (128 if K == 4096 else 208) < M <= 256 and N > 256 * CUS and K >= 4096 and K & (K - 1) == 0


def linear_tile(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None,
                bias: torch.Tensor | None = None, glu: int = 0, defer_reduce: bool = False, prompt: bool = False):
    """Prefill / lm_head GEMM on the compute-bound gfx950 tile kernels (fused bias or gated (``glu``: SILU /
    GELU_TANH) epilogue): tiles of 96 to 256 rows (``tile_rows``), of few rows of prompts also narrower ones (``prompt_tile``), for few rows with K
    slices (``mid_plan``).
    ``defer_reduce``: K slices come back as fp32 slabs (:class:`SplitK`); ``prompt``: rows a prefill graph may pad."""
    M, K = x.shape
    N = w.shape[0]
    defer = defer_reduce and out is None and not glu
    S, rows, cols = None, 256, 256
    if (out is None or (out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0)) and (
            bias is None or (bias.is_contiguous() and bias.data_ptr() % 16 == 0)):   # gemm_mid's 16-B accesses
        S = mid_plan(M, N, K, defer, out is None or out.stride(0) == out.shape[1], prompt)   # the reduce pass has no row stride
        if 128 <= K < 1 << 22 and M < 1 << 24 and N < 1 << 30:   # gemm_mid's
            rows = 256 if not glu and loose_tiles(M, N, K) else tile_rows(M, N, K, S or 1)
            if prompt and (glu or N < LM_HEAD_MIN_N):
                rows, cols = prompt_tile(M, N, K, S or 1, glu)
    part = torch.empty(S * M * N, dtype=torch.float32, device=x.device) if S is not None and S > 1 else None
    opt = {} if rows == 128 else {"rows": rows}
    if cols != 256:
        opt["cols"] = cols
    if part is not None and defer:
        kernels().gemm_mid(x, w, None, bias, part, S, **opt)
        return SplitK(part, S, M, N)
    y = out if out is not None else torch.empty(M, N // 2 if glu else N, dtype=x.dtype, device=x.device)
    if rows < 192 or cols < 256:
        kernels().gemm_mid(x, w, y, bias, part, S or 1, glu, **opt)
    else:
        kernels().gemm_tile(x, w, y, bias, glu, 1 if not glu and loose_tiles(M, N, K) else 0, rows=rows)
    return y


def f32_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Shapes the fp32 GEMM (gemm_f32) takes."""
    return (x.dtype == torch.float32 and w.dtype == torch.float32 and x.dim() == 2 and x.is_contiguous()
            and w.is_contiguous() and x.shape[1] % 16 == 0)


def f32_plan_rows(M: int, prompt: bool) -> int:
    """Rows whose K slices an fp32 product takes: a prompt's are those of its padded prefill graph (see mid_plan), so its
    numbers are the same padded or not; up to 32 rows have plans of their own."""
    return -(-M // 512) * 512 if prompt and M > SKINNY_MAX_M else M


# us, fitted to 4300 products of 17 to 3000 rows of 16 shapes on one MI355X (rms 5 %). The split kernel's tiles of 64 rows, one and two to a CU, of
# 128 and of 256: a 32-column step with one CU busy, and what it takes more with all of them (power); then the fp32 instruction's, with one, two
# and three tiles to a CU.
_F32_SPLIT = {64: (0.69, 0.14), 128: (0.94, 0.40), 256: (1.76, 0.56)}
_F32_PAIR = 1.37   # two 64-row tiles
_F32_PLAIN = (0.66, 1.16, 1.70)


def _f32_slabs(M: int, N: int, S: int, glu: int) -> float:
    return 2.2 + 1.3e-6 * M * N * (S + (0.5 if glu else 1)) if S > 1 else 0.0


def _f32_split_us(rows: int, S: int, M: int, N: int, K: int, glu: int) -> float:
    one, busy = _F32_SPLIT[rows]
    full, last = divmod(-(-M // rows) * -(-N // 128) * S, 2 * CUS if rows == 64 else CUS)
    t = full * (_F32_PAIR if rows == 64 else one + busy)
    if last:
        t += _F32_PAIR if last > CUS else one + busy * last / CUS
    t = 6 + -(-K // (32 * S)) * t + 1.1 * (full + (last > 0) - 1)
    return max(t, 6 + 4e-6 * N * K / 4.5) + _f32_slabs(M, N, S, glu)


def _f32_plain_us(M: int, N: int, K: int, glu: int, S: int) -> float:
    full, last = divmod(-(-(-(-M // 64) * -(-(N // 2 if glu else N) // 64) * S) // CUS), 3)
    t = 3.2 + -(-K // (32 * S)) * (2 if glu else 1) * (full * _F32_PLAIN[2] + (_F32_PLAIN[last - 1] if last else 0))
    return max(t, 3.2 + 4e-6 * N * K / 4) + _f32_slabs(M, N, S, glu)


@functools.lru_cache(maxsize=4096)
def f32_split_slices(M: int, N: int, K: int, glu: int) -> int | None:
    """K slices in which ``M`` rows (f32_plan_rows) run on the split kernel (gemm_f32_split.hip), or None: on the fp32 matrix instruction
    (f32.hip), on its few-row kernel (up to 16 rows, 32 of less than 2048 columns) and where the split kernel, whose steps wait for more before the first, is not
    estimated 10 % faster (32 rows of 28672 x 4096 gated 161 us, 127 split, of 32000 x 2048 92 and 69, of 4096 x 14336 78 and 67; 512 rows of 2048 x 288 9 us against 14, of 2048 x 768 24 and 24, of 2048 x 2048 50 and 37; 2000 rows of 2048 x 288 27 and 20). No fewer slices than
    the fp32 instruction would have: sums that are as long are closer to the 64-bit result (0.86 of its distance), but one slice in the place of four is
    further off (3200 x 1376 gated 1.8 times).

    A prompt's rows are padded to a multiple of 512 for its plan, but run as they are: slices count that are no slower at the fewest rows of that
    plan either (33 rows of 6144 x 2048 in one slice 56 us against 46, in two 33; of 2912 x 560 19 and 11 whatever the slices)."""
    if M <= F32_ROWS_MAX_M or (M <= SKINNY_MAX_M and K < 2048):   # gemm_f32's few-row kernel
        return None
    former = kernels().gemm_f32_splits(M, N, K, glu)
    few = M if M % 512 else max(M - 511, SKINNY_MAX_M + 1)
    us = lambda m, s: min(_f32_split_us(r, s, m, N, K, glu) for r in _F32_SPLIT)  # noqa: E731
    limit = _f32_plain_us(few, N, K, glu, former)
    cost, S = min(((us(M, s), s) for s in range(former, 9) if (s == 1 or (N % 4 == 0 and K // 32 // s >= 4)) and us(few, s) <= limit),
                  default=(float("inf"), 1))
    return S if cost < 0.9 * _f32_plain_us(M, N, K, glu, former) else None


@functools.lru_cache(maxsize=4096)
def f32_split_rows(M: int, N: int, K: int, S: int, glu: int) -> int:
    """Rows of the split kernel's tiles: the sums, and so the bits, are the same for all (the choices take 0.5 % more than the best slices and
    rows of 318 products)."""
    return min((_f32_split_us(r, S, M, N, K, glu), r) for r in _F32_SPLIT)[1]


@functools.lru_cache(maxsize=4096)
def f32_rows_plan(M: int, N: int, K: int, glu: int) -> tuple[int, int] | None:
    """(K slices, workgroups of a slice) in which one to sixteen fp32 rows run on the row-streaming kernel (gemm_f32_rows.hip), or None for gemm_f32: rows too
    long for its registers, and those under 768 columns (1024 of nine rows and more), which leave it idle lanes and little to stream (one and eight rows, us, here
    and on gemm_f32: 2048 x 768 4.9, 5.1 and 5.2, 5.6; 4096 x 512 5.1, 5.8 and 4.6, 4.7; sixteen: 2048 x 768 6.2 and 6.0).

    Up to eight rows one workgroup per CU up to 3e7 weights (2048 x 8192 13.3 us, 15.0 on three, 6144 x 4096 18.6 and 19.4), three past that (28672 x 4096
    gated 76 and 72, 32000 x 2048 of eight rows 46 on two, 45 on three), and where one per CU starts at rows of the same memory channels (_rows_in_step: 8128
    x 4096 32.3 and 22.6, 16256 x 2048 32.2 and 24.0). Nine to sixteen keep the vector units busy: slices of up to 2048 columns, whose X four waves hold, on one
    workgroup per CU or, past 2e7 weights and in slices, two, which is what a CU has room for (sixteen, us: 16384 x 2048 gated 33, 40 on three and 41 on gemm_f32;
    2048 x 8192 in four slices 23 and 37; 2048 x 2048 8.3 and 10.8; 3072 x 2048 10.2, 12.5 on two and 12.4; 32000 x 2048 63 and 77; 28672 x 4096
    gated, of eight waves, 156 and 133)."""
    if not 1 <= M <= F32_ROWS_MAX_M or K % 16 or K < (768 if M <= ROWS_MAX_M else 1024) or N * K < 5e5 or (glu and N % 128):
        return None
    S = 1 if M <= ROWS_MAX_M else -(-K // 2048)
    if K % (16 * S) or S > 8 or (S > 1 and (glu or N % 4)):
        return None
    waves = kernels().f32_rows_waves(M, K // S)
    if not waves or (M > ROWS_MAX_M and waves > 4):
        return None
    if M > ROWS_MAX_M:
        B = CUS if S == 1 and N * K < 2e7 else 2 * CUS // S
    else:
        counts = (CUS, 3 * CUS) if N * K < 3e7 else (3 * CUS, 4 * CUS)
        B = next((b for b in counts if not _rows_in_step(N, 2 * K, b, bool(glu))), counts[0])
    lds = 16 * waves << (M - 1).bit_length()   # bytes of a row's sums
    while (-(-(N // 2 if glu else N) // B) * (2 if glu else 1) + 8) * lds > 48 << 10:
        B *= 2
    return S, B


def linear_f32(x: torch.Tensor, w: torch.Tensor, glu: int = 0, prompt: bool = False) -> torch.Tensor:
    """x @ w^T with 32-bit operands and sums, optionally with the gated epilogue (SILU / GELU_TANH) over a 64-row
    interleaved gate|up weight. ``prompt``: as for ``linear``."""
    M, K = x.shape
    N = w.shape[0]
    y = torch.empty(M, N // 2 if glu else N, dtype=x.dtype, device=x.device)
    if (rows := f32_rows_plan(M, N, K, glu)) is not None:
        S, blocks = rows
        part = torch.empty(S * M * N, dtype=torch.float32, device=x.device) if S > 1 else None
        kernels().gemm_f32(x, w, y, glu, partial=part, splits=S, blocks=blocks)
        return y
    plan = f32_plan_rows(M, prompt)
    S = f32_split_slices(plan, N, K, glu) if M else None
    rows = 0 if S is None else f32_split_rows(M, N, K, S, glu)
    if S is None:
        S = kernels().gemm_f32_splits(plan, N, K, glu)
    part = torch.empty(S * M * N, dtype=torch.float32, device=x.device) if S > 1 else None
    kernels().gemm_f32(x, w, y, glu, partial=part, splits=S, rows=rows)
    return y


def linear(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor | None = None, splits: int | None = None,
           partial: torch.Tensor | None = None, bn: int | None = None, bm: int | None = None,
           defer_reduce: bool = False, stages: int | None = None, bias: torch.Tensor | None = None, prompt: bool = False):
    """y = x @ w^T (+ bias) in bf16 on the gfx950 kernels: up to 8 rows on gemm_rows (rows_plan), up to 32 on gemm_skinny, or on
    gemm_mid where the rows cost more than its tile (_mid_beats_skinny); 64, 128, 192 and 256 rows on the LDS-staged
    split-K gemm_decode (the measured table, else _decode_tiles; vocabularies _vocab_plan, of 9 to 127 rows vocab_rows_plan) or where it is estimated
    faster gemm_mid; everything else (prompts, the lm_head of many of them, biased projections) on gemm_mid's tiles of 96 to 160 rows,
    with K slices where mid_plan has them, or gemm_tile's of 192 to 256 (tile_rows). ``defer_reduce``: K
    slices come back as fp32 slabs (:class:`SplitK`). fp32 operands: linear_f32. hipBLASLt only
    for shapes none of them takes (K % 64 != 0, N % 16 != 0, non-bf16), for decode shapes the
    tuned table measured it fastest on, or under OAMD_PREFILL_BLAS=1 (A/B); CPU tensors on torch.
    ``prompt``: rows of prompts, which a prefill graph pads (mid_plan)."""
    M, K = x.shape
    N = w.shape[0]
    plan = None
    if isinstance(x, Normed):
        y = torch.empty(M, N, dtype=torch.float32 if defer_reduce else w.dtype, device=w.device)
        x.into(w, *((None, y) if defer_reduce else (y, None)))
        return SplitK(y, 1, M, N) if defer_reduce else y
    if x.is_cuda and bias is None and out is None and f32_ok(x, w):
        return linear_f32(x, w, prompt=prompt)
    if bias is not None:
        if tile_ok(x, w) and tile_out_ok(out):
            return linear_tile(x, w, out, bias, defer_reduce=defer_reduce, prompt=prompt)
        return _blas(x, w, out, bias)
    if x.is_cuda and bm is None and bn is None and splits is None and _measured_blas(M, N, K):
        return _blas(x, w, out, None)
    if PREFILL_BLAS and x.is_cuda and M > 256 and N < LM_HEAD_MIN_N and splits is None and x.dtype == torch.bfloat16:
        return _blas(x, w, out, None, planned=True)
    if (not prompt and out is None and bm is None and bn is None and splits is None and x.is_cuda and x.dtype == w.dtype == torch.bfloat16
            and x.is_contiguous() and w.is_contiguous() and (x.data_ptr() | w.data_ptr()) % 16 == 0 and (part := vocab_rows_plan(M, N, K)) is not None):
        y = torch.empty(M, N, dtype=x.dtype, device=x.device)
        kernels().gemm_decode(x, w, y, None, 1, part[1], part[0], False, False, part[3] if len(part) > 3 else 3)
        return y
    if (x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous() and M <= SKINNY_MAX_M
            and bm is None and bn is None):
        S = splits or skinny_plan(M, N, K)
        rows = rows_plan(M, N, K) if splits is None and S is not None and (out is None or out.is_contiguous()) else None
        if rows is not None:
            deferred = defer_reduce and out is None   # in fp32, of one slice too
            S = rows[0]
            p = torch.empty(S * M * N, dtype=torch.float32, device=x.device) if deferred or S > 1 else None
            y = None if deferred else out if out is not None else torch.empty(M, N, dtype=x.dtype, device=x.device)
            kernels().gemm_skinny(x, w, y, p, S, 0, rows[1])
            return SplitK(p, S, M, N) if deferred else y
        if (S is not None and splits is None and out is None and _mid_beats_skinny(M, N, K, defer_reduce) and tile_ok(x, w)
                and (x.data_ptr() | w.data_ptr()) % 16 == 0):
            return linear_tile(x, w, defer_reduce=defer_reduce)
        if S is not None:
            if S > 1 and (partial is None or partial.numel() < S * M * N):
                partial = torch.empty(S * M * N, dtype=torch.float32, device=x.device)
            if defer_reduce and S > 1 and out is None:
                kernels().gemm_skinny(x, w, None, partial, S, False)
                return SplitK(partial, S, M, N)
            y = out if out is not None else torch.empty(M, N, dtype=x.dtype, device=x.device)
            kernels().gemm_skinny(x, w, y, partial if S > 1 else None, S, False)
            return y
    if x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous() and w.is_contiguous():
        plan = gemm_plan(M, N, K, defer_reduce and out is None)
        if plan is None and (splits or bn or bm) and M % 64 == 0 and M <= 256 and N % 64 == 0 and K % 64 == 0:
            plan = (row_tile(M), 64, 1)  # explicit request (tests / tuning)
    if plan is None:
        if tile_ok(x, w) and tile_out_ok(out):
            return linear_tile(x, w, out, defer_reduce=defer_reduce, prompt=prompt)
        return _blas(x, w, out, None)
    bm, bn, S = bm or plan[0], bn or plan[1], splits or plan[2]
    ns = stages or (plan[3] if len(plan) > 3 else 3)
    if S > 1 and (partial is None or partial.numel() < S * M * N):
        partial = torch.empty(S * M * N, dtype=torch.float32, device=x.device)
    if defer_reduce and S > 1 and out is None:
        kernels().gemm_decode(x, w, None, partial, S, bn, bm, False, False, ns)
        return SplitK(partial, S, M, N)
    y = out if out is not None else torch.empty(M, N, dtype=x.dtype, device=x.device)
    kernels().gemm_decode(x, w, y, partial if S > 1 else None, S, bn, bm, False, False, ns)
    return y


FP8_MAX = 448.0  # OCP e4m3fn


def quantize_fp8(x: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Per-row e4m3fn quantization: (q [M, K] float8_e4m3fn, s [M] fp32), x ~= q * s."""
    M, K = x.shape
    if x.is_cuda and x.dtype == torch.bfloat16 and K % 8 == 0:
        q = torch.empty(M, K, dtype=torch.float8_e4m3fn, device=x.device)
        sx = torch.empty(M, dtype=torch.float32, device=x.device)
        kernels().quantize_fp8(x.contiguous(), q, sx)
        return q, sx
    xf = x.float()
    amax = xf.abs().amax(1)
    sx = torch.where(amax > 0, amax / FP8_MAX, torch.ones_like(amax))
    return (xf / sx[:, None]).to(torch.float8_e4m3fn), sx


def silu_quantize_fp8(gu, block: int | None = GU_BLOCK) -> tuple[torch.Tensor, torch.Tensor]:
    """quantize_fp8(silu_mul(gu, block)) — on the GPU one kernel for 64-feature
    interleaved gate|up rows (the SwiGLU never round-trips HBM as bf16). ``gu`` may be
    the gate|up GEMM's split-K slabs (:class:`SplitK`), summed inside the kernel."""
    M, N2 = gu.shape
    inter = N2 // 2
    if gu.is_cuda and block == GU_BLOCK and inter <= 32768 and N2 % 128 == 0:
        q = torch.empty(M, inter, dtype=torch.float8_e4m3fn, device=gu.device)
        sx = torch.empty(M, dtype=torch.float32, device=gu.device)
        if isinstance(gu, SplitK):
            kernels().silu_quantize_fp8(torch.empty(M, N2, dtype=torch.bfloat16, device=gu.device), q, sx,
                                        gu.p, gu.S)
            return q, sx
        if gu.stride(1) == 1 and (inter <= 16384 or gu.stride(0) % 8 == 0):   # long rows: as silu_mul takes them
            kernels().silu_quantize_fp8(gu, q, sx)
            return q, sx
    if isinstance(gu, SplitK):
        gu = gu.materialize()
    return quantize_fp8(silu_mul(gu, block=block))


def _fp8_overrides() -> dict:
    """OAMD_FP8_PLANS="NxK=bm,bn,S;..." (A/B of fp8 decode plans): (N, K) -> (bm, bn, S)."""
    out = {}
    for item in filter(None, os.environ.get("OAMD_FP8_PLANS", "").split(";")):
        shape, plan = item.split("=")
        n, k = (int(v) for v in shape.split("x"))
        out[(n, k)] = tuple(int(v) for v in plan.split(","))
    return out


_FP8_OVERRIDES = _fp8_overrides()


def _fp8_slices(M: int, N: int, K: int) -> tuple[int, int, int]:
    """(rows, columns, K slices) of an fp8 projection: a power of two of slices until blocks of (64, 128 or 256) rows and
    64 columns (128 of wide N) reach one per CU. Both kernels keep to the slices, whatever the tile: they fix the order
    of a sum, and rows whose rounding to e4m3fn turns on its last bit come out visibly different further on."""
    bm = 64 if M <= 64 else 128 if M <= 128 else 256
    bn = 128 if N % 128 == 0 and N // 128 >= 192 else 64
    S = 1
    for s in (1, 2, 4, 8):
        if K % (128 * s):
            break
        S = s
        if (N // bn) * s * -(-M // bm) >= CUS:
            break
    return bm, bn, S


# Estimates of the two fp8 kernels by tile (rows, columns): us to start and to store, us of a 128-column step on a CU and what it takes more
# with every CU busy, us between rounds, us per million fp32 slab elements. gemm_fp8_tile has the tiles of 256 columns. Fitted to 673 products of
# 25 shapes, 65 to 9000 rows, weights from HBM: the choices take 0.6 % more than the best ones, 3 of them 3 to 7 % more than the fixed steps chosen before
_FP8_US = {(64, 64): (3.5, 0.06, 0.29, 0.4, 0.24), (64, 128): (8.3, 0.26, 0.24, 0.7, 0.20), (128, 64): (4.7, 0.13, 0.39, 1.0, 0.24),
           (128, 128): (9.3, 0.45, 0.15, 5.6, 0.32), (256, 64): (8.5, 0.45, 0.22, 5.7, 0.26), (256, 128): (13.1, 0.73, 0.26, 10.0, 0.19),
           (96, 256): (7.3, 0.71, 0.00, 2.0, 0.34), (128, 256): (7.4, 0.72, 0.06, 3.7, 0.54), (160, 256): (8.6, 0.79, 0.14, 4.3, 0.55)}


def _fp8_us(rows: int, cols: int, M: int, N: int, K: int, S: int) -> float:
    start, one, busy, between, slabs = _FP8_US[rows, cols]
    units = -(-M // rows) * -(-N // cols) * S
    full, last = divmod(units, CUS)
    rounds = full * (one + busy) + (one + busy * last / CUS if last else 0)
    return start + -(-(K // 128) // S) * rounds + between * ((units - 1) // CUS) + (slabs * S * M * N * 1e-6 if S > 1 else 0)


@functools.lru_cache(maxsize=4096)
def _fp8_tiles(M: int, N: int, K: int):
    """(estimate in us, (bm, bn, S)) of gemm_fp8: the fastest tile (128 rows of 10240 x 8192 in 128 x 128
    tiles: one round of 160 workgroups 30 us, two of 128 x 64 35). Up to 64 rows two or three workgroups share a CU and
    the narrow tile stays (1 row: 20.5 against 21.3), of wide N too where the CU with the most of them takes in no more (16 rows of
    40960 x 8192: 640 workgroups 71 us, 320 of 128 columns 82; of 57344 x 8192 896 99, 448 92)."""
    bm, bn, S = _fp8_slices(M, N, K)
    if M <= 64:
        if bn == 128 and -(-(N // 64) * S // CUS) * (64 + 64) <= -(-(N // 128) * S // CUS) * (64 + 128):
            bn = 64
        return 0.0, (bm, bn, S)
    return min(((_fp8_us(r, c, M, N, K, S), (r, c, S)) for r, c in _FP8_US if c < 256 and N % c == 0), default=(float("inf"), (bm, bn, S)))


def fp8_plan(M: int, N: int, K: int) -> tuple[int, int, int]:
    """(bm, bn, splits) for gemm_fp8."""
    return _FP8_OVERRIDES.get((N, K)) or _fp8_tiles(M, N, K)[1]


@functools.lru_cache(maxsize=4096)
def fp8_tile_rows(M: int, N: int, K: int, S: int) -> tuple[float, int]:
    """(estimate in us, rows of the tiles, 256 columns wide) of gemm_fp8_tile: those whose rounds of one workgroup per CU
    take least, as tile_rows (700 rows of 8192 x 8192: 192 tiles of 128 rows 57 us, 256 of 96 48; 1200 rows of 8192 x 28672: 320
    tiles of 128 rows 354 us, 256 of 160 215)."""
    return min((_fp8_us(rows, 256, M, N, K, S), rows) for rows in (96, 128, 160))


def fp8_tile_plan(M: int, N: int, K: int) -> int | None:
    """The slices where gemm_fp8_tile is faster than gemm_fp8, whose bits it gives, else None: 512 rows of
    57344 x 8192 306 -> 218 us, 4096 rows of 8192 x 8192 384 -> 203 (2.7 PFLOP/s), 256 rows of 10240 x 8192 57 -> 33, 700 rows of 3072 x 2048
    16 -> 14; but 128 rows of 4096 x 4096 in 4 slices 13.3, against 10.6, and up to 64 rows the weights' stream is all there is
    (57344 x 8192: 104, against 90)."""
    S = _fp8_slices(M, N, K)[2]
    if M <= 64 or N % 64 or K // 128 // S < 3 or (N, K) in _FP8_OVERRIDES:
        return None
    return S if fp8_tile_rows(M, N, K, S)[0] < _fp8_tiles(M, N, K)[0] else None


def linear_fp8(x: torch.Tensor | tuple[torch.Tensor, torch.Tensor], w8: torch.Tensor, sw: torch.Tensor,
               out: torch.Tensor | None = None, plan: tuple[int, int, int] | None = None,
               defer_reduce: bool = False):
    """y = x @ (w8 * sw)^T with x quantized per token to e4m3fn (W8A8, fp32 accumulate).
    ``x`` may already be quantized: a (q, sx) pair from quantize_fp8 / silu_quantize_fp8.
    ``defer_reduce``: a split-K plan returns its fp32 slabs (:class:`SplitK`) for a
    consumer that sums them (rope_kv, rmsnorm, the fused all-reduce + norm, SwiGLU)."""
    q, sx = x if isinstance(x, tuple) else quantize_fp8(x)
    M, K = q.shape
    N = w8.shape[0]
    if not q.is_cuda:
        y = (q.float() * sx[:, None]) @ (w8.float() * sw[:, None]).t()
        return out.copy_(y) if out is not None else y.to(torch.bfloat16 if isinstance(x, tuple) else x.dtype)
    defer = defer_reduce and out is None
    if plan is None and M and (out is None or (out.is_contiguous() and out.data_ptr() % 16 == 0)) and (
            S := fp8_tile_plan(M, N, K)) is not None and (q.data_ptr() | w8.data_ptr()) % 16 == 0:
        part = torch.empty(S * M * N, dtype=torch.float32, device=q.device) if S > 1 else None
        y = None if defer and S > 1 else out if out is not None else torch.empty(M, N, dtype=torch.bfloat16, device=q.device)
        kernels().gemm_fp8_tile(q, w8, sx, sw, y, part, S, rows=fp8_tile_rows(M, N, K, S)[1])
        return SplitK(part, S, M, N) if y is None else y
    bm, bn, S = plan or fp8_plan(M, N, K)
    y = out if out is not None else torch.empty(M, N, dtype=torch.bfloat16, device=q.device)
    part = torch.empty(S * M * N, dtype=torch.float32, device=q.device) if S > 1 else None
    if defer and S > 1:
        kernels().gemm_fp8(q, w8, sx, sw, y, part, S, bn, bm, False)
        return SplitK(part, S, M, N)
    kernels().gemm_fp8(q, w8, sx, sw, y, part, S, bn, bm)
    return y


def decode_splits(max_context: int, batch: int = 1, kv_heads: int = 8, min_tokens: int | None = None, rows: int | None = None) -> int:
    """Workgroups per (sequence, kv-head) for decode attention: split only while
    ``batch * kv_heads`` workgroups cannot fill the GPU, never into pieces shorter
    than ``min_tokens`` (256; measured on MI355X, B=16 ctx=1024: 1 split 25.9 us, 4 splits
    23.7 us, 16 splits 47.8 us). Powers of two, so a graph captured per value
    covers every context length with few captures.

    ``rows``: how many of the batch's are sequences, where the others are padding, whose workgroups end at once: a bucket of 64 that holds 9 to 32 is cut
    as far as its sequences still come to one workgroup per CU (two layers, whole steps, us: 16 x 3000 tokens of 28 / 4 heads 593 in one split, 539 in four; 24 x 3000 601 and, in two,
    567; 12 x 3000 of 32 / 8 545 and, in two, 518; 9 to 31 x 1000 0 to 4 % less). Not further: 24 x 3000 of 32 / 8 535 and, in two, 571."""
    want = max(-(-DECODE_TARGET_BLOCKS // max(1, batch * kv_heads)), DECODE_TARGET_BLOCKS // max(1, (rows or batch) * kv_heads))
    cap = -(-max(1, int(max_context)) // (min_tokens or DECODE_MIN_SPLIT_TOKENS))
    ns = max(1, min(want, cap, 256))
    # the power of two at or BELOW: splits of 256-512 tokens, not 128-256 (B = 64, one kv-head,
    # ctx 1100: 4 splits 15.2 us vs 8 splits 19.9 us with the combine, profiles/attn_decode_tp8_splits_r5.jsonl)
    return 1 << (ns.bit_length() - 1)


def decode_workspace(B: int, Hq: int, num_splits: int, device, D: int = 128):
    """(o_part fp32, ml_part fp32) partial buffers for attn_decode (unused when num_splits == 1)."""
    n = max(1, B * Hq * num_splits) if num_splits > 1 else 1
    return (torch.empty(n * D, dtype=torch.float32, device=device),
            torch.empty(n * 2, dtype=torch.float32, device=device))


def attn_decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, block_tables: torch.Tensor,
                seq_lens: torch.Tensor, scale: float, num_splits: int, out: torch.Tensor | None = None,
                workspace: tuple[torch.Tensor, torch.Tensor] | None = None, variant: int | None = None,
                k_scale: float = 1.0, v_scale: float = 1.0, quant: bool = False):
    """Paged decode attention; ``num_splits`` workgroups per (sequence, kv-head)
    (``decode_splits``). Any value >= 1 is correct; it only changes the schedule.
    The cache is bf16, or e4m3fn holding x / k_scale and x / v_scale.
    ``quant``: return the [B, Hq*D] output rows as per-token e4m3fn ``(q, sx)`` for an
    fp8 o-projection, produced by the split-combine kernel itself (== quantize_fp8)."""
    if not q.is_cuda:
        r = reference.attn_decode(q, k_cache, v_cache, block_tables, seq_lens, scale, k_scale, v_scale)
        if out is not None:
            out.copy_(r)
            r = out
        return quantize_fp8(r.reshape(r.shape[0], -1)) if quant else r
    B, Hq, D = q.shape
    variant = DECODE_ATTN_VARIANT if variant is None else variant
    o = out if out is not None else torch.empty_like(q)
    if workspace is None:
        workspace = decode_workspace(B, Hq, num_splits, q.device)
    q8 = sx = None
    if quant:
        q8 = torch.empty(B, Hq * D, dtype=torch.float8_e4m3fn, device=q.device)
        sx = torch.empty(B, dtype=torch.float32, device=q.device)
    kernels().attn_decode(q, k_cache, v_cache, block_tables, seq_lens, o, workspace[0], workspace[1],
                          num_splits, scale, variant, k_scale, v_scale, q8, sx)
    return (q8, sx) if quant else o


# decode RoPE + KV-cache write folded into decode attention (OAMD_FUSED_ROPE=0: rope_kv, then attn_decode),
# for batches of at most FUSED_ROPE_MAX_SEQ_HEADS (sequence, kv-head) pairs: there attention is
# latency-bound and the fold removes a launch (TP=8 70B fp8 B=64: 6.85 -> 6.64 ms/step); at the
# 8B flagship's 256 x 8 pairs attention streams HBM and every workgroup would pay the fold's
# slab reads and store drain up front (-1.3 % analyses/s, profiles/fused_decode_rope_ab_r5.jsonl)
FUSED_DECODE_ROPE = os.environ.get("OAMD_FUSED_ROPE", "1") != "0"
FUSED_ROPE_MAX_SEQ_HEADS = int(os.environ.get("OAMD_FUSED_ROPE_MAX", "256"))


def attn_decode_rope(qkv, pos: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, Hq: int, k_cache: torch.Tensor,
                     v_cache: torch.Tensor, slots: torch.Tensor, block_tables: torch.Tensor, seq_lens: torch.Tensor,
                     scale: float, num_splits: int, workspace: tuple[torch.Tensor, torch.Tensor] | None = None,
                     bias: torch.Tensor | None = None, k_scale: float = 1.0, v_scale: float = 1.0,
                     quant: bool = False, variant: int | None = None):
    """One decode step's ``rope_kv`` (want_kv=False) + ``attn_decode`` as ONE kernel: every
    attention workgroup rotates its q from the QKV projection (``qkv``: bf16 rows or the
    GEMM's :class:`SplitK` slabs, + the Qwen2 bias), and the workgroup holding each
    sequence's last token writes that token's rotated K and its V into the cache before
    reading it (csrc/kernels/attn_decode.hip, ``DecRope``). Same numerics as the two
    kernels; one launch and the q round trip fewer per layer."""
    Hkv = k_cache.shape[1]
    if not (qkv.is_cuda and FUSED_DECODE_ROPE and qkv.shape[0] * Hkv <= FUSED_ROPE_MAX_SEQ_HEADS):
        q, _, _ = rope_kv(qkv, pos, cos, sin, Hq, Hkv, k_cache, v_cache, slots, want_kv=False, bias=bias,
                          k_scale=k_scale, v_scale=v_scale)
        return attn_decode(q, k_cache, v_cache, block_tables, seq_lens, scale, num_splits, workspace=workspace,
                           variant=variant, k_scale=k_scale, v_scale=v_scale, quant=quant)
    B = qkv.shape[0]
    D = cos.shape[1] * 2
    variant = DECODE_ATTN_VARIANT if variant is None else variant
    o = torch.empty(B, Hq, D, dtype=torch.bfloat16, device=qkv.device)
    if workspace is None:
        workspace = decode_workspace(B, Hq, num_splits, qkv.device)
    q8 = sx = None
    if quant:
        q8 = torch.empty(B, Hq * D, dtype=torch.float8_e4m3fn, device=qkv.device)
        sx = torch.empty(B, dtype=torch.float32, device=qkv.device)
    rx, S = (qkv.p, qkv.S) if isinstance(qkv, SplitK) else (qkv, 1)
    kernels().attn_decode(o, k_cache, v_cache, block_tables, seq_lens, o, workspace[0], workspace[1], num_splits,
                          scale, variant, k_scale, v_scale, q8, sx, rx, S, pos, cos, sin, slots, bias)
    return (q8, sx) if quant else o


# temperature bits of a row whose token nobody reads: it gets token 0, its logits are not read (csrc/kernels/sample.hip;
# the CPU reference samples it like any NaN, greedily)
NO_SAMPLE_BITS = 0x7FC5A5A5


def sample(logits: torch.Tensor, temperature: torch.Tensor, seeds: torch.Tensor, positions: torch.Tensor,
           out: torch.Tensor | None = None, col_offset: int = 0, out_val: torch.Tensor | None = None) -> torch.Tensor:
    """Temperature / Gumbel-max sampling (greedy rows where temperature <= 0).

    For a vocab shard pass ``col_offset`` (global id of column 0) and ``out_val``
    (receives each row's winning perturbed value) and take the max over shards.
    """
    if not logits.is_cuda:
        tok, val = reference.sample_shard(logits, temperature, seeds, positions, col_offset)
        if out_val is not None:
            out_val.copy_(val)
        if out is not None:
            out.copy_(tok)
            return out
        return tok
    o = out if out is not None else torch.empty(logits.shape[0], dtype=torch.long, device=logits.device)
    rows = logits.shape[0]
    parts = kernels().sample_parts(rows, logits.shape[1])   # workgroups per row, merged by a second kernel
    part = torch.empty(2 * rows * parts, dtype=torch.float32, device=logits.device) if parts > 1 else None
    kernels().sample(logits, temperature, seeds, positions, o, col_offset, out_val, part)
    return o


def sample_candidates(logits: torch.Tensor, temperature: torch.Tensor, seeds: torch.Tensor, positions: torch.Tensor,
                      given: torch.Tensor | None = None, dst: torch.Tensor | None = None) -> dict:
    """``sample`` as far as the next kernel takes it: decode_advance's ``tok``, or ``part`` [rows, parts, 2] where several workgroups share a
    row, whose best that kernel takes itself. ``given`` [2] (on the device: the address of fp32 rows, 0: none, and their number): rows that are
    not sampled (NO_SAMPLE_BITS) go to its rows ``dst``."""
    rows = logits.shape[0]
    parts = kernels().sample_parts(rows, logits.shape[1])
    tok = torch.empty(rows, dtype=torch.long, device=logits.device)
    if parts <= 1:
        kernels().sample(logits, temperature, seeds, positions, tok, 0, None, None, True, given, dst)
        return {"tok": tok}
    part = torch.empty(rows, parts, 2, dtype=torch.float32, device=logits.device)
    kernels().sample(logits, temperature, seeds, positions, tok, 0, None, part, False, given, dst)
    return {"tok": None, "part": part, "temperature": temperature}


from . import decoder  # noqa: E402 - uses SplitK and prefill_work_list above
