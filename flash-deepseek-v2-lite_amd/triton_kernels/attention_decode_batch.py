"""Absorbed-MLA decode attention, batch family (reference:
triton_kernels/attention_decode_batch.py:25-35, 214-237, 672-846).

Documented deviation from the reference interface: ``key_cache`` is the
COMPRESSED cache [B, L, 576] bf16 (kv-normalised latent | rotated k_pe) and
``value_cache`` must be None -- the reference caches expanded per-head K/V
[B, 16, L, 192] / [B, 16, L, 128].  Row b's new token is written at
``cache_position`` and attends positions 0..cache_position (src/run.py:196-202).
"""

from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from . import _hip
from ._checks import require_contiguous, require_cuda

NH, NOPE, ROPE, VD, LAT, HID = 16, 128, 64, 128, 512, 2048
QKVA = NH * (NOPE + ROPE) + LAT + ROPE  # 3648
ROW = LAT + ROPE  # 576


@dataclass
class AttentionPackedWeights:
    w_qkva: torch.Tensor        # [3648, 2048] = cat(q_proj, kv_a_proj_with_mqa)
    kv_norm_weight: torch.Tensor  # [512]
    kv_norm_eps: float
    w_uk: torch.Tensor          # [16, 128, 512]
    w_ukt: torch.Tensor         # [16, 512, 128]
    w_uv: torch.Tensor          # [16, 128, 512]
    w_o: torch.Tensor           # [2048, 2048]


def pack_attention_weights(attn: torch.nn.Module) -> AttentionPackedWeights:
    """Pack an HF DeepseekV2Attention (q_lora_rank=None) for the HIP kernels."""
    if getattr(attn, "q_lora_rank", None) is not None:
        raise NotImplementedError("pack_attention_weights supports q_lora_rank=None (DeepSeek-V2-Lite)")
    q = attn.q_proj.weight.detach()
    kva = attn.kv_a_proj_with_mqa.weight.detach()
    kvb = attn.kv_b_proj.weight.detach().reshape(NH, NOPE + VD, LAT)
    ln = attn.kv_a_layernorm
    eps = float(getattr(ln, "variance_epsilon", getattr(ln, "eps", 1e-6)))
    w_uk = kvb[:, :NOPE].contiguous()
    return AttentionPackedWeights(torch.cat((q, kva)).contiguous(), ln.weight.detach().contiguous(), eps, w_uk,
                                  w_uk.transpose(1, 2).contiguous(), kvb[:, NOPE:].contiguous(),
                                  attn.o_proj.weight.detach().contiguous())


# caches up to this many tokens per row take one split per row: the engine then runs the
# one-launch decode (dsv2_mla_decode_rows) and no split merge
ONE_SPLIT_MAX_CTX = 256


# one split per row also up to this cache length where rows alone leave under a third of the CUs idle
IDLE_CU_ONE_SPLIT_CTX = 512


def plan_splits(rows: int, max_ctx: int, target_wgs: int = 256) -> tuple[int, int]:
    """(split_tokens, max_splits) for the split-KV decode: one split per row for caches of at
    most ONE_SPLIT_MAX_CTX tokens (measured on MI355X, whole decode steps, against the
    multi-split plan below: bsz=64 x 57-token caches 2.809 -> 2.726 ms, bsz=64 x 233 6.958 ->
    6.901, bsz=128 x 233 7.941 -> 7.832; at 433 tokens one split loses, 7.013 -> 7.101);
    else the most splits per row (at most 64, split_tokens a multiple of 32) that leave at most
    target_wgs workgroups: 256 = one per CU, each streaming its split with two tiles in flight.
    A few more than 256 make some CUs run two while the rest run one (70 rows x 1,600 tokens 39
    us with 4, 33 with 3; 40 x 4,096 52 with 7, 40 with 6).  Where that leaves one or two splits per
    row and CUs idle, a long row among short ones would end the launch alone, so there are more:
      under 128 rows, two workgroups per CU (decode + merge of 96 rows x 3,300 tokens, 2 / 3 / 5
      splits: equal lengths 72 / 82 / 69 us, lengths from an eighth 64 / 61 / 51, one full row among
      sixteenths 62 / 45 / 31; 110 x 2,048 with 2 / 3 / 4: 50 / 60 / 54, 45 / 47 / 41, 43 / 32 / 27);
      under 171, three (140 x 1,600: 57 us, 66 with 2);
      under 256, two past IDLE_CU_ONE_SPLIT_CTX tokens (200 x 2,048, 1 / 2 / 3 splits: 86 / 89 / 101,
      72 / 68 / 75, 69 / 46 / 39; but 200 x 512 25 / 34 / 40, 23 / 30 / 31, 21 / 20 / 21).
    More than that suits lengths spread as wide as 128 rows of U[256,8192] (1,664-token splits 126
    us, 4,096-token ones 150), which a caller plans with a larger target_wgs."""
    if max_ctx <= ONE_SPLIT_MAX_CTX:
        return max(32, math.ceil(max_ctx / 32) * 32), 1
    per_row = max(1, min(64, target_wgs // max(rows, 1)))
    if per_row == 2 and 2 * rows < target_wgs:
        per_row = 2 * target_wgs // rows
    elif per_row == 1 and rows < target_wgs:
        per_row = 3 if 3 * rows <= 2 * target_wgs else (2 if max_ctx > IDLE_CU_ONE_SPLIT_CTX else 1)
    split = max(32, math.ceil(math.ceil(max_ctx / per_row) / 32) * 32)
    split = max(split, math.ceil(max_ctx / 64 / 32) * 32)
    return split, math.ceil(max_ctx / split)


# the small family runs the absorb path (dsv2_qkva_absorb_bf16 + dsv2_mla_attend_parts) while
# the cache is this short; longer caches take the split-KV decode (from 640 tokens its kernels are
# the faster ones, but these calls launch eagerly and two launches more cost the host 11 us)
FUSED_MAX_CTX = 2048


@dataclass
class AttentionDecodeWorkspace:
    """Per-(device, B, L) buffers of one attention call, cached on the packed weights like
    the reference's workspace (attention_decode_batch.py:641-669); the returned output
    aliases ``out`` and is overwritten by the next call with the same key."""

    pos: torch.Tensor      # [B] int32
    base: torch.Tensor     # [B] int64
    cap: torch.Tensor      # [B] int32
    status: torch.Tensor   # [1] int32: DSV2_DEVERR_* bits of every call so far
    qkva: torch.Tensor     # [B, 3648]
    qlat_part: torch.Tensor  # [B, 16, 8, 512] fp32: partial absorbed queries (small family)
    q: torch.Tensor        # [B, 16, 576]
    split: int
    nsplit: int
    part_o: torch.Tensor   # [B, nsplit, 16, 512] fp32
    part_ml: torch.Tensor  # [B, nsplit, 16, 2] fp32
    olat: torch.Tensor     # [B, 16, 512]
    attn: torch.Tensor     # [B, 2048]
    out: torch.Tensor      # [B, 1, 2048]


def _workspace(packed: AttentionPackedWeights, dev: torch.device, B: int, L: int) -> AttentionDecodeWorkspace:
    key = (dev.index if dev.index is not None else 0, B, L)
    cache = packed.__dict__.setdefault("workspace_by_key", {})
    ws = cache.get(key)
    if ws is None:
        e = lambda *shape, dt=torch.bfloat16: torch.empty(*shape, dtype=dt, device=dev)  # noqa: E731
        split, nsplit = plan_splits(B, L)
        ws = AttentionDecodeWorkspace(
            pos=e(B, dt=torch.int32), base=e(B, dt=torch.int64), cap=e(B, dt=torch.int32),
            status=torch.zeros(1, dtype=torch.int32, device=dev), qkva=e(B, QKVA),
            qlat_part=e(B, NH, NOPE // 16, LAT, dt=torch.float32), q=e(B, NH, ROW), split=split,
            nsplit=nsplit, part_o=e(B, nsplit, NH, LAT, dt=torch.float32), part_ml=e(B, nsplit, NH, 2, dt=torch.float32),
            olat=e(B, NH, LAT), attn=e(B, HID), out=e(B, 1, HID))
        cache[key] = ws
    return ws


def check_cache_status(packed: AttentionPackedWeights) -> None:
    """Raise if an attention call on these weights tried to write its new token at or past
    the cache length L (nothing was written there; synchronises).  The reference raises on
    a cache overflow (src/run.py:131-134)."""
    for ws in packed.__dict__.get("workspace_by_key", {}).values():
        if int(ws.status.item()) & 1:  # DSV2_DEVERR_CACHE_FULL
            ws.status.zero_()
            raise RuntimeError("attention decode: cache_position reached the cache length; the new token was not "
                               "written")


def _attention_decode(family: str, hidden_states, cos, sin, position_ids, cache_position, key_cache, value_cache,
                      packed: AttentionPackedWeights, softmax_scale: float) -> torch.Tensor:
    name = f"attention_decode[{family}]"
    require_cuda(name, hidden_states, cos, sin, cache_position, key_cache)
    if hidden_states.dtype != torch.bfloat16 or key_cache.dtype != torch.bfloat16:
        raise NotImplementedError(f"{name} supports bf16 only")
    if hidden_states.ndim != 3 or hidden_states.shape[1] != 1 or hidden_states.shape[2] != HID:
        raise ValueError(f"{name} expects hidden_states [B, 1, 2048]")
    B = hidden_states.shape[0]
    if value_cache is not None:
        raise ValueError(f"{name} reads the compressed cache only; pass value_cache=None")
    if key_cache.ndim != 3 or key_cache.shape[0] != B or key_cache.shape[2] != ROW:
        raise ValueError(f"{name} expects key_cache [B, L, 576] (compressed)")
    if cos.dtype != torch.bfloat16 or sin.dtype != torch.bfloat16 or cos.shape[-1] != ROPE or cos.shape != sin.shape:
        raise ValueError(f"{name} expects bf16 cos/sin tables [L, 64]")
    if cache_position.numel() != 1 or cache_position.dtype != torch.long:
        raise ValueError("cache_position must be an int64 tensor with one element")
    require_contiguous(name, key_cache, cos, sin)
    dev = hidden_states.device
    L = key_cache.shape[1]
    cos2, sin2 = cos.reshape(-1, ROPE), sin.reshape(-1, ROPE)
    max_pos = min(cos2.shape[0], L)
    x = hidden_states.reshape(B, HID).contiguous()
    ws = _workspace(packed, dev, B, L)
    attn2, out2 = ws.attn, ws.out.view(B, HID)
    st = _hip.stream_ptr(dev)
    call = _hip.call
    P = lambda t: t.data_ptr()  # noqa: E731
    call("dsv2_fill_positions", P(cache_position), P(ws.pos), P(ws.base), P(ws.cap), L, B, st)
    if family == "small":
        if L <= FUSED_MAX_CTX:
            # the engine's default small-batch MLA: the projection also forms the absorbed query
            call("dsv2_qkva_absorb_bf16", P(x), HID, B, P(packed.w_qkva), None, 0.0, P(packed.w_uk), P(ws.qkva), QKVA,
                 P(ws.qlat_part), P(key_cache), P(ws.base), P(ws.pos), P(ws.cap), st)
            call("dsv2_mla_attend_parts", P(ws.qkva), QKVA, B, P(ws.pos), P(ws.base), P(ws.cap),
                 P(packed.kv_norm_weight), packed.kv_norm_eps, P(cos2), P(sin2), max_pos, P(ws.qlat_part),
                 P(packed.w_uv), P(key_cache), float(softmax_scale), P(attn2), HID, P(ws.status), st)
        else:
            call("dsv2_gemv_bf16", P(x), HID, B, HID, P(packed.w_qkva), QKVA, None, 0.0, None, 0, P(ws.qkva), QKVA, 0,
                 st)
            call("dsv2_mla_prepare", P(ws.qkva), QKVA, B, P(ws.pos), P(ws.base), P(ws.cap), P(packed.kv_norm_weight),
                 packed.kv_norm_eps, P(cos2), P(sin2), max_pos, P(packed.w_ukt), P(key_cache), P(ws.q), P(ws.status),
                 st)
            call("dsv2_mla_decode", P(ws.q), P(key_cache), P(ws.base), P(ws.pos), P(ws.cap), B, ws.split, ws.nsplit,
                 float(softmax_scale), P(ws.part_o), P(ws.part_ml), st)
            call("dsv2_mla_combine", P(ws.part_o), P(ws.part_ml), P(ws.pos), P(ws.cap), B, ws.split, ws.nsplit,
                 P(packed.w_uv), P(attn2), HID, st)
        call("dsv2_gemv_bf16", P(attn2), HID, B, HID, P(packed.w_o), HID, None, 0.0, None, 0, P(out2), HID, 0, st)
        return ws.out
    call("dsv2_gemm_bf16", P(x), HID, 0, B, HID, P(packed.w_qkva), 0, QKVA, 1, None, 0, P(ws.qkva), QKVA, 0, 0, st)
    # the new cache row, RoPE and the W_UK absorption in one launch; one split per row needs no merge
    call("dsv2_mla_prepare_qlat", P(ws.qkva), QKVA, B, P(ws.pos), P(ws.base), P(ws.cap), P(packed.kv_norm_weight),
         packed.kv_norm_eps, P(cos2), P(sin2), max_pos, P(packed.w_ukt), P(key_cache), P(ws.q), P(ws.status), st)
    if ws.nsplit == 1:
        call("dsv2_mla_decode_rows", P(ws.q), P(key_cache), P(ws.base), P(ws.pos), P(ws.cap), B, float(softmax_scale),
             P(ws.olat), NH * LAT, st)
    else:
        call("dsv2_mla_decode", P(ws.q), P(key_cache), P(ws.base), P(ws.pos), P(ws.cap), B, ws.split, ws.nsplit,
             float(softmax_scale), P(ws.part_o), P(ws.part_ml), st)
        call("dsv2_mla_combine", P(ws.part_o), P(ws.part_ml), P(ws.pos), P(ws.cap), B, ws.split, ws.nsplit, None,
             P(ws.olat), NH * LAT, st)
    call("dsv2_gemm_bf16", P(ws.olat), NH * LAT, LAT, B, LAT, P(packed.w_uv), VD * LAT, VD, NH, None, 0, P(attn2),
         HID, VD, 0, st)
    call("dsv2_gemm_bf16", P(attn2), HID, 0, B, HID, P(packed.w_o), 0, HID, 1, None, 0, P(out2), HID, 0, 0, st)
    return ws.out


def batched_attention_decode_q1_triton(query_states: torch.Tensor, key_states: torch.Tensor,
                                       value_states: torch.Tensor, cache_position: torch.Tensor,
                                       softmax_scale: float) -> torch.Tensor:
    """q_len=1 attention over an expanded per-head cache: query [B, H, 1, Dq], keys
    [B, H, L, Dq], values [B, H, L, Dv] (bf16, last dim contiguous) -> [B, H, 1, Dv]:
    softmax over positions 0..cache_position of scale * q.k, times v, fp32 math.  Positions
    at or past L are not read (the reference reads them unchecked); the call then attends
    the L rows and the overflow is reported by check_expanded_status.
    Reference: attention_decode_batch.py:345-401."""
    require_cuda("batched_attention_decode_q1_triton", query_states, key_states, value_states, cache_position)
    if query_states.dtype != torch.bfloat16 or key_states.dtype != torch.bfloat16 or \
            value_states.dtype != torch.bfloat16:
        raise NotImplementedError("batched_attention_decode_q1_triton supports bf16 only")
    q, k, v = query_states, key_states, value_states
    qs, ks, vs = q.shape, k.shape, v.shape
    if len(qs) != 4 or len(ks) != 4 or len(vs) != 4:
        raise ValueError("query/key/value states must be rank-4 tensors")
    B, H, q_len, Dq = qs
    if q_len != 1:
        raise ValueError("batched_attention_decode_q1_triton only supports q_len=1")
    if cache_position.numel() != 1 or cache_position.dtype != torch.long:
        raise ValueError("cache_position must be CUDA int64 tensor with one element")
    L, Dv = ks[2], vs[3]
    if ks != (B, H, L, Dq) or vs[:3] != (B, H, L):
        raise ValueError("key/value states must be [B, H, L, Dq] / [B, H, L, Dv] matching the query")
    q_st, k_st, v_st = q.stride(), k.stride(), v.stride()
    if q_st[3] != 1 or k_st[3] != 1 or v_st[3] != 1:
        raise NotImplementedError("batched_attention_decode_q1_triton needs a contiguous last dimension")
    dev = q.device
    out = torch.empty((B, H, 1, Dv), device=dev, dtype=torch.bfloat16)
    if B == 0 or L == 0:
        return out
    ns = expanded_splits(B * H, L)
    part = torch.empty(B * H * ns * (Dv + 2), dtype=torch.float32, device=dev) if ns > 1 else None
    _hip.call("dsv2_attention_decode_expanded_split", q.data_ptr(), q_st[0], q_st[1], k.data_ptr(), k_st[0], k_st[1],
              k_st[2], v.data_ptr(), v_st[0], v_st[1], v_st[2], out.data_ptr(), H * Dv, Dv, B, H, Dq, Dv, L,
              cache_position.data_ptr(), float(softmax_scale), ns, None if part is None else part.data_ptr(),
              _expanded_status(dev).data_ptr(), _hip.stream_ptr(dev))
    return out


def expanded_splits(pairs: int, length: int) -> int:
    """Token ranges per (row, head) of the expanded-cache attention: several only where the
    pairs leave most CUs idle and the cache is long enough to pay for the merge launch and its
    buffer.  Measured on MI355X (whole calls, one range against the best of 2..16; pairs x cached
    tokens): 16 x 4000 49.2 -> 20.9 us with 8, 32 x 3000 40.7 -> 21.3 with 8, 64 x 3900 53.2 ->
    33.0 with 4; but 16 x 900 16.3 -> 20.3, 64 x 800 15.4 -> 19.6, 128 x 2000 33.3 -> 32.4 and
    192 x 1380 29.2 -> 35.9.  The position is known on the device only, so a short one in a long cache
    pays for the second launch too: 60 tokens 3.8 us with one range, 6.1 with several, and 4 us of
    host time, which the wrapper keeps within what one launch cost it by asking torch for less."""
    if pairs > 96 or length < 1536:
        return 1
    return min(8, length // 512, 256 // max(pairs, 1))


_EXPANDED_STATUS: dict = {}


def _expanded_status(dev: torch.device) -> torch.Tensor:
    k = dev.index or 0
    st = _EXPANDED_STATUS.get(k)
    if st is None:
        st = _EXPANDED_STATUS[k] = torch.zeros(1, dtype=torch.int32, device=dev)
    return st


def check_expanded_status(device: torch.device | str = "cuda") -> None:
    """Raise if a batched_attention_decode_q1_triton call on `device` had cache_position
    outside [0, L) (synchronises)."""
    st = _expanded_status(torch.device(device))
    if int(st.item()) & 1:  # DSV2_DEVERR_CACHE_FULL
        st.zero_()
        raise RuntimeError("batched_attention_decode_q1_triton: cache_position outside the cache")


def attention_decode_triton(hidden_states, cos, sin, position_ids, cache_position, key_cache, value_cache, packed,
                            softmax_scale: float) -> torch.Tensor:
    """q_len=1 MLA decode for normalised hidden states [B,1,2048] -> o_proj output [B,1,2048]."""
    return _attention_decode("batch", hidden_states, cos, sin, position_ids, cache_position, key_cache, value_cache,
                             packed, softmax_scale)
