"""Continuous batching under one captured graph (DecodeEngine.insert / retire): a retired
slot keeps decoding throw-away tokens inside its own cache rows without ever stopping the
batch, and a new sequence inserted into it decodes bitwise like the same sequence inserted
into a fresh engine -- nothing of the retired sequence leaks into it -- while the other rows'
caches are untouched by the insertion.  2-layer full-width model (dense + MoE), full vocab."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def weights():
    import dsv2lite

    return dsv2lite.init_weights(dsv2lite.DSV2Config(n_layers=2), device="cuda", seed=0)


def _prompts(lens, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, 102400, (n,), generator=g).cuda() for n in lens]


@pytest.mark.parametrize("family", ["small", "batch"])
def test_retired_slot_reuse_matches_a_fresh_engine_bitwise(weights, family):
    import dsv2lite

    caps = [48, 40, 64, 56]
    tile = 16 if family == "batch" else None
    A = dsv2lite.DecodeEngine(weights, caps, family=family, moe_tile=tile)
    A.prefill(_prompts([10, 7, 20, 12], 1))
    A.capture()
    for _ in range(5):
        A.replay()
    A.retire(2)
    assert A.free_slots == [2]
    for _ in range(3):
        A.replay()  # slot 2 decodes throw-away tokens
    others = {b: A.cache.data[:, int(A.cache.base[b]):int(A.cache.base[b]) + caps[b]].clone() for b in (0, 1, 3)}
    pos_before = A.cache.pos.clone()
    q = _prompts([9], 2)[0]
    first = A.insert(2, q)
    torch.cuda.synchronize()
    assert A.free_slots == [] and int(A.cache.pos[2]) == 9
    for b, t in others.items():  # the insertion touched slot 2's rows only
        assert torch.equal(A.cache.data[:, int(A.cache.base[b]):int(A.cache.base[b]) + caps[b]], t), b
        assert int(A.cache.pos[b]) == int(pos_before[b])
    got = [(first, A.logits[2].clone())]
    for _ in range(6):
        A.replay()
        got.append((int(A.ids[2]), A.logits[2].clone()))
    A.check_errors()

    B = dsv2lite.DecodeEngine(weights, caps, family=family, moe_tile=tile)
    B.capture()
    ref = [(B.insert(2, q), B.logits[2].clone())]
    for _ in range(6):
        B.replay()
        ref.append((int(B.ids[2]), B.logits[2].clone()))
    for i, ((ta, la), (tb, lb)) in enumerate(zip(got, ref)):
        assert ta == tb and torch.equal(la, lb), (family, i)


def test_retired_slot_wraps_inside_its_capacity(weights):
    """A retired slot with a small capacity restarts at 0 whenever it would reach it; the
    active rows decode on, and no kernel ever flags a write past a row's capacity."""
    import dsv2lite

    eng = dsv2lite.DecodeEngine(weights, [80, 12], family="small")
    eng.prefill(_prompts([6, 5], 3))
    eng.capture()
    eng.replay()
    eng.retire(1)
    for _ in range(40):  # > 3 wraps of slot 1's 12 rows
        eng.replay()
        assert 0 <= eng._host_pos[1] <= 12
    torch.cuda.synchronize()
    assert int(eng.cache.pos[0]) == 6 + 41 and int(eng.cache.pos[1]) == eng._host_pos[1]
    eng.check_errors()
    with pytest.raises(ValueError, match="does not fit"):
        eng.insert(1, _prompts([12], 4)[0])
    assert eng.insert(1, _prompts([4], 4)[0]) >= 0 and eng.free_slots == []


@pytest.mark.parametrize("where", ["host", "mixed"])
def test_prefill_takes_prompts_from_host_or_device_alike(weights, where):
    """Prompts on the host (sent in one copy with the chunk plan) give bitwise the state of the
    same prompts on the device, over chunks in which no, one and several prompts end."""
    import dsv2lite

    prompts = _prompts([40, 3, 5, 17], 3)
    other = [p.cpu() if where == "host" or i % 2 else p for i, p in enumerate(prompts)]
    states = []
    for ps in (prompts, other):
        eng = dsv2lite.DecodeEngine(weights, [64] * 4, family="batch", max_prefill_rows=16, moe_tile=16)
        eng.prefill(ps)
        torch.cuda.synchronize()
        states.append((eng.logits.clone(), eng.ids.clone(), eng.cache.pos.clone(), eng.cache.data.clone()))
    for a, b in zip(*states):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows", [4, 5, 8, 17, 40])
def test_small_family_rows_do_not_depend_on_their_batch(weights, rows):
    """The small family below and from the row count at which its step runs the batch family's
    kernels: graph replay equals the eager step bitwise, and a sequence decodes to the same bits
    whatever prompts share its batch -- prompts that spread over the experts (two sets of them) or
    one repeated token, whose rows all go to the same experts."""
    import dsv2lite

    mine = _prompts([11], 7)[0]
    got = []
    lens = [3 + i % 20 for i in range(rows - 1)]
    for others in (_prompts(lens, 8), _prompts(lens, 9), [torch.full((n,), 77).cuda() for n in lens]):
        eng = dsv2lite.DecodeEngine(weights, [32] * rows, family="small")
        eng.prefill([mine] + others)
        snap = eng.snapshot()
        eng.step()
        eager = eng.logits.clone()
        eng.restore(snap)
        eng.capture()
        eng.restore(snap)
        for i in range(3):
            eng.replay()
            if i == 0:
                assert torch.equal(eng.logits, eager)
        eng.check_errors()
        got.append(eng.logits[0].clone())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.parametrize("family,rows", [("batch", 3), ("small", 5), ("small", 24)])
def test_moe_tile_is_honoured_on_every_batch_kernel_step(weights, family, rows):
    """moe_tile fixes the grouped tile of any engine whose step runs the batch family's kernels,
    through capture and replay; a tile the launches do not have is refused."""
    import dsv2lite

    for tile in (16, 32, 64, 256):
        eng = dsv2lite.DecodeEngine(weights, [32] * rows, family=family, moe_tile=tile)
        eng.prefill(_prompts([4 + i % 9 for i in range(rows)], 21))
        eng.capture()
        eng.replay()
        torch.cuda.synchronize()
        assert eng.buf.tile_tokens == tile
        assert torch.isfinite(eng.logits).all()
    with pytest.raises(ValueError, match="tile_tokens"):
        dsv2lite.DecodeEngine(weights, [32] * rows, family=family, moe_tile=48)


@pytest.mark.parametrize("rows,cap", [(4, 40), (5, 40), (8, 400), (40, 40), (40, 400)])
def test_small_family_keeps_the_latent_output_in_fp32(rows, cap):
    """The small family applies W_UV to the fp32 latent output at every row count.  With zero
    queries all scores are 0, the softmax weights are exact and o_lat is the mean of the row's
    latents, which fp32 holds almost exactly and bf16 does not: bf16(W_UV o_lat) then equals the
    float64 result but for values next to a rounding boundary (fp32 sums of 512 terms: within
    512 * 2^-24 of the sum of magnitudes, about 2^-11 of a bf16 step's width here), where a bf16
    o_lat moves a large share of them."""
    import dsv2lite

    cfg = dsv2lite.DSV2Config(n_layers=1)
    w = dsv2lite.init_weights(cfg, device="cuda", seed=0)
    L = w.layers[0]
    L.w_qkva[:cfg.n_heads * (cfg.qk_nope + cfg.qk_rope)].zero_()
    eng = dsv2lite.DecodeEngine(w, [cap] * rows, family="small")
    lens = [3 + (7 * i) % (cap - 8) for i in range(rows)]
    eng.prefill(_prompts(lens, 12))
    eng.step()
    torch.cuda.synchronize()
    eng.check_errors()
    cache, w_uv = eng.cache.layer(0), L.w_uv.double().reshape(cfg.n_heads * cfg.v_dim, cfg.kv_rank)
    differ = total = 0
    for b, n in enumerate(lens):
        base = int(eng.cache.base[b])
        olat = cache[base:base + n + 1, :cfg.kv_rank].double().mean(0)
        want = (w_uv @ olat).to(torch.bfloat16)
        differ += int((eng.buf.attn[b] != want).sum())
        total += want.numel()
    print(f"{rows} rows, capacity {cap}: {differ} of {total} differ from bf16 of the float64 result", flush=True)
    assert differ <= 0.02 * total


def test_small_family_absorb_and_split_decode_agree_at_the_threshold(weights):
    """The small family's attention just below and above the capacity at which "absorb" hands over
    to the split-KV decode: same prompt, logits within the 2e-2 parity bar of each other."""
    import dsv2lite
    from dsv2lite.engine import ABSORB_MAX_CTX

    prompt = _prompts([ABSORB_MAX_CTX - 30], 11)
    got = []
    for cap in (ABSORB_MAX_CTX, ABSORB_MAX_CTX + 1):
        eng = dsv2lite.DecodeEngine(weights, [cap], family="small")
        assert eng.absorb_mla == (cap == ABSORB_MAX_CTX)
        eng.prefill(prompt)
        for _ in range(3):
            eng.ids.fill_(77)  # the same tokens whatever the logits say
            eng.step()
        eng.check_errors()
        got.append(eng.logits.float().clone())
    assert float((got[0] - got[1]).abs().max() / got[0].abs().max()) < 2e-2


def test_one_row_takes_the_path_of_its_length(weights, monkeypatch):
    """A lone row in a cache with room to grow runs the absorb step while few tokens are cached and
    the split-KV one from ABSORB_ROW_CTX, eagerly and replayed alike (bitwise), over the crossing and
    after a short prompt takes the slot again."""
    import dsv2lite
    import dsv2lite.engine as E

    calls, call = [], E.call
    monkeypatch.setattr(E, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    start = E.ABSORB_ROW_CTX - 3
    eng = dsv2lite.DecodeEngine(weights, [1000], family="small")
    eng.prefill(_prompts([start], 13))
    snap = eng.snapshot()
    eager = []
    for i in range(6):
        calls.clear()
        eng.step()
        assert ("dsv2_qkva_absorb_bf16" in calls) == (i < 3) and ("dsv2_mla_decode" in calls) == (i >= 3), i
        eager.append((eng.logits.clone(), eng.ids.clone()))
    for at in (0, 4):  # captured on either side
        eng.restore(snap)
        for i in range(at):
            eng.step()
        eng.capture()
        for i in range(at, 6):
            calls.clear()
            eng.replay()
            assert not calls
            assert torch.equal(eng.logits, eager[i][0]) and torch.equal(eng.ids, eager[i][1]), (at, i)
    eng.insert(0, _prompts([9], 14)[0])
    snap = eng.snapshot()
    eng.replay()
    got = eng.logits.clone()
    eng.restore(snap)
    calls.clear()
    eng.step()
    assert "dsv2_qkva_absorb_bf16" in calls and torch.equal(got, eng.logits)
    eng.check_errors()
