"""GPU tests of decode attention and KV-cached generation.

The decode kernel against the oracle (the last row of the causal forward over
the cached positions; bf16 O max-abs <= 2e-2 as for the forward), and the
cached ``generate`` of the HIP routes against the reference's full-recompute
loop on the same weights: teacher-forced logits within 2e-2 relative (both
run the attention in bf16 through different kernels), greedy tokens equal
wherever the recompute's top-2 logit gap is clear of that tolerance.
"""

from __future__ import annotations

import importlib

import numpy as np
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu

mta = importlib.import_module("mega-trading_amd")
model_mod = importlib.import_module("mega-trading_amd.model")

DECODE_CASES = [
    # (B, Hq, Hkv, L, D, dtype, capacity)
    (2, 8, 2, 1, 64, torch.bfloat16, 16),
    (3, 16, 4, 255, 64, torch.bfloat16, 300),
    (1, 4, 4, 256, 128, torch.float16, 256),
    (2, 8, 1, 1000, 64, torch.bfloat16, 1024),
    (1, 32, 8, 4096, 128, torch.bfloat16, 4096),
    (4, 6, 3, 517, 32, torch.float16, 600),
    (32, 8, 2, 1024, 64, torch.bfloat16, 1024),  # BASELINE config 5 layer at the end of the window
    # up to 16 splits of 64 keys (8 at head_dim 128, group sizes up to 5 there) take the fused
    # one-launch kernel, longer caches and larger head_dim-128 groups the split + combine pair
    (2, 8, 2, 1025, 64, torch.bfloat16, 1100),
    (2, 16, 2, 300, 128, torch.bfloat16, 320),
    (3, 10, 2, 450, 128, torch.float16, 512),
    (2, 7, 1, 129, 32, torch.bfloat16, 129),
]


@pytest.mark.parametrize("b,hq,hkv,length,d,dt,cap", DECODE_CASES)
def test_decode_attention_vs_oracle(b, hq, hkv, length, d, dt, cap):
    g = torch.Generator().manual_seed(length + d)
    q = (torch.randn(b, hq, 1, d, generator=g) * 0.5).to(dt)
    kc = (torch.randn(b, hkv, cap, d, generator=g) * 0.5).to(dt)
    vc = torch.randn(b, hkv, cap, d, generator=g).to(dt)
    kc[:, :, length:] = float("nan")  # past the length: never read
    out = mta.decode_attention(q.cuda(), kc.cuda(), vc.cuda(), length, repeats=hq // hkv)
    torch.cuda.synchronize()
    ref = orc.decode_attention(q[:, :, 0].double().numpy(), kc.double().numpy(), vc.double().numpy(), length, hq // hkv)
    err = np.abs(out[:, :, 0].double().cpu().numpy() - ref).max()
    assert out.shape == (b, hq, 1, d) and out.dtype == dt
    assert err <= 2e-2, err


def test_decode_attention_strided_views_and_errors():
    # the caches are views of a [B, T, H, D] buffer (the projections' layout)
    g = torch.Generator().manual_seed(5)
    base = (torch.randn(2, 64, 2, 64, generator=g) * 0.5).to(torch.bfloat16).cuda()
    kc, vc = base.transpose(1, 2), (base * 0.5).transpose(1, 2)
    q = (torch.randn(2, 8, 1, 64, generator=g) * 0.5).to(torch.bfloat16).cuda()
    out = mta.decode_attention(q, kc, vc, 40, repeats=4)
    ref = orc.decode_attention(q[:, :, 0].double().cpu().numpy(), kc.double().cpu().numpy(),
                               vc.double().cpu().numpy(), 40, 4)
    assert np.abs(out[:, :, 0].double().cpu().numpy() - ref).max() <= 2e-2
    with pytest.raises(ValueError, match="length"):
        mta.decode_attention(q, kc, vc, 65, repeats=4)
    with pytest.raises(ValueError, match="repeats"):
        mta.decode_attention(torch.zeros(1, 24, 1, 64, device="cuda", dtype=torch.bfloat16),
                             torch.zeros(1, 2, 8, 64, device="cuda", dtype=torch.bfloat16),
                             torch.zeros(1, 2, 8, 64, device="cuda", dtype=torch.bfloat16), 4, repeats=16)
    with pytest.raises(RuntimeError, match="float16 and bfloat16"):
        mta.decode_attention(q.float(), kc, vc, 4, repeats=4)


@pytest.mark.parametrize("hq,hkv,length", [(32, 2, 300), (12, 1, 77), (28, 4, 513)])
def test_decode_attention_groups_larger_than_one_launch(hq, hkv, length):
    # more than 8 query heads per KV head (the reference's modal config has 7; any
    # R works there): the group runs as several launches of at most 8 heads
    g = torch.Generator().manual_seed(hq + length)
    b, d, cap = 2, 64, 600
    q = (torch.randn(b, hq, 1, d, generator=g) * 0.5).to(torch.bfloat16).cuda()
    kc = (torch.randn(b, hkv, cap, d, generator=g) * 0.5).to(torch.bfloat16).cuda()
    vc = (torch.randn(b, hkv, cap, d, generator=g) * 0.5).to(torch.bfloat16).cuda()
    r = hq // hkv
    ref = orc.decode_attention(q[:, :, 0].double().cpu().numpy(), kc.double().cpu().numpy(),
                               vc.double().cpu().numpy(), length, r)
    for ln in (length, torch.tensor([length], dtype=torch.int32, device="cuda")):
        out = mta.decode_attention(q, kc, vc, ln, repeats=r)
        assert out.shape == (b, hq, 1, d)
        assert np.abs(out[:, :, 0].double().cpu().numpy() - ref).max() <= 2e-2


@pytest.mark.parametrize("cap", [1024, 1088])
def test_decode_device_length_fused_and_split_paths(cap):
    # a device-side length makes the launch cover the capacity: 16 splits decode in the fused kernel,
    # 17 in the split + combine pair; every length must give the oracle's row either way
    g = torch.Generator().manual_seed(cap)
    b, hq, hkv, d = 3, 8, 2, 64
    q = (torch.randn(b, hq, 1, d, generator=g) * 0.5).to(torch.bfloat16)
    kc = (torch.randn(b, hkv, cap, d, generator=g) * 0.5).to(torch.bfloat16)
    vc = torch.randn(b, hkv, cap, d, generator=g).to(torch.bfloat16)
    qd, kd, vd = q.cuda(), kc.cuda(), vc.cuda()
    length = torch.zeros(1, dtype=torch.int32, device="cuda")
    for ln in (1, 63, 64, 65, 700, 1024, cap):
        length.fill_(ln)
        out = mta.decode_attention(qd, kd, vd, length, repeats=hq // hkv)
        ref = orc.decode_attention(q[:, :, 0].double().numpy(), kc.double().numpy(), vc.double().numpy(), ln,
                                   hq // hkv)
        assert np.abs(out[:, :, 0].double().cpu().numpy() - ref).max() <= 2e-2, ln


def _model(backend, block_size=64, seed=0, **kw):
    torch.manual_seed(seed)
    cfg = dict(vocab_size=128, block_size=block_size, hidden_dim=512, layers=2, attention_heads=8, kv_heads=2,
               dropout=0.0, rope_theta=10_000.0, attention_backend=backend)
    cfg.update(kw)
    return model_mod.TradingModel(**cfg).cuda().eval()


def _rel(a, b):
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("backend", ["hip", "triton"])
def test_cached_logits_match_full_recompute(backend):
    m = _model(backend)
    g = torch.Generator().manual_seed(11)
    tokens = torch.randint(0, 128, (3, 40), generator=g).cuda()
    with torch.no_grad():
        logits, cache, _ = m._prefill(tokens[:, :10])
        assert _rel(logits, m(tokens[:, :10])[:, -1, :]) < 2e-2
        for pos in range(10, 40):  # teacher forcing: feed the true next token
            step = m._decode(tokens[:, pos:pos + 1], cache, pos)
            full = m(tokens[:, :pos + 1])[:, -1, :]
            assert _rel(step, full) < 2e-2, pos


def test_generate_greedy_matches_recompute_and_crosses_the_window():
    # the cached HIP generation against the reference's loop (model.py:134-147) on
    # the same weights, recomputed through the HIP route and through the SDPA
    # route: greedy tokens equal wherever the recompute's top-2 gap is clear of
    # the bf16 attention's rounding
    m = _model("hip", block_size=32)
    for p in m.output.parameters():  # sharper logits: fewer near-ties between top-2 tokens
        p.data.mul_(25.0)
    sdpa = _model("auto", block_size=32)
    sdpa.load_state_dict(m.state_dict())
    g = torch.Generator().manual_seed(12)
    prompt = torch.randint(0, 128, (4, 12), generator=g).cuda()
    out = m.generate(prompt, max_new_tokens=30, top_k=1)  # 12 + 30 > 32: the window slides
    assert out.shape == (4, 42) and torch.equal(out[:, :12], prompt)
    with torch.no_grad():
        for ref_model in (m, sdpa):
            for t in range(12, 42):
                full = ref_model(out[:, max(0, t - 32):t])[:, -1, :]
                top2 = full.topk(2, dim=-1).values
                clear = (top2[:, 0] - top2[:, 1]) > 5e-2 * top2[:, 0].abs().clamp_min(1.0)
                assert torch.equal(out[clear, t], full.argmax(-1)[clear]), (ref_model.operator_backend, t)


def test_generate_sampling_runs_at_c5_shape():
    wl = importlib.import_module("mega-trading_amd.workload")
    m = wl.build_model("hip", seed=0, device="cuda").eval()
    ids, _ = wl.zipf_batch(8, 256, wl.C5_MODEL["vocab_size"])
    torch.manual_seed(0)
    out = m.generate(ids.cuda(), max_new_tokens=16, top_k=16)
    assert out.shape == (8, 272) and int(out.max()) < wl.C5_MODEL["vocab_size"] and int(out.min()) >= 0


@pytest.mark.parametrize("in_dt", [torch.float32, torch.bfloat16])
def test_decode_rope_append_matches_torch_rotation(in_dt):
    attn = importlib.import_module("mega-trading_amd.attention")
    g = torch.Generator().manual_seed(21)
    b, hq, hkv, d, cap, pos = 3, 8, 2, 64, 40, 17
    proj_q = torch.randn(b, 1, hq * d, generator=g).to(in_dt).cuda()
    proj_kv = torch.randn(b, 1, 2 * hkv * d, generator=g).to(in_dt).cuda()
    q = proj_q.view(b, 1, hq, d).transpose(1, 2)               # strided views, as the model passes them
    k = proj_kv[..., : hkv * d].view(b, 1, hkv, d).transpose(1, 2)
    v = proj_kv[..., hkv * d:].view(b, 1, hkv, d).transpose(1, 2)
    rope = model_mod.RotaryEmbedding(d, 64, theta=10_000.0).cuda()
    kc = torch.zeros(b, hkv, cap, d, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    q_rot = attn.decode_rope_append(q, k, v, rope.cos, rope.sin, pos, kc, vc)
    c, s = rope.cos[0, 0, pos:pos + 1], rope.sin[0, 0, pos:pos + 1]
    ref_q = model_mod.rotate(q.to(torch.bfloat16).float(), c, s).to(torch.bfloat16)
    ref_k = model_mod.rotate(k.to(torch.bfloat16).float(), c, s).to(torch.bfloat16)
    for got, ref in ((q_rot, ref_q), (kc[:, :, pos:pos + 1], ref_k)):
        assert float((got == ref).float().mean()) > 0.99  # last-ulp fp32 differences may flip a rounding
        torch.testing.assert_close(got.float(), ref.float(), rtol=2 ** -7, atol=1e-6)
    assert torch.equal(vc[:, :, pos], v[:, :, 0].to(torch.bfloat16))
    assert not kc[:, :, :pos].any() and not kc[:, :, pos + 1:].any()  # only row pos written


def test_decode_rope_append_validates_its_arguments():
    attn = importlib.import_module("mega-trading_amd.attention")
    b, hq, hkv, d, cap = 2, 8, 2, 64, 16
    q = torch.zeros(b, hq, 1, d, device="cuda", dtype=torch.bfloat16)
    k = torch.zeros(b, hkv, 1, d, device="cuda", dtype=torch.bfloat16)
    kc = torch.zeros(b, hkv, cap, d, device="cuda", dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    rope = model_mod.RotaryEmbedding(d, 32, theta=10_000.0).cuda()
    # a 16-bit table (a model cast with .to(dtype)) is read as fp32: same rotation as the fp32 table
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    kr = torch.randn(b, hkv, 1, d, device="cuda").to(torch.bfloat16)
    attn.decode_rope_append(q, kr, kr, rope.cos, rope.sin, 3, kc, vc)
    attn.decode_rope_append(q, kr, kr, rope.cos.to(torch.bfloat16).float(), rope.sin.to(torch.bfloat16).float(), 3,
                            kc2, vc2)
    kc3, vc3 = torch.zeros_like(kc), torch.zeros_like(vc)
    attn.decode_rope_append(q, kr, kr, rope.cos.to(torch.bfloat16), rope.sin.to(torch.bfloat16), 3, kc3, vc3)
    assert torch.equal(kc3, kc2) and torch.equal(vc3, vc)
    with pytest.raises(ValueError, match="head_dim/2"):
        attn.decode_rope_append(q, k, k, rope.cos[..., :16], rope.sin[..., :16], 3, kc, vc)
    with pytest.raises(ValueError, match="unit last-dim stride"):
        attn.decode_rope_append(q, k, torch.zeros(b, hkv, 1, 2 * d, device="cuda", dtype=torch.bfloat16)[..., ::2],
                                rope.cos, rope.sin, 3, kc, vc)
    with pytest.raises(ValueError, match="outside the cache"):
        attn.decode_rope_append(q, k, k, rope.cos, rope.sin, cap, kc, vc)
    with pytest.raises(RuntimeError, match="one device"):
        attn.decode_rope_append(q, k, k, rope.cos.cpu(), rope.sin.cpu(), 3, kc, vc)
    with pytest.raises(RuntimeError, match="ROCm GPU"):
        attn.decode_rope_append(q.cpu(), k.cpu(), k.cpu(), rope.cos, rope.sin, 3, kc, vc)


def test_graph_decode_replays_match_eager_decode():
    # one recorded decode step, replayed per position (device-side token and position), against
    # the eager step with a host position, token for token, with eager work between the replays
    m = _model("hip")
    g = torch.Generator().manual_seed(31)
    tokens = torch.randint(0, 128, (4, 30), generator=g).cuda()
    with torch.no_grad():
        _, cache_a, _ = m._prefill(tokens[:, :12])
        cache_b = [(k.clone(), v.clone()) for k, v in cache_a]
        step = model_mod._DecodeGraph(m, cache_b, 4, tokens.device)
        for pos in range(12, 30):
            eager = m._decode(tokens[:, pos:pos + 1], cache_a, pos)
            torch.cuda.synchronize()
            replay = step(tokens[:, pos:pos + 1], pos).clone()
            torch.cuda.synchronize()
            assert torch.equal(replay, eager), pos
        for (ka, va), (kb, vb) in zip(cache_a, cache_b):
            assert torch.equal(ka[:, :, :30], kb[:, :, :30]) and torch.equal(va[:, :, :30], vb[:, :, :30])


def test_generate_with_graphs_equals_without():
    m = _model("hip", block_size=48)
    g = torch.Generator().manual_seed(32)
    prompt = torch.randint(0, 128, (3, 10), generator=g).cuda()
    m.decode_graphs = False
    a = m.generate(prompt, max_new_tokens=45, top_k=1)  # crosses block_size 48 at the end
    m.decode_graphs = True
    b = m.generate(prompt, max_new_tokens=45, top_k=1)
    assert torch.equal(a, b)


def test_generate_reuses_the_recorded_step_across_calls():
    # a second generate call with the same batch prefills into the kept caches
    # and replays the same recording; its tokens equal a fresh model's and the
    # eager (graph-free) path's; another batch size records anew
    m = _model("hip", block_size=48)
    g = torch.Generator().manual_seed(33)
    p1 = torch.randint(0, 128, (3, 10), generator=g).cuda()
    p2 = torch.randint(0, 128, (3, 14), generator=g).cuda()
    first = m.generate(p1, max_new_tokens=20, top_k=1)
    state = m._gen_state
    assert state is not None and state[0][0] == 3
    second = m.generate(p2, max_new_tokens=20, top_k=1)
    assert m._gen_state is state  # same caches and recording
    fresh = _model("hip", block_size=48)
    fresh.decode_graphs = False
    assert torch.equal(first, fresh.generate(p1, max_new_tokens=20, top_k=1))
    assert torch.equal(second, fresh.generate(p2, max_new_tokens=20, top_k=1))
    p3 = torch.randint(0, 128, (5, 9), generator=g).cuda()
    third = m.generate(p3, max_new_tokens=8, top_k=1)
    assert m._gen_state is not state and m._gen_state[0][0] == 5
    assert torch.equal(third, fresh.generate(p3, max_new_tokens=8, top_k=1))


def test_generate_records_anew_after_weight_or_precision_changes():
    # a recording reads the weights by address and bakes in a dtype and an
    # autocast path: after .to(bfloat16), load_state_dict(assign=True) or a
    # different autocast state the next call records again, and its tokens equal
    # the graph-free path on the model as it now is
    g = torch.Generator().manual_seed(36)
    prompt = torch.randint(0, 128, (3, 10), generator=g).cuda()

    def eager(model):
        model.decode_graphs = False
        try:
            return model.generate(prompt, max_new_tokens=16, top_k=1)
        finally:
            model.decode_graphs = True

    m = _model("hip", block_size=48)
    m.generate(prompt, max_new_tokens=16, top_k=1)
    state = m._gen_state
    m.to(torch.bfloat16)
    after_cast = m.generate(prompt, max_new_tokens=16, top_k=1)
    assert m._gen_state is not state
    assert torch.equal(after_cast, eager(m))
    state = m._gen_state
    other = _model("hip", block_size=48, seed=7).to(torch.bfloat16)
    m.load_state_dict(other.state_dict(), assign=True)
    after_load = m.generate(prompt, max_new_tokens=16, top_k=1)
    assert m._gen_state is not state
    assert torch.equal(after_load, eager(other))
    m2 = _model("hip", block_size=48)
    m2.generate(prompt, max_new_tokens=16, top_k=1)
    state = m2._gen_state
    with torch.autocast("cuda", dtype=torch.bfloat16):
        under_amp = m2.generate(prompt, max_new_tokens=16, top_k=1)
        assert m2._gen_state is not state
        assert torch.equal(under_amp, eager(m2))


def test_recorded_sampling_reproduces_the_eager_draw():
    # the recorded step samples with torch.multinomial's one-sample draw minus
    # its host-synchronising check: the same tokens for the same seed, for the
    # draw alone and for whole top-k 16 generations (recording call and reuse)
    g = torch.Generator().manual_seed(35)
    logits = (torch.randn(6, 128, generator=g) * 3).cuda()
    for k in (1, 16, 0):
        torch.manual_seed(9)
        x = model_mod._sample_next(logits, k)
        torch.manual_seed(9)
        y = model_mod._sample_recorded(logits, k)
        assert torch.equal(x, y), k
    m = _model("hip", block_size=64)
    prompt = torch.randint(0, 128, (3, 10), generator=g).cuda()
    torch.manual_seed(5)
    m.decode_graphs = False
    eager = m.generate(prompt, max_new_tokens=20, top_k=16)
    m.decode_graphs = True
    torch.manual_seed(5)
    recorded = m.generate(prompt, max_new_tokens=20, top_k=16)
    torch.manual_seed(5)
    reused = m.generate(prompt, max_new_tokens=20, top_k=16)
    assert torch.equal(eager, recorded) and torch.equal(recorded, reused)


def test_recorded_decode_with_a_large_vocabulary_samples_like_the_eager_step():
    # over a 16 k vocabulary torch.topk takes its multi-block path, which clears counters with
    # hipMemsetAsync; the sampling therefore runs after each replay, outside the recording.  32 rollouts
    # x 24 tokens with the recorded step (recording call and reuse) against the eager step, same seed
    g = torch.Generator().manual_seed(41)
    m = _model("hip", block_size=64, vocab_size=16384, hidden_dim=128, attention_heads=4, kv_heads=1)
    prompt = torch.randint(0, 16384, (32, 12), generator=g).cuda()
    torch.manual_seed(3)
    m.decode_graphs = False
    eager = m.generate(prompt, max_new_tokens=24, top_k=16)
    m.decode_graphs = True
    for _ in range(2):
        torch.manual_seed(3)
        recorded = m.generate(prompt, max_new_tokens=24, top_k=16)
        torch.cuda.synchronize()
        assert torch.equal(recorded, eager)


@pytest.mark.parametrize("b,hq,hkv,d,cap,pos,in_dt,dev", [
    (3, 8, 2, 64, 40, 17, torch.float32, False),
    (2, 8, 2, 64, 512, 511, torch.float32, True),      # the last position of one 8-wave workgroup
    (2, 6, 2, 32, 513, 512, torch.bfloat16, True),     # the first of a second workgroup
    (33, 4, 2, 64, 1024, 1023, torch.float32, True),   # 66 (batch, KV head) pairs: one 16-wave workgroup
    (32, 4, 2, 64, 1025, 1024, torch.float32, False),  # 4-wave workgroups and the merge
    (2, 7, 1, 128, 300, 64, torch.float16, True),
    (1, 8, 1, 128, 2048, 63, torch.float32, False),
    (2, 9, 1, 64, 128, 5, torch.float32, False),       # a group of 9 heads: the two calls
])
def test_decode_append_attention_equals_the_two_calls(b, hq, hkv, d, cap, pos, in_dt, dev):
    attn = importlib.import_module("mega-trading_amd.attention")
    dt = torch.float16 if in_dt == torch.float16 else torch.bfloat16
    g = torch.Generator().manual_seed(cap + pos)
    qkv = torch.randn(b, 1, (hq + 2 * hkv) * d, generator=g).to(in_dt).cuda()  # a packed projection
    q, k, v = (t.view(b, 1, -1, d).transpose(1, 2) for t in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    rope = model_mod.RotaryEmbedding(d, cap, theta=10_000.0).cuda()
    kc, vc = (torch.randn(b, hkv, cap, d, generator=g).to(dt).cuda() for _ in range(2))
    at = torch.tensor([pos], dtype=torch.int32, device="cuda") if dev else pos
    for length in {pos + 1, max(1, pos // 2), min(cap, pos + 70)}:  # also lengths that are not pos + 1
        n = torch.tensor([length], dtype=torch.int32, device="cuda") if dev else length
        k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        k2[:, :, pos] = v2[:, :, pos] = float("nan")  # the stale rows are never used
        ref = attn.decode_attention(attn.decode_rope_append(q, k, v, rope.cos, rope.sin, at, k1, v1), k1, v1, n,
                                    repeats=hq // hkv)
        got = attn.decode_append_attention(q, k, v, rope.cos, rope.sin, at, n, k2, v2, repeats=hq // hkv)
        assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(ref, got), length


@pytest.mark.parametrize("which", ["query", "value", "cos", "value_cache"])
@pytest.mark.parametrize("dev", [False, True])
def test_decode_append_attention_takes_misaligned_tensors(which, dev):
    """A tensor that starts 8 bytes past a 16-byte boundary: the values of the two calls, which refuse such
    a table or cache."""
    attn = importlib.import_module("mega-trading_amd.attention")
    b, hq, hkv, d, cap, pos = 3, 8, 2, 64, 80, 66

    def place(t, name):
        if name != which:
            return t.cuda()
        shift = 8 // t.element_size()
        flat = torch.empty(t.numel() + shift, dtype=t.dtype, device="cuda")[shift:]
        return flat.copy_(t.reshape(-1)).view(t.shape)

    g = torch.Generator().manual_seed(11)
    rope = model_mod.RotaryEmbedding(d, cap, theta=10_000.0)
    q, k, v = (place(torch.randn(b, n, 1, d, generator=g), name) for n, name in ((hq, "query"), (hkv, "key"), (hkv, "value")))
    cos, sin = place(rope.cos, "cos"), rope.sin.cuda()
    kc, vc = (torch.randn(b, hkv, cap, d, generator=g).bfloat16() for _ in range(2))
    at, n = ((torch.tensor([x], dtype=torch.int32, device="cuda") for x in (pos, pos + 1)) if dev else (pos, pos + 1))
    k1, v1, k2, v2 = place(kc, "key_cache"), place(vc, "value_cache"), kc.cuda(), vc.cuda()
    if which in ("cos", "value_cache"):
        with pytest.raises(RuntimeError, match="16-byte aligned"):
            attn.decode_append_attention(q, k, v, cos, sin, at, n, k1, v1, repeats=hq // hkv)
        return
    got = attn.decode_append_attention(q, k, v, cos, sin, at, n, k1, v1, repeats=hq // hkv)
    ref = attn.decode_attention(attn.decode_rope_append(q, k, v, cos, sin, at, k2, v2), k2, v2, n, repeats=hq // hkv)
    assert torch.equal(k1, k2) and torch.equal(v1, v2) and torch.equal(got, ref)


@pytest.mark.parametrize("dev", [False, True])
def test_compiled_decode_step_equals_the_eager_one(dev):
    """One functionalized graph that writes the caches: values and caches of the eager step, three steps in a row."""
    attn = importlib.import_module("mega-trading_amd.attention")
    b, hq, hkv, d, cap = 3, 8, 2, 64, 48
    g = torch.Generator(device="cuda").manual_seed(21)
    rope = model_mod.RotaryEmbedding(d, cap, theta=10_000.0).cuda()
    k1, v1 = (torch.randn(b, hkv, cap, d, generator=g, device="cuda").bfloat16() for _ in range(2))
    k2, v2 = k1.clone(), v1.clone()
    torch._dynamo.reset()
    step = torch.compile(attn.decode_append_attention, fullgraph=True, backend="aot_eager")
    for pos in (17, 18, 19):
        q, k, v = (torch.randn(b, n, 1, d, generator=g, device="cuda") for n in (hq, hkv, hkv))
        at, n = ((torch.tensor([x], dtype=torch.int32, device="cuda") for x in (pos, pos + 1)) if dev else (pos, pos + 1))
        with torch.no_grad():
            got = step(q, k, v, rope.cos, rope.sin, at, n, k1, v1, repeats=hq // hkv)
            ref = attn.decode_append_attention(q, k, v, rope.cos, rope.sin, at, n, k2, v2, repeats=hq // hkv)
        assert torch.equal(got, ref) and torch.equal(k1, k2) and torch.equal(v1, v2), pos
