"""The patched attention forward / model routing on the GPU: cache bookkeeping,
prefill quantisation of the strided wqkv views, decode through the fused kernel."""
import math
import os

import numpy as np
import pytest
import torch

from oracle import cq_oracle as O
from tests.util import to_np

pytestmark = pytest.mark.gpu


def _tiny_model(layers=2, seed=0, vit=None):
    from calibquant_amd.internlm2 import InternLM2Config, InternVLChatStandIn
    torch.manual_seed(seed)
    m = InternVLChatStandIn(InternLM2Config.tiny(layers), vit=vit).cuda().to(torch.bfloat16).eval()
    return m


def test_patched_forward_decode_matches_oracle_on_one_layer():
    """Prefill S + T + text tokens, then one decode step: the layer's attention output equals
    wo(oracle attention) built from the module's own packed state and fp window."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    torch.manual_seed(1)
    cfg = InternLM2Config.tiny()
    att = InternLM2Attention(cfg).cuda().to(torch.bfloat16)
    att.cq_sprompt_len, att.cq_image_token_num = 5, 200
    B, S, T, TXT = 2, 5, 200, 11
    N = S + T + TXT
    x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    pos = torch.arange(N, device="cuda")[None].expand(B, N)
    with torch.no_grad():
        out_p, _, past = pi.forward_internlm2_calibquant(att, x, None, pos, None, False, True)
        assert out_p.shape == (B, N, cfg.hidden_size)
        assert past[0].shape == (B, cfg.num_key_value_heads, S + TXT, 128)
        assert att.encoded_features_k.shape == (B, cfg.num_key_value_heads, T, 16)
        assert att.scale_key.shape == (B, cfg.num_attention_heads, 1, 128)
        # the packed state equals the oracle's quantisation of the post-RoPE image keys / raw values
        q, k, v = att.split_qkv(x)
        cos, sin = att.rotary_emb(v, seq_len=N)
        qr, kr = pi.apply_rotary_pos_emb(q.transpose(1, 2), k.transpose(1, 2), cos, sin, pos)
        ck, sk, zk = O.quantize_pack(to_np(kr[:, :, S:S + T].transpose(1, 2)), 1, 0.5, "bf16")
        cv, sv, zv = O.quantize_pack(to_np(v[:, S:S + T]), 1, 0.3, "bf16")
        assert np.array_equal(att.encoded_features_k.cpu().numpy(), ck)
        assert np.array_equal(att.encoded_features_v.cpu().numpy(), cv)
        # one decode step with an additive mask that hides two positions
        xd = torch.randn(B, 1, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
        posd = torch.full((B, 1), N, device="cuda", dtype=torch.long)
        mask = torch.zeros(B, 1, 1, N + 1, device="cuda", dtype=torch.bfloat16)
        mask[0, 0, 0, 2] = mask[1, 0, 0, S + 7] = torch.finfo(torch.bfloat16).min
        out_d, _, past2 = pi.forward_internlm2_calibquant(att, xd, mask, posd, past, False, True)
        assert past2[0].shape[2] == S + TXT + 1 and past2[0].data_ptr() == past[0].data_ptr()
        qd, kd, vd = att.split_qkv(xd)
        cos, sin = att.rotary_emb(vd, seq_len=N + 1)
        qd, kd = pi.apply_rotary_pos_emb(qd.transpose(1, 2), kd.transpose(1, 2), cos, sin, posd)
        want = O.decode_attention(to_np(qd[:, :, 0]), ck, cv, sk, zk, sv, zv, to_np(past2[0]), to_np(past2[1]),
                                  S, 1, mask=to_np(mask[:, 0, 0]))
        want = torch.from_numpy(want).cuda().to(torch.bfloat16).reshape(B, 1, -1)
        ref = att.wo(want)
        err = (out_d.float() - ref.float()).abs()
        assert err.max().item() < 2e-2 and err.mean().item() < 2e-3


def test_masked_steady_state_decode_of_a_left_padded_batch():
    """A batch whose second sample is left-padded by four positions: prefill with the (B, kv) padding mask,
    then eight decode steps that each pass the additive (B, 1, 1, kv) mask the reference adds per step
    (patch_internvl.py:404-410).  Every step's attention output equals wo(oracle attention with that mask) on
    the module's own packed state and window; the step times with and without the mask are printed (a masked
    step cannot take the prepared-call fast path: its call object is rebuilt every step)."""
    import time
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    torch.manual_seed(7)
    cfg = InternLM2Config.tiny()
    B, S, T, TXT, PAD, STEPS = 2, 5, 200, 11, 4, 8
    N = S + T + TXT
    lo = torch.finfo(torch.bfloat16).min

    def run(masked):
        torch.manual_seed(8)
        att = InternLM2Attention(cfg).cuda().to(torch.bfloat16)
        att.cq_sprompt_len, att.cq_image_token_num = S, T
        x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
        pos = torch.arange(N, device="cuda")[None].expand(B, N).clone()
        pad = None
        if masked:
            pad = torch.ones(B, N, device="cuda", dtype=torch.bool)
            pad[1, :PAD] = False
            pos[1] = (pos[1] - PAD).clamp_(min=0)
        outs, times = [], []
        with torch.no_grad():
            _, _, past = pi.forward_internlm2_calibquant(att, x, pad, pos, None, False, True)
            ck, cv = att.encoded_features_k.cpu().numpy(), att.encoded_features_v.cpu().numpy()
            sk, zk, sv, zv = (to_np(t) for t in att._cq_stats)
            for i in range(STEPS):
                xd = torch.randn(B, 1, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
                posd = pos[:, -1:] + 1 + i
                mask = None
                if masked:
                    mask = torch.zeros(B, 1, 1, N + 1 + i, device="cuda", dtype=torch.bfloat16)
                    mask[1, 0, 0, :PAD] = lo
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                out_d, _, past = pi.forward_internlm2_calibquant(att, xd, mask, posd, past, False, True)
                torch.cuda.synchronize()
                times.append(time.perf_counter() - t0)
                qd, kd, vd = att.split_qkv(xd)
                cos, sin = att.rotary_emb(vd, seq_len=N + 1 + i)
                qd, _ = pi.apply_rotary_pos_emb(qd.transpose(1, 2), kd.transpose(1, 2), cos, sin, posd)
                m = None if mask is None else to_np(mask[:, 0, 0])
                want = O.decode_attention(to_np(qd[:, :, 0]), ck, cv, sk, zk, sv, zv, to_np(past[0]), to_np(past[1]), S, 1, mask=m)
                ref = att.wo(torch.from_numpy(want).cuda().to(torch.bfloat16).reshape(B, 1, -1))
                err = (out_d.float() - ref.float()).abs()
                assert err.max().item() < 2e-2 and err.mean().item() < 2e-3, (masked, i, err.max().item())
                outs.append(out_d)
        return outs, sorted(times)[len(times) // 2]

    _, t_mask = run(True)
    _, t_plain = run(False)
    print(f"\nmasked decode step {t_mask * 1e6:.0f} us, unmasked {t_plain * 1e6:.0f} us per layer (host-inclusive, tiny layer)")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_decode_step_equals_the_unfused_op_chain(dtype):
    """Several decode steps through the one-launch split + rotary + append path - once driven by the host
    shim's `LayerStep` (the default), once by the Python call objects - and through the chain of torch ops
    (forced by int32 position ids): same outputs and same window, bit for bit."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    cfg = InternLM2Config.tiny()
    B, S, T, TXT = 3, 4, 130, 9
    N = S + T + TXT
    outs, wins = [], []
    for fused, shim in ((True, True), (True, False), (False, False)):
        torch.manual_seed(7)
        att = InternLM2Attention(cfg).cuda().to(dtype)
        att.cq_sprompt_len, att.cq_image_token_num = S, T
        att.cq_no_step_shim = not shim
        x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=dtype)
        pos = torch.arange(N, device="cuda")[None].expand(B, N)
        with torch.no_grad():
            _, _, past = pi.forward_internlm2_calibquant(att, x, None, pos, None, False, True)
            step_out = []
            for i in range(300):   # beyond the first window capacity: the buffers are regrown on the way
                xd = torch.randn(B, 1, cfg.hidden_size, device="cuda", dtype=dtype)
                posd = torch.full((B, 1), N + i, device="cuda", dtype=torch.long)
                o, _, past = pi.forward_internlm2_calibquant(att, xd, None, posd if fused else posd.int(), past,
                                                            False, True)
                if i % 37 == 0 or i == 299:
                    step_out.append(o.clone())
        assert hasattr(att, "_cq_rope_call") == fused
        if shim:    # every step after the first went through the shim, which regrew the window on the way
            step = att._cq_step[0]
            assert step.steps == 299 and step.length == S + TXT + 300 and step.capacity >= step.length
        else:
            assert "_cq_step" not in att.__dict__
        outs.append(torch.stack(step_out))
        wins.append((past[0].clone(), past[1].clone()))
    assert wins[0][0].shape == (B, cfg.num_key_value_heads, S + TXT + 300, 128)
    for other in (1, 2):
        assert torch.equal(wins[0][0], wins[other][0]) and torch.equal(wins[0][1], wins[other][1])
        assert torch.equal(outs[0], outs[other])


def test_fused_decode_step_on_a_chunked_context():
    """A context whose packed tokens take several chunks (a call with a workspace): the steady-state decode step
    goes through the host shim and the re-aimed call object all the same, and both give the bits of the path that
    prepares a new call on every step."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    cfg = InternLM2Config.tiny()
    dtype = torch.bfloat16
    B, S, T, TXT = 2, 4, 20000, 9
    N = S + T + TXT
    outs = []
    for mode in ("shim", "call", "fresh"):
        torch.manual_seed(11)
        att = InternLM2Attention(cfg).cuda().to(dtype)
        att.cq_sprompt_len, att.cq_image_token_num = S, T
        att.cq_no_step_shim = mode != "shim"
        x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=dtype)
        pos = torch.arange(N, device="cuda")[None].expand(B, N)
        with torch.no_grad():
            _, _, past = pi.forward_internlm2_calibquant(att, x, None, pos, None, False, True)
            step_out = []
            for i in range(12):
                xd = torch.randn(B, 1, cfg.hidden_size, device="cuda", dtype=dtype)
                posd = torch.full((B, 1), N + i, device="cuda", dtype=torch.long)
                if mode == "fresh":
                    att._cq_call = None     # a new prepared call (and plan) on every step
                o, _, past = pi.forward_internlm2_calibquant(att, xd, None, posd, past, False, True)
                step_out.append(o.clone())
                if i == 0:
                    plan = att._cq_call.plan()
                    assert plan["chunks"] > 1 and att._cq_call.workspace_bytes > 0
        if mode == "shim":
            assert att._cq_step[0].steps == 11
        else:
            assert "_cq_step" not in att.__dict__
        outs.append(torch.stack(step_out))
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_patched_model_without_image_tokens_equals_the_fp_model():
    """With zero packed tokens the quantised path is plain attention over the fp window."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention
    from calibquant_amd.internlm2 import InternVLChatStandIn
    m = _tiny_model()
    lm = m.language_model
    fp_forward, fp_generate = InternLM2Attention.forward, InternVLChatStandIn.generate
    ids = torch.randint(0, 500, (2, 40), device="cuda")
    nxt = torch.randint(0, 500, (2, 1), device="cuda")
    pos = torch.arange(40, device="cuda")[None].expand(2, 40)
    pos1 = torch.full((2, 1), 40, device="cuda", dtype=torch.long)

    def two_steps():
        emb = lm.get_input_embeddings()
        l0, past = lm.forward_step(emb(ids), pos, None)
        l1, past = lm.forward_step(emb(nxt), pos1, past)
        return l0.float(), l1.float()

    try:
        with torch.no_grad():
            b0, b1 = two_steps()
            pi.patch_model(m, "calibquant", sprompt_len=0)
            for layer in lm.model.layers:
                layer.attention.cq_image_token_num = 0
            p0, p1 = two_steps()
        assert torch.allclose(b0, p0, atol=3e-2, rtol=3e-2)
        assert torch.allclose(b1, p1, atol=3e-2, rtol=3e-2)
    finally:
        InternLM2Attention.forward, InternVLChatStandIn.generate = fp_forward, fp_generate


@pytest.mark.parametrize("tower", ["stand-in", "internvit"])
def test_patch_model_and_custom_generate_end_to_end(tower):
    """Synthetic tiles -> 256 image tokens each, quantised at prefill, 8 greedy tokens.  With the
    InternViT-shaped tower the 12 tiles go through `extract_feature` in two chunks (10 + 2), as the
    reference's `custom_generate` runs them (patch_internvl.py:53-65)."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternVLChatStandIn
    from calibquant_amd.internvit import InternViTConfig
    fp_forward, fp_generate = InternLM2Attention.forward, InternVLChatStandIn.generate
    m = _tiny_model(seed=3, vit=InternViTConfig.tiny() if tower == "internvit" else None)
    B, S, tiles, txt = (2, 41, 6, 9) if tower == "internvit" else (2, 41, 2, 9)
    T = tiles * 256
    ids = torch.randint(0, 500, (B, S + T + txt), device="cuda")
    ids[:, S:S + T] = m.img_context_token_id
    pix = torch.rand(B * tiles, 3, 448, 448, device="cuda", dtype=torch.bfloat16)
    try:
        pi.patch_model(m, "calibquant")
        os.environ.pop("IMAGE_TOKEN_NUM", None)
        out = m.generate(pixel_values=pix, input_ids=ids, max_new_tokens=8)
        assert out.shape == (B, 8)
        assert os.environ["IMAGE_TOKEN_NUM"] == str(T)
        att = m.language_model.model.layers[0].attention
        assert att.encoded_features_k.shape == (B, 2, T, 16) and att.encoded_features_k.dtype == torch.uint8
        assert att._cq_step[0].length == S + txt + 7
        out2 = m.generate(pixel_values=pix, input_ids=ids, max_new_tokens=8)
        assert torch.equal(out, out2)
    finally:
        InternLM2Attention.forward, InternVLChatStandIn.generate = fp_forward, fp_generate


def _prefill(m, ids, pix=None):
    """Prompt embeddings (image features spliced in) -> last-position logits and the per-layer cache."""
    lm = m.language_model
    emb = lm.get_input_embeddings()(ids)
    if pix is not None:
        vit = m.extract_feature(pix)
        emb = emb.clone()
        emb[ids == m.img_context_token_id] = vit.reshape(-1, emb.shape[-1]).to(emb.dtype)
    B, N = ids.shape
    pos = torch.arange(N, device=ids.device)[None].expand(B, N)
    return lm.forward_step(emb, pos, None)


@pytest.mark.parametrize("quantized,fp_kernel,width", [(True, False, "tiny"), (False, False, "tiny"), (False, True, "tiny"),
                                                       (True, False, "26b")])
def test_static_decoder_graph_replays_equal_eager_steps(quantized, fp_kernel, width):
    """The recorded decode step, replayed per token, produces the tokens of the same step run
    eagerly, and its first step agrees with the model's own eager step.  `26b`: two layers of the
    InternLM2-20B width (hidden 6 144, 48 query / 8 kv heads: units of three heads) at batch 6."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.graph_decode import StaticDecoder
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config, InternVLChatStandIn
    fp_forward, fp_generate = InternLM2Attention.forward, InternVLChatStandIn.generate
    if width == "26b":
        torch.manual_seed(5)
        cfg = InternLM2Config(vocab_size=512, hidden_size=6144, intermediate_size=16384, num_hidden_layers=2,
                              num_attention_heads=48, num_key_value_heads=8, max_position_embeddings=8192)
        m = InternVLChatStandIn(cfg).cuda().to(torch.bfloat16).eval()
    else:
        m = _tiny_model(seed=5)
    lm = m.language_model
    B, S, tiles, txt, NEW = (6 if width == "26b" else 2), 41, 2, 9, 12
    T = tiles * 256
    ids = torch.randint(0, 500, (B, S + T + txt), device="cuda")
    ids[:, S:S + T] = m.img_context_token_id
    pix = torch.rand(B * tiles, 3, 448, 448, device="cuda", dtype=torch.bfloat16)
    N = ids.shape[1]
    try:
        with torch.no_grad():
            if quantized:
                pi.patch_model(m, "calibquant")
                for layer in lm.model.layers:
                    layer.attention.cq_image_token_num = T
            runs = []
            for use_graph in (False, True):
                logits, past = _prefill(m, ids, pix)
                first = logits[:, -1].argmax(-1)
                dec = StaticDecoder(lm, past, N, NEW, fp_kernel=fp_kernel)
                toks = dec.generate(first, NEW, use_graph=use_graph)
                torch.cuda.synchronize()
                assert (dec.graph is not None) == use_graph
                runs.append(toks)
            assert torch.equal(runs[0], runs[1])
            # first decode step against the model's eager forward_step (different norm kernel,
            # same arithmetic up to rounding)
            logits, past = _prefill(m, ids, pix)
            first = logits[:, -1].argmax(-1)
            dec = StaticDecoder(lm, past, N, 2, fp_kernel=fp_kernel)
            dec.tok.copy_(first)
            x = lm.get_input_embeddings()(first)[:, None]
            pos1 = torch.full((B, 1), N, device="cuda", dtype=torch.long)
            want, _ = lm.forward_step(x, pos1, past)
            lay = lm.model.layers
            got_tok = dec.step().clone()
            assert runs[0][:, 1].tolist() == got_tok.tolist()
            # the eager model's choice has (near-)maximal logit under the static step as well
            w = want[:, -1].float()
            assert ((w.max(-1).values - w.gather(1, got_tok[:, None])[:, 0]) < 0.15).all()
    finally:
        InternLM2Attention.forward, InternVLChatStandIn.generate = fp_forward, fp_generate


def test_patched_model_with_per_token_values():
    """`patch_model(..., v_mode="token")`: values quantised per token at prefill, decoded by the
    fused kernel; one layer's decode output against the oracle on the module's own state."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    torch.manual_seed(9)
    cfg = InternLM2Config.tiny()
    att = InternLM2Attention(cfg).cuda().to(torch.bfloat16)
    att.cq_sprompt_len, att.cq_image_token_num, att.cq_v_mode = 4, 300, "token"
    B, S, T, TXT = 2, 4, 300, 6
    N = S + T + TXT
    x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
    pos = torch.arange(N, device="cuda")[None].expand(B, N)
    with torch.no_grad():
        _, _, past = pi.forward_internlm2_calibquant(att, x, None, pos, None, False, True)
        assert att.encoded_features_v.dtype == torch.int32 and att.encoded_features_v.shape == (B, 2, T, 4)
        assert att.scale_value.shape == (B, cfg.num_attention_heads, T, 4)
        _, _, v = att.split_qkv(x)
        w_ref, s_ref, m_ref = O.kivi_quantize_pack(to_np(v[:, S:S + T].transpose(1, 2)), 32, 1, "bf16")
        assert np.array_equal(att.encoded_features_v.cpu().numpy(), w_ref)
        xd = torch.randn(B, 1, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
        posd = torch.full((B, 1), N, device="cuda", dtype=torch.long)
        out_d, _, past2 = pi.forward_internlm2_calibquant(att, xd, None, posd, past, False, True)
        qd, kd, vd = att.split_qkv(xd)
        cos, sin = att.rotary_emb(vd, seq_len=N + 1)
        qd, kd = pi.apply_rotary_pos_emb(qd.transpose(1, 2), kd.transpose(1, 2), cos, sin, posd)
        ks, kz, _, _ = att._cq_stats
        want = O.decode_attention(to_np(qd[:, :, 0]), att.encoded_features_k.cpu().numpy(), w_ref, to_np(ks), to_np(kz),
                                  s_ref, m_ref, to_np(past2[0]), to_np(past2[1]), S, 1, v_token_group=32)
        ref = att.wo(torch.from_numpy(want).cuda().to(torch.bfloat16).reshape(B, 1, -1))
        err = (out_d.float() - ref.float()).abs()
        assert err.max().item() < 2e-2 and err.mean().item() < 2e-3


def test_two_prefills_follow_the_environment_variable(monkeypatch):
    """Two prompts through the patched forward with only IMAGE_TOKEN_NUM updated in between
    (no custom_generate, no attribute): each prefill quantises its own image slice, and a 4-D
    prefill mask is refused instead of being dropped."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd._lib import CalibQuantError
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    torch.manual_seed(3)
    cfg = InternLM2Config.tiny()
    att = InternLM2Attention(cfg).cuda().to(torch.bfloat16)
    att.cq_sprompt_len = 3
    B = 2
    with torch.no_grad():
        for T in (200, 72):
            monkeypatch.setenv("IMAGE_TOKEN_NUM", str(T))
            N = 3 + T + 5
            x = torch.randn(B, N, cfg.hidden_size, device="cuda", dtype=torch.bfloat16)
            pos = torch.arange(N, device="cuda")[None].expand(B, N)
            _, _, past = pi.forward_internlm2_calibquant(att, x, None, pos, None, False, True)
            assert att.image_token_num == T and att.encoded_features_k.shape[2] == T
            assert past[0].shape[2] == N - T
            q, k, v = att.split_qkv(x)
            cv, _, _ = O.quantize_pack(to_np(v[:, 3:3 + T]), 1, 0.3, "bf16")
            assert np.array_equal(att.encoded_features_v.cpu().numpy(), cv)
        with pytest.raises(CalibQuantError):
            pi.forward_internlm2_calibquant(att, x, torch.zeros(B, 1, N, N, device="cuda"), pos, None, False, True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 2048, 8), (2, 2560, 24), (3, 4096, 520), (4, 4096, 6144), (5, 6144, 1032), (8, 4096, 4096),
                                   (1, 4096, 6144), (7, 2048, 6144), (8, 8192, 40), (2, 16896, 16)])
def test_linear_rows(shape, dtype):
    """Dot products (one row, two) and one to three tiles a workgroup, pieces and slices beside the eight in flight, rows of x apart; against 64 bits, no further off than
    the library's product beyond one unit of the sums' last places."""
    import ctypes as C
    from calibquant_amd import _lib
    M, K, N = shape
    print(f"case linear rows {shape} {dtype}", flush=True)
    lib = _lib.load()
    assert lib.cq_linear_rows_takes(M, K, N)
    g = torch.Generator(device="cuda").manual_seed(K + M)
    x = torch.randn((M, 2, K), generator=g, device="cuda", dtype=dtype)[:, 1]
    w = torch.randn((N, K), generator=g, device="cuda", dtype=dtype) * K ** -0.5
    out = torch.full((M + 1, N), 7.0, device="cuda", dtype=dtype)
    rc = lib.cq_linear_rows(C.c_void_p(x.data_ptr()), x.stride(0), _lib.CQ_BF16 if dtype == torch.bfloat16 else _lib.CQ_FP16, M, K,
                            C.c_void_p(w.data_ptr()), N, C.c_void_p(out.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    assert (out[M] == 7).all()
    want = x.double() @ w.double().T
    err = lambda t: ((t.double() - want).norm() / want.norm()).item()
    ours, library = err(out[:M]), err(torch.nn.functional.linear(x, w))
    print(f"rel. distance to 64 bits {ours:.4e}, library {library:.4e}")
    # (both are the rounding of the result, 2^-9 or 2^-12 of it at most; fp32 sums of K products are within K * 2^-24 of their size)
    assert ours <= library + K * 2.0 ** -24 * 1e-2
    assert not lib.cq_linear_rows_takes(9, K, N) and not lib.cq_linear_rows_takes(M, K + 8, N) and not lib.cq_linear_rows_takes(M, K, N + 4)
    assert not lib.cq_linear_rows_takes(M, 1536, N)


def test_small_batch_step_takes_its_projections_along():
    """The steady-state step of a few rows runs both projections in the shim; a hook, autograd or autocast, which want the module called, keep the
    module call, and the results agree to the rounding of the projections."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    cfg = InternLM2Config.internvl2_5_8b()
    B, S, T, TXT = 3, 4, 130, 9
    N, dtype = S + T + TXT, torch.bfloat16
    att = InternLM2Attention(cfg).cuda().to(dtype)
    att.cq_sprompt_len, att.cq_image_token_num = S, T
    x = torch.randn(B, N + 6, cfg.hidden_size, device="cuda", dtype=dtype)
    pos = torch.arange(N + 6, device="cuda")[None].expand(B, N + 6)
    seen = []

    def steps(hook):
        seen.clear()
        h = att.wqkv.register_forward_hook(lambda *a: seen.append(1)) if hook else None
        outs = []
        with torch.no_grad():
            _, _, past = pi.forward_internlm2_calibquant(att, x[:, :N], None, pos[:, :N], None, False, True)
            for i in range(N, N + 6):
                o, _, past = pi.forward_internlm2_calibquant(att, x[:, i:i + 1], None, pos[:, i:i + 1], past, False, True)
                outs.append(o)
        if h:
            h.remove()
        step = att._cq_step[0]
        assert step.steps == 5 and step.row_steps == (0 if hook else 5)
        return torch.stack(outs).float(), past

    with torch.no_grad():
        assert pi._plain_products(att.wqkv, att.wo)
        with torch.autocast("cuda", dtype=dtype):
            assert not pi._plain_products(att.wqkv, att.wo)
    assert not pi._plain_products(att.wqkv, att.wo)
    a, pa = steps(False)
    b, pb = steps(True)
    assert len(seen) == 7                                     # prefill and six steps
    assert (a - b).norm() / b.norm() < 8e-3                   # two roundings to bf16 (2^-9 each) and the attention between them
    assert (pa[0].float() - pb[0].float()).norm() / pb[0].float().norm() < 4e-3


def _stepped_layer(B=3, dtype=torch.bfloat16, cfg=None):
    """An attention layer (8B-shaped) after its prefill and first token: the module with its step object, the next token's hidden row and position, the
    window."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    cfg = cfg or InternLM2Config.internvl2_5_8b()
    S, T, TXT = 4, 130, 9
    N = S + T + TXT
    att = InternLM2Attention(cfg).cuda().to(dtype)
    att.cq_sprompt_len, att.cq_image_token_num = S, T
    x = torch.randn(B, N + 2, cfg.hidden_size, device="cuda", dtype=dtype)
    pos = torch.arange(N + 2, device="cuda")[None].expand(B, N + 2)
    with torch.no_grad():
        _, _, past = pi.forward_internlm2_calibquant(att, x[:, :N], None, pos[:, :N], None, False, True)
        _, _, past = pi.forward_internlm2_calibquant(att, x[:, N:N + 1], None, pos[:, N:N + 1], past, False, True)
    return att, x[:, N + 1:].contiguous(), pos[:, N + 1:].contiguous(), past


def test_step_with_projections_declines_what_it_does_not_read_as_it_is():
    """Rows and weights whose memory is not what a product would read (a lazy sign, no storage, a layout or type of their own, off 16 bytes), and what is not
    the next token of the window: None, and nothing has happened."""
    from calibquant_amd import ops
    att, x, pos, past = _stepped_layer()
    step, wqkv, wo = att._cq_step[0], att.wqkv.weight.detach(), att.wo.weight.detach()
    K = x.shape[2]
    off = torch.empty(x.numel() + 1, device="cuda", dtype=x.dtype)[1:].view(x.shape).copy_(x)
    apart = torch.empty((x.shape[0], 1, K + 4), device="cuda", dtype=x.dtype)[:, :, :K].copy_(x)
    inner = torch.empty((*x.shape, 2), device="cuda", dtype=x.dtype)[..., 0].copy_(x)
    turned = lambda w: w.t().contiguous().t()
    empty = lambda w: torch.sparse_coo_tensor(size=w.shape, dtype=w.dtype, device="cuda")
    length = step.length
    cases = {
        "hidden, lazy sign": (torch._neg_view(x), wqkv, wo, pos, past[0]),
        "hidden, sparse": (empty(x), wqkv, wo, pos, past[0]),
        "hidden off 16 bytes": (off, wqkv, wo, pos, past[0]),
        "hidden rows off 16 bytes": (apart, wqkv, wo, pos, past[0]),
        "hidden strided": (inner, wqkv, wo, pos, past[0]),
        "hidden of another type": (x.half(), wqkv, wo, pos, past[0]),
        "hidden on the host": (x.cpu(), wqkv, wo, pos, past[0]),
        "wqkv, lazy sign": (x, torch._neg_view(wqkv), wo, pos, past[0]),
        "wqkv, sparse": (x, empty(wqkv), wo, pos, past[0]),
        "wqkv turned": (x, turned(wqkv), wo, pos, past[0]),
        "wo, lazy sign": (x, wqkv, torch._neg_view(wo), pos, past[0]),
        "wo, sparse": (x, wqkv, empty(wo), pos, past[0]),
        "wo turned": (x, wqkv, turned(wo), pos, past[0]),
        "wo of another type": (x, wqkv, wo.half(), pos, past[0]),
        "positions of another type": (x, wqkv, wo, pos.int(), past[0]),
        "a position too few": (x, wqkv, wo, pos[1:], past[0]),
        "a shorter window": (x, wqkv, wo, pos, past[0][:, :, 1:]),
        "another window": (x, wqkv, wo, pos, past[0].clone()),
    }
    for name, args in cases.items():
        print("case", name, flush=True)
        assert step.step_rows(*args) is None, name
        assert step.length == length
        if name.startswith(("hidden", "wqkv", "wo")):   # (the other routes of a step ask this)
            assert not ops.linear_rows_pays(*args[:3]), name
    assert ops.linear_rows_pays(x, wqkv, wo)
    out, k, v = step.step_rows(x, wqkv, wo, pos, past[0])
    assert step.length == length + 1 and k.shape[2] == length + 1 and torch.isfinite(out).all()


def test_step_of_rows_with_a_lazy_sign():
    """The step of a hidden row that is held as another tensor and a sign is the step of its values."""
    from calibquant_amd import patch_internvl as pi
    att, x, pos, past = _stepped_layer()
    length = att._cq_step[0].length
    with torch.no_grad():
        a, _, pa = pi.forward_internlm2_calibquant(att, torch._neg_view(x.neg()), None, pos, past, False, True)
        want = torch.nn.functional.linear(x, att.wqkv.weight).view(x.shape[0], 8, 6, 128)[:, :, 5]   # the value row
    assert att._cq_step[0].length == length + 1
    assert (pa[1][:, :, -1].float() - want.float()).norm() / want.float().norm() < 4e-3   # (one rounding to bf16 each)


@pytest.mark.parametrize("B", [2, 3, 8])
def test_step_takes_its_projections_along_only_where_that_pays(B):
    """The 26B-shaped layer's projections: of two rows they go along, from three on the modules' products are no slower and stay."""
    from calibquant_amd.internlm2 import InternLM2Config
    att, x, pos, past = _stepped_layer(B, cfg=InternLM2Config.internvl2_5_26b())
    got = att._cq_step[0].step_rows(x, att.wqkv.weight.detach(), att.wo.weight.detach(), pos, past[0])
    assert (got is not None) == (B == 2)


@pytest.mark.parametrize("B", [1, 3, 8])
def test_routes_of_a_step_of_few_rows_give_the_same_bits(B):
    """Steps of an 8B-shaped layer that take the projections along: through the host shim, through the Python call objects and through torch's
    operations around the kernels (int32 positions)."""
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config
    cfg, dtype = InternLM2Config.internvl2_5_8b(), torch.bfloat16
    S, T, TXT = 4, 130, 9
    N = S + T + TXT
    outs, wins = [], []
    for route in ("shim", "calls", "operations"):
        print("case route", route, B, flush=True)
        torch.manual_seed(17)
        att = InternLM2Attention(cfg).cuda().to(dtype)
        att.cq_sprompt_len, att.cq_image_token_num, att.cq_no_step_shim = S, T, route != "shim"
        x = torch.randn(B, N + 5, cfg.hidden_size, device="cuda", dtype=dtype)
        pos = torch.arange(N + 5, device="cuda")[None].repeat(B, 1)
        with torch.no_grad():
            _, _, past = pi.forward_internlm2_calibquant(att, x[:, :N], None, pos[:, :N], None, False, True)
            steps = []
            for i in range(N, N + 5):
                p = pos[:, i:i + 1].int() if route == "operations" else pos[:, i:i + 1]
                o, _, past = pi.forward_internlm2_calibquant(att, x[:, i:i + 1], None, p, past, False, True)
                steps.append(o)
        assert ("_cq_step" in att.__dict__) == (route == "shim")
        outs.append(torch.stack(steps))
        wins.append(torch.stack(past))
    for other in (1, 2):
        assert torch.equal(outs[0], outs[other]) and torch.equal(wins[0], wins[other])


@pytest.mark.parametrize("width, B", [("8b", 1), ("8b", 4), ("8b", 8), ("8b", 9), ("26b", 2), ("26b", 4)])
def test_recorded_step_of_few_rows_gives_the_eager_steps_bits(width, B):
    """Two layers of the model's width: the recorded step, replayed, leaves the tokens and the window rows of the model's own eager steps, bit for bit."""
    import contextlib
    import io
    from calibquant_amd import patch_internvl as pi
    from calibquant_amd.graph_decode import StaticDecoder
    from calibquant_amd.internlm2 import InternLM2Attention, InternLM2Config, InternVLChatStandIn
    fp_forward, fp_generate = InternLM2Attention.forward, InternVLChatStandIn.generate
    hidden, heads = (4096, 32) if width == "8b" else (6144, 48)
    cfg = InternLM2Config(vocab_size=512, hidden_size=hidden, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=heads,
                          num_key_value_heads=8, max_position_embeddings=2048)
    torch.manual_seed(5)
    m = InternVLChatStandIn(cfg).cuda().to(torch.bfloat16).eval()
    lm = m.language_model
    S, T, TXT, NEW = 41, 256, 9, 7
    N = S + T + TXT
    try:
        with contextlib.redirect_stdout(io.StringIO()):
            pi.patch_model(m, "calibquant")
        for layer in lm.model.layers:
            layer.attention.cq_image_token_num = T
        emb = torch.randn(B, N, hidden, device="cuda", dtype=torch.bfloat16)
        pos = torch.arange(N, device="cuda")[None].expand(B, N)
        with torch.no_grad():
            logits, past = lm.forward_step(emb, pos, None)
            toks = [logits[:, -1].argmax(-1)]
            for i in range(NEW - 1):
                logits, past = lm.forward_step(lm.get_input_embeddings()(toks[-1])[:, None], torch.full((B, 1), N + i, device="cuda"), past)
                toks.append(logits[:, -1].argmax(-1))
            want = [torch.stack(p) for p in past]
            _, past = lm.forward_step(emb, pos, None)
            dec = StaticDecoder(lm, past, N, NEW)
            got = dec.generate(toks[0], NEW)
        assert dec.graph is not None and torch.equal(got, torch.stack(toks, 1))
        for st, w in zip(dec.state, want):
            R = w.shape[3]
            assert torch.equal(st.kbuf[:, :, :R], w[0]) and torch.equal(st.vbuf[:, :, :R], w[1])
    finally:
        InternLM2Attention.forward, InternVLChatStandIn.generate = fp_forward, fp_generate
