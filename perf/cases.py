"""What the framework's speed is measured on.

A user of this framework turns camera images, a prompt and a robot state into
action chunks: whole ``predict_action`` calls, at batch 1 on one robot and
batched in a server, with and without real-time chunking, in bf16 and with fp8
weights.  The layers of the three towers behind that call are measured by
themselves as well, through the public op layer (``fluxvla_amd.kernels``) and
the reference-named pipeline functions, in the HIP graphs that such callers
replay.  Sizes are those of the PI0 / PI0.5 configurations in
``fluxvla_amd/config.py``: 1 to 3 views of 224 x 224 (256 tokens each), prompts
of up to 180 tokens (ProcessPrompts' length), chunks of 50 actions, batches of
1 to 32.

Kinds:
  norm     fused RMSNorm + residual of activation rows, an eager call
  siglip   SigLIP-So400m encoder layers over a number of images
  prefix   Gemma-2B layers over image and prompt tokens, filling the K/V cache
  expert   action-expert layers against the cached prefix (one Euler step)
  decoder  the reference-named PI0.5 decoder loop over its weights / buffers
  chunk    a whole predict_action call
"""
import hashlib
import math

import torch
import torch.nn.functional as F

from fluxvla_amd import kernels as K
from fluxvla_amd import pi05_flowmatching_inference as P5
from fluxvla_amd._lib import ACT_GELU_TANH
from fluxvla_amd.config import PI0Config
from fluxvla_amd.pi0_inference import (PI0Inference, attention_groups,
                                       suffix_att_pattern)
from fluxvla_amd.weight_layout import NKWeight

BF16 = torch.bfloat16
DEV = 'cuda'
INT32_MAX = 2**31 - 1
EPS = 1e-6
THETA = 10000.0
PATCHES = 256                                    # tokens per view
VIT, VIT_MLP, VIT_HEADS = 1152, 4304, 16         # SigLIP-So400m/14
LLM, LLM_MLP = 2048, 16384                       # Gemma-2B
EXP, EXP_MLP = 1024, 4096                        # Gemma-300M action expert
HEADS, HD = 8, 256                               # one key / value head
NQKV = (HEADS + 2) * HD
ACTIONS, ADIM, VOCAB = 50, 32, 257152


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the fused norm op on its own (the RMSNorm benchmark shape)
        {'name': 'norm 1024x2048', 'kind': 'norm', 'rows': 1024, 'cols': 2048},
        # one robot's three cameras; a server's batch of 8 requests
        {'name': 'siglip 3 images', 'kind': 'siglip', 'images': 3, 'layers': 4},
        {'name': 'siglip 24 images', 'kind': 'siglip', 'images': 24, 'layers': 4},
        # the prompt pass of one request, of a batch of 8 with prompts of
        # unequal lengths, and of an fp8 server's batch of 32 with two views
        # and the full-length prompt
        {'name': 'prefix bs1', 'kind': 'prefix', 'batch': 1, 'views': 3,
         'prompt': 48, 'weights': 'bf16', 'layers': 2},
        {'name': 'prefix bs8', 'kind': 'prefix', 'batch': 8, 'views': 3,
         'prompt': 48, 'weights': 'bf16', 'layers': 2},
        {'name': 'prefix fp8 bs32', 'kind': 'prefix', 'batch': 32, 'views': 2,
         'prompt': 180, 'weights': 'fp8', 'layers': 1},
        # one Euler step: all 18 layers for one request, a batch of 8
        {'name': 'expert bs1', 'kind': 'expert', 'batch': 1, 'views': 3,
         'prompt': 48, 'weights': 'bf16', 'layers': 18},
        {'name': 'expert bs8', 'kind': 'expert', 'batch': 8, 'views': 3,
         'prompt': 48, 'weights': 'bf16', 'layers': 6},
        # a program written against the reference's decoder function
        {'name': 'decoder', 'kind': 'decoder', 'views': 3, 'prompt': 48,
         'layers': 18, 'steps': 2},
        # the headline call: one PI0 request, full depth
        {'name': 'chunk pi0 bs1', 'kind': 'chunk', 'model': 'pi0', 'batch': 1,
         'views': 3, 'prompt': 48, 'weights': 'bf16', 'rtc': 'none',
         'vit_layers': 27, 'layers': 18},
        # a PI0.5 server with fp8 weights (every layer kind, fewer of each)
        {'name': 'chunk pi05 fp8 bs8', 'kind': 'chunk', 'model': 'pi05',
         'batch': 8, 'views': 3, 'prompt': 48, 'weights': 'fp8', 'rtc': 'none',
         'vit_layers': 6, 'layers': 4},
        # real-time chunking with the correction pulled back through the
        # expert: forward and backward at every Euler step
        {'name': 'chunk pi0 guided', 'kind': 'chunk', 'model': 'pi0', 'batch': 1,
         'views': 2, 'prompt': 48, 'weights': 'bf16', 'rtc': 'guidance_vjp',
         'vit_layers': 2, 'layers': 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['norm', 'siglip', 'siglip', 'prefix', 'prefix', 'prefix',
                       'expert', 'expert', 'expert', 'decoder', 'chunk', 'chunk'])
    views, prompt = rng.randint(1, 3), rng.randint(8, 180)
    if kind == 'norm':
        return {'kind': kind, 'rows': _log(rng, 51, 20000),
                'cols': rng.choice([1024, 2048])}
    if kind == 'siglip':
        return {'kind': kind, 'images': _log(rng, 1, 96),
                'layers': rng.randint(2, 4)}
    if kind == 'prefix':
        batch = _log(rng, 1, 32)
        return {'kind': kind, 'batch': batch, 'views': min(views, 2) if
                batch > 24 else views, 'prompt': prompt,
                'weights': rng.choice(['bf16', 'bf16', 'fp8']),
                'layers': 1 if batch > 8 else rng.randint(1, 2)}
    if kind == 'expert':
        batch = _log(rng, 1, 32)
        return {'kind': kind, 'batch': batch, 'views': views, 'prompt': prompt,
                'weights': rng.choice(['bf16', 'bf16', 'fp8']),
                'layers': rng.randint(4, 18) if batch < 4 else rng.randint(2, 6)}
    if kind == 'decoder':
        return {'kind': kind, 'views': views, 'prompt': prompt,
                'layers': rng.randint(2, 18), 'steps': rng.randint(1, 2)}
    rtc = rng.choice(['none', 'none', 'prefix', 'guidance', 'guidance_vjp'])
    return {'kind': kind, 'model': rng.choice(['pi0', 'pi05']),
            'batch': _log(rng, 1, 8) if rtc == 'none' else rng.randint(1, 2),
            'views': views, 'prompt': prompt,
            'weights': rng.choice(['bf16', 'bf16', 'fp8']), 'rtc': rtc,
            'vit_layers': rng.randint(1, 6), 'layers': rng.randint(2, 4)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
class _Rand:
    """bf16 (or fp32) normal tensors on the GPU from one seed."""

    def __init__(self, seed, tag):
        h = hashlib.sha256(f'{seed}:{tag}'.encode()).digest()
        self.g = torch.Generator(device=DEV).manual_seed(
            int.from_bytes(h[:7], 'little'))

    def __call__(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(shape, generator=self.g, device=DEV,
                        dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype)

    def ints(self, hi, *shape, lo=0):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV)


def _in_norm(c, r):
    rows, cols = c['rows'], c['cols']
    return {'x': r(rows, cols), 'res': r(rows, cols),
            'w': r(cols, std=0.1, mean=1.0)}


def _in_siglip(c, r):
    n = c['images'] * PATCHES
    return {'x': r(n, VIT), 'layers': [
        {'ln1_w': r(VIT, std=0.05, mean=1.0), 'ln1_b': r(VIT, std=0.02),
         'qkv_w': r(3 * VIT, VIT, std=0.02), 'qkv_b': r(3 * VIT, std=0.02),
         'o_w': r(VIT, VIT, std=0.02), 'o_b': r(VIT, std=0.02),
         'ln2_w': r(VIT, std=0.05, mean=1.0), 'ln2_b': r(VIT, std=0.02),
         'fc1_w': r(VIT_MLP, VIT, std=0.02), 'fc1_b': r(VIT_MLP, std=0.02),
         'fc2_w': r(VIT, VIT_MLP, std=0.02), 'fc2_b': r(VIT, std=0.02)}
        for _ in range(c['layers'])]}


def _gemma_layers(r, n, hid, mlp):
    return [{'qkv_w': r(NQKV, hid, std=0.02), 'o_w': r(hid, HEADS * HD, std=0.02),
             'gate_w': r(mlp, hid, std=0.02), 'up_w': r(mlp, hid, std=0.02),
             'down_w': r(hid, mlp, std=0.02)} for _ in range(n)]


def _pad_mask(c, r, batch):
    """All image tokens valid, prompts of unequal lengths."""
    S = c['views'] * PATCHES + c['prompt']
    lens = r.ints(c['prompt'] + 1, batch, lo=max(1, c['prompt'] // 2))
    return (torch.arange(S, device=DEV)[None] <
            (c['views'] * PATCHES + lens)[:, None])


def _in_prefix(c, r):
    pad = _pad_mask(c, r, c['batch'])
    return {'x': r(c['batch'], pad.shape[1], LLM), 'pad': pad,
            'layers': _gemma_layers(r, c['layers'], LLM, LLM_MLP)}


def _in_expert(c, r):
    B, n = c['batch'], c['layers']
    pad = _pad_mask(c, r, B)
    S = pad.shape[1]
    return {'x': r(B, ACTIONS + 1, EXP), 'pad': pad, 'k': r(n, B, S, HD),
            'v': r(n, B, S, HD), 'layers': _gemma_layers(r, n, EXP, EXP_MLP)}


def _in_decoder(c, r):
    S, n = c['views'] * PATCHES + c['prompt'], c['layers']
    w = {'time_in_w': r(EXP, EXP, std=0.02), 'time_in_b': r(EXP, std=0.02),
         'time_out_w': r(EXP, EXP, std=0.02), 'time_out_b': r(EXP, std=0.02),
         'in_w': r(EXP, ADIM, std=0.02), 'in_b': r(EXP, std=0.02),
         'out_w': r(ADIM, EXP, std=0.02), 'out_b': r(ADIM, std=0.02),
         'fin_w': r(3 * EXP, EXP, std=0.02), 'fin_b': r(3 * EXP, std=0.02)}
    layers = _gemma_layers(r, n, EXP, EXP_MLP)
    for L in layers:
        L['m1_w'], L['m1_b'] = r(3 * EXP, EXP, std=0.02), r(3 * EXP, std=0.02)
        L['m2_w'], L['m2_b'] = r(3 * EXP, EXP, std=0.02), r(3 * EXP, std=0.02)
    valid = int(r.ints(S + 1, 1, lo=S - c['prompt'] // 2)[0])
    return {'w': w, 'layers': layers, 'k': r(n, S, HD), 'v': r(n, S, HD),
            'noise': r(ACTIONS, ADIM, dtype=torch.float32), 'valid': valid,
            'rope': P5.rope_rows(torch.arange(valid, valid + ACTIONS, device=DEV)),
            'time': P5.time_embeds(10, EXP, device=DEV)[:c['steps']]}


VISION = 'vision_backbone.vision.vision_model'


def _state_dict(c, r):
    """Random parameters under the checkpoint's names."""
    sd = {}

    def lin(name, n, k, bias=True):
        sd[f'{name}.weight'] = r(n, k, std=0.02)
        if bias:
            sd[f'{name}.bias'] = r(n, std=0.02)

    def norm(name, n):
        sd[f'{name}.weight'] = r(n, std=0.05, mean=1.0)
        sd[f'{name}.bias'] = r(n, std=0.02)

    e = f'{VISION}.embeddings'
    sd[f'{e}.patch_embedding.weight'] = r(VIT, 3, 14, 14, std=0.02)
    sd[f'{e}.patch_embedding.bias'] = r(VIT, std=0.02)
    sd[f'{e}.position_embedding.weight'] = r(PATCHES, VIT, std=0.02)
    for i in range(c['vit_layers']):
        pre = f'{VISION}.encoder.layers.{i}'
        norm(f'{pre}.layer_norm1', VIT)
        norm(f'{pre}.layer_norm2', VIT)
        for nm in ('q_proj', 'k_proj', 'v_proj', 'out_proj'):
            lin(f'{pre}.self_attn.{nm}', VIT, VIT)
        lin(f'{pre}.mlp.fc1', VIT_MLP, VIT)
        lin(f'{pre}.mlp.fc2', VIT, VIT_MLP)
    norm(f'{VISION}.post_layernorm', VIT)
    lin('projector.projector', LLM, VIT)
    sd['llm_backbone.embed_tokens.weight'] = r(VOCAB, LLM, std=0.02)
    ada = c['model'] == 'pi05'
    for prefix, hid, mlp, mod in (('llm_backbone', LLM, LLM_MLP, False),
                                  ('llm_expert', EXP, EXP_MLP, ada)):
        def gnorm(name):
            if mod:
                lin(f'{name}.dense', 3 * hid, EXP)
            else:
                sd[f'{name}.weight'] = r(hid, std=0.1)
        for i in range(c['layers']):
            pre = f'{prefix}.layers.{i}'
            gnorm(f'{pre}.input_layernorm')
            gnorm(f'{pre}.post_attention_layernorm')
            lin(f'{pre}.self_attn.q_proj', HEADS * HD, hid, False)
            lin(f'{pre}.self_attn.k_proj', HD, hid, False)
            lin(f'{pre}.self_attn.v_proj', HD, hid, False)
            lin(f'{pre}.self_attn.o_proj', hid, HEADS * HD, False)
            lin(f'{pre}.mlp.gate_proj', mlp, hid, False)
            lin(f'{pre}.mlp.up_proj', mlp, hid, False)
            lin(f'{pre}.mlp.down_proj', hid, mlp, False)
        gnorm(f'{prefix}.norm')
    lin('action_in_proj.projector', EXP, ADIM)
    lin('action_out_proj.projector', ADIM, EXP)
    if ada:
        lin('time_mlp_in.projector', EXP, EXP)
        lin('time_mlp_out.projector', EXP, EXP)
    else:
        lin('state_proj.projector', EXP, ADIM)
        lin('action_time_mlp_in.projector', EXP, 2 * EXP)
        lin('action_time_mlp_out.projector', EXP, EXP)
    return sd


def _in_chunk(c, r):
    B, views = c['batch'], c['views']
    d = {'sd': _state_dict(c, r)}
    lens = r.ints(c['prompt'] + 1, B, lo=max(1, c['prompt'] // 2))
    rtc = {'none': None, 'prefix': {'method': 'prefix'},
           'guidance': {'method': 'guidance'},
           'guidance_vjp': {'method': 'guidance', 'use_vjp': True}}[c['rtc']]
    d['call'] = {
        'images': r.ints(256, B, 3 * views, 224, 224).float() / 127.5 - 1.0,
        'lang_tokens': r.ints(VOCAB, B, c['prompt']),
        'lang_masks': torch.arange(c['prompt'], device=DEV)[None] < lens[:, None],
        'img_masks': torch.ones(B, views, dtype=torch.bool, device=DEV),
        'states': r(B, ADIM, std=0.5),
        'noise': r(B, ACTIONS, ADIM, dtype=torch.float32)}
    if rtc:
        d['call'].update(prev_actions=r(B, 30, ADIM, dtype=torch.float32),
                         prefix_len=5, rtc_config=rtc)
    return d


_INPUTS = {'norm': _in_norm, 'siglip': _in_siglip, 'prefix': _in_prefix,
           'expert': _in_expert, 'decoder': _in_decoder, 'chunk': _in_chunk}


def _inputs(case, seed):
    return _INPUTS[case['kind']](case, _Rand(seed, case['kind']))


# ---------------------------------------------------------------------------
# Prepared state and one pass
# ---------------------------------------------------------------------------
def _graph(fn):
    """``fn``'s launches as one HIP graph (a warm-up call first), with ``fn``
    itself: its closure keeps alive every buffer that the graph addresses."""
    g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        fn()
        torch.cuda.synchronize()
        g.capture_begin()
        fn()
        g.capture_end()
    torch.cuda.current_stream().wait_stream(st)
    return g, fn


def _empty(*shape, dtype=BF16):
    return torch.empty(*shape, dtype=dtype, device=DEV)


def _prep_norm(c, d):
    d['out'], d['sum'] = _empty(*d['x'].shape), _empty(*d['x'].shape)
    return d


def _run_norm(s):
    K.rms_norm_residual(s['x'], s['res'], s['w'], EPS, out=s['out'],
                        residual_out=s['sum'])
    return [s['out'], s['sum']]


def _prep_siglip(c, d):
    """The encoder layers as PI0Inference.vision_encoder runs them."""
    n = d['x'].shape[0]
    xn, qkv, ctx = _empty(n, VIT), _empty(n, 3 * VIT), _empty(n, VIT)
    h, y = _empty(n, VIT_MLP), [_empty(n, VIT) for _ in range(2)]

    def layers():
        x = d['x']
        for L in d['layers']:
            K.layer_norm(x, L['ln1_w'], L['ln1_b'], EPS, out=xn)
            K.gemm(xn, L['qkv_w'], out=qkv, bias=L['qkv_b'])
            K.mha_packed_qkv(qkv, ctx, c['images'], PATCHES, VIT_HEADS,
                             VIT // VIT_HEADS)
            K.gemm(ctx, L['o_w'], out=y[0], bias=L['o_b'], residual=x)
            K.layer_norm(y[0], L['ln2_w'], L['ln2_b'], EPS, out=xn)
            K.gemm(xn, L['fc1_w'], out=h, bias=L['fc1_b'], act=ACT_GELU_TANH)
            K.gemm(h, L['fc2_w'], out=y[1], bias=L['fc2_b'], residual=y[0])
            x = y[1]
    return {'d': d, 'graph': _graph(layers), 'out': [y[1]]}


def _linear(c, w, frag=False):
    """A prepared weight as the pipeline holds it."""
    if c.get('weights') == 'fp8':
        w = K.Fp8Weight.quantize(w)
        return w.pack_frag() if frag else w
    return K.FragB.pack(w) if frag else w


def _caches(n, B, S):
    T = (S + ACTIONS + 1 + 7) // 8 * 8
    return (torch.zeros(n, B, T, HD, dtype=BF16, device=DEV),
            torch.zeros(n, B, HD, T, dtype=BF16, device=DEV), T)


def _prep_prefix(c, d):
    """Prefix layers as PI0Inference.transformer_encoder runs them: row sums
    of squares handed between the GEMMs, keys and transposed values written
    to the caches."""
    B, S = d['pad'].shape
    M = B * S
    kc, vc, T = _caches(c['layers'], B, S)
    pi0 = PI0Config(n_views=c['views'], max_prompt_len=c['prompt'])
    kgrp, qgrp, _, pos, _ = attention_groups(d['pad'], suffix_att_pattern(pi0))
    pos = pos.view(-1).contiguous()
    rope = K.rope_table(T + 8, HD, THETA, device=DEV)
    W = [{nm: _linear(c, w) for nm, w in L.items()} for L in d['layers']]
    q, ctx, h = _empty(B, S, HEADS * HD), _empty(B, S, HEADS * HD), _empty(M, LLM_MLP)
    x0, y = d['x'].view(M, LLM), [_empty(M, LLM) for _ in range(2)]
    ss = [_empty(K.ss_parts(LLM), M, dtype=torch.float32) for _ in range(2)]

    def layers():
        x = x0
        for i, L in enumerate(W):
            K.gemm_qkv_rope(x, L['qkv_w'], rope, pos, q.view(M, -1),
                            kc[i].view(B * T, HD), vc[i], HEADS, HD,
                            rownorm_eps=EPS, row_group=S, row_group_stride=T,
                            v_ld=T, ss_in=ss[1] if i else None)
            K.mqa_attention(q, kc[i][:, :S], vc[i], ctx, kgrp=kgrp[:, :S],
                            qgrp=qgrp, v_transposed=True)
            K.gemm(ctx.view(M, -1), L['o_w'], out=y[0], residual=x, ss_out=ss[0])
            K.gemm_geglu(y[0], L['gate_w'], L['up_w'], out=h, rownorm_eps=EPS,
                         ss_in=ss[0])
            K.gemm(h, L['down_w'], out=y[1], residual=y[0], ss_out=ss[1])
            x = y[1]
    return {'d': d, 'graph': _graph(layers),
            'out': [y[1].view(B, S, LLM), kc[:, :, :S], vc[:, :, :, :S]]}


def _prep_expert(c, d):
    """One Euler step's PI0 expert layers as PI0Inference runs them: fragment-
    major operands and weight prefetch for one request, row-major batches."""
    B, S = d['pad'].shape
    n, Ss = c['layers'], ACTIONS + 1
    M = B * Ss
    kc, vc, T = _caches(n, B, S)
    kc[:, :, :S] = d['k']
    vc[..., :S] = d['v'].transpose(2, 3)
    pi0 = PI0Config(n_views=c['views'], max_prompt_len=c['prompt'])
    kgrp, _, qgrp, _, pos = attention_groups(d['pad'], suffix_att_pattern(pi0))
    pos = pos.view(-1).contiguous()
    rope = K.rope_table(T + 8, HD, THETA, device=DEV)
    fr = M <= 64
    W = [{nm: _linear(c, w, fr) for nm, w in L.items()} for L in d['layers']]
    q, ctx, h = _empty(B, Ss, HEADS * HD), _empty(B, Ss, HEADS * HD), _empty(M, EXP_MLP)
    x0, y = d['x'].view(M, EXP), [_empty(M, EXP) for _ in range(2)]
    if fr:
        x0f, yf0, yf1 = (K.FragA.empty(EXP, DEV).rows(M) for _ in range(3))
        ctxf, hf = (K.FragA.empty(k, DEV).rows(M) for k in (HEADS * HD, EXP_MLP))
        K.pack_frag(x0, x0f)

    def qkv(i, a):
        K.gemm_qkv_rope(a, W[i]['qkv_w'], rope, pos, q.view(M, -1),
                        kc[i].view(B * T, HD)[S:], vc[i][:, :, S:], HEADS, HD,
                        rownorm_eps=EPS, row_group=Ss, row_group_stride=T, v_ld=T)

    def layers_frag():
        x, xf = x0, x0f
        for i, L in enumerate(W):
            j = (i + 1) % n
            qkv(i, xf)
            K.mqa_attention(q, kc[i][:, :S + Ss], vc[i], ctx, kgrp=kgrp, qgrp=qgrp,
                            v_transposed=True, o_frag=ctxf, o_row_major=False,
                            prefetch=[L['o_w'], L['gate_w'], L['up_w'], L['down_w'],
                                      W[j]['qkv_w'], kc[j], vc[j]])
            K.gemm(ctxf, L['o_w'], out=y[0], residual=x, c_frag=yf0)
            K.gemm_geglu(yf0, L['gate_w'], L['up_w'], out=h, rownorm_eps=EPS,
                         c_frag=hf)
            K.gemm(hf, L['down_w'], out=y[1], residual=y[0], c_frag=yf1)
            x, xf = y[1], yf1

    def layers_rows():
        x = x0
        for i, L in enumerate(W):
            qkv(i, x)
            K.mqa_attention(q, kc[i][:, :S + Ss], vc[i], ctx, kgrp=kgrp, qgrp=qgrp,
                            v_transposed=True)
            K.gemm(ctx.view(M, -1), L['o_w'], out=y[0], residual=x)
            K.gemm_geglu(y[0], L['gate_w'], L['up_w'], out=h, rownorm_eps=EPS)
            K.gemm(h, L['down_w'], out=y[1], residual=y[0])
            x = y[1]
    return {'d': d, 'graph': _graph(layers_frag if fr else layers_rows),
            'out': [y[1].view(B, Ss, EXP), kc[:, :, S:S + Ss], vc[..., S:S + Ss]]}


def _run_graph(s):
    s['graph'][0].replay()
    return s['out']


def _prep_decoder(c, d):
    S, n = d['k'].shape[1], c['layers']
    w, Ls = d['w'], d['layers']

    def stack(nm):
        return torch.stack([L[nm] for L in Ls])
    W = {'decoder_time_embeds': d['time'],
         'decoder_time_mlp_in_w': NKWeight(w['time_in_w']),
         'decoder_time_mlp_in_b': w['time_in_b'],
         'decoder_time_mlp_out_w': NKWeight(w['time_out_w']),
         'decoder_time_mlp_out_b': w['time_out_b'],
         'decoder_action_in_proj_w': NKWeight(w['in_w']),
         'decoder_action_in_proj_b': w['in_b'],
         'decoder_action_out_proj_w': NKWeight(w['out_w']),
         'decoder_action_out_proj_b': w['out_b'],
         'decoder_final_norm_mod_w': NKWeight(w['fin_w']),
         'decoder_final_norm_mod_b': w['fin_b'],
         'decoder_pre_attn_norm_mod_w': NKWeight(stack('m1_w')),
         'decoder_pre_attn_norm_mod_b': stack('m1_b'),
         'decoder_pre_ffn_norm_mod_w': NKWeight(stack('m2_w')),
         'decoder_pre_ffn_norm_mod_b': stack('m2_b'),
         'decoder_attn_qkv_w': NKWeight(stack('qkv_w')),
         'decoder_attn_o_w': NKWeight(stack('o_w')),
         'decoder_ffn_gate_w': NKWeight(stack('gate_w')),
         'decoder_ffn_up_w': NKWeight(stack('up_w')),
         'decoder_ffn_down_w': NKWeight(stack('down_w'))}
    b = P5.init_buffers(c['views'], S, ACTIONS, n, device=DEV)
    b['encoder_K'][:, :S] = d['k']
    b['encoder_V'][:, :S] = d['v']
    b['decoder_rope_weights'].copy_(d['rope'])
    b['attn_kgrp'][d['valid']:S] = INT32_MAX
    s = {'d': d, 'W': W, 'b': b, 'steps': c['steps']}
    s['graph'] = _graph(lambda: P5.transformer_decoder(W, b, S, n, c['steps']))
    return s


def _run_decoder(s):
    b = s['b']
    b['diffusion_noise_f32'].copy_(s['d']['noise'])
    b['diffusion_noise'].copy_(s['d']['noise'])
    s['graph'][0].replay()
    return [b['diffusion_noise_f32'], b['decoder_x']]


def _prep_chunk(c, d):
    cfg = PI0Config(n_views=c['views'], max_prompt_len=c['prompt'],
                    vit_layers=c['vit_layers'], llm_layers=c['layers'],
                    exp_layers=c['layers'], pi05=c['model'] == 'pi05')
    return {'model': PI0Inference(cfg, d['sd'], device=DEV, max_batch=c['batch'],
                                  weight_dtype=c['weights']), 'call': d['call']}


def _run_chunk(s):
    return s['model'].predict_action(**s['call'])


_PREP = {'norm': (_prep_norm, _run_norm), 'siglip': (_prep_siglip, _run_graph),
         'prefix': (_prep_prefix, _run_graph), 'expert': (_prep_expert, _run_graph),
         'decoder': (_prep_decoder, _run_decoder),
         'chunk': (_prep_chunk, _run_chunk)}


@torch.no_grad()
def prepare(case, seed):
    prep, run_ = _PREP[case['kind']]
    state = prep(case, _inputs(case, seed))
    state['run'] = run_
    return state


@torch.no_grad()
def run(state):
    return state['run'](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _gemma_work(M, hid, mlp, wb, sq, sk, B):
    """(bytes, flops) of one Gemma layer on M = B * sq rows, sk keys each."""
    n = NQKV * hid + HEADS * HD * hid + 3 * mlp * hid
    return (n * wb + B * sk * HD * 4,
            2.0 * M * n + 4.0 * B * HEADS * sq * sk * HD)


def _siglip_work(images, layers):
    n, M = 4 * VIT * VIT + 2 * VIT * VIT_MLP, images * PATCHES
    return (layers * n * 2.0, layers * (2.0 * M * n + 4.0 * M * PATCHES * VIT))


def work(case):
    c, kind = case, case['kind']
    if kind == 'norm':
        return {'bytes': 8.0 * c['rows'] * c['cols'] + 2 * c['cols'],
                'flops': 6.0 * c['rows'] * c['cols']}
    if kind == 'siglip':
        b, f = _siglip_work(c['images'], c['layers'])
        return {'bytes': b + 4.0 * c['images'] * PATCHES * VIT, 'flops': f}
    S = c['views'] * PATCHES + c['prompt']
    wb = 1 if c.get('weights') == 'fp8' else 2
    if kind == 'prefix':
        B, n = c['batch'], c['layers']
        b, f = _gemma_work(B * S, LLM, LLM_MLP, wb, S, S, B)
        return {'bytes': n * b + 4.0 * B * S * LLM, 'flops': n * f}
    if kind == 'expert':
        B, n, Ss = c['batch'], c['layers'], ACTIONS + 1
        b, f = _gemma_work(B * Ss, EXP, EXP_MLP, wb, Ss, S + Ss, B)
        return {'bytes': n * b + 4.0 * B * Ss * EXP, 'flops': n * f}
    if kind == 'decoder':
        n, steps = c['layers'], c['steps']
        b, f = _gemma_work(ACTIONS, EXP, EXP_MLP, 2, ACTIONS, S + ACTIONS, 1)
        mod = 6 * EXP * EXP
        return {'bytes': steps * n * (b + 2.0 * mod),
                'flops': steps * n * (f + 2.0 * mod)}
    B, Ss, n = c['batch'], ACTIONS + (c['model'] == 'pi0'), c['layers']
    vb, vf = _siglip_work(B * c['views'], c['vit_layers'])
    # the last prefix layer only fills its K/V cache
    pb, pf = _gemma_work(B * S, LLM, LLM_MLP, wb, S, S, B)
    eb, ef = _gemma_work(B * Ss, EXP, EXP_MLP, wb, Ss, S + Ss, B)
    steps = 10 * (2 if c['rtc'] == 'guidance_vjp' else 1)
    return {'bytes': vb + (n - 1) * pb + steps * n * eb,
            'flops': vf + (n - 1) * pf + steps * n * ef}


# about four times the distance from the 64-bit result that bf16 activations
# give: 1.8e-3 (norm), 5.1e-3 (siglip), 4.6e-3 (prefix), up to 1.3e-2 over 18
# expert layers, 3.7e-3 (chunk)
_REL = {'norm': 7e-3, 'siglip': 2e-2, 'prefix': 1.8e-2, 'expert': 3e-2,
        'decoder': 3e-2, 'chunk': 1.5e-2}


def tolerance(case):
    return {'rel': _REL[case['kind']]}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _lin(x, w, b=None):
    y = x @ w.double().t()
    return y if b is None else y + b.double()


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _gelu(x):
    return F.gelu(x, approximate='tanh')


def _fp8(w):
    """Values of a bf16 weight in e4m3 with one fp32 scale per output row."""
    w = w.float()
    s = (w.abs().amax(1) / 448.0).clamp_min(torch.finfo(torch.float32).tiny)
    return (w / s[:, None]).to(torch.float8_e4m3fn).double() * s.double()[:, None]


def _rope_pairs(x, cos, sin):
    """Rotation of adjacent pairs; x [..., tokens, heads, HD]."""
    a, b = x[..., 0::2], x[..., 1::2]
    cos, sin = cos[..., None, :], sin[..., None, :]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)


def _angles(pos):
    inv = 1.0 / THETA**(torch.arange(0, HD, 2, device=DEV).double() / HD)
    ph = pos.double()[..., None] * inv
    return torch.cos(ph), torch.sin(ph)


def _attend(q, k, v, see):
    """q [B, Sq, H, d]; k, v [B, Sk, d]; see [B, Sq, Sk] bool: one shared
    key / value head, sample by sample."""
    out = []
    for i in range(q.shape[0]):
        s = torch.matmul(q[i].transpose(0, 1), k[i].t().contiguous())
        s = s * q.shape[-1]**-0.5
        s = s.masked_fill(~see[i][None], float('-inf'))
        out.append(torch.matmul(torch.softmax(s, -1), v[i]).transpose(0, 1))
    return torch.stack(out).flatten(-2)


def _gemma_layer(x, L, cos, sin, see, past=None, norms=(None, None)):
    """One decoder layer in 64 bits; ``norms``: (scale, shift, gate) of the
    adaptive norms, or None.  Returns (x, k, v, of this call's tokens)."""
    def norm(t, m):
        return _rms(t) if m is None else _rms(t) * (1 + m[0]) + m[1]
    B, S = x.shape[:2]
    y = _lin(norm(x, norms[0]), L['qkv_w'])
    q, k, v = y.split([HEADS * HD, HD, HD], -1)
    q = _rope_pairs(q.reshape(B, S, HEADS, HD), cos, sin)
    k = _rope_pairs(k.reshape(B, S, 1, HD), cos, sin)[:, :, 0]
    kk, vv = (k, v) if past is None else (torch.cat([past[0], k], 1),
                                          torch.cat([past[1], v], 1))
    o = _lin(_attend(q, kk, vv, see), L['o_w'])
    x = x + (o if norms[0] is None else o * norms[0][2])
    z = norm(x, norms[1])
    m = _lin(_gelu(_lin(z, L['gate_w'])) * _lin(z, L['up_w']), L['down_w'])
    return x + (m if norms[1] is None else m * norms[1][2]), k, v


def _weights64(c, layers):
    if c.get('weights') != 'fp8':
        return layers
    return [{nm: _fp8(w) for nm, w in L.items()} for L in layers]


def _siglip64(x, layers, images):
    """Encoder layers on x [images * PATCHES, VIT]."""
    hd = VIT // VIT_HEADS
    for L in layers:
        y = F.layer_norm(x, (VIT,), L['ln1_w'].double(), L['ln1_b'].double(), EPS)
        y = _lin(y, L['qkv_w'], L['qkv_b']).view(images, PATCHES, 3, VIT_HEADS, hd)
        q, k, v = (t.transpose(1, 2).contiguous() for t in y.unbind(2))
        s = torch.matmul(q, k.transpose(2, 3).contiguous()) * hd**-0.5
        a = torch.matmul(torch.softmax(s, -1), v).transpose(1, 2).reshape(-1, VIT)
        x = x + _lin(a, L['o_w'], L['o_b'])
        y = F.layer_norm(x, (VIT,), L['ln2_w'].double(), L['ln2_b'].double(), EPS)
        x = x + _lin(_gelu(_lin(y, L['fc1_w'], L['fc1_b'])), L['fc2_w'], L['fc2_b'])
    return x


def _exact_norm(c, d):
    h = d['x'].double() + d['res'].double()
    return [_rms(h) * d['w'].double(), h]


def _exact_siglip(c, d):
    return [_siglip64(d['x'].double(), d['layers'], c['images'])]


def _exact_prefix(c, d):
    pad, x = d['pad'], d['x'].double()
    cos, sin = _angles(pad.int().cumsum(1) - 1)
    see = pad[:, None, :].expand(-1, pad.shape[1], -1)
    ks, vs = [], []
    for L in _weights64(c, d['layers']):
        x, k, v = _gemma_layer(x, L, cos, sin, see)
        ks.append(k)
        vs.append(v.transpose(1, 2))
    return [x, torch.stack(ks), torch.stack(vs)]


def _suffix_view(pad, Ss, causal_state):
    """Prefix keys by their mask; the state row (PI0) sees only itself among
    the suffix, the action rows see all of it."""
    own = torch.ones(Ss, Ss, dtype=torch.bool, device=DEV)
    if causal_state:
        own[0, 1:] = False
    B = pad.shape[0]
    return torch.cat([pad[:, None].expand(B, Ss, -1), own.expand(B, Ss, Ss)], 2)


def _exact_expert(c, d):
    pad, x, Ss = d['pad'], d['x'].double(), ACTIONS + 1
    cos, sin = _angles(pad.sum(1, keepdim=True) + torch.arange(Ss, device=DEV))
    see = _suffix_view(pad, Ss, True)
    ks, vs = [], []
    for i, L in enumerate(_weights64(c, d['layers'])):
        x, k, v = _gemma_layer(x, L, cos, sin, see,
                               (d['k'][i].double(), d['v'][i].double()))
        ks.append(k)
        vs.append(v.transpose(1, 2))
    return [x, torch.stack(ks), torch.stack(vs)]


def _split3(t):
    return t.split(EXP, -1)


def _exact_decoder(c, d):
    w, S = d['w'], d['k'].shape[1]
    rope = d['rope'].double().view(1, ACTIONS, HD // 2, 2)
    pad = (torch.arange(S, device=DEV) < d['valid'])[None]
    see = _suffix_view(pad, ACTIONS, False)
    xt = d['noise'].double()
    for step in range(c['steps']):
        t = F.silu(_lin(d['time'][step].double(), w['time_in_w'], w['time_in_b']))
        t = F.silu(_lin(t, w['time_out_w'], w['time_out_b']))
        x = _lin(xt, w['in_w'], w['in_b'])[None]
        for i, L in enumerate(d['layers']):
            x, _, _ = _gemma_layer(
                x, L, rope[..., 0], rope[..., 1], see,
                (d['k'][i][None].double(), d['v'][i][None].double()),
                (_split3(_lin(t, L['m1_w'], L['m1_b'])),
                 _split3(_lin(t, L['m2_w'], L['m2_b']))))
        m = _split3(_lin(t, w['fin_w'], w['fin_b']))
        v = _lin(_rms(x[0]) * (1 + m[0]) + m[1], w['out_w'], w['out_b'])
        xt = xt - v / c['steps']
    return [xt, x[0]]


def _chunk_layers(c, sd, prefix):
    """Per layer: the stacked weights with (1 + norm) folded in, Q and K rows
    in pair order, or the adaptive norms' own weights."""
    ada = c['model'] == 'pi05' and prefix == 'llm_expert'
    pairs = torch.arange(HD, device=DEV).view(2, -1).t().reshape(-1)
    fp8 = c['weights'] == 'fp8'
    out = []
    for i in range(c['layers']):
        pre = f'{prefix}.layers.{i}'

        def weight(nm, norm=None):
            w = sd[f'{pre}.{nm}.weight']
            if norm and not ada:
                g = sd[f'{pre}.{norm}.weight']
                # fp8 quantizes the folded bf16 weight
                w = ((w.float() * (1.0 + g.float())).to(BF16) if fp8 else
                     w.double() * (1.0 + g.double()))
            return _fp8(w) if fp8 else w
        a, m = 'input_layernorm', 'post_attention_layernorm'
        q = weight('self_attn.q_proj', a).double()
        q = q.view(HEADS, HD, -1)[:, pairs].reshape(HEADS * HD, -1)
        k = weight('self_attn.k_proj', a).double()[pairs]
        L = {'qkv_w': torch.cat([q, k, weight('self_attn.v_proj', a).double()]),
             'o_w': weight('self_attn.o_proj'),
             'gate_w': weight('mlp.gate_proj', m), 'up_w': weight('mlp.up_proj', m),
             'down_w': weight('mlp.down_proj')}
        if ada:
            L['mod'] = [(sd[f'{pre}.{nm}.dense.weight'], sd[f'{pre}.{nm}.dense.bias'])
                        for nm in (a, m)]
        out.append(L)
    return out


def _exact_chunk(c, d):
    sd, a = d['sd'], d['call']
    B, pi05 = c['batch'], c['model'] == 'pi05'

    def proj(nm, x):
        return _lin(x, sd[f'{nm}.projector.weight'], sd[f'{nm}.projector.bias'])

    # images
    e, n = f'{VISION}.embeddings', B * c['views']
    x = F.unfold(a['images'].double().view(n, 3, 224, 224), 14, stride=14)
    x = _lin(x.transpose(1, 2), sd[f'{e}.patch_embedding.weight'].flatten(1),
             sd[f'{e}.patch_embedding.bias'])
    x = (x + sd[f'{e}.position_embedding.weight'].double()).reshape(-1, VIT)
    vit = []
    for i in range(c['vit_layers']):
        pre = f'{VISION}.encoder.layers.{i}'
        at = [f'{pre}.self_attn.{p}_proj' for p in 'qkv']
        L = {'qkv_w': torch.cat([sd[f'{p}.weight'] for p in at]),
             'qkv_b': torch.cat([sd[f'{p}.bias'] for p in at])}
        for to, nm in (('ln1', 'layer_norm1'), ('ln2', 'layer_norm2'),
                       ('o', 'self_attn.out_proj'), ('fc1', 'mlp.fc1'),
                       ('fc2', 'mlp.fc2')):
            L[f'{to}_w'], L[f'{to}_b'] = (sd[f'{pre}.{nm}.weight'],
                                          sd[f'{pre}.{nm}.bias'])
        vit.append(L)
    x = _siglip64(x, vit, n)
    x = F.layer_norm(x, (VIT,), sd[f'{VISION}.post_layernorm.weight'].double(),
                     sd[f'{VISION}.post_layernorm.bias'].double(), EPS)
    x = proj('projector', x).view(B, -1, LLM)
    # prompt, prefix layers
    t = sd['llm_backbone.embed_tokens.weight'][a['lang_tokens']].double()
    x = torch.cat([x, t * math.sqrt(LLM)], 1)
    pad = torch.cat([a['img_masks'].repeat_interleave(PATCHES, 1), a['lang_masks']], 1)
    cos, sin = _angles(pad.int().cumsum(1) - 1)
    see = pad[:, None, :].expand(-1, pad.shape[1], -1)
    past = []
    for L in _chunk_layers(c, sd, 'llm_backbone'):
        x, k, v = _gemma_layer(x, L, cos, sin, see)
        past.append((k, v))
    # Euler loop
    layers = _chunk_layers(c, sd, 'llm_expert')
    Ss = ACTIONS + (not pi05)
    cos, sin = _angles(pad.sum(1, keepdim=True) + torch.arange(Ss, device=DEV))
    see = _suffix_view(pad, Ss, not pi05)
    period = 4e-3 * 1000.0**torch.linspace(0, 1, EXP // 2, device=DEV,
                                           dtype=torch.float64)

    def velocity(xt, time):
        """time [ACTIONS]: each position's."""
        ph = time[:, None] * 2 * math.pi / period
        te = torch.cat([torch.sin(ph), torch.cos(ph)], -1)
        h = proj('action_in_proj', xt)

        def mod(w, b):
            return tuple(m.expand(B, -1, -1) for m in _split3(_lin(cond, w, b)))
        if pi05:
            cond = F.silu(proj('time_mlp_out', F.silu(proj('time_mlp_in', te))))
        else:
            h = torch.cat([h, te.expand(B, -1, -1)], -1)
            h = proj('action_time_mlp_out', F.silu(proj('action_time_mlp_in', h)))
            h = torch.cat([proj('state_proj', a['states'].double())[:, None], h], 1)
        for L, kv in zip(layers, past):
            norms = tuple(mod(*m) for m in L['mod']) if pi05 else (None, None)
            h, _, _ = _gemma_layer(h, L, cos, sin, see, kv, norms)
        h = _rms(h[:, -ACTIONS:])
        if pi05:
            s, b, _ = mod(sd['llm_expert.norm.dense.weight'],
                          sd['llm_expert.norm.dense.bias'])
            h = h * (1 + s) + b
        else:
            h = h * (1 + sd['llm_expert.norm.weight'].double())
        return proj('action_out_proj', h)

    xt, dt, lock = a['noise'].double(), -0.1, a.get('prefix_len', 0)
    prev = torch.zeros(B, ACTIONS, ADIM, dtype=torch.float64, device=DEV)
    if lock:
        n_prev = a['prev_actions'].shape[1]
        prev[:, :n_prev] = a['prev_actions'].double()
        # 1 on the locked prefix, then an exponential decay of its length
        w = torch.zeros(ACTIONS, 1, dtype=torch.float64, device=DEV)
        w[:lock] = 1
        for i in range(lock):
            w[lock + i] = math.exp(-3.0 * i / max(lock - 1, 1))
        w[n_prev:] = 0
    for step in range(10):
        time = 1.0 + step * dt
        ts = torch.full((ACTIONS,), time, dtype=torch.float64, device=DEV)
        if c['rtc'] == 'prefix':
            xt = torch.cat([prev[:, :lock], xt[:, lock:]], 1)
            ts[:lock] = 0
            xt = xt + dt * velocity(xt, ts)
        elif c['rtc'] == 'none':
            xt = xt + dt * velocity(xt, ts)
        else:
            vjp = c['rtc'] == 'guidance_vjp'
            p = max(1.0 - time, 1e-6)        # progress: 0 noise, 1 clean
            q = max(time, 1e-6)
            gw = min(q / p * (p * p + q * q) / (q * q), 5.0)
            with torch.set_grad_enabled(vjp):
                xg = xt.detach().requires_grad_(vjp)
                v = -velocity(xg, ts)
                clean = xg + v * q
                err = (w * (prev - clean)).detach()
                if vjp:
                    err, = torch.autograd.grad(clean, xg, err)
            xt = xt - dt * (v.detach() + gw * err)
    if c['rtc'] == 'prefix':
        xt = torch.cat([prev[:, :lock], xt[:, lock:]], 1)
    return xt


_EXACT = {'norm': _exact_norm, 'siglip': _exact_siglip, 'prefix': _exact_prefix,
          'expert': _exact_expert, 'decoder': _exact_decoder,
          'chunk': _exact_chunk}


@torch.no_grad()
def exact(case, seed):
    return _EXACT[case['kind']](case, _inputs(case, seed))
