"""The work a user of exn_hip has it do, as cases that can be timed and compared.

A picture takes the prompt encoder (a prompt to states), eight velocities of the DiT (the first
with the prompt's rows, the rest over its kept K/V) and the VAE decoder; an edit also the vision
tower and the VAE encoder on the picture to edit.  Each case is one call of one of these parts
through its public entry point on device pointers, as a host that keeps its tensors on the GPU
calls it.  The encoder runs 4 of its 36 blocks and the DiT 2 of its 32 (both take the number of
blocks when they are made): every block does the same work, and a change of rounding has fewer
blocks to travel through.  The VAE and the tower run whole.

Weights and inputs come from the seed: Q8_0 matrices of uniform codes and |N(0, 2e-4)| scales
(unit gain at these widths), N(0, 1) states, latents and pictures in -1 .. 1.  exact() restates
each part in plain torch in 64 bits.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ex-nihilo_amd"))
import exn_hip as X  # noqa: E402

WIDTH, HEADS, HD, FFN = 4096, 32, 128, 12288
DEV = "cuda"


def listed():
    return [
        # a short prompt, the most usual call of the encoder: launches and the weights' bytes
        {"name": "prompt 24", "kind": "encoder", "tokens": 24, "picture_h": 0, "picture_w": 0, "layers": 4},
        # a long description
        {"name": "prompt 256", "kind": "encoder", "tokens": 256, "picture_h": 0, "picture_w": 0, "layers": 4},
        # an edit's prompt: the picture's 1024 rows and deepstack sets amid 76 tokens of text
        {"name": "edit prompt 1100", "kind": "encoder", "tokens": 1100, "picture_h": 32, "picture_w": 32, "layers": 4},
        # a 512 x 512 draft's first step, the prompt's rows in the pass
        {"name": "first step 512x512", "kind": "dit", "h": 32, "w": 32, "text": 64, "ref_h": 0, "ref_w": 0,
         "kept": False, "mode": "bf16", "layers": 2},
        # the usual picture's steps 2 to 8
        {"name": "step 1024x1024", "kind": "dit", "h": 64, "w": 64, "text": 256, "ref_h": 0, "ref_w": 0,
         "kept": True, "mode": "bf16", "layers": 2},
        # a wide picture where the weights stay Q8_0 only
        {"name": "q8_0 step 1536x1024", "kind": "dit", "h": 64, "w": 96, "text": 256, "ref_h": 0, "ref_w": 0,
         "kept": True, "mode": "q8_0", "layers": 2},
        # the reference's own default arithmetic: int8 products
        {"name": "int8 step 1024x1024", "kind": "dit", "h": 64, "w": 64, "text": 256, "ref_h": 0, "ref_w": 0,
         "kept": True, "mode": "int8", "layers": 2},
        # an edit's first step: text, the reference picture and the image, 8704 rows
        {"name": "edit first step", "kind": "dit", "h": 64, "w": 64, "text": 512, "ref_h": 64, "ref_w": 64,
         "kept": False, "mode": "bf16", "layers": 2},
        # the picture's pixels from its latent
        {"name": "decode 1024x1024", "kind": "decode", "h": 64, "w": 64},
        # the picture to edit, to its latent
        {"name": "encode 1024x1024", "kind": "encode", "h": 64, "w": 64},
        # the picture to edit, as the prompt encoder sees it: a thumbnail and a whole picture
        {"name": "vision 320x256", "kind": "vision", "h": 320, "w": 256},
        {"name": "vision 1024x1024", "kind": "vision", "h": 1024, "w": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("encoder", "encoder", "dit", "dit", "dit", "decode", "encode", "vision"))
    if kind == "encoder":
        g = rng.choice((0, 0, 1))
        ph, pw = (g * rng.randint(4, 32) for _ in range(2))
        return {"kind": kind, "tokens": ph * pw + _log(rng, 8, 640 if not g else 76), "picture_h": ph, "picture_w": pw,
                "layers": rng.randint(2, 4)}
    if kind == "dit":
        h, w = _log(rng, 12, 64), _log(rng, 12, 96)
        ref = rng.choice((0, 0, 0, 1))
        return {"kind": kind, "h": h, "w": w, "text": _log(rng, 8, 512), "ref_h": ref * _log(rng, 12, 48),
                "ref_w": ref * _log(rng, 12, 48), "kept": rng.random() < 0.6,
                "mode": rng.choice(("bf16", "bf16", "q8_0", "int8")), "layers": 2}
    if kind == "vision":
        return {"kind": kind, "h": 32 * _log(rng, 4, 32), "w": 32 * _log(rng, 4, 32)}
    return {"kind": kind, "h": _log(rng, 10, 64), "w": _log(rng, 10, 64)}


# --- weights ---------------------------------------------------------------------------------


class Tensors:
    """A model's tensors by name, each made from (seed, its place in the list) when asked for."""

    def __init__(self, seed, specs):
        self.seed, self.specs = int(seed), specs           # name -> (kind, shape, base, scale)
        self.place = {n: i for i, n in enumerate(specs)}

    def _gen(self, name):
        return torch.Generator(DEV).manual_seed((self.seed * 1000003 + self.place[name] * 7919 + 17) % (1 << 62))

    def _made(self, name):
        kind, shape, base, scale = self.specs[name]
        g = self._gen(name)
        if kind == "q8":
            q = torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8)
            d = (torch.randn(shape[0], shape[1] // 32, generator=g, device=DEV) * scale).abs().half()
            return q, d
        v = base + scale * torch.randn(*shape, generator=g, device=DEV)
        return v.half() if kind == "f16" else v.bfloat16() if kind == "bf16" else v

    def given(self, name):
        """The tensor as a file holds it: (ggml kind, numpy data)."""
        kind, shape = self.specs[name][:2]
        m = self._made(name)
        if kind == "q8":
            q, d = m
            rec = torch.cat([d.reshape(-1, 1).view(torch.uint8), q.reshape(-1, 32).view(torch.uint8)], 1)
            return X.Q8_0, rec.cpu().numpy()
        if kind == "f32":
            return X.F32, m.cpu().numpy()
        return (X.F16 if kind == "f16" else X.BF16), m.view(torch.int16).cpu().numpy().view(np.uint16)

    def __call__(self, name):
        """The tensor in 64 bits."""
        m = self._made(name)
        if self.specs[name][0] != "q8":
            return m.double()
        q, d = m
        return (q.double().reshape(*d.shape, 32) * d.double()[..., None]).reshape(q.shape)


def _q8(rows, cols):
    return ("q8", (rows, cols), 0.0, 2e-4 * math.sqrt(4096 / cols))


def dit_tensors(seed, layers):
    s = {"img_in.weight": _q8(WIDTH, 64), "txt_in.text_norm.weight": ("f32", (WIDTH,), 0.0, 0.05),
         "txt_in.in_layer.weight": _q8(WIDTH, WIDTH), "txt_in.out_layer.weight": _q8(WIDTH, WIDTH),
         "time_text_embed.timestep_embedder.linear_1.weight": _q8(WIDTH, 256),
         "time_text_embed.timestep_embedder.linear_2.weight": _q8(WIDTH, WIDTH),
         "modulation.1.weight": _q8(4 * WIDTH, WIDTH), "norm_out.linear.weight": _q8(WIDTH, WIDTH),
         "proj_out.weight": _q8(64, WIDTH)}
    for i in range(layers):
        b = "transformer_blocks.%d." % i
        s.update({b + "attn.norm_q.weight": ("f32", (HD,), 1.0, 0.05), b + "attn.norm_k.weight": ("f32", (HD,), 1.0, 0.05)})
        s.update({b + "attn.%s.weight" % n: _q8(WIDTH, WIDTH) for n in ("to_q", "to_k", "to_v", "to_out.0")})
        s.update({b + "img_mlp.gate_up.weight": _q8(2 * FFN, WIDTH), b + "img_mlp.out.weight": _q8(WIDTH, FFN)})
    return Tensors(seed, s)


VOCAB = 8192


def encoder_tensors(seed, layers):
    s = {"token_embd.weight": ("f32", (VOCAB, WIDTH), 0.0, 1.0)}
    for i in range(layers):
        b = "blk.%d." % i
        s.update({b + "%s_norm.weight" % n: ("f32", (d,), 1.0, 0.05)
                  for n, d in (("attn", WIDTH), ("attn_q", HD), ("attn_k", HD), ("ffn", WIDTH))})
        s.update({b + n + ".weight": _q8(r, c) for n, r, c in (
            ("attn_q", WIDTH, WIDTH), ("attn_k", 1024, WIDTH), ("attn_v", 1024, WIDTH), ("attn_output", WIDTH, WIDTH),
            ("ffn_gate", FFN, WIDTH), ("ffn_up", FFN, WIDTH), ("ffn_down", WIDTH, FFN))})
    return Tensors(seed, s)


# (in, out, spatial, temporal) of each stage, from the latent's end and from the picture's
UP = ((1152, 1152, 1, 1), (1152, 1152, 1, 1), (1152, 576, 1, 1), (576, 288, 1, 0), (288, 144, 0, 0))
DOWN = ((96, 96, 1, 0), (96, 192, 1, 1), (192, 384, 1, 1), (384, 768, 1, 1), (768, 768, 0, 0))


def vae_tensors(seed):
    s = {}

    def conv(name, o, i, k, frame=True, gain=1.0):
        s[name + ".weight"] = ("bf16", (o, i, 1, k, k) if frame else (o, i, k, k), 0.0, gain / math.sqrt(i * k * k))
        s[name + ".bias"] = ("bf16", (o,), 0.0, 0.02)

    def res(p, i, o):
        s[p + ".residual.0.gamma"] = ("bf16", (i, 1, 1, 1), 1.0, 0.1)
        conv(p + ".residual.2", o, i, 3)
        s[p + ".residual.3.gamma"] = ("bf16", (o, 1, 1, 1), 1.0, 0.1)
        conv(p + ".residual.6", o, o, 3, gain=0.5)
        if i != o:
            conv(p + ".shortcut", o, i, 1)

    def middle(p, c):
        res(p + ".0", c, c)
        s[p + ".1.norm.gamma"] = ("bf16", (c, 1, 1), 1.0, 0.1)
        conv(p + ".1.to_qkv", 3 * c, c, 1, False)
        conv(p + ".1.proj", c, c, 1, False, 0.5)
        res(p + ".2", c, c)

    conv("conv2", 64, 64, 1)
    conv("decoder.conv1", 1152, 64, 3)
    middle("decoder.middle", 1152)
    for n, (i, o, up, _) in enumerate(UP):
        for j in range(3):
            res("decoder.upsamples.%d.upsamples.%d" % (n, j), i if j == 0 else o, o)
        if up:
            conv("decoder.upsamples.%d.upsamples.3.resample.1" % n, o, o, 3, False)
    s["decoder.head.0.gamma"] = ("bf16", (144, 1, 1, 1), 1.0, 0.1)
    conv("decoder.head.2", 4, 144, 3)
    conv("encoder.conv1", 96, 4, 3)
    for n, (i, o, down, _) in enumerate(DOWN):
        for j in range(2):
            res("encoder.downsamples.%d.downsamples.%d" % (n, j), i if j == 0 else o, o)
        if down:
            conv("encoder.downsamples.%d.downsamples.2.resample.1" % n, o, o, 3, False)
    middle("encoder.middle", 768)
    s["encoder.head.0.gamma"] = ("bf16", (768, 1, 1, 1), 1.0, 0.1)
    conv("encoder.head.2", 128, 768, 3)
    conv("conv1", 128, 128, 1)
    return Tensors(seed, s)


VW, VF = 1152, 4304


def vision_tensors(seed):
    s = {}

    def vec(name, n, weight=False):
        s[name] = ("f32", (n,), 1.0 if weight else 0.0, 0.1 if weight else 0.02)

    def linear(name, o, i, gain=1.0):
        s[name + ".weight"] = ("f16", (o, i), 0.0, gain / math.sqrt(i))
        vec(name + ".bias", o)

    for n in ("v.patch_embd.weight", "v.patch_embd.weight.1"):
        s[n] = ("f16", (VW, 3, 16, 16), 0.0, 0.7 / math.sqrt(768))
    vec("v.patch_embd.bias", VW)
    s["v.position_embd.weight"] = ("f16", (48 * 48, VW), 0.0, 1.0)
    for i in range(27):
        b = "v.blk.%d." % i
        for n in ("ln1", "ln2"):
            vec(b + n + ".weight", VW, True)
            vec(b + n + ".bias", VW)
        linear(b + "attn_qkv", 3 * VW, VW, 2.0)
        linear(b + "attn_out", VW, VW, 0.5)
        linear(b + "ffn_up", VF, VW)
        linear(b + "ffn_down", VW, VF, 0.5)
    for norm, fc1, fc2, n in [("v.deepstack.%d.norm" % i, "v.deepstack.%d.fc1" % i, "v.deepstack.%d.fc2" % i, 4 * VW)
                              for i in (8, 16, 24)] + [("v.post_ln", "mm.0", "mm.2", VW)]:
        vec(norm + ".weight", n, True)
        vec(norm + ".bias", n)
        linear(fc1, 4 * VW, 4 * VW)
        linear(fc2, 4096, 4 * VW)
    return Tensors(seed, s)


# --- inputs ----------------------------------------------------------------------------------


def _randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(DEV).manual_seed(int(seed) * 31 + 5), device=DEV)


def dit_inputs(c, seed):
    """(states, latent, reference latent or None, sigma)."""
    p, h, w, rh, rw = c["text"], c["h"], c["w"], c["ref_h"], c["ref_w"]
    ref = _randn(seed + 300, 64, rh, rw) if rh else None
    return _randn(seed + 100, p, WIDTH), _randn(seed + 200, 64, h, w), ref, 0.89508


def ref_a(c):
    """An edit's text rows ahead of its reference picture."""
    return min(8, c["text"]) if c["ref_h"] else 0


def encoder_inputs(c, seed):
    """(ids, positions, a0, merged, deep): the picture after a0 tokens of text, as an edit's prompt."""
    n, gh, gw = c["tokens"], c["picture_h"], c["picture_w"]
    ids = torch.randint(0, VOCAB, (n,), generator=torch.Generator().manual_seed(int(seed) + 9), dtype=torch.int32).numpy()
    m = gh * gw
    a0 = (n - m) // 3 if m else 0
    pos = np.arange(n, dtype=np.int32)[:, None].repeat(3, 1)
    if not m:
        return ids, pos, 0, None, None
    r, k = np.divmod(np.arange(m, dtype=np.int32), gw)
    pos[a0:a0 + m] = np.stack([np.full(m, a0, np.int32), a0 + r, a0 + k], 1)
    pos[a0 + m:] = (a0 + max(gh, gw) + np.arange(n - a0 - m, dtype=np.int32))[:, None]
    z = _randn(seed + 400, 4, m, WIDTH)
    return ids, pos, a0, z[0].contiguous(), z[1:].contiguous()


def picture(seed, h, w):
    px = (0.5 * _randn(seed + 500, h, w, 4)).clamp(-1, 1)
    px[..., 3] = 1.0
    return px


# --- prepare and run -------------------------------------------------------------------------

_context = None


def context():
    global _context
    if _context is None:
        _context = X.Context(0)
    return _context


class Held:
    """A model that goes when its state goes, and the call that is one pass."""

    def __init__(self, model, call, args, keep, out):
        self.model, self.call, self.args, self.keep, self.out = model, call, args, keep, out

    def __del__(self):
        self.model.destroy()


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    if kind == "dit":
        model = X.Dit(ctx, case["layers"])
        t = dit_tensors(seed, case["layers"])
        model.resident(case["mode"] == "bf16")
        for name, (k, shape, _, _) in t.specs.items():
            model.set(name, *t.given(name), (shape[1], shape[0]) if len(shape) > 1 else shape)
        model.w8a8(case["mode"] == "int8")
        states, latent, ref, sigma = dit_inputs(case, seed)
        v = torch.empty_like(latent)
        key = model.prefix_key("prompt") if case["kept"] else 0
        args = (model.h, _p(states), case["text"], _p(latent), case["h"], case["w"], sigma, key, ref_a(case), _p(ref),
                case["ref_h"], case["ref_w"], _p(v))
        torch.cuda.synchronize()
        state = Held(model, "exn_dit_velocity_dev", args, (states, latent, ref), v)
        if case["kept"]:                      # the loop's first step, which keeps the prompt's K/V
            X.call(state.call, *args)
            ctx.sync()
        return state
    if kind == "encoder":
        model = X.Encoder(ctx, case["layers"])
        t = encoder_tensors(seed, case["layers"])
        for name, (k, shape, _, _) in t.specs.items():
            model.set(name, *t.given(name), shape[-1], shape[0] if len(shape) > 1 else 1)
        ids, pos, a0, merged, deep = encoder_inputs(case, seed)
        cs = torch.from_numpy(X.enc_rope_table(len(ids), pos)).to(DEV)
        ids = torch.from_numpy(ids).to(DEV)
        out = torch.empty(len(ids), WIDTH, device=DEV)
        args = (model.h, _p(ids), len(ids), _p(cs), a0, case["picture_h"] * case["picture_w"], _p(merged), _p(deep), _p(out))
        torch.cuda.synchronize()
        return Held(model, "exn_enc_states_dev", args, (ids, cs, merged, deep), out)
    if kind == "vision":
        model, t = X.Vision(ctx), vision_tensors(seed)
        h, w = case["h"], case["w"]
        px, m = picture(seed, h, w), h * w // 1024
        out = {"merged": torch.empty(m, 4096, device=DEV), "deep": torch.empty(3, m, 4096, device=DEV)}
        args, name_of = (model.h, _p(px), h, w, _p(out["merged"]), _p(out["deep"])), "exn_vision_encode_dev"
    else:
        model, t = X.Vae(ctx), vae_tensors(seed)
        h, w = case["h"], case["w"]
        if kind == "decode":
            px, out = _randn(seed + 200, 64, h, w), torch.empty(16 * h, 16 * w, 4, device=DEV)
        else:
            px, out = picture(seed, 16 * h, 16 * w), torch.empty(64, h, w, device=DEV)
            h, w = 16 * h, 16 * w
        args, name_of = (model.h, _p(px), h, w, _p(out)), "exn_vae_%s_dev" % kind
    for name, (k, shape, _, _) in t.specs.items():
        if kind not in ("decode", "encode") or (kind == "encode") == (name.startswith(("encoder.", "conv1."))):
            model.set(name, *t.given(name), shape)
    torch.cuda.synchronize()
    return Held(model, name_of, args, (px,), out)


def run(state):
    X.call(state.call, *state.args)
    return state.out


# --- work ------------------------------------------------------------------------------------


def _resblock(n, i, o):
    return 2 * n * (9 * i * o + 9 * o * o + (i * o if i != o else 0))


def work(case):
    kind = case["kind"]
    if kind == "dit":
        p, nref, nimg, L = case["text"], case["ref_h"] * case["ref_w"], case["h"] * case["w"], case["layers"]
        n0, l, a = p + nref if case["kept"] else 0, p + nref + nimg, ref_a(case)
        # the prefix's rows go through every block but the last, which takes their K and V alone
        pre = 0 if case["kept"] else p + nref
        g = torch.arange(pre)
        pairs = L * nimg * l + (L - 1) * int(torch.where((g >= a) & (g < a + nref), a + nref, g + 1).sum())
        params = 4 * WIDTH * WIDTH + 3 * FFN * WIDTH
        edge = 64 * WIDTH * 2 + 256 * WIDTH + 6 * WIDTH * WIDTH + (0 if case["kept"] else 2 * WIDTH * WIDTH)
        flops = 2 * params * (L * nimg + (L - 1) * pre) + 4 * pre * WIDTH * WIDTH + 4 * HD * HEADS * pairs
        flops += 2 * nimg * 128 * WIDTH + 24 * WIDTH * WIDTH
        if not case["kept"]:
            flops += 4 * p * WIDTH * WIDTH + 2 * nref * 64 * WIDTH
        data = 4 * (2 * 64 * nimg + (0 if case["kept"] else p * WIDTH + 64 * nref)) + 4 * L * n0 * WIDTH
        return {"bytes": (L * params + edge) * 34 // 32 + data, "flops": flops}
    if kind == "encoder":
        n, L = case["tokens"], case["layers"]
        params = 2 * WIDTH * WIDTH + 2 * 1024 * WIDTH + 3 * FFN * WIDTH
        m = case["picture_h"] * case["picture_w"]
        return {"bytes": L * params * 34 // 32 + 4 * WIDTH * (2 * n + 3 * m),
                "flops": L * (2 * n * params + 4 * HD * HEADS * n * (n + 1) // 2)}
    if kind == "vision":
        n = case["h"] * case["w"] // 256
        m, t = n // 4, vision_tensors(0)
        params = sum(math.prod(s) for _, s, _, _ in t.specs.values())
        flops = 2 * n * VW * 768 + 27 * (2 * n * VW * (4 * VW + 2 * VF) + 4 * n * n * VW) + 8 * m * 4 * VW * (4 * VW + 4096)
        return {"bytes": 2 * params + 16 * case["h"] * case["w"] + 16 * m * 4096, "flops": flops}
    n, t = case["h"] * case["w"], vae_tensors(0)
    mine = [s for k, (_, s, _, _) in t.specs.items() if (kind == "encode") == k.startswith(("encoder.", "conv1."))]
    top = 1152 if kind == "decode" else 768
    flops = 2 * _resblock(n, top, top) + 8 * n * top * top + 4 * n * n * top
    if kind == "decode":
        flops += 2 * n * 64 * 64 + 2 * n * 64 * top * 9
        for i, o, up, _ in UP:
            flops += _resblock(n, i, o) + 2 * _resblock(n, o, o)
            if up:
                n *= 4
                flops += 18 * n * o * o
        flops += 2 * n * 144 * 4 * 9
    else:
        flops += 2 * n * top * 128 * 9 + 2 * n * 128 * 128
        n *= 256
        flops += 18 * n * 4 * 96
        for i, o, down, _ in DOWN:
            flops += _resblock(n, i, o) + _resblock(n, o, o)
            if down:
                n //= 4
                flops += 18 * n * o * o
    return {"bytes": 2 * sum(math.prod(s) for s in mine) + 4 * case["h"] * case["w"] * (64 + 1024), "flops": flops}


def tolerance(case):
    # about four times the distance seen from exact() over drawn cases.  encoder 4.7e-3, dit 5.6e-4:
    # bf16 operands, fp16 attention and 32-bit sums over their blocks; int8 3.8e-3: codes of 8 bits a
    # block of 32; decode and encode 4.9e-3: bf16 activations over some 30 convolutions; vision 6.6e-5:
    # 32-bit arithmetic over 27 blocks
    kind = "int8" if case.get("mode") == "int8" else case["kind"]
    return {"rel": {"encoder": 1.8e-2, "dit": 2.2e-3, "int8": 1.5e-2, "vision": 2.6e-4}.get(kind, 2e-2)}


# --- the same in 64 bits -----------------------------------------------------------------------


def _ln(x, eps=1e-6):
    m = x.mean(-1, keepdim=True)
    return (x - m) / ((x - m).square().mean(-1, keepdim=True) + eps).sqrt()


def _rms(x, w, eps=1e-6):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _attend(q, k, v, lim=None):
    """q (n, heads, d), k and v (l, kv heads, d); row t sees the keys 0 .. lim[t]."""
    n, heads, d = q.shape
    rep, out = heads // k.shape[1], torch.empty_like(q)
    hidden = None if lim is None else torch.arange(k.shape[0], device=DEV)[None, :] > lim[:, None]
    for h in range(heads):
        s = q[:, h] @ k[:, h // rep].t().contiguous() / math.sqrt(d)
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // rep].contiguous()
    return out.reshape(n, heads * d)


def _grid(frame, h, w):
    r, c = np.meshgrid(np.arange(h), np.arange(w), indexing="ij")
    return np.stack([np.full(h * w, frame), (r - (h - h // 2)).ravel(), (c - (w - w // 2)).ravel()], 1)


def _same3(first, n):
    return np.repeat(first + np.arange(n)[:, None], 3, 1)


def exact_dit(c, seed):
    t = dit_tensors(seed, c["layers"])
    states, latent, ref, sigma = (x.double() if torch.is_tensor(x) else x for x in dit_inputs(c, seed))
    p, a, nref, nimg = c["text"], ref_a(c), c["ref_h"] * c["ref_w"], c["h"] * c["w"]

    def mm(name, x):
        if c["mode"] == "int8" and len(x) >= 16:      # activations in codes of 8 bits a block of 32, scales fp16
            b = x.reshape(len(x), -1, 32)
            d = b.abs().amax(-1, keepdim=True) / 127
            q = torch.sign(b) * torch.floor(b.abs() / torch.where(d > 0, d, torch.ones_like(d)) + 0.5)
            x = (q * d.half().double()).reshape(x.shape)
        return x @ t(name).t().contiguous()

    f = torch.exp(-math.log(10000.0) * torch.arange(128, device=DEV, dtype=torch.float64) / 128)
    e = torch.stack([torch.cat([torch.cos(s * f), torch.sin(s * f)]) for s in (1000 * sigma, 0.0)])
    e = _silu(_silu(e @ t("time_text_embed.timestep_embedder.linear_1.weight").t())
              @ t("time_text_embed.timestep_embedder.linear_2.weight").t())
    mod = (e @ t("modulation.1.weight").t()).reshape(2, 4, WIDTH)
    img = mm("img_in.weight", latent.reshape(64, -1).t().contiguous())
    txt = mm("txt_in.in_layer.weight", _rms(states, 1.0 + t("txt_in.text_norm.weight")))
    txt = mm("txt_in.out_layer.weight", _gelu(txt))
    if ref is None:
        x = torch.cat([txt, img])
        pos = np.concatenate([_same3(0, p), _grid(p, c["h"], c["w"])])
    else:
        x = torch.cat([txt[:a], mm("img_in.weight", ref.reshape(64, -1).t().contiguous()), txt[a:], img])
        after = a + max(c["ref_h"], c["ref_w"])
        pos = np.concatenate([_same3(0, a), _grid(a, c["ref_h"], c["ref_w"]), _same3(after, p - a),
                              _grid(after + p - a, c["h"], c["w"])])
    ang = np.concatenate([pos[:, i:i + 1] * (10000.0 ** -(np.arange(0, d, 2) / d)) for i, d in enumerate((16, 56, 56))], 1)
    cos, sin = (torch.from_numpy(fn(ang)).to(DEV)[:, None, :] for fn in (np.cos, np.sin))
    rows = torch.arange(len(x), device=DEV)
    prefix = p + nref
    lim = torch.where(rows >= prefix, len(x) - 1, torch.where((rows >= a) & (rows < a + nref), a + nref - 1, rows))
    mod = mod[(rows < prefix).long()]

    def turned(y, w):
        y = _rms(y.reshape(len(y), HEADS, HD), w)
        u, v = y[..., 0::2], y[..., 1::2]
        return torch.stack([u * cos - v * sin, u * sin + v * cos], -1).reshape(y.shape)

    for i in range(c["layers"]):
        b = "transformer_blocks.%d." % i
        y = _ln(x) * (1.0 + mod[:, 0])
        q = turned(mm(b + "attn.to_q.weight", y), t(b + "attn.norm_q.weight"))
        k = turned(mm(b + "attn.to_k.weight", y), t(b + "attn.norm_k.weight"))
        v = mm(b + "attn.to_v.weight", y).reshape(len(y), HEADS, HD)
        x = x + torch.tanh(mod[:, 1]) * mm(b + "attn.to_out.0.weight", _attend(q, k, v, lim))
        g, u = mm(b + "img_mlp.gate_up.weight", _ln(x) * (1.0 + mod[:, 2])).chunk(2, 1)
        x = x + torch.tanh(mod[:, 3]) * mm(b + "img_mlp.out.weight", _silu(g) * u)
    y = _ln(x[prefix:]) * (1.0 + e[:1] @ t("norm_out.linear.weight").t())
    return mm("proj_out.weight", y).t().reshape(64, c["h"], c["w"]).contiguous()


def exact_encoder(c, seed):
    t = encoder_tensors(seed, c["layers"])
    ids, pos, a0, merged, deep = encoder_inputs(c, seed)
    x = t("token_embd.weight")[torch.from_numpy(ids).to(DEV).long()]
    n, m = len(ids), c["picture_h"] * c["picture_w"]
    if m:
        x[a0:a0 + m] = merged.double()
    j = np.arange(64)
    ang = pos[:, np.where(j < 60, j % 3, 0)].astype(np.float64) * 5e6 ** (-2.0 * j / 128)
    cos, sin = (torch.from_numpy(fn(ang)).to(DEV)[:, None, :].repeat(1, 1, 2) for fn in (np.cos, np.sin))
    lim = torch.arange(n, device=DEV)

    def turned(y, w):
        y = _rms(y.reshape(n, -1, HD), w)
        return y * cos + torch.cat([-y[..., 64:], y[..., :64]], -1) * sin

    for i in range(c["layers"]):
        b = "blk.%d." % i
        h = _rms(x, t(b + "attn_norm.weight"))
        q = turned(h @ t(b + "attn_q.weight").t(), t(b + "attn_q_norm.weight"))
        k = turned(h @ t(b + "attn_k.weight").t(), t(b + "attn_k_norm.weight"))
        v = (h @ t(b + "attn_v.weight").t()).reshape(n, -1, HD)
        x = x + _attend(q, k, v, lim) @ t(b + "attn_output.weight").t()
        h = _rms(x, t(b + "ffn_norm.weight"))
        x = x + (_silu(h @ t(b + "ffn_gate.weight").t()) * (h @ t(b + "ffn_up.weight").t())) @ t(b + "ffn_down.weight").t()
        if m and i < 3:
            x[a0:a0 + m] += deep[i].double()
    return x


def _conv(t, p, x, step=1):
    """x (H, W, C), 3 x 3 'same' or 1 x 1; STEP 2: zeros only below and to the right."""
    w, b = t(p + ".weight"), t(p + ".bias")
    w = w.reshape(w.shape[0], w.shape[1], w.shape[-2], w.shape[-1])
    if w.shape[-1] == 1:
        return x @ w[:, :, 0, 0].t() + b
    h, wd, c = x.shape
    lo = 1 if step == 1 else 0
    xp = torch.nn.functional.pad(x, (0, 0, lo, 1, lo, 1))
    ho, wo = h // step, wd // step
    y = b.expand(ho * wo, -1).clone()
    for dy in range(3):
        for dx in range(3):
            tap = xp[dy:dy + step * ho:step, dx:dx + step * wo:step].reshape(-1, c)
            y.addmm_(tap, w[:, :, dy, dx].t().contiguous())
    return y.reshape(ho, wo, -1)


def _norm(t, name, x):
    return x / x.square().sum(-1, keepdim=True).sqrt().clamp_min(1e-12) * math.sqrt(x.shape[-1]) * t(name).reshape(-1)


def _res(t, p, x):
    y = _conv(t, p + ".residual.2", _silu(_norm(t, p + ".residual.0.gamma", x)))
    y = _conv(t, p + ".residual.6", _silu(_norm(t, p + ".residual.3.gamma", y)))
    return y + (_conv(t, p + ".shortcut", x) if p + ".shortcut.weight" in t.specs else x)


def _middle(t, p, x):
    x = _res(t, p + ".0", x)
    h, w, c = x.shape
    qkv = _conv(t, p + ".1.to_qkv", _norm(t, p + ".1.norm.gamma", x)).reshape(h * w, 1, 3 * c)
    a = _attend(qkv[..., :c], qkv[..., c:2 * c], qkv[..., 2 * c:])
    return _res(t, p + ".2", _conv(t, p + ".1.proj", a.reshape(h, w, c)) + x)


def exact_decode(c, seed):
    t = vae_tensors(seed)
    x = _randn(seed + 200, 64, c["h"], c["w"]).double().permute(1, 2, 0)
    x = _middle(t, "decoder.middle", _conv(t, "decoder.conv1", _conv(t, "conv2", x)))
    for n, (i, o, up, frames) in enumerate(UP):
        x0 = x
        for j in range(3):
            x = _res(t, "decoder.upsamples.%d.upsamples.%d" % (n, j), x)
        if up:
            ft = 1 + frames
            h, w, _ = x0.shape
            twice = x.repeat_interleave(2, 0).repeat_interleave(2, 1)
            short = x0.repeat_interleave(o * ft * 4 // i, -1).reshape(h, w, o, ft, 2, 2)[:, :, :, ft - 1]
            x = _conv(t, "decoder.upsamples.%d.upsamples.3.resample.1" % n, twice)
            x = x + short.permute(0, 3, 1, 4, 2).reshape(2 * h, 2 * w, o)
    return _conv(t, "decoder.head.2", _silu(_norm(t, "decoder.head.0.gamma", x))).clamp(-1, 1)


def exact_encode(c, seed):
    t = vae_tensors(seed)
    x = _conv(t, "encoder.conv1", picture(seed, 16 * c["h"], 16 * c["w"]).double())
    for n, (i, o, down, frames) in enumerate(DOWN):
        x0 = x
        for j in range(2):
            x = _res(t, "encoder.downsamples.%d.downsamples.%d" % (n, j), x)
        if down:
            ft = 1 + frames
            h, w = x0.shape[0] // 2, x0.shape[1] // 2
            full = torch.zeros(h, w, i, ft, 2, 2, device=DEV, dtype=torch.float64)
            full[:, :, :, ft - 1] = x0.reshape(h, 2, w, 2, i).permute(0, 2, 4, 1, 3)
            x = _conv(t, "encoder.downsamples.%d.downsamples.2.resample.1" % n, x, 2)
            x = x + full.reshape(h, w, o, -1).mean(-1)
        else:
            x = x + x0
    x = _silu(_norm(t, "encoder.head.0.gamma", _middle(t, "encoder.middle", x)))
    x = _conv(t, "conv1", _conv(t, "encoder.head.2", x))
    return x[..., :64].permute(2, 0, 1).contiguous()


def exact_vision(c, seed):
    t = vision_tensors(seed)
    gh, gw = c["h"] // 16, c["w"] // 16
    n = gh * gw

    def linear(name, x):
        return x @ t(name + ".weight").t() + t(name + ".bias")

    def ln(name, x):
        return _ln(x) * t(name + ".weight") + t(name + ".bias")

    # patches in merge-block order: block row, block column, then the 2 x 2 inside
    order = np.arange(n).reshape(gh // 2, 2, gw // 2, 2).transpose(0, 2, 1, 3).ravel()
    rows, cols = np.divmod(order, gw)
    px = picture(seed, c["h"], c["w"]).double()[..., :3]
    pat = px.reshape(gh, 16, gw, 16, 3).permute(0, 2, 4, 1, 3).reshape(n, 768)[torch.from_numpy(order).to(DEV)]
    x = pat @ (t("v.patch_embd.weight") + t("v.patch_embd.weight.1")).reshape(VW, 768).t() + t("v.patch_embd.bias")
    table = t("v.position_embd.weight").reshape(48, 48, VW)

    def taps(i, size):
        s = i * 47.0 / max(size - 1, 1)
        lo = np.minimum(np.floor(s).astype(np.int64), 47)
        return lo, np.minimum(lo + 1, 47), torch.from_numpy(s - lo).to(DEV)[:, None]

    r0, r1, fr = taps(rows, gh)
    c0, c1, fc = taps(cols, gw)
    x = x + (1 - fr) * ((1 - fc) * table[r0, c0] + fc * table[r0, c1]) + fr * ((1 - fc) * table[r1, c0] + fc * table[r1, c1])
    inv = 10000.0 ** -(np.arange(18) / 18)
    ang = np.concatenate([rows[:, None] * inv, cols[:, None] * inv], 1)
    cos, sin = (torch.from_numpy(fn(ang)).to(DEV)[:, None, :].repeat(1, 1, 2) for fn in (np.cos, np.sin))

    def turned(y):
        return y * cos + torch.cat([-y[..., 36:], y[..., :36]], -1) * sin

    def merger(y, fc1, fc2):
        return linear(fc2, torch.nn.functional.gelu(linear(fc1, y)))

    deep = []
    for i in range(27):
        b = "v.blk.%d." % i
        qkv = linear(b + "attn_qkv", ln(b + "ln1", x)).reshape(n, 3, 16, 72)
        x = x + linear(b + "attn_out", _attend(turned(qkv[:, 0]), turned(qkv[:, 1]), qkv[:, 2]))
        x = x + linear(b + "ffn_down", _gelu(linear(b + "ffn_up", ln(b + "ln2", x))))
        if i in (8, 16, 24):
            d = "v.deepstack.%d." % i
            deep.append(merger(ln(d + "norm", x.reshape(-1, 4 * VW)), d + "fc1", d + "fc2"))
    merged = merger(ln("v.post_ln", x).reshape(-1, 4 * VW), "mm.0", "mm.2")
    return {"merged": merged, "deep": torch.stack(deep)}


def exact(case, seed):
    return {"dit": exact_dit, "encoder": exact_encoder, "decode": exact_decode, "encode": exact_encode,
            "vision": exact_vision}[case["kind"]](case, seed)
