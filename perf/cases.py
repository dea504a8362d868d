"""The work that this framework is timed on: scoring, prompt passes and pooled decoding of its three model families through the entry points a
program calls (`positional_entropies`, `model(ids)`, `DecodePool.admit / advance / release`), at the layer sizes of the 7B models and a depth of four
layers, random weights.  `listed()` are fixed cases, `draw(rng)` gives others of the same ranges; `prepare` builds what a program holds before
the call, `run` is one pass, `exact` the same outputs in 64 bits from plain torch."""
import math

import torch
import torch.nn.functional as F

from evo_amd.models import architecture_of
from evo_amd.pool import DecodePool
from evo_amd.scoring import positional_entropies
from evo_amd.tokenizer import CharLevelTokenizer

DEV = "cuda:0"
WIDTH, HEADS, VOCAB, EPS = 4096, 32, 512, 1e-6
FF, PLAIN_FF = 11008, 16384
INNER = 10928                      # StripedHyena's own inner size at width 4096
LAYERS = 4
BF16, FP32 = "bf16", "fp32"


# ------------------------------------------------------------------------------------------------ cases
def _case(name, model, what, n, nt, ragged=0, steps=0, dtype=BF16):
    """`n` sequences of at most `nt` nucleotides (tokens), the i-th shorter than the first by up to `ragged` percent; `steps` decoded tokens."""
    c = dict(model=model, what=what, n=n, nt=nt, ragged=ragged, steps=steps, dtype=dtype)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        _case("evo score 1 x 160", "evo", "entropies", 1, 160),                        # one short element: a promoter, a guide, a primer
        _case("evo score 8 x <=900", "evo", "entropies", 8, 900, ragged=60),           # a batch of genes of unequal length, padded by the scorer
        _case("evo score 8 x 8192", "evo", "entropies", 8, 8192),                      # the 8k model's full context, the benchmark's batch
        _case("evo logits 1 x 131072", "evo131k", "logits", 1, 131072),                # the 131k model's full context
        _case("evo generate 1 x 3000", "evo", "decode", 1, 3000, steps=48),            # one stream behind a prompt
        _case("evo pool 16 x <=1100", "evo", "decode", 16, 1100, ragged=80, steps=24),  # many prompts sampled together
        _case("vozalorn prompts 6 x <=2500", "vozalorn", "prompts", 6, 2500, ragged=50),   # unequal prompts packed into one pass, every logit wanted
        _case("vozalorn pool 8 x <=1100", "vozalorn", "decode", 8, 1100, ragged=70, steps=32),   # decoding across the window's edge
        _case("vozalorn fp32 3 x <=500", "vozalorn", "decode", 3, 500, ragged=70, steps=6, dtype=FP32),   # a trace replayed in fp32
        _case("batodra prompt 1 x 8190", "batodra", "prompts", 1, 8190),               # one long document
        _case("batodra pool 24 x <=600", "batodra", "decode", 24, 600, ragged=70, steps=24),
        _case("batodra fp32 3 x <=500", "batodra", "decode", 3, 500, ragged=70, steps=6, dtype=FP32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["evo score", "evo score", "evo decode", "prompts", "decode", "fp32"])
    family = rng.choice(["vozalorn", "batodra"])
    if kind == "evo score":            # one sequence of 40 nt to a 32 k batch
        nt = _log(rng, 40, 16000)
        return _case(None, "evo" if nt < 8192 else "evo131k", rng.choice(["entropies", "logits"]), _log(rng, 1, max(1, min(32, 32768 // nt))), nt,
                     ragged=rng.randrange(0, 70))
    if kind == "evo decode":
        return _case(None, "evo", "decode", _log(rng, 1, 32), _log(rng, 40, 1500), ragged=rng.randrange(0, 90), steps=rng.randrange(8, 33))
    if kind == "prompts":
        nt = _log(rng, 64, 8192)
        return _case(None, family, "prompts", _log(rng, 1, max(1, min(24, 16384 // nt))), nt, ragged=rng.randrange(0, 90))
    if kind == "decode":
        return _case(None, family, "decode", _log(rng, 1, 32), _log(rng, 40, 1500), ragged=rng.randrange(0, 90), steps=rng.randrange(8, 33))
    return _case(None, family, "decode", rng.randrange(1, 5), _log(rng, 40, 500), ragged=rng.randrange(0, 90), steps=rng.randrange(2, 9), dtype=FP32)


def _lengths(case):
    n, nt = case["n"], case["nt"]
    return [max(2, nt - nt * case["ragged"] * ((5 * i) % n) // (100 * n)) for i in range(n)]


# ------------------------------------------------------------------------------------------------ models and their weights
def _config(case):
    kind = case["model"]
    if kind.startswith("evo"):
        c = dict(vocab_size=VOCAB, hidden_size=WIDTH, num_layers=LAYERS, attn_layer_idxs=[2], num_attention_heads=HEADS)
        if kind == "evo131k":
            c.update(use_interpolated_rotary_pos_emb=True, rotary_emb_scaling_factor=16, max_seqlen=131072)
        return c
    rot = dict(base=10000.0, dims=128)
    if kind == "vozalorn":
        ff = dict(kind="dense", ff=FF)
        lat = dict(type="latent_attention", mlp=ff, mixer=dict(heads=HEADS, dim=128, rot_dim=64, vdim=128, kv_rank=512, mask=dict(size=1024),
                                                               rot=dict(base=10000.0, dims=64), scale=192 ** -0.5))
        lin = dict(type="lightning", mlp=ff, mixer=dict(heads=HEADS, dim=128, vdim=128, decay=[1 - 2.0 ** (-1 - 9 * h / HEADS) for h in range(HEADS)]))
        return dict(architecture="Vozalorn", vocab=VOCAB, width=WIDTH, norm=dict(eps=EPS), embedding=dict(scale=1.0), layers=[lat, lin, lat, lin][:LAYERS])
    ff = dict(kind="dense", ff=PLAIN_FF)
    win = dict(type="attention_2", mlp=ff, mixer=dict(heads=32, kv_heads=8, dim=128, vdim=128, mask=dict(size=1024, keep_first=4), scale=128 ** -0.5,
                                                      rot=dict(rot, scaling=dict(factor=4.0, original=4096, fast=32.0, slow=1.0))))
    dif = dict(type="attention", mlp=ff, mixer=dict(heads=16, kv_heads=16, dim=128, vdim=256, scale=128 ** -0.5, diff=0.5, rot=rot))
    rec = dict(type="rglru", mlp=ff, mixer=dict(width=WIDTH, blocks=16, conv=4))
    return dict(architecture="Batodra", vocab=VOCAB, width=WIDTH, norm=dict(eps=EPS), postln_alpha=2.0, layers=[win, rec, dif, rec][:LAYERS])


def _weights(case, shapes, seed):
    """{name: tensor} of the checkpoint, on the GPU; `shapes` in a fixed order."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    dtype = torch.float32 if case["dtype"] == FP32 else torch.bfloat16
    out = {}

    def normal(shape, std, mean=0.0):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(mean, std, generator=g)
    evo = case["model"].startswith("evo")
    for name, shape in shapes.items():
        if name == "unembed.weight":
            out[name] = out["embedding_layer.weight"]
        elif name.endswith("inv_freq"):
            out[name] = 1.0 / 10000.0 ** (torch.arange(0, 128, 2, dtype=torch.float32, device=DEV) / 128)
        elif name.endswith("poles"):                              # memories of ten to a hundred thousand steps
            u = torch.rand(2, WIDTH, 8, generator=g, device=DEV)
            mag, ang = 1.0 - 10.0 ** (4.0 * u[0] - 5.0), (2.0 * u[1] - 1.0) * math.pi
            out[name] = torch.stack([mag * ang.cos(), mag * ang.sin()], -1).reshape(shape)
        elif name.endswith("residues"):                           # of about equal energy
            p = out[name.replace("residues", "poles")].reshape(WIDTH, 8, 2)
            r = torch.randn(WIDTH, 8, 2, generator=g, device=DEV) * (1.0 - p.norm(dim=-1, keepdim=True)).clamp_min(1e-6).sqrt()
            out[name] = r.reshape(shape)
        elif evo:
            # the first block writes the stream, the later ones change it by some per cent, as in trained residual stacks
            gain = 1.0 if name.startswith("blocks.0.") else 0.1
            if name.endswith("scale"):
                out[name] = normal(shape, 0.02, 1.0)
            elif name == "embedding_layer.weight":
                out[name] = normal(shape, 2.0 / math.sqrt(WIDTH))
            elif name.endswith("short_filter_weight"):
                out[name] = normal(shape, 0.3)
            elif name.endswith("filter.D"):
                out[name] = normal(shape, 0.5)
            elif name.endswith("bias"):
                out[name] = normal(shape, 0.02 * (gain if "out_" in name else 1.0))
            elif name.endswith(("projections.weight", "Wqkv.weight")):
                out[name] = normal(shape, 0.04)
            elif name.endswith(("out_filter_dense.weight", "out_proj.weight", "l3.weight")):
                out[name] = normal(shape, 0.03 * gain)
            else:
                out[name] = normal(shape, 0.02)
        elif name.endswith(".lam"):                               # decays per token between about 0.8 and 0.99
            out[name] = torch.empty(shape, dtype=dtype, device=DEV).uniform_(-6.0, -3.0, generator=g)
        elif len(shape) == 1:
            one = 1.0 if "norm" in name and (".mix." in name or case["model"] == "batodra") else 0.0
            out[name] = normal(shape, 0.2, one)
        else:
            out[name] = normal(shape, 1.0 if name == "embed" else 1.0 / math.sqrt(shape[-1]))
    return out


def _build(case, seed):
    config = _config(case)
    dtype = torch.float32 if case["dtype"] == FP32 else torch.bfloat16
    if case["model"].startswith("evo"):
        model = architecture_of(config)(config)
        shapes = {k: tuple(t.shape) for k, t in list(model.named_parameters(remove_duplicate=False)) + list(model.named_buffers())}
    else:
        model = architecture_of(config)(config, dtype=dtype)
        shapes = model.tensor_shapes()
    return model, _weights(case, shapes, seed)


def _tokens(case, seed):
    """Uniform nucleotides: one id vector per sequence (and the decoded ones behind it)."""
    g = torch.Generator().manual_seed(seed + 1)
    letters = torch.tensor(list(b"ACGT"), dtype=torch.int64)
    return [letters[torch.randint(0, 4, (n + case["steps"],), generator=g)] for n in _lengths(case)]


def prepare(case, seed):
    model, weights = _build(case, seed)
    model.load_state_dict(weights, strict=True)
    if case["model"].startswith("evo"):
        model.to_bfloat16_except_poles_residues()
        model = model.to(DEV).eval()
        model.prepare()
    else:
        model = model.to(DEV).eval()
    tokenizer = CharLevelTokenizer(VOCAB)
    tokens, lens, what = _tokens(case, seed), _lengths(case), case["what"]
    state = dict(what=what, model=model, tokenizer=tokenizer)
    if what == "entropies":
        state["seqs"] = [bytes(t.tolist()).decode() for t in tokens]
    elif what == "logits":                                        # BOS in front, pads behind
        ids = torch.full((len(lens), max(lens) + 1), tokenizer.pad_id, dtype=torch.int64)
        ids[:, 0] = tokenizer.eod_id
        for i, t in enumerate(tokens):
            ids[i, 1:1 + t.numel()] = t
        state["ids"] = ids.to(DEV)
    else:
        state["pool"] = DecodePool(model, tokenizer, n_slots=case["n"])
        state["prompts"] = [t[:n].to(DEV) for t, n in zip(tokens, lens)]
        state["next"] = [t[n:].tolist() for t, n in zip(tokens, lens)]
        state["steps"] = case["steps"]
    return state


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    what = state["what"]
    if what == "entropies":
        return torch.cat([torch.from_numpy(e) for e in positional_entropies(state["seqs"], state["model"], state["tokenizer"], device=DEV)])
    if what == "logits":
        with torch.inference_mode():
            return state["model"](state["ids"])[0]
    pool, prompts = state["pool"], state["prompts"]
    if what == "prompts":
        slots, logits = pool.admit(prompts, want=[list(range(p.numel())) for p in prompts])
        for s in slots:
            pool.release(s)
        return torch.cat(logits)
    slots, last = pool.admit(prompts, reserve=state["steps"])
    order = torch.tensor(slots, device=DEV)
    out = [torch.cat(last)]
    for k in range(state["steps"]):
        out.append(pool.advance({s: t[k] for s, t in zip(slots, state["next"])})[order])
    for s in slots:
        pool.release(s)
    return torch.stack(out)                                       # [1 + steps, sequences, vocabulary]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _layer_sizes(case):
    """-> (weights of the dense layers and maps, [attended keys' window or None, flops per (query, key) pair], flops per token of the mixers,
    bytes that one token adds to the caches and a decoded token reads of each earlier one)"""
    D, e = WIDTH, 4 if case["dtype"] == FP32 else 2
    if case["model"].startswith("evo"):
        dense = LAYERS * (4 * D * D + 3 * D * INNER)
        return dense, [(None, 4 * D)], (LAYERS - 1) * D * 8 * 8, 2 * D * e
    if case["model"] == "vozalorn":
        half = LAYERS // 2
        dense = LAYERS * 3 * D * FF + half * (5 * D * D) + half * (HEADS * 192 * D + 576 * D + 2 * HEADS * 128 * 512 + D * D)
        return dense, [(1024, 2 * HEADS * (192 + 128))] * half, half * HEADS * 128 * 128 * 4, half * 576 * e
    dense = LAYERS * 2 * D * PLAIN_FF + (D * 6144 + D * D) + (D * (4096 + 4096 + 4096) + D * D) + 2 * (3 * D * D + 2 * D * 256)
    return dense, [(1024, 2 * 32 * 256), (None, 2 * 16 * (2 * 128 + 2 * 256))], 2 * D * 20, (2 * 1024 + 2 * 4096) * e


def work(case):
    e = 4 if case["dtype"] == FP32 else 2
    dense, pairs, per_token, per_key = _layer_sizes(case)
    lens, steps = _lengths(case), case["steps"]
    if case["what"] in ("entropies", "logits"):
        lens = [max(lens) + 1] * len(lens)                        # (the scorer's padded batch)

    def seen(a, b, w):                                            # keys seen by the tokens a .. b - 1
        return sum(min(t + 1, w or t + 1) for t in range(a, b))
    tokens = sum(lens) + steps * len(lens)
    flops = tokens * (2 * dense + per_token) + sum(f * seen(0, n + steps, w) for w, f in pairs for n in lens)
    outputs = {"entropies": sum(_lengths(case)), "logits": sum(lens) * VOCAB, "prompts": sum(lens) * VOCAB, "decode": (1 + steps) * len(lens) * VOCAB}[case["what"]]
    flops += 2 * WIDTH * (sum(lens) * VOCAB if case["what"] == "entropies" else outputs)
    keys = sum(min(n, pairs[0][0] or n) + steps / 2 for n in lens)
    return {"bytes": (1 + steps) * (dense + VOCAB * WIDTH) * e + steps * keys * per_key + outputs * 4 + tokens * 8, "flops": flops}


def tolerance(case):
    if case["dtype"] == FP32:
        return {"rel": 2e-5}
    # (bf16 models are 1.8e-3, entropies, and 5e-3 to 8e-3, logits, from their values in 64 bits; fp32 ones 2.3e-6 to 2.7e-6)
    return {"rel": 6e-3} if case["what"] == "entropies" else {"rel": 2e-2}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _rms(x, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, window=None, keep=0, sink=None):
    """q [T, H, n], k [T, G, n], v [T, G, dv] of one sequence -> [T, H, dv]; a block of queries at a time."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = q.new_empty(T, H, v.shape[2])
    step = max(64, min(T, (1 << 28) // T))
    for h in range(H):
        g = h * G // H
        for a in range(0, T, step):
            b = min(T, a + step)
            lo = 0 if window is None or keep else max(0, a - window + 1)
            s = (q[a:b, h] @ k[lo:b, g].T) * scale
            d = torch.arange(a, b, device=q.device)[:, None] - torch.arange(lo, b, device=q.device)[None]
            hide = d < 0
            if window is not None:
                hide |= (d >= window) & (torch.arange(lo, b, device=q.device)[None] >= keep)
            s.masked_fill_(hide, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(b - a, 1)], 1)
            p = torch.softmax(s, -1)
            out[a:b, h] = p[:, :b - lo] @ v[lo:b, g]
    return out


def _turn(x, freq, amp=1.0):
    """x [T, heads, n]: pairs (i, i + len(freq)) turned by position * freq[i]."""
    half = freq.numel()
    a = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None, None] * freq
    c, s, u, v = a.cos() * amp, a.sin() * amp, x[..., :half], x[..., half:2 * half]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * half:]], -1)


def _freq(dims, base=10000.0):
    return torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float32).double().to(DEV)


def _evo64(case, w, ids):
    B, T = ids.shape
    D, H, hd = WIDTH, HEADS, WIDTH // HEADS
    x = w["embedding_layer.weight"].double()[ids]                 # [B, T, D]

    def norm(x, s):
        return x / (x.norm(dim=-1, keepdim=True) * D ** -0.5 + EPS) * s.double()

    def get(i, k):
        return w[f"blocks.{i}.{k}"].double()
    for i in range(LAYERS):
        for b in range(B):
            u = norm(x[b], get(i, "pre_norm.scale"))
            if i == 2:
                q, k, v = (u @ get(i, "inner_mha_cls.Wqkv.weight").T + get(i, "inner_mha_cls.Wqkv.bias")).view(T, 3, H, hd).unbind(1)
                pos = torch.arange(T, dtype=torch.float32, device=DEV) / (16.0 if case["model"] == "evo131k" else 1.0)
                a = torch.outer(pos, 1.0 / 10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float32, device=DEV) / hd))
                c, s = (t.bfloat16().double()[:, None] for t in (a.cos(), a.sin()))      # (the model's table is a bf16 one)
                q, k = (torch.cat([t[..., :64] * c - t[..., 64:] * s, t[..., :64] * s + t[..., 64:] * c], -1) for t in (q, k))
                y = _attend(q, k, v, hd ** -0.5).reshape(T, D)
                del q, k, v
                y = y @ get(i, "inner_mha_cls.out_proj.weight").T + get(i, "inner_mha_cls.out_proj.bias")
            else:
                y = torch.empty(T, D, dtype=torch.float64, device=DEV)
                p, r = (torch.view_as_complex(get(i, "filter." + k).reshape(D, 8, 2).contiguous()) for k in ("poles", "residues"))
                wp, bp, fw, fb, skip = (get(i, k) for k in ("projections.weight", "projections.bias", "filter.short_filter_weight", "filter.short_filter_bias", "filter.D"))
                t = torch.arange(T, dtype=torch.float64, device=DEV)
                for h in range(H):                                # (a head's columns are x2 | x1 | v)
                    cols, ch = slice(3 * hd * h, 3 * hd * (h + 1)), slice(hd * h, hd * (h + 1))
                    z = F.pad(u @ wp[cols].T + bp[cols], (0, 0, 2, 0))
                    z = sum(z[k:k + T] * fw[cols, 0, k] for k in range(3)) + fb[cols]
                    x1v = (z[:, hd:2 * hd] * z[:, 2 * hd:]).T.contiguous()
                    filt = torch.zeros(hd, T, dtype=torch.float64, device=DEV)
                    for m in range(8):
                        filt += (r[ch, m, None] * torch.exp(torch.log(p[ch, m, None]) * t)).real
                    conv = torch.fft.irfft(torch.fft.rfft(x1v, n=2 * T) * torch.fft.rfft(filt, n=2 * T), n=2 * T)[:, :T]
                    y[:, ch] = (conv + x1v * skip[ch, None]).T * z[:, :hd]
                y = y @ get(i, "out_filter_dense.weight").T + get(i, "out_filter_dense.bias")
            x[b] += y
            del y, u
            for a in range(0, T, 16384):
                n = norm(x[b, a:a + 16384], get(i, "post_norm.scale"))
                x[b, a:a + 16384] += (F.gelu(n @ get(i, "mlp.l1.weight").T) * (n @ get(i, "mlp.l2.weight").T)) @ get(i, "mlp.l3.weight").T
    return norm(x, w["norm.scale"]) @ w["unembed.weight"].double().T


def _vozalorn64(case, w, ids):
    config, out = _config(case), []
    for row in ids:                                               # each sequence of its own
        x, T = w["embed"].double()[row], row.numel()
        for i, layer in enumerate(config["layers"]):
            m, H = layer["mixer"], HEADS

            def get(k):
                return w[f"l{i}.{k}"].double()
            if layer["type"] == "lightning":
                q, k, v = (F.silu(x @ get("mix." + n).T).view(T, H, 128) for n in "qkv")
                o, t = torch.empty_like(v), torch.arange(T, device=DEV, dtype=torch.float64)
                for h in range(H):
                    a = torch.tensor(m["decay"][h], dtype=torch.float32).double().item()
                    for b in range(0, T, 2048):
                        e = min(T, b + 2048)
                        d = t[b:e, None] - t[None, :e]
                        s = (q[b:e, h] @ k[:e, h].T) * torch.where(d >= 0, a ** d.clamp_min(0), 0.0)
                        o[b:e, h] = s @ v[:e, h]
                y = _rms(o.reshape(T, -1)) * get("mix.norm") * torch.sigmoid(x @ get("mix.g").T)
            else:
                f = _freq(64)
                q = (x @ get("mix.q").T).view(T, H, 192)
                q = torch.cat([q[..., :128], _turn(q[..., 128:], f)], -1)
                down = x @ get("mix.dkv").T
                c, kr = _rms(down[:, :512]) * get("mix.dkv.norm"), _turn(down[:, None, 512:], f)
                k = torch.cat([(c @ get("mix.uk").T).view(T, H, 128), kr.expand(T, H, 64)], -1)
                y = _attend(q, k, (c @ get("mix.uv").T).view(T, H, 128), m["scale"], m["mask"]["size"], 0, get("mix.sink")).reshape(T, -1)
            x = x + _rms(y @ get("mix.o").T) * (1.0 + get("norm1"))
            y = (F.silu(x @ get("mlp.gate").T) * (x @ get("mlp.up").T)) @ get("mlp.down").T
            x = x + _rms(y) * (1.0 + get("norm2"))
        out.append((_rms(x) * (1.0 + w["final.norm"].double())) @ w["head"].double().T)
    return out


def _batodra64(case, w, ids):
    config, out = _config(case), []
    for row in ids:
        x, T = w["embed"].double()[row], row.numel()
        for i, layer in enumerate(config["layers"]):
            m = layer["mixer"]

            def get(k):
                return w[f"l{i}.{k}"].double()
            if layer["type"] == "rglru":
                y = F.gelu(x @ get("mix.y").T + get("mix.y.b"), approximate="tanh")
                z, taps = F.pad(x @ get("mix.x").T + get("mix.x.b"), (0, 0, 3, 0)), get("mix.conv")
                u = sum(z[j:j + T] * taps[:, j] for j in range(4)) + get("mix.conv.b")
                r, g = (torch.sigmoid(torch.einsum("tbi,boi->tbo", u.view(T, 16, 256), get("mix." + k)) + get(f"mix.{k}.b")).reshape(T, -1) for k in ("ra", "ri"))
                log_a = -8.0 * r * F.softplus(get("mix.lam"))
                a, add = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * g * u
                S, d = add, 1                                     # scan by doubling: S_t = a_t S_{t-1} + add_t
                while d < T:
                    S = torch.cat([S[:d], S[d:] + a[d:] * S[:-d]])
                    a = torch.cat([a[:d], a[d:] * a[:-d]])
                    d *= 2
                y = S * y
            else:
                maps, dv, H, G = (2, 256, 16, 16) if layer["type"] == "attention" else (1, 128, 32, 8)
                q, k = (x @ get("mix.q").T).view(T, H * maps, 128), (x @ get("mix.k").T).view(T, G * maps, 128)
                v, f = (x @ get("mix.v").T).view(T, G, dv), _freq(128)
                if maps == 2:
                    q, k = (_turn(_rms(t) * get(n), f).view(T, -1, 2, 128) for t, n in ((q, "mix.q.norm"), (k, "mix.k.norm")))
                    l1, l2 = ((get("mix.lq" + n) * get("mix.lk" + n)).sum().exp() for n in "12")
                    a1, a2 = (_attend(q[:, :, j], k[:, :, j], v, m["scale"]) for j in (0, 1))
                    y = _rms(a1 - (l1 - l2 + m["diff"]) * a2) * (1.0 - m["diff"])
                else:
                    s = m["rot"]["scaling"]                       # pairs that turn seldom over the original length are slowed
                    lo, hi = (128 * math.log(s["original"] / (2 * math.pi * n)) / (2 * math.log(10000.0)) for n in (s["fast"], s["slow"]))
                    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), 127)
                    ramp = ((torch.arange(64, dtype=torch.float64, device=DEV) - lo) / max(hi - lo, 1e-3)).clamp(0.0, 1.0)
                    f, amp = f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0
                    y = _attend(_rms(_turn(q, f, amp)), _rms(_turn(k, f, amp)), v, m["scale"], m["mask"]["size"], m["mask"]["keep_first"])
                y = y.reshape(T, -1)
            x = _rms(2.0 * x + y @ get("mix.o").T) * get("norm1")
            x = _rms(2.0 * x + F.relu(x @ get("mlp.up").T).square() @ get("mlp.down").T) * get("norm2")
        out.append((_rms(x) * w["final.norm"].double()) @ w["head"].double().T)
    return out


def exact(case, seed):
    if case["n"] * case["nt"] > 70000:                            # (over half a minute in 64 bits)
        return None
    _, w = _build(case, seed)
    tokens, lens = _tokens(case, seed), _lengths(case)
    with torch.inference_mode():
        if case["what"] in ("entropies", "logits"):
            ids = torch.full((len(lens), max(lens) + 1), 1, dtype=torch.int64)
            ids[:, 0] = 0
            for i, t in enumerate(tokens):
                ids[i, 1:1 + t.numel()] = t
            logits = _evo64(case, w, ids.to(DEV))
            if case["what"] == "logits":
                return logits
            lsm = torch.log_softmax(logits, -1)
            entropy = -(lsm.exp() * lsm).sum(-1)
            return torch.cat([entropy[i, :n] for i, n in enumerate(lens)])
        rows = [t.to(DEV) for t in tokens]
        if case["model"] == "evo":
            logits = [_evo64(case, w, t[None])[0] for t in rows]
        else:
            logits = (_vozalorn64 if case["model"] == "vozalorn" else _batodra64)(case, w, rows)
        if case["what"] == "prompts":
            return torch.cat(logits)
        return torch.stack([lg[n - 1:] for lg, n in zip(logits, lens)], 1)
