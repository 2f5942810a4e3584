"""The work whose time this framework is judged by: one denoising step and its parts, through the public entry points.

A case names a path (``kind``) and the sizes it runs at:
  sampler      every update of a sampling schedule (guidance combine + UniPC), without the model
  stack        ``DMStack`` forward of the joint sequence text | video | action
  graph        the same forward recorded once and replayed (``DMStack.capture``)
  context      ``DMStack.precompute_context``: the prompt's keys and values, once per prompt (prefill)
  transformer  ``DMTransformer`` forward, latents in and velocity out, against a kept context (one denoising step)
  production   conditional + unconditional ``DMTransformer`` forward and the sampler's update, two steps
  attention    ``ops.attention`` with the rotation applied inside
  processor    ``DMAttnProcessor`` on a diffusers-style joint-attention module
Widths are those of the repository's configurations (1024 = 16 x 64, 4096 = 32 x 128) and one between; stacks are cut
to a few blocks where every block does the same work, so that a pass stays short.
"""
import torch

from cosmos_amd import DMAttnProcessor, DMConfig, DMStack, DMTransformer, UniPCStepper, ops, rotary

SECTIONS = {64: (16, 24, 24), 128: (32, 48, 48)}
# (d_model, heads, head_dim, hidden)
SMALL, MEDIUM, LARGE = (1024, 16, 64, 4096), (2048, 16, 128, 8192), (4096, 32, 128, 16384)
MAX_FLOPS = 1.6e14                      # of a drawn case; the largest listed one has 1.67e14


def _case(kind, width, blocks=1, grid=(0, 0, 0), text=0, action=0, branches=1, kv=None, fp8=False, qk_norm=False, name=None):
    d, heads, hd, hidden = width
    c = dict(kind=kind, d=d, heads=heads, head_dim=hd, hidden=hidden, blocks=blocks, t=grid[0], h=grid[1], w=grid[2], text=text,
             action=action, branches=branches, kv=heads if kv is None else kv, fp8=fp8, qk_norm=qk_norm)
    if name:
        c["name"] = name
    return c


def _sampler(t, h, w, steps, order, name=None):
    c = dict(kind="sampler", channels=16, t=t, h=h, w=w, steps=steps, order=order)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # what a sampler adds to the model's forwards: 35 updates of the latents of 16 x 44 x 80 tokens (720p, 61 frames)
        _sampler(16, 88, 160, 35, 2, name="sampler_35"),
        # smallest stack of the configurations, called eagerly: latency, launches and host work
        _case("stack", SMALL, 1, (4, 16, 16), name="small_eager"),
        # the same shape as a serving loop runs it
        _case("graph", SMALL, 1, (4, 16, 16), name="small_graph"),
        # a prompt's keys and values for all 28 layers: few rows, every weight read once
        _case("context", LARGE, 28, (16, 44, 80), text=512, name="prompt_512"),
        # one image (a single 44 x 80 frame) per step against its kept prompt
        _case("transformer", LARGE, 4, (1, 44, 80), text=512, name="image"),
        # the same sequence in one joint forward, e4m3 weights and activations
        _case("stack", LARGE, 2, (1, 44, 80), text=512, fp8=True, name="image_fp8"),
        # the layout of a released checkpoint - grouped K/V heads, QK-norm - through guided steps of a short clip
        _case("production", LARGE, 2, (4, 44, 80), text=333, kv=8, qk_norm=True, name="guided_clip"),
        # three weight sets over text, 8 frames of video and a run of actions in one joint sequence
        _case("stack", LARGE, 2, (8, 44, 80), text=1024, action=256, branches=3, name="mixture_action"),
        # the full video sequence, bf16
        _case("stack", LARGE, 2, (16, 44, 80), text=512, name="video"),
        # the full video sequence, e4m3 linears
        _case("stack", LARGE, 2, (16, 44, 80), text=512, fp8=True, name="video_fp8"),
        # rotation and attention alone at the full video grid, for users of the operator
        _case("attention", LARGE, 1, (16, 44, 80), name="attention_video"),
        # attention layer of somebody else's model with this processor installed; ragged context, odd grid
        _case("processor", MEDIUM, 1, (1, 39, 40), text=77, kv=8, qk_norm=True, name="adopted_layer"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _grid(rng, lo, hi):
    """A grid of about lo .. hi tokens (spread over the logarithm), any aspect ratio up to 2."""
    n = _log_int(rng, lo, hi)
    t = rng.choice([1, 1, 2, 3, 4, 5, 8, 11, 16])
    t = min(t, max(1, n // 64))
    h = max(4, int(round((n / t / rng.uniform(0.6, 2.0)) ** 0.5)))
    return t, h, max(4, int(round(n / t / h)))


def draw(rng):
    while True:
        kind = rng.choice(["sampler", "stack", "stack", "graph", "context", "transformer", "transformer", "production",
                           "attention", "processor"])
        if kind == "sampler":
            return _sampler(rng.randint(1, 16), 2 * rng.randint(8, 44), 2 * rng.randint(8, 80), rng.randint(8, 50), rng.choice([1, 2, 2, 3]))
        width = rng.choice([SMALL, MEDIUM, LARGE, LARGE])
        kv = rng.choice([width[1], width[1], width[1] // 4])
        qk = rng.random() < 0.4
        fp8 = kind == "stack" and rng.random() < 0.4
        text = _log_int(rng, 16, 1024)
        blocks = rng.randint(1, 4)
        if kind == "stack":
            blocks = min(blocks, 2) if fp8 else blocks
            branches = rng.choice([1, 1, 2, 3])
            action = _log_int(rng, 8, 256) if branches == 3 else 0
            c = _case(kind, width, blocks, _grid(rng, 256, 56320), rng.choice([0, 64, 512, text]), action, branches, kv, fp8, qk)
        elif kind == "graph":
            c = _case(kind, rng.choice([SMALL, MEDIUM]), blocks, _grid(rng, 256, 4096), rng.choice([0, 64, text]), 0, 1, None, False, qk)
        elif kind == "context":
            c = _case(kind, width, rng.randint(8, 28), (1, 16, 16), text, 0, 1, kv, False, qk)
        elif kind in ("transformer", "production"):
            c = _case(kind, width, blocks, _grid(rng, 256, 28160), text, 0, rng.choice([1, 2]), kv, False, qk)
        elif kind == "attention":
            c = _case(kind, width, 1, _grid(rng, 256, 56320), 0, 0, 1, kv, False, qk)
        else:
            c = _case(kind, width, 1, _grid(rng, 256, 14080), text, 0, 1, kv, False, qk)
        if work(c)["flops"] <= MAX_FLOPS:
            return c


# ----------------------------------------------------------------------------- inputs, models, plans
def _config(c):
    return DMConfig("perf", c["d"], c["heads"], c["head_dim"], c["hidden"], c["blocks"], (c["t"], c["h"], c["w"]), n_text=c["text"],
                    n_action=c["action"], n_branches=c["branches"], mrope_sections=SECTIONS[c["head_dim"]], fp8=c["fp8"],
                    qk_norm=c["qk_norm"], hybrid_mask=c["kind"] in ("context", "transformer", "production"), n_kv_heads=c["kv"])


def _as_trained(module, g, fp8):
    """Norm weights and modulation as a trained model has them: norms around one, shifts, scales and gates of a few
    tenths.  (An e4m3 stack keeps the small gates of the random initialisation: any other order of a sum flips codes of
    the quantiser, a few percent of every update, and large gates would carry that noise into the output.)"""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if "norm" in name:
                p.copy_(1.0 + 0.1 * torch.randn(p.shape, generator=g, device=p.device))
            elif name.endswith("adaLN_modulation.bias") and not fp8:
                p.copy_(0.3 * torch.randn(p.shape, generator=g, device=p.device))


class _Norm(torch.nn.Module):
    def __init__(self, dim):
        super().__init__()
        self.weight, self.eps = torch.nn.Parameter(torch.ones(dim, device="cuda"), requires_grad=False), 1e-6


class _JointAttention(torch.nn.Module):
    """An attention layer as diffusers' joint-attention models name its parts."""

    def __init__(self, d, heads, kv, qk_norm):
        super().__init__()
        hd = d // heads
        lin = lambda o: torch.nn.Linear(d, o, bias=False, device="cuda", dtype=torch.bfloat16)
        self.heads = heads
        self.to_q, self.to_k, self.to_v, self.to_out = lin(d), lin(kv * hd), lin(kv * hd), torch.nn.ModuleList([lin(d)])
        self.add_q_proj, self.add_k_proj, self.add_v_proj, self.to_add_out = lin(d), lin(kv * hd), lin(kv * hd), lin(d)
        if qk_norm:
            self.norm_q, self.norm_k, self.norm_added_q, self.norm_added_k = (_Norm(hd) for _ in range(4))
        self.processor = DMAttnProcessor()

    def forward(self, hidden_states, encoder_hidden_states=None, image_rotary_emb=None):
        return self.processor(self, hidden_states, encoder_hidden_states=encoder_hidden_states, image_rotary_emb=image_rotary_emb)


@torch.no_grad()
def prepare(case, seed):
    c, kind = case, case["kind"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    randn = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    tokens = lambda n: randn(1, n, c["d"]).to(torch.bfloat16)
    if kind == "sampler":
        lat = (1, c["channels"], c["t"], c["h"], c["w"])
        return dict(kind=kind, steps=c["steps"], order=c["order"], noise=randn(*lat), v_cond=randn(*lat).to(torch.bfloat16),
                    v_uncond=randn(*lat).to(torch.bfloat16))
    n_video = c["t"] * c["h"] * c["w"]
    if kind in ("attention", "processor"):
        n = n_video + (c["text"] if kind == "processor" else 0)
        pos, _ = rotary.build_positions(n - n_video, (c["t"], c["h"], c["w"]))
        rot = rotary.rotary_tables(pos, c["head_dim"], SECTIONS[c["head_dim"]], device="cuda")
        if kind == "processor":
            attn = _JointAttention(c["d"], c["heads"], c["kv"], c["qk_norm"])
            for name, p in attn.named_parameters():
                p.copy_(1.0 + 0.1 * randn(*p.shape) if "norm" in name else 0.02 * randn(*p.shape))
            return dict(kind=kind, attn=attn, x=tokens(n_video), ctx=tokens(c["text"]), rot=rot)
        dq, dkv = c["d"], c["kv"] * c["head_dim"]
        scale = 1.0 if c["qk_norm"] else c["head_dim"] ** -0.5
        qkv = (randn(n, dq + 2 * dkv) * scale).to(torch.bfloat16)
        norm = None
        if c["qk_norm"]:
            norm = (1.0 + 0.1 * randn(1, c["head_dim"]), 1.0 + 0.1 * randn(1, c["head_dim"]), (n,), 1e-6)
        return dict(kind=kind, q=qkv[:, :dq], k=qkv[:, dq:dq + dkv], v=qkv[:, dq + dkv:], heads=c["heads"], kv=c["kv"],
                    head_dim=c["head_dim"], rot=rot, norm=norm, out=torch.empty((n, dq), dtype=torch.bfloat16, device="cuda"),
                    workspace=torch.empty(ops.attn_workspace_total_bytes(n, c["heads"], c["kv"], c["head_dim"]), dtype=torch.uint8,
                                          device="cuda"))
    cfg = _config(c)
    model = (DMTransformer if kind in ("transformer", "production") else DMStack)(cfg, device="cuda")
    model.reset_parameters(seed)
    _as_trained(model, g, c["fp8"])
    stack = model.stack if isinstance(model, DMTransformer) else model
    s = dict(kind=kind, model=model, stack=stack, t=torch.rand(1, generator=g, device="cuda") * 1000.0)
    if c["text"]:
        s["ctx"] = tokens(c["text"])
    if kind in ("stack", "graph"):
        s["x"] = tokens(n_video)
        s["action"] = tokens(c["action"]) if c["action"] else None
        if kind == "graph":
            s["graph"] = stack.capture(s["x"], s["t"], encoder_hidden_states=s.get("ctx"))
    elif kind == "context":
        s["kv"], s["head_dim"] = c["kv"], c["head_dim"]
    else:
        s["latents"] = randn(1, 16, c["t"], 2 * c["h"], 2 * c["w"])
        s["cond"] = stack.precompute_context(s["ctx"])
        if kind == "production":
            s["uncond"] = stack.precompute_context(tokens(c["text"]))
    return s


# ----------------------------------------------------------------------------- one pass
def _images(img, n, kv, hd):
    """A layer's kept keys and values as typed views of its buffer: (K and V tiles, largest key norm of every tile)."""
    tiles = (n + 63) // 64
    size = 2 * tiles * 64 * kv * hd * 2
    return img[:size].view(torch.bfloat16), img[size:size + 4 * tiles * kv].view(torch.float32)


def run(s):
    kind = s["kind"]
    if kind == "sampler":
        stepper = UniPCStepper.from_flow_shift(s["steps"], 10.0, guidance_scale=6.0, solver_order=s["order"])
        x = s["noise"].clone()
        for _ in range(s["steps"]):
            stepper.step(s["v_cond"], s["v_uncond"], x)
        return x, stepper.last_sample, stepper.m_hist
    if kind == "stack":
        return s["model"](s["x"], s["t"], encoder_hidden_states=s.get("ctx"), action_states=s["action"])
    if kind == "graph":
        return s["graph"](s["x"], s["t"], encoder_hidden_states=s.get("ctx"))
    if kind == "context":
        cache = s["model"].precompute_context(s["ctx"])
        return [_images(img, cache.n_tokens, s["kv"], s["head_dim"]) for img in cache.images]
    if kind == "transformer":
        return s["model"](s["latents"], s["t"], context_cache=s["cond"])
    if kind == "production":
        stepper = UniPCStepper.from_flow_shift(35, 10.0, guidance_scale=6.0)
        x = s["latents"].clone()
        for _ in range(2):
            t = torch.full((1,), stepper.timesteps[stepper.index], device="cuda")
            v_cond = s["model"](x, t, context_cache=s["cond"])[0]
            v_uncond = s["model"](x, t, context_cache=s["uncond"])[0]
            stepper.step(v_cond, v_uncond, x)
        return x, v_cond, v_uncond
    if kind == "attention":
        return ops.attention(s["q"], s["k"], s["v"], s["heads"], s["head_dim"], out=s["out"], workspace=s["workspace"], cos=s["rot"][0],
                             sin=s["rot"][1], qk_norm=s["norm"], n_kv_heads=s["kv"])
    return s["attn"](s["x"], encoder_hidden_states=s["ctx"], image_rotary_emb=s["rot"])


# ----------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    c, kind = case, case["kind"]
    n_video = c["t"] * c["h"] * c["w"]
    if kind == "sampler":
        n = c["channels"] * n_video
        # per update: latents, two bf16 predictions and the kept tensors in; latents, data prediction, corrected latents out
        return {"bytes": float(c["steps"] * n * (4 + 2 + 2 + 4 * (1 + c["order"]) + 12)), "flops": float(c["steps"] * n * 2 * 3 * (3 + c["order"]))}
    d, h, dkv = c["d"], c["hidden"], c["kv"] * c["head_dim"]
    wb = 1 if c["fp8"] else 2
    qkv, out, mlp = d * (d + 2 * dkv), d * d, 3 * d * h
    if kind == "attention":
        return {"bytes": 2.0 * n_video * (2 * d + 2 * dkv) + 4.0 * n_video * c["head_dim"], "flops": 4.0 * n_video * n_video * d}
    if kind == "processor":
        n = n_video + c["text"]
        return {"bytes": 2.0 * 2 * (qkv + out) + 2.0 * 2 * n * d + 4.0 * n * c["head_dim"], "flops": 2.0 * n * (qkv + out) + 4.0 * n * n * d}
    L, P = c["blocks"], c["text"]
    if kind == "context":
        # the last layer only contributes its keys and values
        gemm, attn = 2.0 * P * ((L - 1) * (qkv + out + mlp) + d * 2 * dkv), (L - 1) * 2.0 * P * P * d
        weights = wb * ((L - 1) * (qkv + out + mlp) + d * 2 * dkv)
        return {"bytes": float(weights + 2 * P * d + L * 4 * P * dkv), "flops": gemm + attn}
    n = n_video + c["action"] + (0 if kind in ("transformer", "production") else P)
    keys = n_video + c["action"] + P
    used = min(c["branches"], (1 if kind in ("transformer", "production") else bool(P)) + 1 + bool(c["action"]))
    if kind in ("transformer", "production"):
        used = 1
    flops = L * (2.0 * n * (qkv + out + mlp) + 4.0 * n * keys * d)
    weights = L * (wb * used * (qkv + out + mlp) + 2 * 6 * d * d)
    if kind in ("stack", "graph"):
        return {"bytes": float(weights + 2 * n * d + 2 * n_video * d), "flops": flops}
    kept = L * 4 * P * dkv
    one = weights + kept + 64 * n_video * (4 + 2)
    if kind == "transformer":
        return {"bytes": float(one), "flops": flops + 4.0 * n * d * 64}
    return {"bytes": float(4 * one + 2 * 64 * n_video * 32), "flops": 4 * (flops + 4.0 * n * d * 64)}


def tolerance(case):
    """About four times what two forms of the attention kernel (32 or 64 query rows per wave, row maxima always or only where
    needed) move the outputs by - the linears' sums come out the same in both of their kernels -, and against the same
    updates in 64 bits for the sampler.  Measured: sampler 1e-7; bf16 stack 2e-3; one forward with its context 7e-3; two
    guided steps 6e-3; attention alone 5e-4, and 1.5e-3 where bf16 partial results are merged; a prompt through 28
    un-modulated layers 1.5e-2, and e4m3 stacks (a last-bit change flips codes) 4e-3 - 1.5e-2, where 3e-2 is the limit."""
    kind = case["kind"]
    if kind == "sampler":
        return {"rel": 1e-6}
    if kind in ("attention", "processor"):
        return {"rel": 6e-3}
    if kind == "context" or case["fp8"]:
        return {"rel": 0.03}
    return {"rel": 8e-3 if kind in ("stack", "graph") else 0.028}
