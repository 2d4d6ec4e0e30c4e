"""The work that users of rollfast_amd have it do, as timed cases.

A case is one call (or one optimizer step) through the public API on inputs
that are already on the GPU: the fused 8-bit AdamW step over parameter trees
from a few small leaves to Llama-7B-wide layers, with each option that
changes the work (stochastic rounding of params and of moments, block size,
f32 params, clipping, the fine-tune composition, gradient accumulation,
full-precision moments), the two-call Optax form, and the standalone
quantize_blocks / dequantize_blocks.

A parameter tree's buffers are laid out the way a restored checkpoint's are:
one arena per kind (params, grads, codes, scales, unquantized moments), each
leaf a 256-byte aligned view.  The moments are those of a run in progress
(first moments a fraction of the gradient scale, second moments around its
square), quantized to the codebooks in plain torch.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import rollfast_amd as rf

MIN_SIZE = 4096  # adamw8's default: smaller leaves keep unquantized moments
B1, B2, EPS = 0.9, 0.999, 1e-8
LR, DECAY = 1e-3, 0.01
COUNT = 100  # steps taken before the timed ones
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
CLIP = 1.0
MICRO_STEPS = 4
# finetune's groups: learning rate and decay by leaf-name prefix
GROUPS = {"a": (1e-3, 0.05), "b": (2e-3, 0.0)}


def listed():
    return [
        # the work of a full training step of a 7B model's eight layers and
        # embeddings: large matrices, bf16, nearest rounding
        {"name": "step_llama_8_layers", "kind": "step", "tree": "llama", "hidden": 4096, "ffn": 11008, "vocab": 32000,
         "layers": 8, "dtype": "bf16", "block_size": 2048, "param_sr": False, "moment_sr": False, "bits": "jax",
         "clip": False},
        # a small language model with adamw8_step's default stochastic
        # rounding of the bf16 params; LayerNorm vectors on f32 moments
        {"name": "step_gpt2_small_sr", "kind": "step", "tree": "gpt2", "hidden": 768, "vocab": 50304, "layers": 12,
         "dtype": "bf16", "block_size": 2048, "param_sr": True, "moment_sr": False, "bits": "jax", "clip": False},
        # unbiased 8-bit state: moments and params both stochastically rounded
        {"name": "step_llama_layer_all_sr", "kind": "step", "tree": "llama", "hidden": 4096, "ffn": 11008, "vocab": 0,
         "layers": 1, "dtype": "bf16", "block_size": 2048, "param_sr": True, "moment_sr": True, "bits": "jax",
         "clip": False},
        # finer quantization blocks, for outlier-heavy gradients
        {"name": "step_llama_layer_block256", "kind": "step", "tree": "llama", "hidden": 4096, "ffn": 11008,
         "vocab": 0, "layers": 1, "dtype": "bf16", "block_size": 256, "param_sr": False, "moment_sr": False,
         "bits": "jax", "clip": False},
        # the smallest models: a few leaves of odd sizes in f32, where the
        # call's latency counts
        {"name": "step_mlp_small", "kind": "step", "tree": "mlp", "hidden": 301, "ffn": 517, "vocab": 10, "layers": 4,
         "dtype": "f32", "block_size": 2048, "param_sr": False, "moment_sr": False, "bits": "jax", "clip": False},
        # many leaves of every size, most of them below min_size, with
        # global-norm clipping and the cheaper packed rounding bits
        {"name": "step_ragged_clip", "kind": "step", "tree": "ragged", "vectors": 2000, "matrices": 256, "most": 2048,
         "dtype": "bf16", "block_size": 2048, "param_sr": True, "moment_sr": False, "bits": "packed", "clip": True},
        # an existing Optax program: tx.update, then apply_updates, f32 master params
        {"name": "optax_gpt2_small_f32", "kind": "optax", "tree": "gpt2", "hidden": 768, "vocab": 50304, "layers": 12,
         "dtype": "f32", "block_size": 2048, "param_sr": False, "moment_sr": False, "bits": "jax", "clip": False},
        # adamw with stochastically rounded bf16 moments
        {"name": "adamw_llama_layer_bf16", "kind": "adamw", "tree": "llama", "hidden": 4096, "ffn": 11008, "vocab": 0,
         "layers": 1, "dtype": "bf16", "moments": "bf16", "param_sr": True, "bits": "jax"},
        # fine-tuning adapters: low-rank pairs beside frozen weights, two
        # parameter groups, clipping and the non-finite guard
        {"name": "finetune_lora", "kind": "finetune", "tree": "lora", "hidden": 4096, "rank": 16, "layers": 32,
         "dtype": "bf16", "block_size": 2048, "param_sr": False},
        # a window of four micro-steps into an f32 accumulator
        {"name": "accumulate_gpt2_small", "kind": "accumulate", "tree": "gpt2", "hidden": 768, "vocab": 50304,
         "layers": 12, "dtype": "bf16", "block_size": 2048, "param_sr": False},
        # moments or checkpoints into 8-bit blocks and back
        {"name": "quantize_2p26", "kind": "quantize", "size": (1 << 26) + 1000, "dtype": "f32", "block_size": 2048,
         "quantizer": "dynamic_signed", "sr": False},
        {"name": "dequantize_2p26", "kind": "dequantize", "size": (1 << 26) + 1000, "dtype": "f32",
         "block_size": 2048, "quantizer": "dynamic_unsigned"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _block_size(rng):
    return 2048 if rng.random() < 0.5 else rng.choice([128, 256, 512, 1024, 4096, 1000])


def _draw_tree(rng):
    """A tree of 50 thousand to about 400 million parameters."""
    style = rng.choice(["llama", "gpt2", "mlp", "ragged", "lora"])
    if style == "llama":
        h = _log_int(rng, 256, 4096) // 8 * 8 + rng.choice([0, 0, 0, 4])
        return {"tree": "llama", "hidden": h, "ffn": int(h * rng.uniform(2.5, 4.0)),
                "vocab": rng.choice([0, 8000, 32000]) if h <= 2048 else 0, "layers": rng.randint(1, 2)}
    if style == "gpt2":
        return {"tree": "gpt2", "hidden": _log_int(rng, 128, 1280), "vocab": rng.choice([1000, 50257, 50304]),
                "layers": rng.randint(2, 12)}
    if style == "mlp":
        return {"tree": "mlp", "hidden": _log_int(rng, 65, 3000), "ffn": _log_int(rng, 65, 6000),
                "vocab": rng.randint(2, 1000), "layers": rng.randint(2, 8)}
    if style == "lora":
        return {"tree": "lora", "hidden": _log_int(rng, 512, 8192), "rank": rng.choice([4, 8, 16, 64]),
                "layers": rng.randint(4, 40)}
    return {"tree": "ragged", "vectors": _log_int(rng, 100, 2000), "matrices": _log_int(rng, 10, 256),
            "most": _log_int(rng, 256, 2048)}


def draw(rng):
    kind = rng.choice(["step", "step", "step", "step", "optax", "adamw", "finetune", "accumulate", "quantize",
                       "dequantize"])
    if kind in ("quantize", "dequantize"):
        return {"kind": kind, "size": _log_int(rng, 5000, 1 << 28), "dtype": rng.choice(["f32", "f32", "bf16"]),
                "block_size": _block_size(rng),
                "quantizer": rng.choice(["dynamic_signed", "dynamic_unsigned", "symmetric_int8"]),
                **({"sr": rng.random() < 0.3} if kind == "quantize" else {})}
    case = {"kind": kind, **_draw_tree(rng), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if case["dtype"] == "f32" and rng.random() < 0.4:
        case["grads"] = "bf16"  # mixed precision: f32 master params
    if kind == "adamw":
        case["moments"] = rng.choice(["bf16", "f32"])
        case["bits"] = rng.choice(["jax", "packed"])
    else:
        case["block_size"] = _block_size(rng)
    case["param_sr"] = case["dtype"] == "bf16" and rng.random() < 0.5
    if kind in ("step", "optax"):
        case["moment_sr"] = rng.random() < 0.25
        case["bits"] = rng.choice(["jax", "packed"])
        case["clip"] = kind == "step" and rng.random() < 0.25
    return case


# ------------------------------------------------------------- the trees ---
def _shapes(case):
    """[(leaf name, shape)] of the case's parameter tree."""
    tree, out = case["tree"], []
    if tree == "llama":
        h, f, v = case["hidden"], case["ffn"], case["vocab"]
        if v:
            out += [("embed", (v, h)), ("lm_head", (v, h)), ("norm", (h,))]
        for i in range(case["layers"]):
            out += [("layer%02d.%s" % (i, n), s) for n, s in (
                ("q", (h, h)), ("k", (h, h)), ("v", (h, h)), ("o", (h, h)), ("gate", (f, h)), ("up", (f, h)),
                ("down", (h, f)), ("attn_norm", (h,)), ("mlp_norm", (h,)))]
    elif tree == "gpt2":
        d = case["hidden"]
        out += [("wte", (case["vocab"], d)), ("ln_f", (d,))]
        for i in range(case["layers"]):
            out += [("h%02d.%s" % (i, n), s) for n, s in (
                ("qkv", (d, 3 * d)), ("proj", (d, d)), ("fc", (d, 4 * d)), ("fc_proj", (4 * d, d)), ("ln1", (d,)),
                ("ln2", (d,)))]
    elif tree == "mlp":
        widths = [case["hidden"]] + [case["ffn"]] * (case["layers"] - 1) + [case["vocab"]]
        for i, (a, b) in enumerate(zip(widths, widths[1:])):
            out += [("fc%d.w" % i, (a, b)), ("fc%d.b" % i, (b,))]
    elif tree == "lora":
        h, r = case["hidden"], case["rank"]
        for i in range(case["layers"]):
            for n in ("q", "v"):
                out += [("a.layer%02d.%s" % (i, n), (r, h)), ("b.layer%02d.%s" % (i, n), (h, r))]
    else:
        pick = np.random.default_rng(0)
        sizes = lambda lo, hi, n: np.exp(pick.uniform(math.log(lo), math.log(hi), n)).astype(int)  # noqa: E731
        out += [("v%04d" % i, (int(n),)) for i, n in enumerate(sizes(16, 4096, case["vectors"]))]
        rows, cols = (sizes(64, case["most"], case["matrices"]) for _ in range(2))
        out += [("m%03d" % i, (int(r), int(c))) for i, (r, c) in enumerate(zip(rows, cols))]
    return out


def _quantized(case, n):
    return case["kind"] != "adamw" and n >= MIN_SIZE


def _blocks(case, n):
    return -(-n // case["block_size"])


class _Arena:
    """One buffer with a 256-byte aligned place per leaf."""

    def __init__(self, sizes, dtype):
        step = 256 // torch.empty((), dtype=dtype).element_size()
        self.at, n = {}, 0
        for name, size in sizes:
            self.at[name] = (n, size)
            n += -(-size // step) * step
        self.flat = torch.zeros(n, dtype=dtype, device="cuda")

    def __getitem__(self, name):
        at, size = self.at[name]
        return self.flat[at: at + size]


def _codebook(signed):
    """The dynamic 8-bit map: seven decades of evenly spaced bin means, 0 and 1."""
    data = []
    for i in range(7):
        edges = np.linspace(0.1, 1.0, (1 << (i if signed else i + 1)) + 1)
        means = (edges[:-1] + edges[1:]) / 2.0 * 10.0 ** (i - 6)
        data += list(means) + (list(-means) if signed else [])
    return torch.tensor(sorted(data + [0.0, 1.0]), dtype=torch.float32, device="cuda")


def _to_codes(x, block_size, signed):
    """(codes, scales) of a flat f32 tensor: block absmax scales, nearest codes."""
    nb = -(-x.numel() // block_size)
    blocks = torch.nn.functional.pad(x, (0, nb * block_size - x.numel())).view(nb, block_size)
    scales = blocks.abs().amax(1)
    scales = torch.where(scales > 0, scales, torch.ones_like(scales))
    cb = _codebook(signed)
    codes = torch.bucketize(blocks / scales[:, None], (cb[1:] + cb[:-1]) / 2, out_int32=True)
    return codes.to(torch.uint8).view(-1), scales


class _Tree:
    """A case's parameter tree with its gradients and moments, from the seed."""

    def __init__(self, case, seed, gradients=1):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        self.case = case
        self.shapes = dict(_shapes(case))
        sizes = [(k, math.prod(s)) for k, s in self.shapes.items()]
        self.sizes = dict(sizes)
        dtype = DTYPES[case["dtype"]]
        self.grads = [_Arena(sizes, DTYPES[case.get("grads", case["dtype"])]) for _ in range(gradients)]
        # gradient scales differ by leaf
        pick = np.random.default_rng(seed)
        scale = {k: float(10.0 ** pick.uniform(-4.5, -2.5)) for k, _ in sizes}
        for g in self.grads:
            for k, n in sizes:
                g[k].copy_(torch.randn(n, generator=gen, device="cuda") * scale[k])
        self.params = _Arena(sizes, dtype)
        for k, n in sizes:
            self.params[k].copy_(torch.randn(n, generator=gen, device="cuda") * 0.02)
        quant = [(k, n) for k, n in sizes if _quantized(case, n)]
        plain = [(k, n) for k, n in sizes if not _quantized(case, n)]
        self.codes = [_Arena([(k, _blocks(case, n) * case["block_size"]) for k, n in quant], torch.uint8)
                      for _ in range(2 if quant else 0)]
        self.scales = [_Arena([(k, _blocks(case, n)) for k, n in quant], torch.float32)
                       for _ in range(2 if quant else 0)]
        self.moments = [_Arena(plain, DTYPES[case.get("moments", "f32")]) for _ in range(2 if plain else 0)]
        for k, n in sizes:
            m = torch.randn(n, generator=gen, device="cuda") * (0.3 * scale[k])
            v = torch.exp(torch.randn(n, generator=gen, device="cuda") * 0.4) * scale[k] ** 2
            for i, x in enumerate((m, v)):
                if _quantized(case, n):
                    codes, scales = _to_codes(x, case["block_size"], i == 0)
                    self.codes[i][k].copy_(codes)
                    self.scales[i][k].copy_(scales)
                else:
                    self.moments[i][k].copy_(x)

    def tree(self, arena):
        return {k: arena[k].view(s) for k, s in self.shapes.items()}

    def restore(self, state):
        """The optimizer state of tx.init with this tree's moments and step count in it."""
        if hasattr(state, "mu") and hasattr(state, "nu"):
            return state._replace(count=np.asarray(COUNT, dtype=np.int32),
                                  **{f: {k: self._moment(i, k, x) for k, x in getattr(state, f).items()}
                                     for i, f in enumerate(("mu", "nu"))})
        if isinstance(state, tuple) and hasattr(state, "_fields"):
            return type(state)(*[self.restore(x) for x in state])
        if isinstance(state, tuple):
            return tuple(self.restore(x) for x in state)
        if isinstance(state, dict):
            return {k: self.restore(x) for k, x in state.items()}
        return state

    def _moment(self, i, name, leaf):
        if isinstance(leaf, rf.QuantizedBlocks):
            children, aux = leaf.tree_flatten()
            return rf.QuantizedBlocks.tree_unflatten(
                aux, (self.codes[i][name].view(children[0].shape), self.scales[i][name]))
        return self.moments[i][name].view(leaf.shape) if isinstance(leaf, torch.Tensor) else leaf

    def outputs(self):
        out = {"params": self.params.flat}
        for what, arenas in (("codes", self.codes), ("scales", self.scales), ("moments", self.moments)):
            for i, a in enumerate(arenas):
                out["%s_%s" % (("mu", "nu")[i], what)] = a.flat
        return out


def _transformation(case):
    key = rf.prng.PRNGKey(7)
    kind = case["kind"]
    if kind == "adamw":
        return rf.adamw(LR, b1=B1, b2=B2, eps=EPS, weight_decay=DECAY, key=key, sr_bits=case["bits"],
                        mu_dtype=DTYPES["bf16"] if case["moments"] == "bf16" else None)
    if kind == "finetune":
        groups = {g: rf.adamw8(lr, b1=B1, b2=B2, eps=EPS, weight_decay=wd, block_size=case["block_size"],
                               key=rf.prng.PRNGKey(i)) for i, (g, (lr, wd)) in enumerate(GROUPS.items())}
        labels = {k: _group(k) for k, _ in _shapes(case)}
        groups = {g: tx for g, tx in groups.items() if g in labels.values()}
        tx = rf.chain(rf.clip_by_global_norm(CLIP), rf.multi_transform(groups, labels))
        return rf.apply_if_finite(tx, max_consecutive_errors=1)
    tx = rf.adamw8(LR, b1=B1, b2=B2, eps=EPS, weight_decay=DECAY, block_size=case["block_size"], key=key,
                   stochastic_rounding=case.get("moment_sr", False), sr_bits=case.get("bits", "jax"))
    if kind == "accumulate":
        return rf.MultiSteps(tx, every_k_schedule=MICRO_STEPS, accumulator_dtype=torch.float32)
    return tx


def _group(name):
    return "b" if name.startswith("b.") else "a"


class _State:
    pass


# -------------------------------------------------------------- the cases --
def prepare(case, seed):
    s = _State()
    s.case = case
    s.key = rf.prng.PRNGKey(seed % (1 << 31))
    if case["kind"] in ("quantize", "dequantize"):
        s.x = _values(case, seed)
        if case["kind"] == "dequantize":
            s.x = _quantized_blocks(case, s.x)
        return s
    s.tree = _Tree(case, seed, MICRO_STEPS if case["kind"] == "accumulate" else 1)
    s.grads = [s.tree.tree(g) for g in s.tree.grads]
    s.params = s.tree.tree(s.tree.params)
    s.tx = _transformation(case)
    s.opt_state = s.tree.restore(s.tx.init(s.params))
    if case["kind"] == "accumulate":
        s.acc = _Arena(list(s.tree.sizes.items()), torch.float32)
        s.opt_state = s.opt_state._replace(acc_grads=s.tree.tree(s.acc))
    return s


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "quantize":
        q = rf.quantize_blocks(s.x, block_size=case["block_size"], quantizer=case["quantizer"],
                               stochastic_rounding=case["sr"], key=s.key if case["sr"] else None)
        return {"codes": q.values, "scales": q.scales}
    if kind == "dequantize":
        return {"x": rf.dequantize_blocks(s.x, dtype=DTYPES[case["dtype"]])}
    if kind == "optax":
        updates, s.opt_state = s.tx.update(s.grads[0], s.opt_state, s.params)
        s.params = rf.apply_updates(s.params, updates, key=s.key, stochastic=case["param_sr"], sr_bits=case["bits"])
        return s.tree.outputs()
    step = rf.adamw_step if kind == "adamw" else rf.adamw8_step
    more = {"clip_global_norm": CLIP} if case.get("clip") else {}
    for g in s.grads:
        s.params, s.opt_state = step(s.tx, s.params, g, s.opt_state, key=s.key, stochastic=case["param_sr"], **more)
    out = s.tree.outputs()
    if kind == "accumulate":
        out["acc"] = s.acc.flat
    return out


def _values(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n = case["size"]
    x = torch.randn(n, generator=gen, device="cuda") * torch.exp(torch.randn(n, generator=gen, device="cuda") - 7.0)
    if case["quantizer"] == "dynamic_unsigned":
        x = x * x
    return x.to(DTYPES[case["dtype"]]) if case["kind"] == "quantize" else x


def _quantized_blocks(case, x):
    if case["quantizer"] == "symmetric_int8":
        nb = _blocks(case, case["size"])
        blocks = torch.nn.functional.pad(x, (0, nb * case["block_size"] - x.numel())).view(nb, -1)
        scales = blocks.abs().amax(1) / 127.0
        return rf.QuantizedBlocks(torch.round(blocks / scales[:, None]).to(torch.int8), scales, (case["size"],),
                                  case["size"], case["block_size"], "blockwise_symmetric_int8",
                                  rf.SYMMETRIC_INT8_CODEBOOK_ID, -127, 127, 0)
    signed = case["quantizer"] == "dynamic_signed"
    codes, scales = _to_codes(x, case["block_size"], signed)
    ids = rf.DYNAMIC_SIGNED_CODEBOOK_ID if signed else rf.DYNAMIC_UNSIGNED_CODEBOOK_ID
    return rf.QuantizedBlocks(codes.view(-1, case["block_size"]), scales, (case["size"],), case["size"],
                              case["block_size"], "blockwise_%s_8bit" % case["quantizer"], ids, 0, 255,
                              127 if signed else 0)


def work(case):
    """Bytes: each input read and each output written once, params and state
    in place.  Operations: about 30 per parameter for an Adam step with
    requantization, 3 per element for a conversion."""
    width = 4 if case["dtype"] == "f32" else 2
    if case["kind"] in ("quantize", "dequantize"):
        n = case["size"]
        return {"bytes": n * width + n + 4 * _blocks(case, n), "flops": 3 * n}
    sizes = [math.prod(s) for _, s in _shapes(case)]
    n = sum(sizes)
    grad = 4 if case.get("grads", case["dtype"]) == "f32" else 2
    total = n * (2 * width + grad)  # params read and written, grads read
    if case["kind"] == "accumulate":
        total += (MICRO_STEPS - 1) * n * grad + 8 * n  # more grads; the accumulator read and written
    moment = 2 if case.get("moments") == "bf16" else 4
    for k in sizes:
        total += 4 * k + 16 * _blocks(case, k) if _quantized(case, k) else 4 * moment * k
    return {"bytes": total, "flops": 30 * n}


def tolerance(case):
    """Codes and conversions are exact.  A 16-bit param may land on the
    neighbouring value where the direction's last f32 bits differ (one unit
    in the last place, on few elements); f32 params differ in their last
    bits.  About four times the difference between the default direction and
    exact=True: bf16 params 1.2e-5 (largest 2^-7 of a value), f32 params
    3.7e-9 (largest 2^-23)."""
    if case["kind"] in ("quantize", "dequantize"):
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 5e-8, "max": 5e-7, "differ": 0.0}
    return {"rel": 5e-5, "max": 8e-3, "differ": 0.0}


# -------------------------------------------------------------- in 64 bits --
def exact(case, seed):
    """run()'s floating outputs for a new state in plain torch float64,
    before any rounding to 16 bits; None in the place of codes."""
    kind = case["kind"]
    if kind == "quantize":
        x = _values(case, seed).double()
        nb = _blocks(case, case["size"])
        scales = torch.nn.functional.pad(x, (0, nb * case["block_size"] - x.numel())).view(nb, -1).abs().amax(1)
        if case["quantizer"] == "symmetric_int8":
            scales = scales / 127.0
        return {"codes": None, "scales": torch.where(scales > 0, scales, torch.ones_like(scales))}
    if kind == "dequantize":
        q = _quantized_blocks(case, _values(case, seed))
        if case["quantizer"] == "symmetric_int8":
            v = q.values.double()
        else:
            v = _codebook(case["quantizer"] == "dynamic_signed").double()[q.values.long()]
        return {"x": (v * q.scales.double()[:, None]).view(-1)[: case["size"]]}

    t = _Tree(case, seed, MICRO_STEPS if kind == "accumulate" else 1)
    grads = {k: sum(g[k].double() for g in t.grads) / len(t.grads) for k in t.shapes} if len(t.grads) > 1 else None
    grad = (lambda k: grads[k]) if grads else (lambda k: t.grads[0][k].double())
    factor = 1.0
    if kind == "finetune" or case.get("clip"):
        norm = math.sqrt(sum(float(grad(k).square().sum()) for k in t.shapes))
        factor = min(1.0, CLIP / (norm + 1e-6))
    books = [_codebook(True).double(), _codebook(False).double()]
    out = {}
    wide = {name: torch.zeros_like(a, dtype=torch.float64) if a.is_floating_point() else None
            for name, a in t.outputs().items()}
    c1, c2 = 1.0 - B1 ** (COUNT + 1), 1.0 - B2 ** (COUNT + 1)
    for k, n in t.sizes.items():
        lr, wd = GROUPS[_group(k)] if kind == "finetune" else (LR, DECAY)
        g = grad(k) * factor
        old = []
        for i in range(2):
            if _quantized(case, n):
                block = books[i][t.codes[i][k].long()].view(-1, case["block_size"])
                old.append((block * t.scales[i][k].double()[:, None]).view(-1)[:n])
            else:
                old.append(t.moments[i][k].double())
        new = [B1 * old[0] + (1.0 - B1) * g, B2 * old[1] + (1.0 - B2) * g * g]
        p = t.params[k].double()
        u = new[0] / c1 / (torch.sqrt(new[1] / c2) + EPS) + wd * p
        _place(wide["params"], t.params, k, p - lr * u)
        for i, what in enumerate(("mu", "nu")):
            if _quantized(case, n):
                bs = case["block_size"]
                x = torch.nn.functional.pad(new[i], (0, _blocks(case, n) * bs - n)).view(-1, bs).abs().amax(1)
                _place(wide[what + "_scales"], t.scales[i], k, torch.where(x > 0, x, torch.ones_like(x)))
            else:
                _place(wide[what + "_moments"], t.moments[i], k, new[i])
    out.update(wide)
    if kind == "accumulate":
        out["acc"] = torch.zeros(_Arena(list(t.sizes.items()), torch.float32).flat.numel(), dtype=torch.float64)
    return out


def _place(flat, arena, name, values):
    at, size = arena.at[name]
    flat[at: at + size] = values
