"""Performance cases: what a user of this framework has it do, through its public entry points, over the range of sizes
it is used at.

  products   the four matrix shapes of a decoder layer (query / output, key / value, gate or up, down) as `q_mat_mul` calls:
             1 row (a decode step), 2 - 16 rows (a small batch), hundreds to thousands of rows (a prompt), f32 or bf16
             activations, every block format of GGUF files that the library tiles
  attention  `flash_attention` of a whole prompt, causal
  cached     `flash_attention` of one new token against a filled cache, several layers' caches one after the other
  llama      a Llama-architecture decoder from Q4_K_M weights: a prompt, or a prompt and a greedy or sampled continuation
  hybrid     the same for layer-list decoders (Fidasun, Zovovik) with bf16 weights

Weights of models are made once per process and kept, as a program keeps its model; prompts, activations, matrices and
caches come from the seed.  `exact` restates every path in 64 bits with plain torch operations."""
from __future__ import annotations

import math

import numpy as np
import torch

from kalosm_amd import bench_hybrid, synth
from kalosm_amd.fusor import Device, GpuMirostat2SamplerParams, MaskKind, QMatrix, Tensor
from kalosm_amd.hybrid import HybridModel
from kalosm_amd.llama import Model

BLOCKS = {"Q4_0": (2, 32, 18), "Q5_0": (6, 32, 22), "Q8_0": (8, 32, 34), "Q4_K": (12, 256, 144), "Q5_K": (13, 256, 176),
          "Q6_K": (14, 256, 210)}  # type, weights and bytes of a block
TYPE_NAME = {t: n for n, (t, _, _) in BLOCKS.items()}
GPU = "cuda"


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one decode step's matrices, three layers of an 8B model: the smallest calls, bound by launches and latency
        dict(name="products_q4k_1row", kind="products", weights="Q4_K", act="f32", rows=1, width=4096, ffn=14336, layers=3),
        # a small batch of sequences decoded together
        dict(name="products_q4k_16rows", kind="products", weights="Q4_K", act="f32", rows=16, width=4096, ffn=14336, layers=3),
        # a prompt of ordinary length through 6-bit matrices with bf16 activations
        dict(name="products_q6k_bf16_512rows", kind="products", weights="Q6_K", act="bf16", rows=512, width=4096, ffn=14336,
             layers=1),
        # a long prompt through 8-bit matrices
        dict(name="products_q8_0_bf16_2048rows", kind="products", weights="Q8_0", act="bf16", rows=2048, width=4096, ffn=14336,
             layers=1),
        # attention of a prompt, grouped heads, f16
        dict(name="attention_causal_2048", kind="attention", dtype="f16", heads=32, kv_heads=8, dim=128, tokens=2048),
        # one new token against a long conversation
        dict(name="attention_cached_16384", kind="cached", heads=32, kv_heads=8, dim=128, tokens=16384, layers=4),
        # a long document read by the 8B model (time to first token)
        dict(name="llama_8b_prompt_2048", kind="llama", model="8b", kv="f32", prompt=2048, new=0, sampled=False),
        # a chat turn: ordinary prompt, greedy answer
        dict(name="llama_8b_512_and_128", kind="llama", model="8b", kv="f32", prompt=512, new=128, sampled=False),
        # a short odd prompt and a sampled answer of a small model: launches and host work count
        dict(name="llama_small_37_and_64_sampled", kind="llama", model="small", kv="f32", prompt=37, new=64, sampled=True),
        # mixture-of-experts decoder: long prompt, logits of the last 16 places (scoring)
        dict(name="fidasun_w4096_prompt_2048", kind="hybrid", model="fidasun_w4096", prompt=2048, new=0, places=16),
        # the smaller one: a chat turn
        dict(name="fidasun_w2048_512_and_64", kind="hybrid", model="fidasun_w2048", prompt=512, new=64, places=1),
        # recurrent and windowed layers: long prompt and a short answer
        dict(name="zovovik_w4096_2048_and_32", kind="hybrid", model="zovovik_w4096", prompt=2048, new=32, places=1),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["products", "products", "products", "attention", "cached", "llama", "llama", "hybrid", "hybrid"])
    if kind == "products":
        width, ffn = rng.choice([(2048, 5632), (2048, 8192), (3072, 8192), (4096, 11008), (4096, 14336)])
        weights = rng.choice(sorted(BLOCKS))
        band = rng.choice(["one", "batch", "prompt", "prompt"])
        rows = {"one": 1, "batch": rng.randint(2, 16), "prompt": _spread(rng, 17, 2048)}[band]
        return dict(kind=kind, weights=weights, act=rng.choice(["f32", "bf16"]) if band == "prompt" else "f32", rows=rows,
                    width=width, ffn=ffn, layers=rng.randint(2, 4) if rows <= 16 else 1)
    if kind == "attention":
        kv = rng.choice([2, 4, 8])
        return dict(kind=kind, dtype=rng.choice(["f16", "f16", "f32"]), heads=kv * rng.choice([1, 2, 4]), kv_heads=kv,
                    dim=rng.choice([64, 128, 128]), tokens=_spread(rng, 33, 4096))
    if kind == "cached":
        kv = rng.choice([4, 8])
        return dict(kind=kind, heads=kv * rng.choice([1, 4, 8]), kv_heads=kv, dim=128, tokens=_spread(rng, 60, 16384),
                    layers=rng.randint(2, 5))
    if kind == "llama":
        model = rng.choice(["8b", "small", "small"])
        new = rng.choice([0, rng.randint(2, 100)])
        return dict(kind=kind, model=model, kv=rng.choice(["f32", "f32", "f16"]) if model == "small" else "f32",
                    prompt=_spread(rng, 5, 2000 if model == "small" or not new else 500), new=new,
                    sampled=bool(new) and rng.random() < 0.5)
    new = rng.choice([0, rng.randint(2, 64)])
    return dict(kind="hybrid", model=rng.choice(["fidasun_w2048", "fidasun_w4096", "zovovik_w2048", "zovovik_w4096"]),
                prompt=_spread(rng, 17, 2048), new=new, places=1 if new else rng.randint(4, 16))


# ---------------------------------------------------------------- inputs
_held = {}


def _once(key, make):
    if key not in _held:
        _held[key] = make()
    return _held[key]


def _device():
    return _once("device", lambda: Device.gpu(0))


def _generator(seed, *what):
    h = 1469598103934665603
    for ch in repr((int(seed),) + what).encode():
        h = (h ^ ch) * 1099511628211 % (1 << 62)
    return torch.Generator(device=GPU).manual_seed(h)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=GPU)


class _Memory:
    """What torch needs to see a tensor of the library as its own; holds the tensor as long as torch holds this."""

    def __init__(self, t, typestr):
        self.owner = t
        self.__cuda_array_interface__ = dict(shape=t.shape, typestr=typestr, data=(t.ptr, False), version=2)


def _tensor(shape, dtype, values=None):
    """A tensor of the library and, over the same memory, a torch view of it that keeps it alive."""
    t = Tensor(_device(), shape, dtype)
    view = torch.as_tensor(_Memory(t, {"f32": "<f4", "f16": "<f2", "bf16": "<i2"}[dtype]), device=GPU)
    if dtype == "bf16":
        view = view.view(torch.bfloat16)
    view.owner = t
    if values is not None:
        view.copy_(values)
    return t, view


def _blocks(weights, n, k, sigma, g):
    """Random blocks of a GGUF matrix [n, k] on the GPU: uniform codes and sub-scales, normal super-scales."""
    _, elems, size = BLOCKS[weights]
    b = torch.randint(0, 256, (n * k // elems, size), generator=g, device=GPU, dtype=torch.uint8)

    def scale():
        return (sigma * _normal(g, b.shape[0], 1)).half().view(torch.uint8)

    if weights == "Q6_K":
        b[:, 208:210] = scale()
    else:
        b[:, 0:2] = scale()
        if weights in ("Q4_K", "Q5_K"):
            b[:, 2:4] = scale()
        if weights == "Q8_0":
            codes = b[:, 2:]
            codes[codes == 128] = 0  # -128 is not a code that quantization writes
    return b


def _values(weights, b):
    """The weights that blocks stand for, in 64 bits, one row of values per block."""
    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    def i(x):
        return x.to(torch.int16)

    if weights == "Q8_0":
        return half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    if weights in ("Q4_0", "Q5_0"):
        qs = i(b[:, -16:])
        codes = torch.cat([qs & 15, qs >> 4], 1)
        if weights == "Q5_0":
            bit = torch.arange(32, device=GPU)
            high = (i(b[:, 2:6])[:, bit // 8] >> (bit % 8).to(torch.int16)) & 1
            return half(0) * (codes + 16 * high - 16).double()
        return half(0) * (codes - 8).double()
    if weights == "Q6_K":
        lo, hi, sc = i(b[:, :128]).view(-1, 2, 64), i(b[:, 128:192]).view(-1, 2, 1, 32), b[:, 192:208].contiguous().view(torch.int8)
        lo = torch.cat([lo & 15, lo >> 4], 2).view(-1, 2, 4, 32)
        shift = torch.tensor([0, 2, 4, 6], device=GPU, dtype=torch.int16).view(1, 1, 4, 1)
        codes = (lo | (((hi >> shift) & 3) << 4)).reshape(-1, 16, 16) - 32
        return half(208) * (sc.double().unsqueeze(2) * codes.double()).reshape(-1, 256)
    p = i(b[:, 4:16])
    sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
    qs = i(b[:, -128:]).view(-1, 4, 1, 32)
    codes = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
    if weights == "Q5_K":
        bit = torch.arange(8, device=GPU, dtype=torch.int16).view(1, 8, 1)
        codes = codes + 16 * ((i(b[:, 16:48]).unsqueeze(1) >> bit) & 1)
    w = (half(0) * sc).unsqueeze(2) * codes.double() - (half(2) * mn).unsqueeze(2)
    return w.reshape(-1, 256)


def _shapes(case):
    d, f = case["width"], case["ffn"]
    return [(d, d), (d // 4, d), (f, d), (d, f)]


def _rows(case, seed):
    """Activations of each matrix shape's input width."""
    out = {}
    for k in (case["width"], case["ffn"]):
        x = _normal(_generator(seed, "rows", k), case["rows"], k)
        out[k] = x.bfloat16() if case["act"] == "bf16" else x
    return out


def _matrix(case, seed, layer, n, k):
    return _blocks(case["weights"], n, k, 0.002, _generator(seed, "matrix", layer, n, k))


def _prepare_products(case, seed):
    x = {k: _tensor(v.shape, case["act"], v)[0] for k, v in _rows(case, seed).items()}
    todo = []
    for layer in range(case["layers"]):
        for n, k in _shapes(case):
            raw = _matrix(case, seed, layer, n, k).cpu().numpy()
            w = QMatrix.from_raw_bytes(_device(), (n, k), raw, BLOCKS[case["weights"]][0])
            todo.append((x[k], w, *_tensor((case["rows"], n), "f32")))
    return dict(kind="products", todo=todo)


def _heads(case, seed, layer=0):
    h, g, d, t = case["heads"], case["kv_heads"], case["dim"], case["tokens"]
    gen, dt = _generator(seed, "heads", layer), torch.float32 if case.get("dtype") == "f32" else torch.float16
    q = _normal(gen, 1, h, t if case["kind"] == "attention" else 1, d).to(dt)
    return q, _normal(gen, 1, g, t, d).to(dt), _normal(gen, 1, g, t, d).to(dt)


def _prepare_attention(case, seed):
    todo = []
    for layer in range(case.get("layers", 1)):
        q, k, v = _heads(case, seed, layer)
        dt = "f32" if q.dtype == torch.float32 else "f16"
        todo.append((*[_tensor(x.shape, dt, x)[0] for x in (q, k, v)], *_tensor(q.shape, dt)))
    return dict(kind=case["kind"], todo=todo, scale=case["dim"] ** -0.5, mask=MaskKind.Causal if case["kind"] == "attention" else None)


# models ---------------------------------------------------------
def _llama_config(model):
    if model == "8b":
        return dict(synth.LLAMA3_8B)
    s = bench_hybrid.SIZES["w2048"]  # the Llama decoder that the layer-list ones are measured beside
    return bench_hybrid.llama_config(bench_hybrid.config(**s), s["heads"], s["top"], s["ff"])


def _llama_tensors(model):
    for name, ty, n, k in synth.llama_tensor_specs(_llama_config(model)):
        g = _generator(7, model, name)
        yield name, ty, n, k, 1.0 + 0.1 * _normal(g, n) if ty == 0 else _blocks(TYPE_NAME[ty], n, k, 1e-4, g)


def _llama(model, kv):
    m = Model(_device(), _llama_config(model), kv_dtype=kv)
    for name, ty, n, k, data in _llama_tensors(model):
        m.load_tensor(name, ty, n, k, data.cpu().numpy())
    m.finalize()
    return m


def _hybrid_config(model):
    family, size = model.split("_")
    if family == "fidasun":
        return bench_hybrid.config(**bench_hybrid.SIZES[size])
    return bench_hybrid.zovovik_config(**bench_hybrid.ZOVOVIK[size])


def _hybrid_tensors(model):
    """Rows of matrices with a norm near one, decays and step sizes spread over useful ranges.  The head answers a token
    with another fixed one beside noise: a model predicts with a margin, which a random head does not."""
    cfg = _hybrid_config(model)
    plus = cfg["architecture"] == "Fidasun"
    embed = None
    for name, n, k in synth.hybrid_tensor_specs(cfg):
        g, last = _generator(7, model, name), name.rsplit(".", 1)[-1]
        shape = (n, k) if k else (n,)
        uniform = lambda lo, hi: lo + (hi - lo) * torch.rand(*shape, generator=g, device=GPU)  # noqa: E731
        if last == "A_log":
            x = uniform(-3.0, 1.0)
        elif last == "dt_bias":
            x = uniform(-3.0, 0.5)
        elif last in ("norm1", "norm2") or name == "final.norm":
            x = (0.0 if plus else 1.0) + 0.2 * _normal(g, n)
        elif last == "w0":
            x = uniform(-6.0, 1.0)
        elif last == "u":
            x = 0.7 * _normal(g, n, k)
        elif ".mu." in name:
            x = uniform(0.0, 1.0)
        elif name == "pos":
            x = 0.3 * _normal(g, n, k)
        elif last in ("norm", "D"):
            x = 1.0 + 0.2 * _normal(g, n)
        elif last in ("sink", "b") and k == 0:
            x = 0.5 * _normal(g, n)
        elif name == "embed":
            x = embed = _normal(g, n, k).bfloat16()
        elif name == "head":
            x = (embed[(torch.arange(n, device=GPU) * 5 + 1) % n].float() + 0.5 * _normal(g, n, k)) / math.sqrt(k)
        else:
            x = _normal(g, n, k) / math.sqrt(k) * (2.0 if last == "router" else 1.0)
        yield name, n, k, x.bfloat16()


def _hybrid(model):
    m = HybridModel(_device(), _hybrid_config(model), ctx=8192)
    m.load_all((name, n, k, x.view(torch.int16).cpu().numpy().view(np.uint16)) for name, n, k, x in _hybrid_tensors(model))
    return m


def _vocab(case):
    return (_llama_config(case["model"]) if case["kind"] == "llama" else _hybrid_config(case["model"]))["vocab"]


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, _vocab(case), case["prompt"]).astype(np.uint32)


def _sampler():
    """The reference's default generation parameters over the 64 best candidates."""
    return GpuMirostat2SamplerParams(64, 0.8, 1.3, 5.0, 0.1, 0.0)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "products":
        return _prepare_products(case, seed)
    if kind in ("attention", "cached"):
        return _prepare_attention(case, seed)
    if kind == "llama":
        m = _once(("llama", case["model"], case["kv"]), lambda: _llama(case["model"], case["kv"]))
    else:
        m = _once(("hybrid", case["model"]), lambda: _hybrid(case["model"]))
    return dict(kind="model", model=m, prompt=_prompt(case, seed), new=case["new"], sampled=case.get("sampled", False),
                places=case.get("places", 1), seed=seed)


# ---------------------------------------------------------------- one pass
def run(state):
    if state["kind"] == "products":
        for x, w, y, _ in state["todo"]:
            x.q_mat_mul(w, out=y)
        return [view for _, _, _, view in state["todo"]]
    if state["kind"] in ("attention", "cached"):
        for q, k, v, out, _ in state["todo"]:
            q.flash_attention(k, v, state["scale"], state["mask"], out=out)
        return [view for *_, view in state["todo"]]
    m, prompt, new = state["model"], state["prompt"], state["new"]
    m.reset()
    if not new:
        n = len(prompt)
        return m.forward(prompt, want=range(max(0, n - state["places"]), n))
    if state["sampled"]:
        tokens = m.generate(prompt, new, _sampler(), seed=state["seed"])
        return dict(tokens=tokens.astype(np.int64), after=m.forward(tokens[-1:]))
    first = m.forward(prompt)
    tokens, _ = m.decode_greedy(int(np.argmax(first)), new)
    return dict(prompt=first, tokens=tokens.astype(np.int64), after=m.forward(tokens[-1:]))


# ---------------------------------------------------------------- work and tolerance
def _llama_work(case):
    c = _llama_config(case["model"])
    nbytes = flops = head = 0.0
    for name, ty, n, k in synth.llama_tensor_specs(c):
        if ty and not name.startswith("token_embd"):
            _, elems, size = BLOCKS[TYPE_NAME[ty]]
            b, f = n * k / elems * size, 2.0 * n * k
            if name.startswith("output"):
                head = f
            else:
                flops += f
            nbytes += b
    t, new = case["prompt"], case["new"] + (1 if case["new"] else 0)
    row = c["n_layers"] * 2 * c["n_kv_heads"] * c["head_dim"] * (2 if case["kv"] == "f16" else 4)
    pair = c["n_layers"] * 4.0 * c["n_heads"] * c["head_dim"]
    steps = sum(t + i for i in range(new))
    return dict(bytes=nbytes * (1 + new) + row * (t + new + steps) + 4.0 * c["vocab"] * (2 if new else 1),
                flops=flops * (t + new) + head * (1 + new) + pair * (t * (t + 1) / 2 + steps))


def _hybrid_work(case):
    c = _hybrid_config(case["model"])
    t, new, places = case["prompt"], case["new"] + (1 if case["new"] else 0), case["places"]
    once = step = flops = head = 0.0
    for name, n, k in synth.hybrid_tensor_specs(c):
        if name in ("embed", "pos"):
            continue
        size, part, share = 2.0 * n * max(k, 1), name.split("."), 1.0
        if name == "head":
            head = 2.0 * n * k
        elif len(part) > 2 and part[1] == "mlp" and part[2][0] == "e" and part[2][1:].isdigit():
            r = c["layers"][int(part[0][1:])]["mlp"]["router"]
            share = r["top"] / r["experts"]
        if name != "head" and k:
            flops += 2.0 * n * k * share
        once += size * min(1.0, share * t)
        step += size * share
    pairs = 0.0  # multiply-adds of attention, per query and visible key; states of the recurrences in f32
    state = cache = 0.0
    for layer in c["layers"]:
        a = layer["mixer"]
        if layer["type"] == "latent_attention":
            w = a["mask"]["size"]
            pairs += 2.0 * a["heads"] * (a["dim"] + a["rot_dim"] + a["vdim"]) * sum(min(i + 1, w) for i in range(t + new))
            cache += 2.0 * (a["kv_rank"] + a["rot_dim"]) * min(t, w)
        elif layer["type"] == "parallel":
            w, l = a["left"]["mask"]["size"] + a["left"]["mask"]["keep_first"], a["left"]
            pairs += 4.0 * l["heads"] * l["dim"] * sum(min(i + 1, w) for i in range(t + new))
            cache += 4.0 * l["kv_heads"] * l["dim"] * min(t, w)
            state += 4.0 * a["right"]["heads"] * a["right"]["dim"] ** 2
        elif layer["type"] == "retention":
            state += 4.0 * a["heads"] * a["dim"] * a["vdim"]
        elif layer["type"] == "delta":
            state += 4.0 * a["heads"] * a["dim"] * a["vdim"]
        else:
            state += 4.0 * a["heads"] * a["state"] * a["vdim"]
    flops = flops * (t + new) + head * (places + new) + pairs + 2.0 * state * (t + new)
    return dict(bytes=once + (step + cache + 2.0 * state) * new + 4.0 * c["vocab"] * (places + (1 if new else 0)), flops=flops)


def work(case):
    kind = case["kind"]
    if kind == "products":
        _, elems, size = BLOCKS[case["weights"]]
        esz = 2 if case["act"] == "bf16" else 4
        m, layers, shapes = case["rows"], case["layers"], _shapes(case)
        return dict(bytes=layers * sum(n * k / elems * size + 4.0 * m * n for n, k in shapes) + esz * m * (case["width"] + case["ffn"]),
                    flops=layers * sum(2.0 * m * n * k for n, k in shapes))
    if kind in ("attention", "cached"):
        h, g, d, t = case["heads"], case["kv_heads"], case["dim"], case["tokens"]
        esz, q = 4 if case.get("dtype") == "f32" else 2, t if kind == "attention" else 1
        pairs = t * (t + 1) / 2 if kind == "attention" else t
        layers = case.get("layers", 1)
        return dict(bytes=layers * esz * 2.0 * (h * q * d + g * t * d), flops=layers * 4.0 * h * d * pairs)
    return _llama_work(case) if kind == "llama" else _hybrid_work(case)


def tolerance(case):
    """About four times the largest error against 64 bits seen over the ranges."""
    kind = case["kind"]
    if kind == "products":  # 32-bit sums: 8e-7
        return {"rel": 4e-6}
    if kind in ("attention", "cached"):  # f16 weights and outputs: 2.6e-4
        return {"rel": 5e-6 if case.get("dtype") == "f32" else 1e-3}
    if kind == "llama":  # 32-bit sums through 32 layers: 8e-4; through four: 2e-5; an f16 cache rounds on its own
        return {"rel": 4e-3 if case["kv"] == "f16" or case["model"] == "8b" else 1e-4}
    return {"rel": 2.7e-2}  # bf16 operands: 6.7e-3


# ---------------------------------------------------------------- the same in 64 bits
def _attend(q, k, v, scale, visible, sink=None):
    """q [h, t, d], k, v [h, s, d], visible [t, s]: softmax attention; exp(sink) [h] joins the denominators."""
    out = torch.empty(*q.shape[:2], v.shape[2], dtype=q.dtype, device=GPU)
    for at in range(0, q.shape[1], 1024):  # blocks of queries, so that the scores fit
        z = (q[:, at:at + 1024] @ k.transpose(1, 2)) * scale
        if visible is not None:
            z = z.masked_fill(~visible[at:at + 1024], -math.inf)
        top = z.amax(2, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink.view(-1, 1, 1))
        e = torch.exp(z - top)
        total = e.sum(2, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink.view(-1, 1, 1) - top)
        out[:, at:at + 1024] = (e / total) @ v
    return out


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _angles(start, count, freq):
    """Angles as the tables hold them: 32-bit products of the position and the 32-bit frequency."""
    p = torch.arange(start, start + count, device=GPU, dtype=torch.float32)
    return (p[:, None] * freq.float()[None]).double()


def _rotate(x, angle, amp=1.0):
    """x [.., t, d]: neighbouring pairs of the first 2 * angle.shape[1] dimensions."""
    n = 2 * angle.shape[1]
    c, s = torch.cos(angle) * amp, torch.sin(angle) * amp
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    out = x.clone()
    out[..., 0:n:2], out[..., 1:n:2] = u * c - v * s, v * c + u * s
    return out


def _rotate_halves(x, angle):
    n = angle.shape[1]
    c, s = torch.cos(angle), torch.sin(angle)
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], -1)


class _Llama64:
    def __init__(self, model, kv):
        self.c, self.kv, self.w = _llama_config(model), kv, {}
        for name, ty, n, k, data in _llama_tensors(model):
            self.w[name] = data.double() if ty == 0 else _values(TYPE_NAME[ty], data).reshape(n, k)
        half, theta = self.c["head_dim"] // 2, np.float32(self.c["theta"])
        freq = [np.float32(1.0) / np.power(theta, np.float32(2 * i) / np.float32(2 * half), dtype=np.float32) for i in range(half)]
        self.freq = torch.tensor(np.array(freq, np.float32), device=GPU)
        self.cache = [(None, None)] * self.c["n_layers"]
        self.at = 0

    def forward(self, tokens, places=1):
        c, w, t, at = self.c, self.w, len(tokens), self.at
        h, g, d, eps = c["n_heads"], c["n_kv_heads"], c["head_dim"], float(np.float32(c["eps"]))
        x = w["token_embd.weight"][torch.as_tensor(np.asarray(tokens, np.int64), device=GPU)]
        angle = _angles(at, t, self.freq)
        visible = None if t == 1 else torch.ones(t, at + t, dtype=torch.bool, device=GPU).tril(at)
        for i in range(c["n_layers"]):
            l = lambda name: w["blk.%d.%s.weight" % (i, name)]  # noqa: E731,B023
            n = _rms(x, eps) * l("attn_norm")
            q, k, v = ((n @ l("attn_" + s).T).view(t, -1, d).transpose(0, 1) for s in "qkv")
            q, k = _rotate(q, angle), _rotate(k, angle)
            if self.kv == "f16":
                k, v = k.half().double(), v.half().double()
            if at:
                k, v = torch.cat([self.cache[i][0], k], 1), torch.cat([self.cache[i][1], v], 1)
            self.cache[i] = (k, v)
            if t == 1:  # the heads of a group as rows of one product
                o = _attend(q.reshape(g, h // g, d), k, v, d ** -0.5, None).reshape(1, -1)
            else:
                o = _attend(q, k.repeat_interleave(h // g, 0), v.repeat_interleave(h // g, 0), d ** -0.5, visible)
                o = o.transpose(0, 1).reshape(t, -1)
            x = x + o @ l("attn_output").T
            n = _rms(x, eps) * l("ffn_norm")
            x = x + (_silu(n @ l("ffn_gate").T) * (n @ l("ffn_up").T)) @ l("ffn_down").T
        self.at += t
        return (_rms(x[-places:], eps) * w["output_norm.weight"]) @ w["output.weight"].T


class _Hybrid64:
    def __init__(self, model):
        self.c = _hybrid_config(model)
        self.w = {name: x.double() for name, _, _, x in _hybrid_tensors(model)}
        self.eps, self.at, self.kept = self.c["norm"]["eps"], 0, {}

    def behind(self, key, x, keep):
        """x with the last `keep` rows of what came before it (zeros ahead of the first token) in front."""
        old = self.kept.get(key)
        if old is None:
            old = torch.zeros(keep, *x.shape[1:], dtype=x.dtype, device=GPU)
        whole = torch.cat([old, x])
        self.kept[key] = whole[len(whole) - keep:]
        return whole

    def cached(self, key, k, v):
        if key in self.kept:
            k, v = torch.cat([self.kept[key][0], k], 1), torch.cat([self.kept[key][1], v], 1)
        self.kept[key] = (k, v)
        return k, v

    def state(self, key, *shape):
        if key not in self.kept:
            self.kept[key] = torch.zeros(*shape, dtype=torch.float64, device=GPU)
        return self.kept[key]

    def visible(self, t, size, first=0):
        i, j = torch.arange(self.at, self.at + t, device=GPU)[:, None], torch.arange(self.at + t, device=GPU)[None]
        return (j <= i) & ((i - j < size) | (j < first))

    def conv(self, key, x, taps, bias=None):
        n = taps.shape[1]
        whole = self.behind(key, x, n - 1)
        out = sum(whole[i:i + len(x)] * taps[:, i] for i in range(n))
        return _silu(out if bias is None else out + bias)

    @staticmethod
    def frequencies(rot):
        n, base, s = rot["dims"], float(rot["base"]), rot.get("scaling")
        i = np.arange(n // 2)
        f = base ** (-2.0 * i / n)
        if not s:
            return torch.tensor(f.astype(np.float32), device=GPU), 1.0
        at = [n * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base)) for turns in (s["fast"], s["slow"])]
        lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), n - 1)
        ramp = np.clip((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        return torch.tensor((f / s["factor"] * ramp + f * (1.0 - ramp)).astype(np.float32), device=GPU), 0.1 * math.log(s["factor"]) + 1.0

    def latent_attention(self, p, x, a):
        w, t, h, dn, r = self.w, len(x), a["heads"], a["dim"], a["kv_rank"]
        freq, amp = self.frequencies(a["rot"])
        angle = _angles(self.at, t, freq)
        q = (x @ w[p + "q"].T).view(t, h, -1).transpose(0, 1)
        c = x @ w[p + "dkv"].T
        lat, kr = _rms(c[:, :r], self.eps) * w[p + "dkv.norm"], _rotate(c[:, r:], angle, amp)
        k = torch.cat([(lat @ w[p + "uk"].T).view(t, h, dn).transpose(0, 1), kr.expand(h, -1, -1)], 2)
        v = (lat @ w[p + "uv"].T).view(t, h, -1).transpose(0, 1)
        q = torch.cat([q[..., :dn], _rotate(q[..., dn:], angle, amp)], 2)
        k, v = self.cached(p, k, v)
        o = _attend(q, k, v, a["scale"], self.visible(t, a["mask"]["size"]), w[p + "sink"])
        return o.transpose(0, 1).reshape(t, -1) @ w[p + "o"].T

    def delta(self, p, x, a):
        w, t, h, g, d = self.w, len(x), a["heads"], a["kv_heads"], a["dim"]
        q, k, v = (self.conv(p + n, x @ w[p + n].T, w[p + n + ".conv"]).view(t, -1, d if n != "v" else a["vdim"]) for n in "qkv")
        q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        q, k = (q * d ** -0.5).repeat_interleave(h // g, 1), k.repeat_interleave(h // g, 1)
        beta = torch.sigmoid(x @ w[p + "b"].T)
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * torch.nn.functional.softplus(x @ w[p + "a"].T + w[p + "dt_bias"]))
        s, o = self.state(p, h, d, a["vdim"]), torch.empty_like(v)
        for i in range(t):
            s = s * decay[i].view(h, 1, 1)
            u = (v[i] - (k[i].unsqueeze(1) @ s).squeeze(1)) * beta[i].unsqueeze(1)
            s = s + k[i].unsqueeze(2) * u.unsqueeze(1)
            o[i] = (q[i].unsqueeze(1) @ s).squeeze(1)
        self.kept[p] = s
        o = _rms(o, self.eps) * w[p + "norm"] * _silu(x @ w[p + "g"].T).view(t, h, -1)
        return o.reshape(t, -1) @ w[p + "o"].T

    def mamba2(self, p, x, a):
        w, t, h, dv, n, g = self.w, len(x), a["heads"], a["vdim"], a["state"], a["groups"]
        inner = h * dv
        z, xbc, dt = (x @ w[p + "in"].T).split([inner, inner + 2 * g * n, h], 1)
        xbc = self.conv(p + "in", xbc, w[p + "conv"], w[p + "conv.b"])
        v = xbc[:, :inner].view(t, h, dv)
        b, c = (xbc[:, inner + i * g * n:inner + (i + 1) * g * n].reshape(t, g, n).repeat_interleave(h // g, 1) for i in (0, 1))
        dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"])
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * dt)
        s, o = self.state(p, h, n, dv), torch.empty_like(v)
        for i in range(t):
            s = s * decay[i].view(h, 1, 1) + (b[i] * dt[i].unsqueeze(1)).unsqueeze(2) * v[i].unsqueeze(1)
            o[i] = (c[i].unsqueeze(1) @ s).squeeze(1)
        self.kept[p] = s
        o = (o + w[p + "D"].unsqueeze(1) * v).reshape(t, inner) * _silu(z)
        return (_rms(o.view(t, a["norm_groups"], -1), self.eps).reshape(t, inner) * w[p + "norm"]) @ w[p + "o"].T

    def retention(self, p, x, a):
        w, t, h, d = self.w, len(x), a["heads"], a["dim"]
        angle = _angles(self.at, t, self.frequencies(a["rot"])[0])
        q, k, v = ((x @ w[p + n].T).view(t, h, -1) for n in "qkv")
        q, k = (_rotate_halves(z.transpose(0, 1), angle).transpose(0, 1) for z in (q, k))
        k = k * d ** -0.5
        decay = torch.tensor(a["decay"], dtype=torch.float64, device=GPU).view(h, 1, 1)
        s, o = self.state(p, h, d, a["vdim"]), torch.empty_like(v)
        for i in range(t):
            s = s * decay + k[i].unsqueeze(2) * v[i].unsqueeze(1)
            o[i] = (q[i].unsqueeze(1) @ s).squeeze(1)
        self.kept[p] = s
        return (_rms(o, self.eps).reshape(t, -1) * _silu(x @ w[p + "g"].T)) @ w[p + "o"].T

    def grouped_attention(self, p, x, a):
        w, t, h, g, d = self.w, len(x), a["heads"], a["kv_heads"], a["dim"]
        angle = _angles(self.at, t, self.frequencies(a["rot"])[0])
        q, k, v = ((x @ w[p + n].T).view(t, -1, d).transpose(0, 1) for n in "qkv")
        q, k = _rotate(_rms(q, self.eps) * w[p + "q.norm"], angle), _rotate(_rms(k, self.eps) * w[p + "k.norm"], angle)
        k, v = self.cached(p, k, v)
        o = _attend(q, k.repeat_interleave(h // g, 0), v.repeat_interleave(h // g, 0), a["scale"],
                    self.visible(t, a["mask"]["size"], a["mask"]["keep_first"]), w[p + "sink"])
        return o.transpose(0, 1).reshape(t, -1) @ w[p + "o"].T

    def time_mixing(self, p, x, a):
        w, t, h, d = self.w, len(x), a["heads"], a["dim"]
        before = self.behind(p + "x", x, 1)[:-1]
        mixed = {n: x + (before - x) * w[p + "mu." + n] for n in "rkvgw"}
        r, k, v = ((mixed[n] @ w[p + n].T).view(t, h, d) for n in "rkv")
        z = torch.tanh(mixed["w"] @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"]
        decay, bonus = torch.exp(-torch.exp(z)).view(t, h, d, 1), w[p + "u"].unsqueeze(2)
        s, o = self.state(p, h, d, d), torch.empty_like(v)
        for i in range(t):
            kv = k[i].unsqueeze(2) * v[i].unsqueeze(1)
            o[i] = (r[i].unsqueeze(1) @ (s + bonus * kv)).squeeze(1)
            s = decay[i] * s + kv
        self.kept[p] = s
        return (_rms(o, self.eps).reshape(t, -1) * w[p + "norm"] * _silu(mixed["g"] @ w[p + "g"].T)) @ w[p + "o"].T

    def parallel(self, p, x, a):
        return (a["left_scale"] * self.grouped_attention(p + "left.", x, a["left"])
                + a["right_scale"] * self.time_mixing(p + "right.", x, a["right"]))

    def experts(self, p, x, c):
        w, r = self.w, c["router"]
        one = lambda n, y: (_silu(y @ w[p + n + ".gate"].T) * (y @ w[p + n + ".up"].T)) @ w[p + n + ".down"].T  # noqa: E731
        score, idx = torch.softmax(x @ w[p + "router"].T, 1).topk(r["top"], 1)
        out = one("shared", x)
        for e in sorted(set(idx.flatten().tolist())):
            rows, place = (idx == e).nonzero(as_tuple=True)
            out[rows] += one("e%d" % e, x[rows]) * (score[rows, place] * r["scale"]).unsqueeze(1)
        return out

    def forward(self, tokens, places=1):
        w, eps, t = self.w, self.eps, len(tokens)
        x = w["embed"][torch.as_tensor(np.asarray(tokens, np.int64), device=GPU)]
        after = self.c["architecture"] == "Zovovik"
        if after:
            x = x + w["pos"][self.at:self.at + t]
        for i, l in enumerate(self.c["layers"]):
            p, mixer = "l%d." % i, getattr(self, l["type"])
            if after:
                x = x + _rms(mixer(p + "mix.", x, l["mixer"]), eps) * w[p + "norm1"]
                up = (x @ w[p + "mlp.up"].T).clamp(min=0.0)
                x = x + _rms((up * up) @ w[p + "mlp.down"].T, eps) * w[p + "norm2"]
            else:
                h = _rms(x, eps) * (1.0 + w[p + "norm1"])
                x = x + mixer(p + "mix.", h, l["mixer"]) + self.experts(p + "mlp.", h, l["mlp"])
        self.at += t
        return (_rms(x[-places:], eps) * (w["final.norm"] + (0.0 if after else 1.0))) @ w["head"].T


def _picked(logits, previous, params, random, mu):
    """Mirostat 2 over the processed best candidates: the id and the new state."""
    v = logits.clone()
    seen = torch.as_tensor(sorted(set(int(i) for i in previous)), device=GPU, dtype=torch.int64)
    v[seen] = torch.where(v[seen] <= 0, v[seen] * params.repetition_penalty, v[seen] / params.repetition_penalty)
    top, ids = (v / params.temperature).topk(params.top_k)
    weight = torch.exp(top - top[0]).cpu().numpy()
    ids = ids.cpu().numpy()
    surprise = -np.log2(weight / weight.sum())
    over = np.nonzero(surprise > mu)[0]
    cut = max(int(over[0]), 1) if len(over) else len(ids)
    total = weight[:cut].sum()
    at = min(int(np.searchsorted(np.cumsum(weight[:cut]), float(np.float32(random)) * total)), cut - 1)
    return int(ids[at]), mu - params.eta * (-math.log2(weight[at] / total) - params.tau)


def exact(case, seed):
    with torch.no_grad():
        return _exact(case, seed)


def _exact(case, seed):
    kind = case["kind"]
    if kind == "products":
        x = {k: v.double() for k, v in _rows(case, seed).items()}
        return [x[k] @ _values(case["weights"], _matrix(case, seed, layer, n, k)).reshape(n, k).T
                for layer in range(case["layers"]) for n, k in _shapes(case)]
    if kind in ("attention", "cached"):
        out = []
        for layer in range(case.get("layers", 1)):
            q, k, v = (x[0].double() for x in _heads(case, seed, layer))
            n, t = case["heads"] // case["kv_heads"], case["tokens"]
            visible = torch.ones(t, t, dtype=torch.bool, device=GPU).tril() if kind == "attention" else None
            per = max(1, min(case["kv_heads"], 2 ** 27 // (n * min(t, 1024) * t)))  # heads at a time, so that the scores fit
            out.append(torch.cat([_attend(q[i * n:(i + per) * n], k[i:i + per].repeat_interleave(n, 0), v[i:i + per].repeat_interleave(n, 0),
                                          case["dim"] ** -0.5, visible) for i in range(0, case["kv_heads"], per)]).unsqueeze(0))
        return out
    m = _Llama64(case["model"], case["kv"]) if kind == "llama" else _Hybrid64(case["model"])
    prompt, new = _prompt(case, seed), case["new"]
    if not new:
        return m.forward(prompt, min(case.get("places", 1), len(prompt)))
    first = m.forward(prompt)[0]
    if case.get("sampled"):
        params, mu, window = _sampler(), 10.0, 64
        random = np.random.default_rng(seed).random(new).astype(np.float32)
        token, mu = _picked(first, prompt[-window:], params, random[0], mu)
        tokens, history = [token], list(prompt) + [token]
        for i in range(1, new):
            token, mu = _picked(m.forward(tokens[-1:])[0], history[-window:], params, random[i], mu)
            tokens.append(token)
            history.append(token)
        return dict(tokens=None, after=m.forward(tokens[-1:])[0])
    token = int(first.argmax())
    for _ in range(new):  # whole numbers have no 64-bit value of their own: only the logits are stated
        token = int(m.forward([token])[0].argmax())
    return dict(prompt=first, tokens=None, after=m.forward([token])[0])
