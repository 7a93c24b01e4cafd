"""Performance cases: the work a user of the provider has it do, through its
public entry points (the provider vtables, nf_hip_run_tasks and a HIP graph
captured on nf_hip_get_stream), on device buffers.

Kinds of case:
  linear       one fused dequant + linear dispatch (vtable.dispatch)
  projections  the fused linears of a decode step's layers in one
               nf_hip_run_tasks call, or that call replayed as a HIP graph
  dense        one dense `linear` dispatch (the route of the weight formats
               without a fused op)
  dequant      one dequant_<fmt> dispatch (weights converted at load time)
  attention    one flash_attention_cached dispatch, prefill or decode
  model        a whole llama step, embedding to logits, in one
               nf_hip_run_tasks call (prefill or one decode token)
"""
import ctypes
import math

import torch

from neurofabric_amd import abi, hiprt
from neurofabric_amd import plugin
from neurofabric_amd import synthetic as syn

BLOCK = {"q4_0": 18, "q8_0": 34}
QTYPE = {"q4_0": abi.NF_DTYPE_Q4_0, "q8_0": abi.NF_DTYPE_Q8_0}
ATYPE = {"f32": abi.NF_DTYPE_F32, "f16": abi.NF_DTYPE_F16, "i32": abi.NF_DTYPE_I32, "u8": abi.NF_DTYPE_U8}
TORCH = {"f32": torch.float32, "f16": torch.float16}
SIZE = {"f32": 4, "f16": 2}
EPS, THETA = 1e-5, 10000.0

# The largest product of a listed case (prefill_f16), the bound on drawn ones.
MAX_FLOPS = 2 * 2048 * 11008 * 4096


def listed():
    return [
        # The smallest call: one 2048 x 2048 projection of a 1.1B model for one token, where launch
        # and host latency count.
        {"name": "gemv_small", "kind": "linear", "fmt": "q4_0", "act": "f32", "m": 1, "n": 2048, "k": 2048},
        # bench.py's headline: every projection of a TinyLlama-1.1B token, replayed as a captured graph.
        {"name": "decode_step", "kind": "projections", "fmt": "q4_0", "m": 1, "dim": 2048, "kv_dim": 256,
         "ffn": 5632, "layers": 22, "vocab": 32000, "graph": True},
        # Single-token FFN matrix of a 70B model in fp16 mode: the memory-bound decode.
        {"name": "gemv_large", "kind": "linear", "fmt": "q4_0", "act": "f16", "m": 1, "n": 28672, "k": 8192},
        # A batch of 32 sequences on the long-K down projection of the same model.
        {"name": "batch_f16", "kind": "linear", "fmt": "q4_0", "act": "f16", "m": 32, "n": 8192, "k": 28672},
        # Serving 64 sequences: the seven projections of one Llama-3-8B layer, Q8_0, f32 activations.
        {"name": "serve_q8_b64", "kind": "projections", "fmt": "q8_0", "m": 64, "dim": 4096, "kv_dim": 1024,
         "ffn": 14336, "layers": 1, "vocab": 0, "graph": False},
        # Prompt processing in fp16 mode, Llama-2-7B gate/up projection over 2048 tokens.
        {"name": "prefill_f16", "kind": "linear", "fmt": "q4_0", "act": "f16", "m": 2048, "n": 11008, "k": 4096},
        # A prompt of an odd length on a Q8_0 gate/up projection.
        {"name": "prefill_q8_ragged", "kind": "linear", "fmt": "q8_0", "act": "f16", "m": 389, "n": 14336, "k": 4096},
        # Prompt processing with the engine's default f32 activations, down projection.
        {"name": "prefill_f32", "kind": "linear", "fmt": "q4_0", "act": "f32", "m": 512, "n": 4096, "k": 11008},
        # The same for a K-quant model, whose weights are dense f32 after the load-time dequantization.
        {"name": "dense_f32", "kind": "dense", "act": "f32", "m": 256, "n": 11008, "k": 4096},
        # Load-time dequantization of one FFN matrix of a K-quant model in fp16 mode.
        {"name": "dequant_q4_k", "kind": "dequant", "fmt": "q4_k", "act": "f16", "n": 11008, "k": 4096},
        # Prompt attention of a grouped-query model.
        {"name": "attention_prefill", "kind": "attention", "act": "f16", "heads": 32, "kv": 8, "dim": 128,
         "seq": 2048, "pos": 0, "max_seq": 2048},
        # One token of a whole TinyLlama-shaped model at position 500, embedding to logits.
        {"name": "model_decode", "kind": "model", "fmt": "q4_0", "dim": 2048, "heads": 32, "kv": 4, "ffn": 5632,
         "layers": 22, "vocab": 32000, "seq": 1, "pos": 500, "max_seq": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _k(rng, lo, hi):
    """A row length: mostly whole 256-element superblocks as models have them, some multiples of 64, a few of 32."""
    step = rng.choice([256] * 6 + [64] * 3 + [32])
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choices(["linear", "projections", "dense", "dequant", "attention", "model"], [10, 3, 2, 2, 3, 2])[0]
    if kind in ("linear", "dense"):
        c = {"kind": kind, "act": rng.choice(["f32", "f16"]), "m": _log(rng, 1, 2048), "n": _log(rng, 128, 32000),
             "k": _k(rng, 512, 28672)}
        if kind == "linear":
            c["fmt"] = rng.choice(["q4_0", "q8_0"])
        # f32 products and dense weights cost more per unit of work than the fp16 fused path
        most = MAX_FLOPS if kind == "linear" and c["act"] == "f16" else MAX_FLOPS // 8
        while 2 * c["m"] * c["n"] * c["k"] > most:
            c["m"] = max(1, c["m"] // 2)
        return c
    if kind == "projections":
        dim = 256 * _log(rng, 2, 16)
        return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0"]), "m": _log(rng, 1, 96), "dim": dim,
                "kv_dim": dim // rng.choice([1, 4, 8]), "ffn": 256 * _log(rng, 4, 56), "layers": rng.randint(1, 8),
                "vocab": rng.choice([0, 0, 32000, 50257]), "graph": rng.random() < 0.5}
    if kind == "dequant":
        return {"kind": kind, "fmt": rng.choice(sorted(syn.KQ_GEOM)), "act": rng.choice(["f32", "f16"]),
                "n": _log(rng, 256, 16384), "k": 256 * _log(rng, 4, 56)}
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8])
        c = {"kind": kind, "act": rng.choice(["f32", "f16"]), "heads": kv * rng.choice([1, 2, 4]), "kv": kv,
             "dim": rng.choice([64, 128, 128, 96])}
        if rng.random() < 0.5:
            return dict(c, seq=_log(rng, 8, 2048), pos=0, max_seq=2048)
        return dict(c, seq=1, pos=_log(rng, 16, 8191), max_seq=8192)
    heads = rng.choice([8, 16, 32])
    decode = rng.random() < 0.5
    return {"kind": kind, "fmt": rng.choice(["q4_0", "q8_0"]), "dim": 64 * heads, "heads": heads,
            "kv": heads // rng.choice([1, 2, 4, 8]), "ffn": 256 * _log(rng, 4, 22), "layers": rng.randint(2, 12),
            "vocab": _log(rng, 2048, 32000), "seq": 1 if decode else _log(rng, 4, 256),
            "pos": _log(rng, 1, 1000) if decode else 0, "max_seq": 1024}


# ---- inputs -------------------------------------------------------------------

_provider = None


def _prov():
    global _provider
    if _provider is None:
        _provider = plugin.Provider()
        _provider.init()
    return _provider


class State:
    """Tensors, the provider's handles on them and the prepared tasks."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.prov = _prov()
        self.tensors = []
        self.handles = []
        self.tasks = []
        self.outputs = []
        self.graph = None

    def handle(self, t, dtype):
        """A provider buffer on the memory of tensor `t`."""
        desc = abi.make_desc(dtype, t.numel() * t.element_size())
        ops, h = abi.nf_buffer_ops(), ctypes.c_void_p()
        self.prov.check(self.prov.mem.import_buffer(self.prov.handle, t.data_ptr(), abi.NF_MEM_DOMAIN_DEVICE,
                                                    ctypes.byref(desc), ctypes.byref(ops), ctypes.byref(h)),
                        "import_buffer")
        b = plugin.Buffer(self.prov, h.value, ops, dtype, desc.size_bytes)
        self.tensors.append(t)
        self.handles.append(b)
        return b

    def empty(self, act, *shape):
        t = torch.zeros(shape, dtype=TORCH[act], device="cuda")
        return t, self.handle(t, ATYPE[act])

    def normal(self, act, *shape):
        t = torch.randn(shape, generator=self.gen, device="cuda").to(TORCH[act])
        return t, self.handle(t, ATYPE[act])

    def blocks(self, fmt, n, k):
        t = random_blocks(fmt, n * k // syn.KQ_GEOM[fmt][1], self.gen)
        return self.handle(t, QTYPE.get(fmt, abi.NF_DTYPE_U8))

    def add(self, op, ins, outs, m=0, n=0, k=0, **pc):
        raw = plugin.push_constants(m, n, k, **pc) if m or n or k or pc else b""
        self.tasks.append(self.prov.task(op, ins, outs, pc=raw))

    def ready(self, graph=False):
        self.array = (abi.nf_task_desc * len(self.tasks))(*self.tasks)
        torch.cuda.synchronize()  # the provider's stream does not wait for torch's
        if graph:
            self.graph = hiprt.Graph(self.prov.stream(), lambda: self.prov.run_tasks(self.array))
        return self

    def __del__(self):
        self.graph = None
        for b in self.handles:
            b.release()


def random_blocks(fmt, count, gen):
    """Blocks with uniform code and scale bytes and |N(0,1)|-distributed fp16 scales (synthetic.py's statistics)."""
    size, _ = syn.KQ_GEOM[fmt]
    raw = torch.randint(0, 256, (count, size), generator=gen, device="cuda", dtype=torch.uint8)
    scale = 0.002 if fmt == "q8_0" else 0.01
    for off in syn.KQ_F16_FIELDS[fmt]:
        d = (torch.randn(count, generator=gen, device="cuda").abs() * scale).to(torch.float16)
        raw[:, off:off + 2] = d.view(torch.uint8).reshape(count, 2)
    return raw


def _fused(fmt, act):
    return "dequant_%s_linear%s" % (fmt, "_f16" if act == "f16" else "")


def _linear(case, seed):
    s = State(seed)
    m, n, k, act = case["m"], case["n"], case["k"], case["act"]
    s.a, a = s.normal(act, m, k)
    if case["kind"] == "dense":
        s.w = (torch.randn(n, k, generator=s.gen, device="cuda") * 0.05).to(TORCH[act])
        w, op = s.handle(s.w, ATYPE[act]), "linear"
    else:
        w, op = s.blocks(case["fmt"], n, k), _fused(case["fmt"], act)
        s.w = s.tensors[-1]
    c, out = s.empty(act, m, n)
    s.add(op, [a, w], [out], m, n, k)
    s.outputs = [c]
    return s.ready()


def _projections(case, seed):
    s = State(seed)
    m, dim, kvd, ffn, fmt = case["m"], case["dim"], case["kv_dim"], case["ffn"], case["fmt"]
    # per layer: the attention norm's output feeds q, k and v, the attention output o, the FFN norm's output
    # gate and up, the gated product down
    s.x = [s.normal("f32", m, w) for w in (dim, dim, dim, ffn)]
    shapes = [(0, dim, dim), (0, kvd, dim), (0, kvd, dim), (1, dim, dim), (2, ffn, dim), (2, ffn, dim), (3, dim, ffn)]
    s.y = [torch.zeros(case["layers"], m, n, device="cuda") for _, n, _ in shapes]
    s.lin = []
    for layer in range(case["layers"]):
        for y, (x, n, k) in zip(s.y, shapes):
            w = s.blocks(fmt, n, k)
            s.lin.append((s.tensors[-1], x, n, k))
            s.add(_fused(fmt, "f32"), [s.x[x][1], w], [s.handle(y[layer], abi.NF_DTYPE_F32)], m, n, k)
    s.outputs = list(s.y)
    if case["vocab"]:
        w = s.blocks(fmt, case["vocab"], dim)
        s.lin.append((s.tensors[-1], 2, case["vocab"], dim))
        c, out = s.empty("f32", m, case["vocab"])
        s.add(_fused(fmt, "f32"), [s.x[2][1], w], [out], m, case["vocab"], dim)
        s.outputs.append(c)
    return s.ready(case["graph"])


def _dequant(case, seed):
    s = State(seed)
    w = s.blocks(case["fmt"], case["n"], case["k"])
    s.w = s.tensors[-1]
    c, out = s.empty(case["act"], case["n"], case["k"])
    s.add("dequant_%s%s" % (case["fmt"], "_f16" if case["act"] == "f16" else ""), [w], [out])
    s.outputs = [c]
    return s.ready()


def _attention(case, seed):
    s = State(seed)
    act, h, kv, d, seq = case["act"], case["heads"], case["kv"], case["dim"], case["seq"]
    s.q, q = s.normal(act, seq, h, d)
    s.k, k = s.normal(act, seq, kv, d)
    s.v, v = s.normal(act, seq, kv, d)
    s.ck, ck = s.normal(act, kv, case["max_seq"], d)
    s.cv, cv = s.normal(act, kv, case["max_seq"], d)
    c, out = s.empty(act, seq, h, d)
    s.add("flash_attention_cached", [q, k, v, ck, cv], [out], m=kv, seq_len=seq, n_heads=h, head_dim=d,
          step_idx=case["pos"], max_seq_len=case["max_seq"])
    s.outputs = [c, s.ck, s.cv]
    return s.ready()


def _model(case, seed):
    s = State(seed)
    fmt, d, h, kv, ffn, seq, pos = (case[x] for x in ("fmt", "dim", "heads", "kv", "ffn", "seq", "pos"))
    hd, vocab, ms = d // h, case["vocab"], case["max_seq"]
    kvd = kv * hd
    op = _fused(fmt, "f32")
    s.embed, embed = s.normal("f32", vocab, d)
    s.ids = torch.randint(0, vocab, (seq,), generator=s.gen, device="cuda", dtype=torch.int32)
    ids = s.handle(s.ids, ATYPE["i32"])
    act = {name: s.empty("f32", seq, w)[1] for name, w in
           [("normed", d), ("q", d), ("k", kvd), ("v", kvd), ("qr", d), ("kr", kvd), ("att", d), ("proj", d),
            ("res", d), ("gate", ffn), ("up", ffn), ("silu", ffn), ("mul", ffn), ("down", d)]}
    x = s.empty("f32", seq, d)[1]
    s.add("embedding_lookup", [embed, ids], [x], seq_len=seq, head_dim=d)
    s.layers = []
    kc = torch.randn(case["layers"], kv, ms, hd, generator=s.gen, device="cuda")
    vc = torch.randn(case["layers"], kv, ms, hd, generator=s.gen, device="cuda")
    norm = dict(seq_len=seq, n_heads=h, head_dim=d, epsilon=EPS, theta=THETA, step_idx=pos, max_seq_len=ms)
    rope = dict(seq_len=seq, head_dim=hd, theta=THETA, step_idx=pos)

    def weight(n, k):
        return s.blocks(fmt, n, k), s.tensors[-1], n, k

    def project(src, w, dst):
        s.add(op, [src, w[0]], [dst], seq, w[2], w[3])

    for i in range(case["layers"]):
        n1, g1 = s.normal("f32", d)
        n2, g2 = s.normal("f32", d)
        q, k, v, o = weight(d, d), weight(kvd, d), weight(kvd, d), weight(d, d)
        gate, up, down = weight(ffn, d), weight(ffn, d), weight(d, ffn)
        s.layers.append((n1, n2, [w[1:] for w in (q, k, v, o, gate, up, down)], kc[i], vc[i]))
        s.add("rms_norm", [x, g1], [act["normed"]], **norm)
        project(act["normed"], q, act["q"])
        project(act["normed"], k, act["k"])
        project(act["normed"], v, act["v"])
        s.add("rope_batch", [act["q"]], [act["qr"]], n_heads=h, **rope)
        s.add("rope_batch", [act["k"]], [act["kr"]], n_heads=kv, **rope)
        s.add("flash_attention_cached", [act["qr"], act["kr"], act["v"], s.handle(kc[i], ATYPE["f32"]),
                                         s.handle(vc[i], ATYPE["f32"])], [act["att"]], m=kv, seq_len=seq, n_heads=h,
              head_dim=hd, step_idx=pos, max_seq_len=ms)
        project(act["att"], o, act["proj"])
        s.add("metal_vector_add", [x, act["proj"]], [act["res"]])
        s.add("rms_norm", [act["res"], g2], [act["normed"]], **norm)
        project(act["normed"], gate, act["gate"])
        project(act["normed"], up, act["up"])
        s.add("silu", [act["gate"]], [act["silu"]])
        s.add("elementwise_mul", [act["silu"], act["up"]], [act["mul"]])
        project(act["mul"], down, act["down"])
        x = s.empty("f32", seq, d)[1]
        s.add("metal_vector_add", [act["res"], act["down"]], [x])
    s.norm, g = s.normal("f32", d)
    s.add("rms_norm", [x, g], [act["normed"]], **norm)
    head = weight(vocab, d)
    s.head = head[1:]
    logits, out = s.empty("f32", seq, vocab)
    project(act["normed"], head, out)
    s.outputs = [logits]
    return s.ready()


_MAKE = {"linear": _linear, "dense": _linear, "projections": _projections, "dequant": _dequant,
         "attention": _attention, "model": _model}


def prepare(case, seed):
    return _MAKE[case["kind"]](case, seed)


def run(state):
    if state.graph is not None:
        state.graph.launch()
    elif len(state.tasks) > 1:
        state.prov.run_tasks(state.array)
    else:
        state.prov.check(state.prov.dispatch_task(state.tasks[0]), "dispatch")
    return state.outputs


# ---- work ---------------------------------------------------------------------

def _linear_work(m, n, k, weight_bytes, elt):
    return {"bytes": weight_bytes + elt * m * (n + k), "flops": 2 * m * n * k}


def _attention_work(h, kv, d, seq, pos, elt):
    keys = pos + 1 if pos else seq
    pairs = keys if pos else seq * (seq + 1) // 2
    new = 2 * seq * kv * d * elt  # the appended rows: read, and written into the cache
    cache = 2 * (keys - seq) * kv * d * elt if pos else 0
    return {"bytes": 2 * new + cache + 2 * seq * h * d * elt, "flops": 4 * pairs * h * d}


def _sum(works):
    works = list(works)
    return {key: sum(w[key] for w in works) for key in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return _linear_work(case["m"], case["n"], case["k"], case["n"] * case["k"] // 32 * BLOCK[case["fmt"]],
                            SIZE[case["act"]])
    if kind == "dense":
        return _linear_work(case["m"], case["n"], case["k"], case["n"] * case["k"] * SIZE[case["act"]],
                            SIZE[case["act"]])
    if kind == "dequant":
        size, elems = syn.KQ_GEOM[case["fmt"]]
        count = case["n"] * case["k"]
        return {"bytes": count // elems * size + count * SIZE[case["act"]], "flops": 2 * count}
    if kind == "attention":
        return _attention_work(case["heads"], case["kv"], case["dim"], case["seq"], case["pos"], SIZE[case["act"]])
    d, ffn, bb = case["dim"], case["ffn"], BLOCK[case["fmt"]]
    m = case["m"] if kind == "projections" else case["seq"]
    kvd = case["kv_dim"] if kind == "projections" else case["kv"] * (d // case["heads"])

    def lin(n, k):
        return _linear_work(m, n, k, n * k // 32 * bb, 4)

    layer = [lin(d, d), lin(kvd, d), lin(kvd, d), lin(d, d), lin(ffn, d), lin(ffn, d), lin(d, ffn)]
    if kind == "model":  # the activations stay on the chip: each layer's are counted once, with its linears
        layer.append(_attention_work(case["heads"], case["kv"], d // case["heads"], case["seq"], case["pos"], 4))
    works = layer * case["layers"]
    if case["vocab"]:
        works.append(lin(case["vocab"], d))
    return _sum(works)


def tolerance(case):
    if case["kind"] == "dequant":
        return "exact"
    # About four times the distance from exact() measured on MI355X: 2.3e-5 through 22 layers in f32, one fp16
    # rounding of each value (2.1e-4) for f16 outputs, 5e-6 for the f32 linears' two-piece bf16 activations.
    if case["kind"] == "model":
        return {"rel": 1e-4, "max": 1e-3}
    if case.get("act") == "f16":
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 2e-5, "max": 2e-4}


# ---- 64-bit results -----------------------------------------------------------

def _half(raw, off):
    return raw[:, off:off + 2].contiguous().view(torch.float16).double()


def _bits(raw, lo, hi, width, count):
    """`count` fields of `width` bits each from bytes lo..hi-1 of every block, lowest bits first."""
    b = raw[:, lo:hi].int()
    parts = [(b >> s) & ((1 << width) - 1) for s in range(0, 8, width)]
    return torch.stack(parts, 2).reshape(raw.shape[0], -1)[:, :count]


def _nib32(raw, off):
    b = raw[:, off:off + 16].int()
    return torch.cat([b & 15, b >> 4], 1)


def _k_scales(raw):
    b = raw[:, 4:16].int()
    s = torch.cat([b[:, :4] & 63, (b[:, 0:4] >> 6) | ((b[:, 8:12] & 15) << 2)], 1)
    m = torch.cat([b[:, 4:8] & 63, (b[:, 4:8] >> 6) | ((b[:, 8:12] >> 4) << 2)], 1)
    return s, m


def dequantize(raw, fmt, f16=False):
    """The blocks' values in 64 bits, [blocks, elements]."""
    if fmt == "q4_0":
        return _half(raw, 0) * (_nib32(raw, 2) - 8)
    if fmt == "q8_0":
        return _half(raw, 0) * raw[:, 2:].contiguous().view(torch.int8)
    if fmt == "q4_1":
        return _half(raw, 0) * _nib32(raw, 4) + _half(raw, 2)
    if fmt in ("q5_0", "q5_1"):
        at = 2 if fmt == "q5_0" else 4
        q = _nib32(raw, at + 4) | (_bits(raw, at, at + 4, 1, 32) << 4)
        return _half(raw, 0) * (q - 16) if fmt == "q5_0" else _half(raw, 0) * q + _half(raw, 2)
    if fmt == "q2_k":
        s, q = raw[:, :16].int(), _bits(raw, 16, 80, 2, 256)
        sc, mn = _half(raw, 80) * (s & 15), _half(raw, 82) * (s >> 4)
        return sc.repeat_interleave(16, 1) * q - mn.repeat_interleave(16, 1)
    if fmt == "q3_k":
        q = (_bits(raw, 32, 96, 2, 256) | (_bits(raw, 0, 32, 1, 256) << 2)) - 4
        if f16:  # the op's documented reading: raw bytes 96..111, two of them the next block's first (zeros at the end)
            nxt = torch.cat([raw[1:, :2], torch.zeros_like(raw[:1, :2])])
            s = torch.cat([raw[:, 96:110], nxt], 1).int() - 32
        else:
            b = raw[:, 96:108].int()
            j = torch.arange(8, device=raw.device)
            top = b[:, 8 + j // 2] >> (4 * (j % 2))
            s = torch.cat([(b[:, :8] & 15) | ((top & 3) << 4), (b[:, :8] >> 4) | (((top >> 2) & 3) << 4)], 1) - 32
        return (_half(raw, 108) * s).repeat_interleave(16, 1) * q
    if fmt in ("q4_k", "q5_k"):
        s, m = _k_scales(raw)
        q = _bits(raw, 16, 144, 4, 256)
        if fmt == "q5_k":
            q = q | (_bits(raw, 144, 176, 1, 256) << 4)
        return (_half(raw, 0) * s).repeat_interleave(32, 1) * q - (_half(raw, 2) * m).repeat_interleave(32, 1)
    q = (_bits(raw, 0, 128, 4, 256) | (_bits(raw, 128, 192, 2, 256) << 4)) - 32
    s = raw[:, 192:208].contiguous().view(torch.int8)
    return (_half(raw, 208) * s).repeat_interleave(16, 1) * q


def _weights(raw, fmt, n, k, f16=False):
    w = dequantize(raw, fmt).reshape(n, k)
    return w.to(torch.float16).double() if f16 else w  # the f16 op rounds each weight to fp16


def _attend(q, k, v, pos):
    """Causal attention of q [seq, heads, dim] on k, v [kv, keys, dim], query i at position pos + i."""
    seq, heads, dim = q.shape
    out = torch.empty(seq, heads, dim, dtype=torch.float64, device=q.device)
    keys = k.shape[1]
    seen = torch.arange(keys, device=q.device)[None] <= torch.arange(pos, pos + seq, device=q.device)[:, None]
    for h in range(heads):
        g = h * k.shape[0] // heads
        p = (q[:, h] @ k[g].T) / math.sqrt(dim)
        out[:, h] = torch.softmax(p.masked_fill(~seen, -math.inf), 1) @ v[g]
    return out


def _rope(x, pos, dim):
    """x [seq, heads, dim]; pairs (i, i + dim/2)."""
    half = dim // 2
    f = THETA ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dim)
    a = torch.arange(pos, pos + x.shape[0], dtype=torch.float64, device=x.device)[:, None, None] * f
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], 2)


def _rms(x, g):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + EPS) * g.double()


def _exact_model(case, s):
    d, seq, pos, fmt = case["dim"], case["seq"], case["pos"], case["fmt"]
    hd = d // case["heads"]

    def lin(x, w):
        return x @ _weights(w[0], fmt, w[1], w[2]).T

    x = s.embed[s.ids.long()].double()
    for n1, n2, (q, k, v, o, gate, up, down), kc, vc in s.layers:
        y = _rms(x, n1)
        qr = _rope(lin(y, q).reshape(seq, -1, hd), pos, hd)
        keys, values = kc.double().clone(), vc.double().clone()
        keys[:, pos:pos + seq] = _rope(lin(y, k).reshape(seq, -1, hd), pos, hd).transpose(0, 1)
        values[:, pos:pos + seq] = lin(y, v).reshape(seq, -1, hd).transpose(0, 1)
        x = x + lin(_attend(qr, keys[:, :pos + seq], values[:, :pos + seq], pos).reshape(seq, d), o)
        y = _rms(x, n2)
        x = x + lin(torch.nn.functional.silu(lin(y, gate)) * lin(y, up), down)
    return [lin(_rms(x, s.norm), s.head)]


def exact(case, seed):
    """What run() returns, from the same inputs, in plain 64-bit torch."""
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return [s.a.double() @ _weights(s.w, case["fmt"], case["n"], case["k"], case["act"] == "f16").T]
    if kind == "dense":
        return [s.a.double() @ s.w.double().T]
    if kind == "dequant":
        return [dequantize(s.w, case["fmt"], case["act"] == "f16").reshape(case["n"], case["k"])]
    if kind == "projections":
        y = [s.x[x][0].double() @ _weights(w, case["fmt"], n, k).T for w, x, n, k in s.lin]
        outs = [torch.stack(y[i:7 * case["layers"]:7]) for i in range(7)]
        return outs + y[7 * case["layers"]:]
    if kind == "attention":
        pos, seq = case["pos"], case["seq"]
        ck, cv = s.ck.double(), s.cv.double()
        ck[:, pos:pos + seq] = s.k.double().transpose(0, 1)
        cv[:, pos:pos + seq] = s.v.double().transpose(0, 1)
        return [_attend(s.q.double(), ck[:, :pos + seq], cv[:, :pos + seq], pos), ck, cv]
    return _exact_model(case, s)
