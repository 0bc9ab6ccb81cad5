"""What this library is used for, as measurable calls: quantised linear layers, plain products,
the gated FFN block, attention and a mixture-of-experts layer, each at prefill and decode sizes
where it has both, through the C entry points on operands that lie in GPU memory.

Every call runs asynchronously on one stream, as a GPU-resident inference program queues its
layers; weights are packed once and kept."""
import ctypes as C
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rocket-userspace_amd"))
import rocketnpu as R  # noqa: E402

EXPERTS = 8   # experts of the mixture layer, two of them a token


def listed():
    return [
        # the smallest product of the library's tests: one launch's latency
        dict(name="fp16_small", op="fp16", M=64, K=256, N=128),
        # W4A8 up-projection of an FFN (3840 -> 15360): a prefill chunk of 512 tokens on rows
        # that are already quantised (several projections share them) ...
        dict(name="w4a8_prefill", op="w4a8", M=512, K=3840, N=15360, group=128, rows="int8"),
        # ... and a decode step of a few sequences, fp32 rows quantised inside the call
        dict(name="w4a8_decode", op="w4a8", M=4, K=3840, N=15360, group=128, rows="fp32"),
        # per-channel int8 projection with int32 results, prefill
        dict(name="int8_prefill", op="int8", M=512, K=4096, N=4096),
        # a mixture-of-experts layer, int8 weights in groups of 32: 4096 tokens of prefill
        # (about 1024 rows an expert, ragged), and a decode batch of 16 (about 4 rows an expert)
        dict(name="moe_prefill", op="moe", tokens=4096, hidden=2048, inter=1408, group=32),
        dict(name="moe_decode", op="moe", tokens=16, hidden=2048, inter=1408, group=32),
        # fp32 operands computed in bf16: a down-projection of 2048 rows, the largest product
        dict(name="bf16_large", op="fp32", M=2048, K=15360, N=3840, math="bf16"),
        # fp32 operands at tf32 precision: a middling product, no size a multiple of a tile
        dict(name="tf32_ragged", op="fp32", M=396, K=2064, N=1936, math="tf32"),
        # fp16 gated FFN block: a prefill chunk, and one token
        dict(name="ffn_prefill", op="ffn", M=512, H=3840, I=15360, act="gelu"),
        dict(name="ffn_decode", op="ffn", M=1, H=3840, I=15360, act="gelu"),
        # grouped-query attention: a causal chunk over a long cache, and one token over a cache
        # whose length is no multiple of a tile
        dict(name="attn_prefill", op="attn", T=512, n_kv=4096, dim=256, heads=16, kv_heads=8, mask=True, softcap=0.0),
        dict(name="attn_decode", op="attn", T=1, n_kv=3000, dim=256, heads=16, kv_heads=8, mask=False, softcap=0.0),
    ]


def draw(rng):
    def size(lo, hi, step=1):   # log-uniform, a multiple of step
        return max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step

    op = rng.choice(["fp16", "w4a8", "int8", "moe", "fp32", "ffn", "attn"])
    while True:
        if op == "fp16":
            c = dict(op=op, M=rng.choice([1, size(4, 1024, 4), size(4, 1024, 4)]), K=size(64, 8192, 32), N=size(64, 16384, 16))
        elif op == "w4a8":
            g = rng.choice([32, 64, 128])
            c = dict(op=op, M=size(4, 1024, 4), K=size(512, 8192, g), N=size(512, 16384, 64), group=g,
                     rows=rng.choice(["int8", "fp32"]))
        elif op == "int8":
            c = dict(op=op, M=size(4, 1024, 4), K=size(256, 8192, 32), N=size(256, 16384, 32))
        elif op == "moe":
            g = rng.choice([32, 32, 64, 128])
            c = dict(op=op, tokens=size(4, 4096), hidden=size(512, 4096, g), inter=size(512, 2048, g), group=g)
        elif op == "fp32":
            c = dict(op=op, M=size(4, 2048, 4), K=size(64, 15360, 32), N=size(64, 8192, 16), math=rng.choice(["bf16", "tf32"]))
        elif op == "ffn":
            c = dict(op=op, M=rng.choice([1, size(4, 512, 4), size(4, 512, 4)]), H=size(256, 4096, 32), I=size(512, 15360, 32),
                     act=rng.choice(["silu", "gelu"]))
        else:
            T = rng.choice([1, size(2, 512), size(2, 512)])
            kv = rng.choice([1, 2, 4, 8])
            c = dict(op=op, T=T, n_kv=max(T, size(64, 8192)), dim=rng.choice([64, 128, 256]), heads=kv * rng.choice([1, 2, 4]),
                     kv_heads=kv, mask=T > 1, softcap=rng.choice([0.0, 0.0, 50.0]))
        if work(c)["flops"] <= 1.2e11:
            return c


# ---- the library, its handles and the stream they run on ------------------------------

_DEV = "cuda"
_own = {}


def _session():
    if not _own:
        lib = R.load()
        stream = torch.cuda.Stream()
        fd = lib.rocket_open()
        assert fd >= 0, "no GPU"
        i4, i8 = lib.rocket_i4_ctx_create(1), lib.rocket_i8_ctx_create(1)
        for h in (fd, lib.rocket_i4_ctx_fd(i4), lib.rocket_i8_ctx_fd(i8)):
            assert lib.rocket_hip_set_stream(h, C.c_void_p(stream.cuda_stream)) == 0
            assert lib.rocket_hip_set_mode(h, R.ROCKET_HIP_ASYNC | R.ROCKET_HIP_DEVICE_OPERANDS) == 0
        _own.update(lib=lib, stream=stream, fd=fd, i4=i4, i8=i8)
    return _own


class _Weight:
    """A resident group-wise or per-channel weight, freed with its last reference."""

    def __init__(self, kind, codes, group):
        o = _session()
        self.lib, self.ctx, self.kind = o["lib"], o[kind], kind
        N, K = codes.shape
        pack = getattr(self.lib, "rocket_%s_weights_pack%s" % (kind, "_gw" if group else ""))
        self.h = pack(self.ctx, 4, K, N, R.ptr(codes), *([group] if group else []))
        assert self.h, "weight not packed"

    def __del__(self):
        if getattr(self, "h", None):
            getattr(self.lib, "rocket_%s_weights_free" % self.kind)(self.ctx, self.h)


class _State:
    """One layer's operands: the entry points to call in order, and the outputs they fill."""

    def __init__(self, calls, out, keep):
        self.calls, self.out, self.keep = calls, out, keep


def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(seed)


def _normal(g, shape, std=1.0, dtype=torch.float32):
    return torch.empty(shape, dtype=torch.float32, device=_DEV).normal_(0.0, std, generator=g).to(dtype)


def _quantised(g, N, K, group, top):
    """Symmetric codes in [-top, top] of N(0, 0.02) weights, one scale per `group` of K."""
    w = _normal(g, (N, K // group, group), 0.02)
    s = (w.abs().amax(2) / top).clamp_min(1e-12)
    return torch.round(w / s[:, :, None]).to(torch.int8).view(N, K), s.contiguous()


def _rows(x):
    """Per-row int8 codes and scales of fp32 rows, by the library's formula (fp32 divisions)."""
    a = x.abs().amax(1, keepdim=True)
    q = torch.round(x * torch.where(a > 0, 127.0 / a, torch.zeros_like(a))).clamp(-128, 127).to(torch.int8)
    return q, (a / 127.0).squeeze(1).contiguous()


def _expert_rows(tokens):
    """Rows an expert gets when every token takes two of EXPERTS at random, in fours."""
    rng, n = random.Random(tokens), [0] * EXPERTS
    for _ in range(tokens):
        for e in rng.sample(range(EXPERTS), 2):
            n[e] += 1
    return [-(-m // 4) * 4 for m in n]


def _inputs(c, seed):
    """The tensors of a case, from the seed alone (what prepare and exact share)."""
    g, op = _gen(seed), c["op"]
    if op == "fp16":
        return dict(A=_normal(g, (c["M"], c["K"]), 1.0, torch.float16), B=_normal(g, (c["N"], c["K"]), 0.02, torch.float16))
    if op == "fp32":
        return dict(A=_normal(g, (c["M"], c["K"])), B=_normal(g, (c["N"], c["K"]), 0.02))
    if op == "int8":
        i = dict(generator=g, dtype=torch.int8, device=_DEV)
        return dict(A=torch.randint(-128, 128, (c["M"], c["K"]), **i), B=torch.randint(-128, 128, (c["N"], c["K"]), **i))
    if op == "w4a8":
        B, s = _quantised(g, c["N"], c["K"], c["group"], 7)
        x = _normal(g, (c["M"], c["K"]))
        q, r = _rows(x)
        return dict(x=x, q=q, r=r, B=B, s=s)
    if op == "ffn":
        H, I = c["H"], c["I"]
        return dict(x=_normal(g, (c["M"], H), 1.0, torch.float16), Wg=_normal(g, (I, H), 0.02, torch.float16),
                    Wu=_normal(g, (I, H), 0.02, torch.float16), Wd=_normal(g, (H, I), 0.02, torch.float16))
    if op == "attn":
        T, n, d, h, kv = c["T"], c["n_kv"], c["dim"], c["heads"], c["kv_heads"]
        t = dict(Q=_normal(g, (h, T, d), 1.0, torch.float16), K=_normal(g, (kv, n, d), 1.0, torch.float16),
                 V=_normal(g, (kv, d, n), 1.0, torch.float16), mask=None)
        if c["mask"]:   # query t stands at position n - T + t
            pos = torch.arange(T, device=_DEV)[:, None] + (n - T)
            t["mask"] = torch.zeros((T, n), device=_DEV).masked_fill_(torch.arange(n, device=_DEV)[None] > pos, -math.inf).half()
        return t
    assert op == "moe"
    H, F, grp = c["hidden"], c["inter"], c["group"]
    t = dict(q=[], r=[], gate=[], up=[], down=[])
    for m in _expert_rows(c["tokens"]):
        q, r = _rows(_normal(g, (m, H)))
        t["q"].append(q)
        t["r"].append(r)
        for k, (n, kk) in (("gate", (F, H)), ("up", (F, H)), ("down", (H, F))):
            t[k].append(_quantised(g, n, kk, grp, 127))
    return t


def prepare(case, seed):
    o, c, op = _session(), case, case["op"]
    lib, fd = o["lib"], o["fd"]
    with torch.cuda.stream(o["stream"]):
        t = _inputs(c, seed)
        new = lambda shape, dtype: torch.empty(shape, dtype=dtype, device=_DEV)  # noqa: E731
        if op in ("fp16", "fp32"):
            M, K, N = c["M"], c["K"], c["N"]
            out = new((M, N), t["A"].dtype)
            fn = lib.rocket_matmul_fp16 if op == "fp16" else getattr(lib, "rocket_matmul_" + c["math"])
            return _State([(fn, (fd, M, K, N, R.ptr(t["A"]), R.ptr(t["B"]), R.ptr(out)))], out, t)
        if op == "int8":
            M, K, N = c["M"], c["K"], c["N"]
            w, out = _Weight("i8", t["B"], 0), new((M, N), torch.int32)
            return _State([(lib.rocket_matmul_int8_prepacked, (o["i8"], M, K, N, R.ptr(t["A"]), R.ptr(out), w.h))], out, (t["A"], w))
        if op == "w4a8":
            M, K, N = c["M"], c["K"], c["N"]
            w, out = _Weight("i4", t["B"], c["group"]), new((M, N), torch.float32)
            if c["rows"] == "fp32":
                call = (lib.rocket_matmul_int4_prepacked_gw_f32in, (o["i4"], M, K, N, R.ptr(t["x"]), R.ptr(t["s"]), R.ptr(out), w.h))
            else:
                call = (lib.rocket_matmul_int4_prepacked_gw_rowscale,
                        (o["i4"], M, K, N, R.ptr(t["q"]), R.ptr(t["r"]), R.ptr(t["s"]), R.ptr(out), w.h))
            del t["B"]
            return _State([call], out, (t, w))
        if op == "ffn":
            act = R.ROCKET_ACTIVATION_SILU if c["act"] == "silu" else R.ROCKET_ACTIVATION_GELU
            out = new((c["M"], c["H"]), torch.float16)
            return _State([(lib.rocket_ffn_fp16, (fd, c["M"], c["H"], c["I"], R.ptr(t["x"]), R.ptr(t["Wg"]), R.ptr(t["Wu"]),
                                                  R.ptr(t["Wd"]), act, R.ptr(out)))], out, t)
        if op == "attn":
            out = new((c["heads"], c["T"], c["dim"]), torch.float16)
            return _State([(lib.rocket_flash_attn_fp16,
                            (fd, c["T"], c["n_kv"], c["dim"], c["dim"], c["heads"], c["kv_heads"], c["dim"] ** -0.5, c["softcap"],
                             R.ptr(t["Q"]), R.ptr(t["K"]), R.ptr(t["V"]), R.ptr(t["mask"]), R.ptr(out)))], out, t)
        # the mixture layer: gate and up of all experts as one grouped call with fp16 results, then
        # the down products on silu(gate) * up
        H, F, E = c["hidden"], c["inter"], EXPERTS
        Ms = _expert_rows(c["tokens"])
        W = {k: [_Weight("i8", codes, c["group"]) for codes, _ in t[k]] for k in ("gate", "up", "down")}
        S = {k: [s for _, s in t[k]] for k in W}
        gate, up = ([new((m, F), torch.float16) for m in Ms] for _ in range(2))
        out = [new((m, H), torch.float32) for m in Ms]
        keep = [t["q"], t["r"], W, S]

        def arr(xs):
            p, k = R.ptr_array([x.h if isinstance(x, _Weight) else x for x in xs])
            keep.append(k)
            return p

        two, one = R.int_array(Ms + Ms), R.int_array(Ms)
        keep += [two, one]
        up_args = (o["i8"], 2 * E, two[0], H, F, arr(t["q"] * 2), arr(t["r"] * 2), arr(S["gate"] + S["up"]), arr(gate + up),
                   arr(W["gate"] + W["up"]))
        down_args = (o["i8"], E, one[0], F, H, arr(gate), arr(up), R.ROCKET_ACTIVATION_SILU, arr(S["down"]), arr(out), arr(W["down"]))
        return _State([(lib.rocket_matmul_int8_prepacked_gw_grouped_rowscale_f16out, up_args),
                       (lib.rocket_matmul_int8_prepacked_gw_grouped_glu_f16in, down_args)],
                      dict(gate=gate, up=up, out=out), keep)


def run(state):
    for fn, args in state.calls:
        rc = fn(*args)
        if rc:
            raise RuntimeError("%s returned %d" % (fn.__name__, rc))
    return state.out


def work(case):
    c, op = case, case["op"]
    if op in ("fp16", "fp32", "int8"):
        M, K, N, e = c["M"], c["K"], c["N"], {"fp16": 2, "fp32": 4, "int8": 1}[op]
        return dict(bytes=e * (M * K + N * K) + (2 if op == "fp16" else 4) * M * N, flops=2 * M * N * K)
    if op == "w4a8":
        M, K, N = c["M"], c["K"], c["N"]
        a = 4 * M * K if c["rows"] == "fp32" else M * K + 4 * M
        return dict(bytes=a + N * K // 2 + 4 * N * (K // c["group"]) + 4 * M * N, flops=2 * M * N * K)
    if op == "ffn":
        M, H, I = c["M"], c["H"], c["I"]
        return dict(bytes=2 * (2 * M * H + 3 * H * I), flops=6 * M * H * I)
    if op == "attn":
        T, n, d, h, kv = c["T"], c["n_kv"], c["dim"], c["heads"], c["kv_heads"]
        pairs = T * n - T * (T - 1) // 2 if c["mask"] else T * n   # a causal query sees no later key
        return dict(bytes=2 * (2 * h * T * d + 2 * kv * n * d + (T * n if c["mask"] else 0)), flops=4 * h * d * pairs)
    H, F, grp = c["hidden"], c["inter"], c["group"]
    Ms = _expert_rows(c["tokens"])
    rows, used = sum(Ms), sum(m > 0 for m in Ms)
    return dict(bytes=used * 3 * H * F * (1 + 4 / grp) + rows * (H + 4 + 2 * 2 * F + 4 * H), flops=6 * rows * H * F)


def tolerance(case):
    """About four times what the path was seen to differ from exact() by."""
    op = case["op"]
    if op == "int8":
        return "exact"
    if op == "fp32":   # fp32 sums of bf16 products (8e-7 at K = 15360); tf32 leaves out the products of the low parts (9e-6)
        return dict(rel=4e-6) if case["math"] == "bf16" else dict(rel=4e-5)
    if op == "w4a8":   # whole group sums folded in fp32 (1e-7); a value of an fp32 row may round to the next code (3e-5)
        return dict(rel=1e-6) if case["rows"] == "int8" else dict(rel=1.2e-4, max=8e-3)
    if op == "moe":    # fp16 gate and up values, a hidden value may round to the next 8-bit code (7e-4)
        return dict(rel=3e-3, max=0.1)
    # fp16 results (2e-4); with an fp16 hidden row, 3e-4; with fp16 probabilities and partial outputs, 3.6e-4
    return dict(rel={"fp16": 8e-4, "ffn": 1.2e-3, "attn": 1.5e-3}[op])


def exact(case, seed):
    c, op = case, case["op"]
    if work(c)["flops"] > 1e12:
        return None
    t = _inputs(c, seed)
    f = lambda x: x.double()  # noqa: E731
    if op == "fp16":
        return f(t["A"]) @ f(t["B"]).t()
    if op == "int8":
        return (f(t["A"]) @ f(t["B"]).t()).to(torch.int32)
    if op == "fp32":   # operands truncated as the entry states: 16 low bits (bf16), 13 (tf32)
        cut = lambda x: (x.view(torch.int32) & (-1 << (16 if c["math"] == "bf16" else 13))).view(torch.float32).double()  # noqa: E731
        return cut(t["A"]) @ cut(t["B"]).t()
    deq = lambda q, s: (f(q).view(s.shape[0], s.shape[1], -1) * f(s)[:, :, None]).view(q.shape)  # noqa: E731
    if op == "w4a8":
        return (f(t["q"]) @ deq(t["B"], t["s"]).t()) * f(t["r"])[:, None]
    if op == "ffn":
        g, u = f(t["x"]) @ f(t["Wg"]).t(), f(t["x"]) @ f(t["Wu"]).t()
        a = torch.nn.functional.silu(g) if c["act"] == "silu" else torch.nn.functional.gelu(g)
        return (a * u) @ f(t["Wd"]).t()
    if op == "attn":
        out = []
        for h in range(c["heads"]):
            k = h // (c["heads"] // c["kv_heads"])
            s = (f(t["Q"][h]) @ f(t["K"][k]).t().contiguous()) * c["dim"] ** -0.5
            if c["softcap"]:
                s = torch.tanh(s / c["softcap"]) * c["softcap"]
            if t["mask"] is not None:
                s = s + f(t["mask"])
            out.append(torch.softmax(s.clamp_min(-30000.0), 1) @ f(t["V"][k]).t().contiguous())
        return torch.stack(out)
    r = dict(gate=[], up=[], out=[])
    for e in range(EXPERTS):
        x = f(t["q"][e]) * f(t["r"][e])[:, None]
        g, u = (x @ deq(*t[k][e]).t() for k in ("gate", "up"))
        r["gate"].append(g)
        r["up"].append(u)
        # the layer's hidden rows are 8-bit codes of silu(gate) * up by definition
        q, s = _rows((torch.nn.functional.silu(g.half().double()) * u.half().double()).float())
        r["out"].append((f(q) * f(s)[:, None]) @ deq(*t["down"][e]).t())
    return r
