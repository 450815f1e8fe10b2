"""The work a user of accel_amd has it do, as cases that can be timed and compared.

Every case goes through the package's public operators on device buffers:

- ``matvec``    one decode token against one int4 matrix (a projection, or the
                vocabulary head): Int4MatVec on the planes, or on a bound copy;
- ``rows``      2..16 decode rows against one int4 matrix: Int4MatMul, planes
                or bound;
- ``step``      the products of a decoder layer at batch 1..16 on bound
                weights, captured once in a graph and replayed, as a serving
                loop does;
- ``linear``    prompt rows (prefill) through Int4Linear, f32 or bf16, with or
                without a bias; extents on and off the tiles' multiples;
- ``moe``       routed rows against int4 experts: Int4GroupedMatMul, planes or
                bound, decode and prefill token counts;
- ``grouped``   routed rows against f32 experts: GroupedMatMul;
- ``int8``      rows against an int8 matrix: QuantMatMul, f32 or f16 rows;
- ``quantize``  a weight packed on the device into the int4 format (load time).

Sizes are those of the repository's benchmark (4096 / 1024 / 14336 layers, 8
experts, the 2048 x 2048 decode product, 2048-row prompts) and generic odd
ones.  Weights are normal with a standard deviation of 0.02, as the benchmark
draws them, packed here by plain torch in the reference's format.
"""
import math

import torch

import accel_amd
from accel_amd import BF16, F16, F32, I8, U32

GROUP = 128      # int4 weights a scale and a zero point cover
BLOCK = 32       # int8 weights a scale covers
EPS = 1e-5

_DTYPES = {torch.float32: F32, torch.float16: F16, torch.bfloat16: BF16, torch.int32: U32,
           torch.int8: I8, torch.int16: F16}
_device = None


def device():
    global _device
    if _device is None:
        _device = accel_amd.Device(0)
    return _device


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the smallest call: one token against a 2048 x 2048 projection, on the
        # planes as they were packed; latency and the host path count
        dict(name="matvec_2048", op="matvec", K=2048, N=2048, form="planes"),
        # one token against a vocabulary head whose width is no multiple of a
        # group, so quantisation groups straddle rows
        dict(name="head_ragged", op="matvec", K=4096, N=32004, form="planes"),
        # a decoder layer's seven products, two norms and SwiGLU for one token
        # in a graph: single-stream generation
        dict(name="step_b1", op="step", M=1, d=4096, kv=1024, f=14336),
        # the same for eight sequences: batched generation
        dict(name="step_b8", op="step", M=8, d=4096, kv=1024, f=14336),
        # a 2048-token prompt through one projection in bf16
        dict(name="prefill_bf16", op="linear", M=2048, K=4096, N=4096, dtype="bf16", bias=False),
        # a prompt of an odd length in f32, with a bias
        dict(name="prefill_f32", op="linear", M=333, K=4096, N=4096, dtype="f32", bias=True),
        # extents off every tile (K % 64, N % 128, odd rows), f32 with a bias
        dict(name="linear_ragged", op="linear", M=100, K=4100, N=4004, dtype="f32", bias=True),
        # 512 prompt tokens routed to two of eight experts, bf16: the largest
        dict(name="moe_prefill", op="moe", T=512, top=2, E=8, K=4096, N=14336, dtype="bf16",
             form="planes"),
        # eight decode tokens routed the same way, f32, bound experts
        dict(name="moe_decode", op="moe", T=8, top=2, E=8, K=4096, N=14336, dtype="f32",
             form="side"),
        # 128 tokens routed to two of eight unquantised f32 experts
        dict(name="grouped_f32", op="grouped", T=128, top=2, E=8, K=2048, N=4096),
        # a 512-token prompt against an int8 matrix
        dict(name="int8_prefill", op="int8", M=512, K=4096, N=4096, dtype="f32"),
        # packing one 4096 x 14336 matrix while a model loads
        dict(name="quantize", op="quantize", n=4096 * 14336),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    op = rng.choice(["matvec", "rows", "step", "linear", "linear", "ragged", "moe", "grouped",
                     "int8", "int8", "quantize"])
    if op == "matvec":
        form = rng.choice(["planes", "planes", "panels", "ragged"])
        if form == "ragged":
            return dict(op="matvec", K=_log(rng, 256, 8192), N=_log(rng, 256, 40000),
                        form="planes")
        return dict(op="matvec", K=_extent(rng, 256, 14336, rng.choice([32, 4])),
                    N=_extent(rng, 256, 14336, 128), form=form)
    if op == "rows":
        return dict(op="rows", M=rng.randint(2, 16), K=_extent(rng, 256, 14336, 32),
                    N=_extent(rng, 256, 14336, 128), form=rng.choice(["planes", "tiles"]))
    if op == "step":
        d = rng.choice([1024, 2048, 4096])
        return dict(op="step", M=rng.randint(1, 16), d=d, kv=d // rng.choice([1, 2, 4]),
                    f=_extent(rng, 2 * d, 4 * d, 128))
    if op == "linear":
        # prompt rows on tile-friendly matrices
        K, N = _extent(rng, 512, 14336, 64), _extent(rng, 512, 14336, 128)
        M = _log(rng, 17, 2048)
        while M * K * N > 2048 * 4096 * 4096:
            M = max(17, M // 2 + 1)
        return dict(op="linear", M=M, K=K, N=N, dtype=rng.choice(["bf16", "f32"]),
                    bias=rng.random() < 0.5)
    if op == "ragged":
        # rows against a matrix of any extents
        return dict(op="linear", M=_log(rng, 2, 512), K=_log(rng, 100, 5000),
                    N=_log(rng, 100, 5000), dtype=rng.choice(["bf16", "f32"]),
                    bias=rng.random() < 0.5)
    if op == "moe":
        dtype = rng.choice(["bf16", "f32"])
        T = _log(rng, 1, 512)
        form = rng.choice(["planes", "side", "panels"] if T <= 32 else ["planes"])
        return dict(op="moe", T=T, top=2, E=rng.choice([4, 8, 16]),
                    K=_extent(rng, 512, 4096, 64), N=_extent(rng, 512, 14336, 128) if T <= 64
                    else _extent(rng, 512, 7168, 128), dtype=dtype, form=form)
    if op == "grouped":
        return dict(op="grouped", T=_log(rng, 1, 512), top=2, E=rng.choice([4, 8]),
                    K=_log(rng, 128, 2048), N=_log(rng, 128, 4096))
    if op == "int8":
        N = _extent(rng, 256, 14336, 32) if rng.random() < 0.75 else _log(rng, 200, 5000)
        K = _log(rng, 256, 8192)
        M = _log(rng, 1, 2048)
        while M * K * N > 512 * 4096 * 4096:
            M = max(1, M // 2)
        return dict(op="int8", M=M, K=K, N=N, dtype=rng.choice(["f32", "f32", "f16"]))
    return dict(op="quantize", n=_log(rng, 10000, 4096 * 14336))


# ---- inputs --------------------------------------------------------------------

class State(dict):
    """A case's inputs, outputs and handles; the handles are freed with it."""

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.get("exec"):
                device().destroy_exec(self["exec"])
            if self.get("stream"):
                device().destroy_stream(self["stream"])
            for h in self.get("handles", ()):
                h.free()
        except Exception:
            pass


def _buffer(t):
    """A torch tensor's memory as a buffer of the package (the tensor is kept
    by the state)."""
    return accel_amd.Buffer(device(), t.data_ptr(), t.numel() * t.element_size(),
                            _DTYPES[t.dtype], tuple(t.shape))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _weight(g, n):
    return _normal(g, n) * 0.02


def _pack4(w):
    """Flat f32 weights in the int4 format: codes, scales, zeros (f16)."""
    n = w.numel()
    groups = -(-n // GROUP)
    if groups * GROUP != n:
        w = torch.cat([w, w[-1:].expand(groups * GROUP - n)])
    v = w.view(groups, GROUP)
    lo, hi = v.amin(1), v.amax(1)
    s = ((hi - lo) / 15).half()
    z = torch.where(s > 0, -lo / s.float(), lo).half()
    q = torch.round(v / s.float().clamp_min(1e-8)[:, None] + z.float()[:, None])
    q = torch.where(s[:, None] > 0, q.clamp(0, 15), torch.zeros_like(q)).to(torch.int32)
    q = q.view(-1, 8)
    codes = torch.zeros(q.shape[0], dtype=torch.int32, device="cuda")
    for j in range(8):
        codes |= q[:, j] << (4 * j)
    return codes[:-(-n // 8)].contiguous(), s, z


def _unpack4(codes, s, z, n):
    """The weights the planes stand for, in 64 bits: (code - z) * s, or z where
    the scale is zero."""
    q = torch.stack([(codes >> (4 * j)) & 15 for j in range(8)], 1).reshape(-1)[:n]
    g = torch.arange(n, device="cuda") // GROUP
    s, z = s.double()[g], z.double()[g]
    return torch.where(s == 0, z, (q.double() - z) * s)


def _pack8(w):
    n = w.numel()
    blocks = -(-n // BLOCK)
    if blocks * BLOCK != n:
        w = torch.cat([w, w.new_zeros(blocks * BLOCK - n)])
    v = w.view(blocks, BLOCK)
    s = (v.abs().amax(1) / 127).half()
    q = torch.round(v / s.float().clamp_min(1e-8)[:, None]).clamp(-127, 127).to(torch.int8)
    return q.view(-1)[:n].contiguous(), s


def _planes(codes, s, z, n):
    return accel_amd.Int4Weights(_buffer(codes), _buffer(s), _buffer(z), n)


def _act(g, M, K, dtype):
    x = _normal(g, M, K)
    return x.to({"bf16": torch.bfloat16, "f16": torch.float16}.get(dtype, torch.float32))


def _matrices(case):
    """The (K, N) of each int4 matrix of a case, in the order they are drawn."""
    if case["op"] == "step":
        d, kv, f = case["d"], case["kv"], case["f"]
        return [(d, d), (d, kv), (d, kv), (d, d), (d, f), (d, f), (f, d)]
    if case["op"] == "moe":
        return [(case["K"], case["N"])] * case["E"]
    return [(case["K"], case["N"])]


def _inputs(case, seed):
    """Everything drawn for a case, from the seed alone."""
    g = _generator(seed)
    op = case["op"]
    r = {}
    if op == "quantize":
        r["w"] = _weight(g, case["n"])
        return r
    if op in ("matvec", "step", "rows"):
        r["x"] = _act(g, case.get("M", 1), case["d"] if op == "step" else case["K"], "f32")
    elif op in ("linear", "int8"):
        r["x"] = _act(g, case["M"], case["K"], case["dtype"])
    else:
        # tokens to `top` experts by a softmax of normal logits, rows sorted by expert
        T, top, E = case["T"], case["top"], case["E"]
        x = _act(g, T, case["K"], case.get("dtype", "f32"))
        chosen = torch.topk(_normal(g, T, E), top, dim=1).indices.reshape(-1)
        order = torch.sort(chosen, stable=True).indices
        r["x"] = x[order // top].contiguous()
        r["counts"] = torch.bincount(chosen, minlength=E).to(torch.int32)
    if op == "int8":
        r["q"], r["s"] = _pack8(_weight(g, case["K"] * case["N"]))
    elif op == "grouped":
        r["w"] = _weight(g, case["E"] * case["K"] * case["N"]).view(
            case["E"], case["K"], case["N"])
    else:
        r["planes"] = [_pack4(_weight(g, K * N)) for K, N in _matrices(case)]
    if op == "step":
        r["gain"] = [1 + 0.1 * _normal(g, case["d"]) for _ in range(2)]
    if case.get("bias"):
        r["bias"] = _normal(g, case["N"]) * 0.02
    return r


def prepare(case, seed):
    dev = device()
    op = case["op"]
    s = State(_inputs(case, seed), op=op, handles=[])
    new = lambda *shape, dtype=torch.float32: torch.empty(  # noqa: E731
        *shape, dtype=dtype, device="cuda")
    if op == "quantize":
        n = case["n"]
        s["out"] = [new(-(-n // 8), dtype=torch.int32), new(-(-n // GROUP), dtype=torch.int16),
                    new(-(-n // GROUP), dtype=torch.int16)]
        s["b"] = [_buffer(t) for t in [s["w"]] + s["out"]]
        s["n"] = n
        return s
    if op == "grouped":
        s["out"] = new(s["x"].shape[0], case["N"])
        s["b"] = [_buffer(s[k]) for k in ("x", "w", "counts", "out")]
        return s
    if op == "int8":
        s["out"] = new(case["M"], case["N"])
        s["q"] = s["q"].view(case["K"], case["N"])
        s["b"] = [_buffer(s[k]) for k in ("x", "q", "s", "out")]
        return s
    if op == "moe":
        K, N, E = case["K"], case["N"], case["E"]
        s["planes"] = [torch.cat(p) for p in zip(*s["planes"])]
        w = _planes(*s["planes"], E * K * N)
        s["out"] = new(s["x"].shape[0], N, dtype=s["x"].dtype)
        s["b"] = [_buffer(s[k]) for k in ("x", "counts", "out")]
        s["E"], s["form"], s["w"] = E, case["form"], w
        torch.cuda.synchronize()
        if case["form"] != "planes":
            s["w"] = dev.prepare_int4_grouped(w, E, K, N, panels=case["form"] == "panels")
            s["handles"].append(s["w"])
        return s
    ws = [_planes(*p, K * N) for p, (K, N) in zip(s["planes"], _matrices(case))]
    if op == "step":
        return _prepare_step(case, s, ws)
    M, N = case.get("M", 1), case["N"]
    if op == "matvec":
        s["x"] = s["x"].view(-1)
    out_dtype = s["x"].dtype
    s["out"] = new(*((N,) if op == "matvec" else (M, N)), dtype=out_dtype)
    s["b"] = [_buffer(s["x"]), _buffer(s["out"])]
    s["bias_b"] = _buffer(s["bias"]) if case.get("bias") else None
    s["w"], s["form"] = ws[0], case.get("form", "planes")
    torch.cuda.synchronize()
    if s["form"] != "planes":
        s["w"] = dev.prepare_int4(ws[0], case["K"], N, tiles=s["form"] == "tiles")
        s["handles"].append(s["w"])
    return s


def _prepare_step(case, s, ws):
    """Binds the layer's weights (panels for one row, side copies for more)
    and captures its launches once."""
    dev = device()
    M, f = case["M"], case["f"]
    torch.cuda.synchronize()
    w = [dev.prepare_int4(p, K, N, tiles=M > 1) for p, (K, N) in zip(ws, _matrices(case))]
    s["handles"] += w
    names = ("n1", "q", "k", "v", "o", "n2", "g", "u", "h", "y")
    d, kv = case["d"], case["kv"]
    widths = dict(n1=d, q=d, k=kv, v=kv, o=d, n2=d, g=f, u=f, h=f, y=d)
    shape = (lambda n: (n,)) if M == 1 else (lambda n: (M, n))
    t = {n: torch.empty(shape(widths[n]), dtype=torch.float32, device="cuda") for n in names}
    s["x"] = s["x"].view(shape(d))
    b = {n: _buffer(v) for n, v in t.items()}
    x, g1, g2 = _buffer(s["x"]), _buffer(s["gain"][0]), _buffer(s["gain"][1])
    st = dev.stream()
    s["stream"] = st

    def issue():
        dev.RMSNorm(x, g1, EPS, b["n1"], st)
        if M == 1:
            dev.Int4MatVecPreparedSet(b["n1"], w[:3], [b["q"], b["k"], b["v"]], st)
            dev.Int4MatVecPrepared(b["q"], w[3], b["o"], st)
            dev.RMSNorm(b["o"], g2, EPS, b["n2"], st)
            dev.Int4MatVecPreparedSwiGLU(b["n2"], w[4], w[5], b["h"], st)
            dev.Int4MatVecPrepared(b["h"], w[6], b["y"], st)
        else:
            dev.Int4MatMulPreparedSet(b["n1"], w[:3], [b["q"], b["k"], b["v"]], st)
            dev.Int4MatMulPrepared(b["q"], w[3], b["o"], st)
            dev.RMSNorm(b["o"], g2, EPS, b["n2"], st)
            dev.Int4MatMulPreparedSet(b["n2"], w[4:6], [b["g"], b["u"]], st)
            dev.SwiGLU(b["g"], b["u"], b["h"], st)
            dev.Int4MatMulPrepared(b["h"], w[6], b["y"], st)

    issue()
    dev.sync(st)
    dev.capture_begin(st)
    issue()
    s["exec"] = dev.capture_end(st)
    s["out"] = [t[n] for n in ("k", "v", "o", "h", "y")]
    s["tensors"] = t
    s["planes"] = None   # the bound copies are what the step reads
    return s


# ---- one pass --------------------------------------------------------------------

def run(s):
    dev = device()
    op, b = s["op"], s.get("b")
    if op == "step":
        dev.launch(s["exec"])
    elif op == "matvec":
        (dev.Int4MatVec if s["form"] == "planes" else dev.Int4MatVecPrepared)(b[0], s["w"], b[1])
    elif op == "rows":
        (dev.Int4MatMul if s["form"] == "planes" else dev.Int4MatMulPrepared)(b[0], s["w"], b[1])
    elif op == "linear":
        dev.Int4Linear(b[0], s["w"], s["bias_b"], b[1])
    elif op == "moe":
        if s["form"] == "planes":
            dev.Int4GroupedMatMul(b[0], s["w"], s["E"], b[1], b[2])
        else:
            dev.Int4GroupedMatMulPrepared(b[0], s["w"], b[1], b[2])
    elif op == "grouped":
        dev.GroupedMatMul(*b)
    elif op == "int8":
        dev.QuantMatMul(*b)
    else:
        dev.int4_quantize(b[0], s["n"], b[1], b[2], b[3])
    return s["out"]


# ---- what a pass cannot do without -------------------------------------------------

def work(case):
    op = case["op"]
    if op == "quantize":
        n = case["n"]
        return {"bytes": 4 * n + n / 2 + 4 * n / GROUP, "flops": 0}
    if op == "step":
        M = case["M"]
        kn = [K * N for K, N in _matrices(case)]
        acts = M * (2 * case["d"] + 2 * case["kv"] + case["f"])
        return {"bytes": sum(kn) * (0.5 + 4 / GROUP) + 4 * acts, "flops": 2 * M * sum(kn)}
    K, N = case["K"], case["N"]
    wide = 4 if case.get("dtype", "f32") == "f32" else 2
    if op in ("moe", "grouped"):
        rows = case["T"] * case["top"]
        # the experts that some token is expected to choose
        used = case["E"] * (1 - (1 - case["top"] / case["E"]) ** case["T"])
        per = K * N * (4 if op == "grouped" else 0.5 + 4 / GROUP)
        return {"bytes": used * per + wide * rows * (K + N), "flops": 2 * rows * K * N}
    M = case.get("M", 1)
    per = K * N * (1 + 2 / BLOCK if op == "int8" else 0.5 + 4 / GROUP)
    out = 4 if op == "int8" else wide
    return {"bytes": per + wide * M * K + out * M * N + (4 * N if case.get("bias") else 0),
            "flops": 2 * M * K * N}


def tolerance(case):
    """f32 paths: sums of up to 14336 products in 32 bits, in another order
    (the start and a 64-bit sum differ by 1e-7 to 2e-6; a step's five outputs
    carry it through four products).  bf16: each result rounded once to 8 bits
    and the weights rounded to bf16 in the tiles (2.6e-3 off the 64-bit
    result)."""
    if case["op"] == "quantize":
        return "exact"
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 0.05}
    return {"rel": 5e-6, "max": 2e-4}


# ---- the same in 64 bits -------------------------------------------------------------

def exact(case, seed):
    op = case["op"]
    if op == "quantize":
        return None
    r = _inputs(case, seed)
    x = r["x"].double()
    if op == "int8":
        K, N = case["K"], case["N"]
        g = torch.arange(K * N, device="cuda") // BLOCK
        w = (r["q"].double() * r["s"].double()[g]).view(K, N)
        return x @ w
    if op in ("moe", "grouped"):
        out = torch.zeros(x.shape[0], case["N"], dtype=torch.float64, device="cuda")
        at = 0
        for e, c in enumerate(r["counts"].tolist()):
            if c:
                w = r["w"][e].double() if op == "grouped" else \
                    _unpack4(*r["planes"][e], case["K"] * case["N"]).view(case["K"], case["N"])
                out[at:at + c] = x[at:at + c] @ w
            at += c
        return out
    if op == "step":
        def product(a, i):
            K, N = _matrices(case)[i]
            return a @ _unpack4(*r["planes"][i], K * N).view(K, N)

        def norm(a, gain):
            return a * torch.rsqrt(a.square().mean(-1, keepdim=True) + EPS) * gain.double()

        n1 = norm(x, r["gain"][0])
        o = product(product(n1, 0), 3)
        n2 = norm(o, r["gain"][1])
        gate = product(n2, 4)
        h = gate / (1 + torch.exp(-gate)) * product(n2, 5)
        out = [product(n1, 1), product(n1, 2), o, h, product(h, 6)]
        return [t.view(-1) for t in out] if case["M"] == 1 else out
    K, N = case["K"], case["N"]
    out = x @ _unpack4(*r["planes"][0], K * N).view(K, N)
    if case.get("bias"):
        out = out + r["bias"].double()
    return out.view(-1) if op == "matvec" else out
