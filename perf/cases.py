"""Performance cases of the quantized-matmul path: what a program that serves a model through this
framework calls, over the range of sizes, token counts and weight types it meets.

Kinds of case:

  proj     one dense projection of `tokens` tokens: a GEMV for up to 8 tokens, a GEMM above that
  ffn      a dense SwiGLU FFN block (gate, up, SwiGLU, down), the same split by token count
  experts  the routed experts of one MoE layer: one fused FFN for one token, the several-token form
           up to 16, the grouped GEMM above that
  layer    a whole MoE layer: router, routing on the host, shared expert, routed experts, sum

Weights are random blocks in GGUF layout whose scales give a weight spread of about 0.02, as in a
trained model, activations N(0,1) as behind a norm; routes are top-k draws from a Zipf(1.1) popularity.
Everything runs on the default stream, on torch's device memory.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "glm-ssd_amd"))

import glmssd as G  # noqa: E402
from glmssd.moe import MoeLayer  # noqa: E402

GEMV_MAX = 8      # tokens a GEMV call takes
TOKENS_MAX = 16   # tokens that run as one-token FFNs, in calls of up to 32 (token, expert) pairs
PAIRS_MAX = 32

# type: id, elements and bytes of a block, byte offsets of its f16 scales and their size
TYPES = {
    "f32": (0, 1, 4, ()), "f16": (1, 1, 2, ()),
    "q8_0": (8, 32, 34, ((0, 3e-4),)),
    "q4_k": (12, 256, 144, ((0, 9e-5), (2, 6.8e-4))),
    "q5_k": (13, 256, 176, ((0, 4.5e-5), (2, 6.8e-4))),
    "q6_k": (14, 256, 210, ((208, 1.5e-5),)),
    "iq2_xxs": (16, 256, 66, ((0, 5e-4),)),
    "iq3_xxs": (18, 256, 98, ((0, 1.3e-4),)),
}


def listed():
    return [
        # the smallest call of a decode step: an attention projection of one token
        {"name": "proj_decode", "kind": "proj", "type": "q8_0", "K": 4096, "rows": 4096, "tokens": 1},
        # a dense layer's FFN: one decoded token, a batch of speculated tokens, a ragged short prompt,
        # a prompt chunk
        {"name": "ffn_decode", "kind": "ffn", "type": "q4_k", "type_down": "q6_k", "n_embd": 4096, "n_ff": 12288, "tokens": 1},
        {"name": "ffn_verify", "kind": "ffn", "type": "q4_k", "type_down": "q6_k", "n_embd": 4096, "n_ff": 12288, "tokens": 5},
        {"name": "ffn_short", "kind": "ffn", "type": "q4_k", "type_down": "q6_k", "n_embd": 4096, "n_ff": 12288, "tokens": 77},
        {"name": "ffn_prompt", "kind": "ffn", "type": "q4_k", "type_down": "q6_k", "n_embd": 4096, "n_ff": 12288, "tokens": 512},
        # the output head of one decoded token: the largest single matrix
        {"name": "head_decode", "kind": "proj", "type": "q6_k", "K": 4096, "rows": 262144, "tokens": 1},
        # one decoded token through the routed experts of four layers (8 of 288 experts each)
        {"name": "experts_decode", "kind": "experts", "type": "iq2_xxs", "type_down": "iq2_xxs", "n_embd": 4096, "n_ff": 1536,
         "n_exp": 288, "top": 8, "tokens": 1, "layers": 4},
        # speculated tokens verified together
        {"name": "experts_verify", "kind": "experts", "type": "iq2_xxs", "type_down": "iq2_xxs", "n_embd": 4096, "n_ff": 1536,
         "n_exp": 288, "top": 8, "tokens": 4, "layers": 1},
        # a ragged short prompt over the mixed expert types and the wider experts of the target model
        {"name": "experts_short", "kind": "experts", "type": "iq2_xxs", "type_down": "iq3_xxs", "n_embd": 4096, "n_ff": 2048,
         "n_exp": 96, "top": 8, "tokens": 37, "layers": 1},
        # a prompt chunk, and a long one: the largest call
        {"name": "experts_prompt", "kind": "experts", "type": "iq2_xxs", "type_down": "iq2_xxs", "n_embd": 4096, "n_ff": 1536,
         "n_exp": 288, "top": 8, "tokens": 512, "layers": 1},
        {"name": "experts_long", "kind": "experts", "type": "iq2_xxs", "type_down": "iq2_xxs", "n_embd": 4096, "n_ff": 1536,
         "n_exp": 288, "top": 8, "tokens": 2048, "layers": 1},
        # a whole MoE layer, host routing included
        {"name": "layer_verify", "kind": "layer", "type": "iq2_xxs", "type_down": "iq3_xxs", "n_embd": 2048, "n_ff": 512,
         "n_ff_shared": 1024, "n_exp": 32, "top": 8, "tokens": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _by(n, step):
    return max(step, int(round(n / step)) * step)


def draw(rng):
    """One more case: row lengths in whole super-blocks, row and token counts of any value."""
    dense = ("q8_0", "q4_k", "q5_k", "q6_k")
    iq = ("iq2_xxs", "iq3_xxs")
    most = max(work(c)["flops"] for c in listed())
    while True:
        kind = rng.choice(["proj", "proj", "ffn", "ffn", "experts", "experts", "experts", "head", "layer"])
        if kind == "proj":
            c = {"kind": "proj", "type": rng.choice(dense + iq + ("f16",)), "K": _by(_log(rng, 512, 12288), 256),
                 "rows": _log(rng, 256, 16384), "tokens": _log(rng, 1, 512)}
        elif kind == "head":
            c = {"kind": "proj", "type": rng.choice(dense), "K": _by(_log(rng, 2048, 4096), 256),
                 "rows": _log(rng, 32768, 262144), "tokens": rng.choice([1, 1, 2, 4, 5, 8])}
        elif kind == "ffn":
            c = {"kind": "ffn", "type": rng.choice(dense), "type_down": rng.choice(dense),
                 "n_embd": _by(_log(rng, 1024, 6144), 256), "n_ff": _by(_log(rng, 1024, 12288), 256), "tokens": _log(rng, 1, 512)}
        elif kind == "experts":
            t = _log(rng, 1, 2048)
            c = {"kind": "experts", "type": rng.choice(iq), "type_down": rng.choice(iq), "n_embd": _by(_log(rng, 1024, 4096), 256),
                 "n_ff": _by(_log(rng, 512, 2048), 256), "n_exp": rng.choice([32, 64, 96, 288]), "top": rng.choice([4, 6, 8, 8]),
                 "tokens": t, "layers": rng.randint(1, 4) if t == 1 else 1}
        else:
            c = {"kind": "layer", "type": "iq2_xxs", "type_down": rng.choice(iq), "n_embd": 256 * rng.randint(4, 8),
                 "n_ff": 256 * rng.randint(2, 4), "n_ff_shared": 256 * rng.randint(2, 6), "n_exp": rng.choice([24, 32]),
                 "top": rng.choice([4, 8]), "tokens": _log(rng, 1, 64)}
        if work(c)["flops"] <= most:
            return c


# ---- sizes ------------------------------------------------------------------------------------
def _row_bytes(ty, K):
    return K // TYPES[ty][1] * TYPES[ty][2]


def _routes(case, seed, layer=0):
    """Experts [tokens][top] drawn without replacement from a Zipf(1.1) popularity over a random order
    of the experts (Gumbel top-k), and combine weights (softmax of N(0,1))."""
    r = np.random.default_rng([seed, 77, layer])
    n, t, k = case["n_exp"], case["tokens"], case["top"]
    score = -1.1 * np.log(np.arange(1, n + 1))[r.permutation(n)] + r.gumbel(size=(t, n))
    experts = np.argsort(-score, axis=1)[:, :k].astype(np.int32)
    w = np.exp(r.standard_normal((t, k)))
    return experts, (w / w.sum(1, keepdims=True)).astype(np.float32)


def _used(case):
    """Distinct experts one layer's call reads (of one draw of routes)."""
    return len(np.unique(_routes(case, 0)[0]))


def work(case):
    t = case["tokens"]
    if case["kind"] == "proj":
        w = case["rows"] * _row_bytes(case["type"], case["K"])
        return {"bytes": w + 4 * t * (case["K"] + case["rows"]), "flops": 2 * t * case["K"] * case["rows"]}
    n, f = case["n_embd"], case["n_ff"]
    up, down = f * _row_bytes(case["type"], n), n * _row_bytes(case["type_down"], f)
    if case["kind"] == "ffn":
        return {"bytes": 2 * up + down + 8 * t * n, "flops": 6 * t * n * f}
    if case["kind"] == "experts":
        one = min(case["n_exp"], _used(case)) * (2 * up + down) + 8 * t * n
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 6 * t * case["top"] * n * f}
    s = case["n_ff_shared"]
    fixed = 3 * n * _row_bytes("q6_k", 256) // 256 * s + 4 * n * case["n_exp"] + 8 * t * n
    used = min(case["n_exp"], t * case["top"])
    return {"bytes": fixed + used * (2 * up + down), "flops": 2 * t * n * (3 * s + case["n_exp"] + 3 * case["top"] * f)}


# ---- inputs -----------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _matrix(g, ty, rows, K):
    """`rows` rows of `K` weights in GGUF layout, as bytes."""
    _, be, bb, halves = TYPES[ty]
    if ty in ("f32", "f16"):
        w = torch.randn(rows * K, generator=g, device="cuda") * 0.02
        return (w.half() if ty == "f16" else w).view(torch.uint8)
    n = rows * K // be
    raw = torch.randint(-2 ** 31, 2 ** 31, (n * bb // 4 + 1,), generator=g, device="cuda", dtype=torch.int32).view(torch.uint8)[: n * bb]
    blk = raw.view(n, bb)
    for off, size in halves:
        d = (torch.rand(n, generator=g, device="cuda") + 0.5) * size
        blk[:, off:off + 2] = d.half().view(torch.uint8).view(n, 2)
    return raw


def _gemm_work(shapes, t):
    need = max(G.ops.gemm_workspace(K, rows, t) for K, rows in shapes) if t > GEMV_MAX else 0
    return torch.empty(max(need, 16), dtype=torch.uint8, device="cuda"), need


def _group(experts, w, n_exp):
    """(token, weight) pairs sorted by expert, tokens in order within one: offsets, tokens, weights."""
    t, k = experts.shape
    e = experts.reshape(-1)
    order = np.argsort(e, kind="stable")
    offs = np.zeros(n_exp + 1, np.int32)
    offs[1:] = np.cumsum(np.bincount(e, minlength=n_exp))
    return offs, (order // k).astype(np.int32), w.reshape(-1)[order]


def _prepare_experts(case, g, seed):
    n, f, t, k, ne, layers = (case[x] for x in ("n_embd", "n_ff", "tokens", "top", "n_exp", "layers"))
    s = {"x": torch.randn(t, n, generator=g, device="cuda"), "y": torch.zeros(layers, t, n, device="cuda"), "layers": []}
    for li in range(layers):
        experts, w = _routes(case, seed, li)
        # the resident experts that this call can reach, in one allocation per matrix kind
        ids = np.unique(experts)
        up, down = f * _row_bytes(case["type"], n), n * _row_bytes(case["type_down"], f)
        gate, upm, dn = (_matrix(g, ty, len(ids) * r, K) for ty, r, K in
                         ((case["type"], f, n), (case["type"], f, n), (case["type_down"], n, f)))
        at = {int(e): i for i, e in enumerate(ids)}
        ptr = lambda e: (gate.data_ptr() + at[e] * up, upm.data_ptr() + at[e] * up, dn.data_ptr() + at[e] * down)  # noqa: E731
        L = {"gate": gate, "up": upm, "down": dn, "ids": ids, "experts": experts, "w": w}
        if t <= TOKENS_MAX:
            L["batches"] = []
            for row, wt in zip(experts.tolist(), w.tolist()):
                b = G.MoeBatch()
                b.n = k
                for j, e in enumerate(row):
                    b.gate[j], b.up[j], b.down[j] = ptr(e)
                    b.w[0][j] = wt[j]
                L["batches"].append(b)
            L["h"] = torch.empty(min(t, max(1, PAIRS_MAX // k)) * k * f, device="cuda")
        else:
            tab = np.zeros((ne, 3), np.int64)
            for e in at:
                tab[e] = ptr(e)
            offs, idx, wp = _group(experts, w, ne)
            L["table"], L["offs"], L["idx"], L["wp"] = (torch.from_numpy(a).cuda() for a in (tab, offs, idx, wp))
            L["bytes"] = G.ops.moe_grouped_workspace(t, t * k, n, f)
            L["work"] = torch.empty(L["bytes"], dtype=torch.uint8, device="cuda")
        s["layers"].append(L)
    return s


def _prepare_layer(case, g):
    n, f, sh, ne = case["n_embd"], case["n_ff"], case["n_ff_shared"], case["n_exp"]
    host = lambda ty, rows, K: _matrix(g, ty, rows, K).cpu().numpy()  # noqa: E731
    router = (torch.randn(ne, n, generator=g, device="cuda") * 0.03).cpu().numpy()
    bias = (torch.randn(ne, generator=g, device="cuda") * 0.1).cpu().numpy()
    shared = [host("q6_k", sh, n), host("q6_k", sh, n), host("q6_k", n, sh)]
    experts = [(host(case["type"], f, n), host(case["type"], f, n), host(case["type_down"], n, f)) for _ in range(ne)]
    m = MoeLayer(router.view(np.uint8).reshape(-1), bias, shared, experts, n, f, TYPES[case["type"]][0],
                 TYPES[case["type_down"]][0], k=case["top"], weights_norm=True, weights_scale=2.5, n_ff_shexp=sh,
                 deterministic=False)
    t = case["tokens"]
    return {"layer": m, "host": (router, bias, shared, experts), "x": torch.randn(t, n, generator=g, device="cuda"),
            "out": torch.empty(t, n, device="cuda")}


_CALLED = set()   # the cases called once in this process


def prepare(case, seed):
    """Inputs, weights, routes and workspaces. The first time in a process it also makes one call: the
    library finds a kernel among its code objects at the kernel's first use, and the lookup can leave
    hipErrorNotFound as the runtime's last error, which torch would raise at its own next launch."""
    s = _prepare(case, seed)
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _CALLED:
        run(s)
        torch.cuda.synchronize()
        G.lib().hipGetLastError()
        _CALLED.add(key)
    return s


def _prepare(case, seed):
    g = _gen(seed)
    t = case["tokens"]
    if case["kind"] == "experts":
        s = _prepare_experts(case, g, seed)
    elif case["kind"] == "layer":
        s = _prepare_layer(case, g)
    elif case["kind"] == "proj":
        K, rows = case["K"], case["rows"]
        s = {"w": _matrix(g, case["type"], rows, K), "x": torch.randn(t, K, generator=g, device="cuda"),
             "y": torch.empty(t, rows, device="cuda")}
        s["work"], s["bytes"] = _gemm_work([(K, rows)], t)
    else:
        n, f = case["n_embd"], case["n_ff"]
        s = {"gate": _matrix(g, case["type"], f, n), "up": _matrix(g, case["type"], f, n),
             "down": _matrix(g, case["type_down"], n, f), "x": torch.randn(t, n, generator=g, device="cuda")}
        s["g"], s["u"], s["y"] = (torch.empty(t, m, device="cuda") for m in (f, f, n))
        s["work"], s["bytes"] = _gemm_work([(n, f), (f, n)], t)
    s["case"] = case
    return s


# ---- one pass ---------------------------------------------------------------------------------
def _mm(s, ty, w, K, rows, x, y, t):
    """The engine's split: a GEMV for up to 8 tokens, a GEMM with the caller's workspace above."""
    tid = TYPES[ty][0]
    if t <= GEMV_MAX:
        G.ops.gemv(tid, w.data_ptr(), _row_bytes(ty, K), K, rows, x.data_ptr(), K, y.data_ptr(), rows, t)
    else:
        G.ops.gemm_ex(tid, w.data_ptr(), _row_bytes(ty, K), K, rows, x.data_ptr(), K, y.data_ptr(), rows, t,
                      work=s["work"].data_ptr() if s["bytes"] else None, work_bytes=s["bytes"])


def _run_experts(s, case):
    n, f, t, k = (case[x] for x in ("n_embd", "n_ff", "tokens", "top"))
    ty, td = TYPES[case["type"]][0], TYPES[case["type_down"]][0]
    rg, rd = _row_bytes(case["type"], n), _row_bytes(case["type_down"], f)
    x = s["x"].data_ptr()
    s["y"].zero_()   # the experts' outputs are added up
    for li, L in enumerate(s["layers"]):
        y = s["y"].data_ptr() + 4 * li * t * n
        if t == 1:
            G.ops.moe_ffn(ty, td, L["batches"][0], 1, rg, n, f, rd, x, L["h"].data_ptr(), y)
        elif t <= TOKENS_MAX:
            per = max(1, PAIRS_MAX // k)
            for t0 in range(0, t, per):
                G.ops.moe_ffn_tokens(ty, td, L["batches"][t0:t0 + per], rg, n, f, rd, x + 4 * n * t0, L["h"].data_ptr(),
                                     y + 4 * n * t0)
        else:
            G.ops.moe_grouped(ty, td, L["table"].data_ptr(), case["n_exp"], L["offs"].data_ptr(), L["idx"].data_ptr(),
                              L["wp"].data_ptr(), t * k, t, rg, n, f, rd, x, y, 0.0, L["work"].data_ptr(), L["bytes"])
    return s["y"]


def run(s):
    case = s["case"]
    t = case["tokens"]
    if case["kind"] == "proj":
        _mm(s, case["type"], s["w"], case["K"], case["rows"], s["x"], s["y"], t)
        return s["y"]
    if case["kind"] == "ffn":
        n, f = case["n_embd"], case["n_ff"]
        _mm(s, case["type"], s["gate"], n, f, s["x"], s["g"], t)
        _mm(s, case["type"], s["up"], n, f, s["x"], s["u"], t)
        G.ops.swiglu(s["g"].data_ptr(), s["u"].data_ptr(), s["g"].data_ptr(), t * f)
        _mm(s, case["type_down"], s["down"], f, n, s["g"], s["y"], t)
        return s["y"]
    if case["kind"] == "experts":
        return _run_experts(s, case)
    s["layer"].forward(s["x"].data_ptr(), s["out"].data_ptr(), t)
    return s["out"]


# ---- tolerances -------------------------------------------------------------------------------
def tolerance(case):
    """Measured against the same path with its 32-bit sums in another order. One matrix: the sums alone.
    Two in a row with q8_1 between (decode sizes): a sum that moves can move one hidden value to the next
    of its 255 steps, 0.02 over the root of the hidden values in the output, stated fivefold. With f16
    between: 1.5e-5 seen, and 7e-5 with the inputs moved by a part in 1e7."""
    t, kind = case["tokens"], case["kind"]
    if kind == "proj":
        return {"rel": 1e-5}
    if t <= (GEMV_MAX if kind == "ffn" else TOKENS_MAX):
        hidden = {"ffn": case["n_ff"], "experts": case["n_ff"] * case.get("top", 1), "layer": case.get("n_ff_shared", 1)}[kind]
        return {"rel": 0.1 / math.sqrt(hidden)}
    return {"rel": 1e-4}


# ---- the same in 64 bits, in plain torch --------------------------------------------------------
# IQ2_XXS grid: 16 bits an entry, 2 bits a value (0, 1, 2 for 8, 25, 43), the first value lowest.
# IQ3_XXS grid: 12 bits an entry, 3 bits a value (0..6 for 4 + 8 v, 7 for 62), the first value lowest.
_IQ2_XXS_GRID = (
    "0000000200050008000a00110014002000220028002a00410044005000580061006400800082008a00a20101010401100115014001840198"
    "020002020222028204010404041004210424044004420448046004810484049004a405000502050805200546056905800591060906100640"
    "068406a40800080508080814082808410844085008520888090409400a020a14100110041010102110401060108410901095110011081120"
    "1150115a1180122412451400140814201425144914801518156216001616180118041810184018811900190519a01a5120002002200a2044"
    "20612080208221292148220022022401240424102440245625002541256426902808282028942a4440014004401040184021402440404048"
    "4056406040814084409041004120416141804185420142104248425642684400440844204480449945124524460048014804481048404845"
    "49004958496149824a454a9050005008501150195020508050885104514251a4529154905492550a56015654580058115819586459405a08"
    "6004601060406068610061556218626064006405651065126584684280008002800a80418082810481188140821184018404841084158440"
    "8460850085468594860986408660880289048a11900490109024904090a1911691809245940094229444955198819920a002a050a085a109"
    "a200a418a850a904"
)
_IQ3_XXS_GRID = (
    "00000200400900b00f01001201902203b03d04104304804a05105505805a06106c07808008208408909009209909b09f0a90af0bd0c10c70"
    "c80ca0d50f810b11f12412f13b13d14114715a16a19d1b41c81cc1ce1e31f120120320820a21121321821a21c22722824024224925025228"
    "128328828a2912982ba2c02c22d02d92e62f63013053283503543663793853d23e040040240940b41041241641942244144344544844a451"
    "45847347747848048248948f49049249f4a04ad4c14c84cc4f84fc51d52b54355756157c5c15c35ce5e560160860a61161362863563a6406"
    "426506596646666816836886956aa6ba6c96db71872773a74074675276d78c79e7b37db7f080480f81d81f82b82f87c89089f8a08b08b68c"
    "78e59049299349559639789c59c89ca9d8a0aa21a38a40a46a56a6da8ca9aabaac2aebb08b13b17b3ab42b59ba8bd4be2c14c24c26c34c51"
    "c71c8fcb4cd8cded24d45d6ad9bdc3dd1e03e05e07e08e1ae2ae56e60e8aea5eaaec0ecdedbef0f11f21f40f42f54f98"
)

def _grid(text, digits, values, bits, lut):
    code = torch.tensor([int(text[i:i + digits], 16) for i in range(0, len(text), digits)], device="cuda")
    return torch.tensor(lut, dtype=torch.float64, device="cuda")[(code[:, None] >> (bits * torch.arange(values, device="cuda"))) & (2 ** bits - 1)]


def _half(b, off):
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _scale_min(b):
    """Six-bit scales and minima of the eight sub-blocks, packed in the bytes 4..15."""
    p = b[:, 4:16].int()
    lo, hi = p[:, 0:4], p[:, 4:8]
    sc = torch.cat([lo & 63, (p[:, 8:12] & 15) | ((lo >> 6) << 4)], 1)
    mn = torch.cat([hi & 63, (p[:, 8:12] >> 4) | ((hi >> 6) << 4)], 1)
    return sc.double(), mn.double()


def _signs(idx):
    """+-1 of eight values from a seven-bit index; the eighth bit makes the parity even."""
    bits = (idx[..., None] >> torch.arange(7, device=idx.device)) & 1
    bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)
    return 1.0 - 2.0 * bits.double()


def _decode(ty, raw):
    """The weights that the bytes of whole blocks hold, in 64 bits."""
    if ty == "f32":
        return raw.view(torch.float32).double()
    if ty == "f16":
        return raw.view(torch.float16).double()
    b = raw.view(-1, TYPES[ty][2])
    n = b.shape[0]
    if ty == "q8_0":
        return (_half(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    if ty in ("q4_k", "q5_k"):
        sc, mn = _scale_min(b)
        qs = b[:, 16:144] if ty == "q4_k" else b[:, 48:176]
        qs = qs.reshape(n, 4, 1, 32).int()
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        if ty == "q5_k":
            q = q + (((b[:, 16:48].int()[:, None, :] >> torch.arange(8, device=b.device)[None, :, None]) & 1) << 4)
        return ((_half(b, 0) * sc)[:, :, None] * q.double() - (_half(b, 2) * mn)[:, :, None]).reshape(-1)
    if ty == "q6_k":
        ql = b[:, 0:128].reshape(n, 2, 2, 32).int()            # [half][low or high 32 bytes]
        qh = b[:, 128:192].reshape(n, 2, 1, 32).int()
        lo = torch.cat([ql & 15, ql >> 4], 2)                  # the four 32-value quarters of a half
        q = (lo | (((qh >> (2 * torch.arange(4, device=b.device)).view(1, 1, 4, 1)) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 16, 1)
        return (_half(b, 208)[:, :, None] * sc * q.reshape(n, 16, 16).double()).reshape(-1)
    if ty == "iq2_xxs":
        u = b[:, 2:66].reshape(n, 8, 8).long()
        aux = u[..., 4] | (u[..., 5] << 8) | (u[..., 6] << 16) | (u[..., 7] << 24)
        grid, idx, f = _grid(_IQ2_XXS_GRID, 4, 8, 2, [8.0, 25.0, 43.0, 0.0]), u[..., :4], 0.25
    else:
        u = b[:, 66:98].reshape(n, 8, 4).long()
        aux = u[..., 0] | (u[..., 1] << 8) | (u[..., 2] << 16) | (u[..., 3] << 24)
        grid, idx, f = _grid(_IQ3_XXS_GRID, 3, 4, 3, [4.0, 12.0, 20.0, 28.0, 36.0, 44.0, 52.0, 62.0]), b[:, 2:66].reshape(n, 8, 8).long(), 0.5
    sign = _signs((aux[..., None] >> (7 * torch.arange(4, device=b.device))) & 127)
    scale = _half(b, 0) * (0.5 + (aux >> 28).double()) * f
    return (scale[..., None, None] * grid[idx].reshape(n, 8, 4, 8) * sign).reshape(-1)


def _mm64(ty, raw, K, rows, x):
    """x [t][K] (64 bits) through the matrix, in slices of rows."""
    rb, step = _row_bytes(ty, K), max(1, (1 << 26) // K)
    out = [x @ _decode(ty, raw[r * rb:min(rows, r + step) * rb]).view(-1, K).t() for r in range(0, rows, step)]
    return torch.cat(out, 1)


def _ffn64(types, raws, n, f, x):
    g, u = (_mm64(types[0], r, n, f, x) for r in raws[:2])
    return _mm64(types[1], raws[2], f, n, torch.nn.functional.silu(g) * u)


def exact(case, seed):
    s = _prepare(case, seed)
    x = s["x"].double()
    if case["kind"] == "proj":
        return _mm64(case["type"], s["w"], case["K"], case["rows"], x)
    n, f = case["n_embd"], case["n_ff"]
    types = (case["type"], case["type_down"])
    if case["kind"] == "ffn":
        return _ffn64(types, (s["gate"], s["up"], s["down"]), n, f, x)
    if case["kind"] == "experts":
        out = []
        for L in s["layers"]:
            y = torch.zeros_like(x)
            sizes = [f * _row_bytes(types[0], n)] * 2 + [n * _row_bytes(types[1], f)]
            for i, e in enumerate(L["ids"]):
                tok, rank = np.nonzero(L["experts"] == e)
                tok_d, w = torch.from_numpy(tok).cuda(), torch.from_numpy(L["w"][tok, rank]).cuda().double()
                raws = [L[m][i * b:(i + 1) * b] for m, b in zip(("gate", "up", "down"), sizes)]
                y.index_add_(0, tok_d, w[:, None] * _ffn64(types, raws, n, f, x[tok_d]))
            out.append(y)
        return torch.stack(out)
    router, bias, shared, experts = s["host"]
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    score = torch.sigmoid(x @ dev(router).double().t())
    top = torch.argsort(score + dev(bias).double(), 1, descending=True)[:, :case["top"]]
    w = score.gather(1, top)
    w = 2.5 * w / w.sum(1, keepdim=True)
    out = _ffn64(("q6_k", "q6_k"), [dev(a) for a in shared], n, case["n_ff_shared"], x)
    for e in top.unique().tolist():
        tok, rank = torch.nonzero(top == e, as_tuple=True)
        out.index_add_(0, tok, w[tok, rank][:, None] * _ffn64(types, [dev(a) for a in experts[e]], n, f, x[tok]))
    return out
