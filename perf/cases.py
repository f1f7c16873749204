"""The work that users of this framework have it do, for measurement.

Six kinds of call, each through a public entry point:

  decode    one pruned decode-attention step over caches already in place: the paged q2 / nvfp4 / nf4
            caches and the contiguous reference layouts, from one short sequence, where latency counts,
            to ragged batches of long ones, where the caches' bytes do.  With `layers` above 1 the step
            is that of several layers, each with its own cache, in one HIP graph, as a serving loop
            replays it; otherwise one eager call
  project   K projection + RoPE + per-channel q2 quantize of a prompt (the reference's fused producer)
  append    K projection + RoPE + g32 quantize of the newest token(s) of every sequence into the
            paged cache (the producer of a serving step, `layers` of them in one HIP graph)
  fill      quantize the K and V of a prompt, projected elsewhere, into a paged cache
  quantize  quantize a prompt's K in a reference layout
  dequant   the paged cache as contiguous K and V, for the exact attention of a prompt's next chunk

Inputs are N(0, 1) keys, values and queries with heavy tokens planted per query head (keys at cosine
0.8 with the query, one inside the first probe window), as in the repository's own benchmark: without
them the threshold would keep nearly everything.
"""
import math
import random
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parents[1] / "ffa-speedtest_amd"
for _p in (str(_ROOT), str(_ROOT / "ffa-q2fp8")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

D = 128
PAGE = 64
HEAVY, COS = 16, 0.8
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_FP8 = {"e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}


# ---------------------------------------------------------------------------- the cases
def _decode(name, fmt, B, lo, hi, HQ=32, HKV=8, BS=64, SBS=64, dtype="bf16", layers=1, mean=False):
    return {"name": name, "kind": "decode", "fmt": fmt, "B": B, "lo": lo, "hi": hi, "HQ": HQ, "HKV": HKV, "BS": BS,
            "SBS": SBS, "dtype": dtype, "layers": layers, "mean": mean}


def listed():
    return [
        # one short conversation: two launches a layer, each far too small to fill the chip
        _decode("decode_b1_2k", "q2", 1, 2000, 2000, layers=16),
        # one long context: the benchmark's headline step, 16 layers of it (more than the last-level cache holds)
        _decode("decode_b1_32k", "q2", 1, 32768, 32768, layers=16),
        # a serving batch of long, ragged contexts, called eagerly
        _decode("decode_b16_ragged", "q2", 16, 8192, 65536),
        # the reference's own layout (per-channel scales, contiguous, e5m2 residual), BS = 128 as its default
        _decode("decode_reference_b2", "q2c", 2, 30001, 30001, BS=128, SBS=128, layers=4),
        # a ragged batch on the 4-bit cache of the benchmark's config 4
        _decode("decode_nf4_b8_ragged", "nf4", 8, 8192, 65536),
        # 64 query heads over 8 KV heads (groups of 8): the two-pass decode
        _decode("decode_group8_b8", "q2", 8, 3000, 16000, HQ=64),
        # the fused producer on a prompt of 4K tokens, 4096 -> 8 x 128
        {"name": "project_4k", "kind": "project", "B": 1, "T": 4096, "H": 4096, "HKV": 8, "D": 128, "dtype": "bf16",
         "cs": "fp32", "bias": False},
        # one new token of each of 64 sequences, projected and appended in each of 16 layers
        {"name": "append_b64", "kind": "append", "B": 64, "Tn": 1, "H": 4096, "HKV": 8, "dtype": "bf16", "layers": 16},
        # a 16K prompt's K and V into the paged q2 cache
        {"name": "fill_q2_16k", "kind": "fill", "fmt": "q2", "B": 1, "T": 16384, "HKV": 8, "dtype": "bf16"},
        # a 32K prompt in the reference layout
        {"name": "quantize_q2_32k", "kind": "quantize", "fmt": "q2", "B": 1, "T": 32768, "HKV": 8, "D": 128,
         "dtype": "bf16", "res": "e5m2"},
        # nvfp4 in the reference layout, an odd length over two sequences
        {"name": "quantize_nvfp4_2x10k", "kind": "quantize", "fmt": "nvfp4", "B": 2, "T": 10001, "HKV": 8, "D": 128,
         "dtype": "bf16", "res": "e5m2"},
        # the cache of four ragged sequences as contiguous keys and values
        {"name": "dequant_b4_8k", "kind": "dequant", "B": 4, "lo": 3000, "hi": 8000, "HKV": 8, "out": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "project", "append", "fill", "quantize", "dequant"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode":
        fmt = rng.choice(["q2", "q2", "q2c", "nvfp4", "nf4", "fp8"])
        B = _log(rng, 1, 16)
        hi = _log(rng, 1000, 65536 if B * 65536 <= 600000 else 600000 // B)
        lo = rng.randint(max(1, hi // 4), hi) if fmt in ("q2", "nvfp4", "nf4") else hi
        G = rng.choice([4, 4, 4, 2, 8])
        HKV = rng.choice([8, 8, 4])
        BS = rng.choice([64, 64, 128])
        case = _decode("", fmt, B, lo, hi, HQ=G * HKV, HKV=HKV, BS=BS, SBS=rng.choice([BS, 64]), dtype=dtype,
                       layers=max(1, min(16, 300000 // (B * hi))), mean=fmt == "q2c" and rng.random() < 0.5)
        del case["name"]
        return case
    if kind == "project":
        H = rng.choice([1024, 2048, 4096])
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "T": _log(rng, 16, 4096), "H": H, "HKV": rng.choice([4, 8]),
                "D": rng.choice([64, 128, 128]), "dtype": dtype, "cs": rng.choice(["fp32", dtype]),
                "bias": rng.random() < 0.3}
    if kind == "append":
        return {"kind": kind, "B": _log(rng, 1, 64), "Tn": rng.choice([1, 1, 1, 4]), "H": rng.choice([2048, 4096]),
                "HKV": rng.choice([4, 8]), "dtype": dtype, "layers": 16}
    if kind == "fill":
        B = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "fmt": rng.choice(["q2", "q2", "nvfp4", "nf4"]), "B": B, "T": _log(rng, 64, 32768 // B),
                "HKV": rng.choice([4, 8]), "dtype": rng.choice([dtype, "fp32"])}
    if kind == "quantize":
        B = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "fmt": rng.choice(["q2", "q2", "fp8", "nvfp4", "nf4"]), "B": B,
                "T": _log(rng, 64, 32768 // B), "HKV": rng.choice([4, 8]), "D": rng.choice([64, 128, 128]),
                "dtype": rng.choice([dtype, "fp32"]), "res": rng.choice(["e5m2", "e4m3"])}
    hi = _log(rng, 100, 8000)
    return {"kind": kind, "B": rng.choice([1, 2, 4]), "lo": rng.randint(max(1, hi // 2), hi), "hi": hi,
            "HKV": rng.choice([4, 8]), "out": rng.choice(["bf16", "fp16", "fp32"])}


def _lens(case):
    """Ragged lengths in [lo, hi] (the longest first), the same for every seed."""
    r = random.Random(case["B"] * 1000003 + case["hi"])
    return [case["hi"]] + [r.randint(case["lo"], case["hi"]) for _ in range(case["B"] - 1)]


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _sequence(q, T, HKV, g, dtype):
    """k, v [T, HKV, D] of one sequence; q [HQ, D] f32.  Heavy keys per query head, one of them in tokens 0..15."""
    G = q.shape[0] // HKV
    k, v = _randn(g, T, HKV, D), _randn(g, T, HKV, D).to(dtype)
    n = min(HEAVY - 1, max(T - 16, 0) // G)
    if T > 16:
        first = torch.rand((HKV, 16), generator=g, device="cuda").argsort(1)[:, :G]
        rest = torch.randperm(T - 16, generator=g, device="cuda")[:G * n]
        shift = torch.arange(HKV, device="cuda")[:, None] * 977
        rest = (16 + (rest[None] + shift) % (T - 16)).view(HKV, G, n)
        pos = torch.cat([first.view(HKV, G, 1), rest], 2)  # distinct within a head
        head = torch.arange(HKV, device="cuda").view(HKV, 1, 1).expand_as(pos)
        qh = (q / q.norm(dim=-1, keepdim=True)).view(HKV, G, 1, D)
        u = _randn(g, *pos.shape, D)
        u = u - (u * qh).sum(-1, keepdim=True) * qh
        u = u / u.norm(dim=-1, keepdim=True)
        norm = k[pos, head].norm(dim=-1, keepdim=True)
        k[pos, head] = norm * (COS * qh + math.sqrt(1 - COS * COS) * u)
    return k.to(dtype), v


def _tables(lens, g):
    """A block table of randomly ordered pages for each length, and how many pages there are."""
    npg = [-(-t // PAGE) for t in lens]
    perm = torch.randperm(sum(npg), generator=g, device="cuda").to(torch.int32)
    bt = torch.zeros((len(lens), max(npg)), dtype=torch.int32, device="cuda")
    o = 0
    for b, n in enumerate(npg):
        bt[b, :n] = perm[o:o + n]
        o += n
    return bt, sum(npg)


def _decode_inputs(case, seed):
    """q [B, HQ, D] and, one after the other, k, v [T_b, HKV, D] of every sequence."""
    dt = _DT[case["dtype"]]
    g = _gen(seed)
    q = _randn(g, case["B"], case["HQ"], D).to(dt)
    return q, [lambda b=b, T=T: _sequence(q[b].float(), T, case["HKV"], _gen(seed * 4099 + 17 * b + 1), dt)
               for b, T in enumerate(_lens(case))]


def _project_inputs(case, seed, tokens):
    """h [B, tokens, H], w_k [HKV * D, H], bias or None."""
    dt, g = _DT[case["dtype"]], _gen(seed)
    d = case.get("D", D)
    h = _randn(g, case["B"], tokens, case["H"]).to(dt)
    w = (_randn(g, case["HKV"] * d, case["H"]) * 0.02).to(dt)
    return h, w, (_randn(g, case["HKV"] * d) * 0.1).to(dt) if case.get("bias") else None


def _angles(pos, d, base=500000.0):
    inv = 1.0 / (base ** (torch.arange(0, d, 2, dtype=torch.float32, device="cuda") / d))
    a = pos.float()[..., None] * inv
    a = torch.cat([a, a], -1)
    return a.cos(), a.sin()


def _kv_inputs(case, seed):
    """k, v [B, T, HKV, D] of a prompt: N(0, 1) with four larger channels, as rotated keys have."""
    g, d = _gen(seed), case.get("D", D)
    k = _randn(g, case["B"], case["T"], case["HKV"], d)
    k[..., torch.randperm(d, generator=g, device="cuda")[:4]] *= 6.0
    dt = _DT[case["dtype"]]
    v = _randn(g, case["B"], case["T"], case["HKV"], d).to(dt) if case["kind"] == "fill" else None
    return k.to(dt), v


def _append_pos(case, seed):
    """Position of the first new token of each sequence, inside a table of two pages each."""
    r = random.Random(seed)
    return [r.randint(0, 2 * PAGE - case["Tn"]) for _ in range(case["B"])]


# ---------------------------------------------------------------------------- prepare and run
class _Replay:
    """A captured graph with what it reads (the steps hold their inputs) and its outputs."""

    def __init__(self, graph, steps, out):
        self.graph, self.steps, self.out = graph, steps, out

    def __call__(self):
        self.graph.replay()
        return self.out


def _captured(steps):
    """The layers' steps as one HIP graph, as serving loops launch it."""
    def step():
        return [s() for s in steps]

    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return _Replay(graph, steps, out)


def _layer_seed(seed, layer):
    return seed + 7919 * layer


def _decode_layer(case, seed):
    from ffa_mi355x.decode import DecodeWorkspace

    q, seqs = _decode_inputs(case, seed)
    lens, HKV, BS, SBS, fmt = _lens(case), case["HKV"], case["BS"], case["SBS"], case["fmt"]
    T, B, HQ = max(lens), case["B"], case["HQ"]
    ws = DecodeWorkspace(B, HQ, HKV, T, BS, SBS, q.device, q.dtype)
    if fmt in ("q2", "nvfp4", "nf4"):
        from ffa_mi355x.paged import PagedQ2Cache
        from ffa_mi355x.paged_kfmt import PagedKfmtCache

        bt, pages = _tables(lens, _gen(seed + 1))
        cache = PagedQ2Cache(pages, HKV, "cuda") if fmt == "q2" else PagedKfmtCache(fmt, pages, HKV, "cuda")
        zero = torch.zeros(1, dtype=torch.int32, device="cuda")
        for b, make in enumerate(seqs):
            k, v = make()
            cache.append(k[None], v[None], zero, bt[b:b + 1])
        seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")

        def step():
            cache.decode(q, bt, seq_lens, T=T, BS=BS, SBS=SBS, workspace=ws)
            return {"o": ws.o, "mask": ws.mask_buf, "threshold": ws.threshold_buf}
    else:
        kv = [make() for make in seqs]
        k, v = torch.stack([x[0] for x in kv]), torch.stack([x[1] for x in kv])
        if fmt == "fp8":
            from ffa_mi355x.dropins import _load
            from ffa_mi355x.kfmt_quant import quantize_fp8fp8

            call = _load("perf_fp8_decode", _ROOT / "ffa-fp8fp8" / "attn_kernel" /
                         "attn_kernel_v1210_fused_bsz_fp8fp8.py").attn_forward_decode_fp8fp8
            base, res = quantize_fp8fp8(k, torch.float8_e5m2)
            q1 = q[:, None].contiguous()

            def step():
                call(q1, base, v, k_residual=res, BS=BS, SBS=SBS, workspace=ws)
                return {"o": ws.o, "mask": ws.mask_buf, "threshold": ws.threshold_buf}
        else:
            from ffa_mi355x.dropins import _load, q2fp8_dropin
            from ffa_mi355x.quant import quantize_per_channel

            mod = q2fp8_dropin() if not case["mean"] else _load(
                "perf_meanv_decode",
                _ROOT / "ffa-q2fp8-meanv" / "attn_kernel" / "attn_kernel_v1210_meanv_bsz_q2fp8.py")
            kq, ks, kz, kr = quantize_per_channel(k, torch.float8_e5m2)
            q1 = q[:, None].contiguous()

            def step():
                mod.attn_forward_decode_quantized(q1, kq, ks, kz, v, k_residual=kr, BS=BS, SBS=SBS, workspace=ws)
                return {"o": ws.o, "mask": ws.mask_buf, "threshold": ws.threshold_buf}
    return step


def _prepare_decode(case, seed):
    steps = [_decode_layer(case, _layer_seed(seed, layer)) for layer in range(case["layers"])]
    return _captured(steps) if len(steps) > 1 else steps[0]


def _append_inputs(case, seed):
    """h, w_k and v of every layer; positions, their angles, and the block table [layers * B, 2] of one pool."""
    B, Tn, L = case["B"], case["Tn"], case["layers"]
    layers = [_project_inputs(case, _layer_seed(seed, layer), Tn)[:2] +
              (_randn(_gen(_layer_seed(seed, layer) + 1), B, Tn, case["HKV"], D).to(torch.float16),)
              for layer in range(L)]
    pos = torch.tensor(_append_pos(case, seed), dtype=torch.int32, device="cuda")
    angles = _angles(pos[:, None] + 65536 + torch.arange(Tn, device="cuda"), D)
    return layers, pos, angles, _tables([2 * PAGE] * (B * L), _gen(seed + 2))


def _prepare_append(case, seed):
    from ffa_mi355x.paged import PagedQ2Cache
    from ffa_mi355x.quant import kproj_rope_q2_append

    layers, pos, (cos, sin), (bt, pages) = _append_inputs(case, seed)
    cache = PagedQ2Cache(pages, case["HKV"], "cuda")

    def layer_step(h, w, v, table):
        kproj_rope_q2_append(cache, h, w, cos, sin, pos, table, v_new=v, validate=False)

    B = case["B"]
    replay = _captured([lambda x=x, i=i: layer_step(*x, bt[i * B:(i + 1) * B]) for i, x in enumerate(layers)])
    return lambda: (replay(), [cache.k_q, cache.k_scale, cache.k_zero, cache.k_res.view(torch.uint8),
                              cache.v])[1]


def _prepare_fill(case, seed):
    from ffa_mi355x.paged import PagedQ2Cache
    from ffa_mi355x.paged_kfmt import PagedKfmtCache

    k, v = _kv_inputs(case, seed)
    bt, pages = _tables([case["T"]] * case["B"], _gen(seed + 1))
    q2 = case["fmt"] == "q2"
    cache = PagedQ2Cache(pages, case["HKV"], "cuda") if q2 else PagedKfmtCache(case["fmt"], pages, case["HKV"], "cuda")
    pos = torch.zeros(case["B"], dtype=torch.int32, device="cuda")

    def step():
        cache.append(k, v, pos, bt)
        return [cache.k_q, cache.k_scale, cache.k_zero, cache.k_res, cache.v] if q2 else \
            [cache.k, cache.k_scale, cache.k_res, cache.v]
    return step


def prepare(case, seed):
    """What the caller holds before the call; here a function that makes it."""
    kind = case["kind"]
    if kind == "decode":
        return _prepare_decode(case, seed)
    if kind == "append":
        return _prepare_append(case, seed)
    if kind == "fill":
        return _prepare_fill(case, seed)
    if kind == "project":
        from fused_kproj_rope_q2fp8 import kproj_rope_quantize_fused

        h, w, bias = _project_inputs(case, seed, case["T"])
        cos, sin = (x.to(_DT[case["cs"]]) for x in _angles(torch.arange(case["T"], device="cuda"), case["D"]))
        def project():
            codes, scale, zero, res = kproj_rope_quantize_fused(h, w, cos, sin, case["HKV"], case["D"], bias=bias)
            return codes, scale, zero, res.view(torch.uint8)
        return project
    if kind == "quantize":
        from ffa_mi355x import kfmt_quant
        from ffa_mi355x.quant import quantize_per_channel

        k, _ = _kv_inputs(case, seed)
        fp8 = _FP8[case["res"]]
        return {"q2": lambda: quantize_per_channel(k, fp8), "fp8": lambda: kfmt_quant.quantize_fp8fp8(k, fp8),
                "nvfp4": lambda: kfmt_quant.encode_nvfp4(k, fp8, 128),
                "nf4": lambda: kfmt_quant.encode_nf4(k, fp8)}[case["fmt"]]
    from ffa_mi355x.paged import PagedQ2Cache

    lens = _lens(case)
    bt, pages = _tables(lens, _gen(seed + 1))
    cache = PagedQ2Cache(pages, case["HKV"], "cuda")
    zero = torch.zeros(1, dtype=torch.int32, device="cuda")
    for b in range(case["B"]):
        k, v = _dequant_kv(case, seed, b)
        cache.append(k[None], v[None], zero, bt[b:b + 1])
    seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    return lambda: cache.dequantize(bt, max(lens), seq_lens, out_dtype=_DT[case["out"]])


def _dequant_kv(case, seed, b):
    g, T = _gen(seed * 4099 + 17 * b + 1), _lens(case)[b]
    return _randn(g, T, case["HKV"], D).to(torch.bfloat16), _randn(g, T, case["HKV"], D).to(torch.bfloat16)


def run(state):
    return state()


# ---------------------------------------------------------------------------- what a pass cannot do without
_EVERY = {"q2": 48, "q2c": 32, "nvfp4": 72, "nf4": 68, "fp8": 128}  # bytes of one token and KV head
_ES = {"bf16": 2, "fp16": 2, "fp32": 4}


def work(case):
    kind, HKV = case["kind"], case["HKV"]
    if kind == "decode":
        G, nbytes, flops = case["HQ"] // HKV, 0.0, 0.0
        for T in _lens(case):
            blocks = -(-T // case["SBS"])
            kept = min(1.0, 1 - (1 - 1 / blocks) ** (HEAVY * G) + 0.01)  # blocks with a heavy token, about
            nbytes += T * HKV * (_EVERY[case["fmt"]] + kept * (D + 2 * D) + (2 * D * (1 - kept) if case["mean"] else 0))
            flops += T * case["HQ"] * 2 * D * (1 + 2 * kept)
        L = case["layers"]
        return {"bytes": L * (nbytes + case["B"] * case["HQ"] * D * 4), "flops": L * flops}
    es = _ES[case.get("dtype") or case["out"]]
    if kind in ("project", "append"):
        d, M = case.get("D", D), case["B"] * case.get("T", case.get("Tn"))
        n = M * HKV * d
        out = n * (1.25 if kind == "project" else 1.25 + 4 * 4 / 128 + 4)  # codes, residual (and scales, V in and out)
        L = case.get("layers", 1)
        return {"bytes": L * (M * case["H"] * es + HKV * d * case["H"] * es + out), "flops": L * 2.0 * n * case["H"]}
    if kind == "dequant":
        n = sum(_lens(case)) * HKV * D
        pages = max(-(-t // PAGE) for t in _lens(case)) * PAGE * case["B"] * HKV * D
        return {"bytes": n * (0.25 + 0.125 + 1 + 2) + 2 * pages * es, "flops": 3.0 * n}
    n = case["B"] * case["T"] * HKV * case.get("D", D)
    if kind == "fill":
        return {"bytes": n * (2 * es + 2 + 1 + {"q2": 0.375, "nvfp4": 0.5625, "nf4": 0.53125}[case["fmt"]]),
                "flops": 8.0 * n}
    return {"bytes": n * (es + 1 + {"q2": 0.25, "fp8": 1, "nvfp4": 0.5, "nf4": 0.5}[case["fmt"]]), "flops": 8.0 * n}


def tolerance(case):
    # decode: 16-bit outputs and a survivor mask.  The decode is 2e-3 off its scores in fp64 (exact); sums in another
    # order move o by less, and flip a block only where its maximum meets the threshold to about 1e-5.
    if case["kind"] == "decode":
        masks = case["B"] * case["HKV"] * -(-case["hi"] // case["SBS"])
        return {"rel": 5e-3, "max": 0.1, "differ": max(1e-3, min(1e-2, 2 / masks))}
    # The projection's 32-bit sums in another order (torch's linear layer against the kernel: scale and zero up to 3e-5
    # apart, 1e-6 of the code bytes and up to 9e-5 of the residual bytes different) move a few 16-bit K by one ulp, with
    # them their residual and now and then a code.  A code that turns takes its residual from one end of the step to the
    # other: residuals are compared as the bytes they are, beside the codes.
    if case["kind"] in ("project", "append"):
        return {"rel": 2e-3, "max": 0.03, "differ": 1e-3}
    # one rounding of a 32-bit sum to the output type
    if case["kind"] == "dequant":
        return {"rel": 1e-6} if case["out"] == "fp32" else {"rel": 1e-3, "max": 0.01}
    return "exact"  # the quantizers' bytes are defined to the bit


# ---------------------------------------------------------------------------- the same in plain torch, 64 bits
_FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
_FP4_MID = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)
_NF4 = (-1.0, -0.6961928009986877, -0.5229921340942383, -0.39491748809814453, -0.28444138169288635,
        -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634,
        0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)


def _t(values):
    return torch.tensor(values, dtype=torch.float32, device="cuda")


def _fp4_levels(x):
    """Nearest e2m1 value of x (midpoints away from zero)."""
    level = _t(_FP4)[torch.bucketize(x.float().abs(), _t(_FP4_MID), right=True)]
    return torch.where(x < 0, -level, level)


def _nf4_levels(x):
    book = _t(_NF4)
    return book[torch.bucketize(x.contiguous(), (book[:-1] + book[1:]) * 0.5)]


def _coarse(fmt, k):
    """K [..., T, HKV, D] as the format's codes and scales hold it (f64), and the scale / zero tensors.  The rounding of
    scales, codes and levels is the format's definition, in the types that it names; sums and products are in 64 bits."""
    f = k.float()
    if fmt == "q2":  # groups of 32 channels, fp16 scale and zero
        x = f.unflatten(-1, (4, 32))
        z = x.amin(-1, keepdim=True).half().float()
        s = ((x.amax(-1, keepdim=True) - z).clamp_min(1e-6) / 3.0).half().float()
        c = torch.round((x - z) / s).clamp(0, 3)
        return (c.double() * s.double() + z.double()).flatten(-2), (s[..., 0], z[..., 0])
    if fmt == "q2c":  # per channel over the tokens, in K's own type
        z = k.amin(-3, keepdim=True)
        s = (k.amax(-3, keepdim=True) - z).clamp_min(1e-6) / 3.0
        c = torch.round((k - z) / s).clamp(0, 3)
        return c.double() * s.double() + z.double(), (s.squeeze(-3), z.squeeze(-3))
    if fmt == "nvfp4":
        x = f.unflatten(-1, (8, 16))
        s = (x.abs().amax(-1, keepdim=True) / 6.0).clamp_max(448.0).to(torch.float8_e4m3fn)
        sf = s.float()
        return (_fp4_levels(torch.where(sf > 0, x / sf, 0.0)).double() * sf.double()).flatten(-2), (s[..., 0],)
    if fmt == "nf4":
        x = f.unflatten(-1, (2, 64))
        s = x.abs().amax(-1, keepdim=True).clamp_min(1e-6).half()
        sf = s.float()
        return (_nf4_levels((x / sf).clamp(-1, 1)).double() * sf.double()).flatten(-2), (s[..., 0],)
    raise ValueError(fmt)


def _residual(k, coarse, fp8):
    return (k.float() - coarse.float()).to(fp8)


def _exact_decode_layer(case, seed):
    q, seqs = _decode_inputs(case, seed)
    HKV, BS, SBS, fmt = case["HKV"], case["BS"], case["SBS"], case["fmt"]
    G, outs, ths = case["HQ"] // HKV, [], []
    unit = math.log2(math.e) / math.sqrt(D)
    for b, make in enumerate(seqs):
        k, v = make()
        T = k.shape[0]
        if fmt == "fp8":
            base = k.to(torch.float8_e5m2).double()
        else:
            base = _coarse(fmt, k)[0]
        fp8 = torch.float8_e5m2 if fmt in ("q2c", "fp8") else torch.float8_e4m3fn
        fine = base + _residual(k, base, fp8).double()
        qh = q[b].double().view(HKV, G, D)
        sc = torch.matmul(qh, base.permute(1, 2, 0).contiguous()) * unit  # [HKV, G, T]
        sf = torch.matmul(qh, fine.permute(1, 2, 0).contiguous()) * unit
        del base, fine
        ntb = -(-T // BS)
        th = sc[..., :16].amax(-1)
        if (ntb - 1) * 16 < T:
            th = torch.maximum(th, sc[..., (ntb - 1) * 16:ntb * 16].amax(-1))
        th = th - 5.0
        pad = -T % SBS
        mx = torch.nn.functional.pad(sc, (0, pad), value=-math.inf).unflatten(-1, (-1, SBS)).amax(-1)
        kept = (mx >= th[..., None]).any(1).repeat_interleave(SBS, -1)[:, :T][:, None]  # [HKV, 1, T]
        s = torch.where(kept, sf, sc if case["mean"] else torch.full_like(sc, -math.inf))
        p = torch.exp2(s - s.amax(-1, keepdim=True))
        vh = v.double().transpose(0, 1).contiguous()
        o = torch.matmul(p * kept, vh)
        if case["mean"]:
            o = o + (p * ~kept).sum(-1, keepdim=True) * vh.mean(1, keepdim=True)
        outs.append((o / p.sum(-1, keepdim=True)).reshape(-1, D))
        ths.append(th.reshape(-1))
    return {"o": torch.stack(outs), "mask": None, "threshold": torch.stack(ths)}


def _exact_decode(case, seed):
    layers = [_exact_decode_layer(case, _layer_seed(seed, layer)) for layer in range(case["layers"])]
    return layers if len(layers) > 1 else layers[0]


def _rotated(case, h, w, bias, cos, sin, heads):
    """RoPE of the projected keys [B, T, heads, D] in the promoted type; the projection is rounded to h's type, as a
    linear layer returns it."""
    x = h.double() @ w.double().t().contiguous()
    x = (x if bias is None else x + bias.double()).to(h.dtype).unflatten(-1, (heads, -1))
    cos, sin = (a[..., :, None, :] for a in (cos, sin))
    turned = torch.stack((-x[..., 1::2], x[..., ::2]), -1).flatten(-2)
    return x * cos + turned * sin


def _tiles():
    """Where the paged pools hold (token, channel) of the residual, (channel, token) of V, (group, token) of scales."""
    t, c = torch.arange(64, device="cuda")[:, None], torch.arange(128, device="cuda")[None]
    res = (((t & 3) * 2 + ((c >> 4) & 1)) * 64 + (c >> 5) * 16 + (t >> 2)) * 16 + (c & 15)
    v = (((c.T >> 4) * 2 + ((t.T >> 3) & 1)) * 64 + (t.T >> 4) * 16 + (c.T & 15)) * 8 + (t.T & 7)
    slot = 16 * (t // 16) + 4 * (t % 4) + (t // 4) % 4
    group = torch.arange(4, device="cuda")[None]
    return res, v, ((((slot >> 3) & 1) * 4 + group) * 4 + (slot >> 4)) * 8 + (slot & 7)


def _exact_pools(case, k, v, pos, bt, pages, fmt):
    """The paged pools (f64; codes left out) after k, v [B, Tn, HKV, D] were appended at pos."""
    res_at, v_at, scale_at = _tiles()
    B, Tn, HKV, _ = k.shape
    coarse, scales = _coarse(fmt, k)
    at = torch.tensor(pos, device="cuda")[:, None] + torch.arange(Tn, device="cuda")
    page = torch.gather(bt.long(), 1, at // PAGE).reshape(-1)  # of each token
    t = (at % PAGE).reshape(-1)
    heads = torch.arange(HKV, device="cuda")[None, :, None]
    where = page[:, None, None], heads

    def pool(n, at_, values):
        p = torch.zeros((pages, HKV, n), dtype=torch.float64, device="cuda")
        p[where[0], where[1], at_[:, None, :].expand(-1, HKV, -1)] = values.flatten(0, 1).double()
        return p

    res = pool(64 * D, res_at[t], k.double() - coarse).view(pages, HKV, 64, D)
    vp = pool(64 * D, v_at.T[t], v.half()).view(pages, HKV, D, 64)
    if fmt == "q2":
        return [None] + [pool(256, scale_at[t], s).view(pages, HKV, 4, 64) for s in scales] + [res, vp]
    n = scales[0].shape[-1]
    own = t[:, None] * n + torch.arange(n, device="cuda")
    return [None, pool(64 * n, own, scales[0].float()).view(pages, HKV, 64, n), res, vp]


def _exact_quantize(case, seed):
    k, _ = _kv_inputs(case, seed)
    fmt = case["fmt"]
    if fmt == "q2":
        coarse, (s, z) = _coarse("q2c", k)
        return (None, s.double(), z.double(), k.double() - coarse)
    if fmt == "fp8":
        base = k.to(_FP8[case["res"]])
        return (k.double(), k.double() - base.double())
    if fmt == "nf4":
        s = k.float().abs().amax(1, keepdim=True).clamp_min(1e-6)
        level = _nf4_levels((k.float() / s).clamp(-1, 1))
        return (None, s.squeeze(1).double(), k.double() - level.double() * s.double())
    x = torch.nn.functional.pad(k, (0, 0, 0, 0, 0, -case["T"] % 128)).unflatten(1, (-1, 128))
    s = (x.abs().amax((2, 4), keepdim=True) / 6.0).clamp_min(1e-6)
    coarse = (_fp4_levels(x / s).to(k.dtype) * s).double()
    return (None, s[:, :, 0, :, 0].double(), (x.double() - coarse).flatten(1, 2)[:, :case["T"]].contiguous())


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "quantize":
        return _exact_quantize(case, seed)
    if kind == "fill":
        k, v = _kv_inputs(case, seed)
        bt, pages = _tables([case["T"]] * case["B"], _gen(seed + 1))
        return _exact_pools(case, k, v, [0] * case["B"], bt, pages, case["fmt"])
    if kind == "project":
        h, w, bias = _project_inputs(case, seed, case["T"])
        cos, sin = (x.to(_DT[case["cs"]]) for x in _angles(torch.arange(case["T"], device="cuda"), case["D"]))
        k = _rotated(case, h, w, bias, cos, sin, case["HKV"])
        _, (s, z) = _coarse("q2c", k)
        return (None, s.double(), z.double(), None)
    if kind == "append":
        layers, pos, angles, (bt, pages) = _append_inputs(case, seed)
        k = torch.cat([_rotated(case, h, w, None, *angles, case["HKV"]) for h, w, _ in layers])
        v = torch.cat([v for _, _, v in layers])
        pools = _exact_pools(case, k, v, pos.tolist() * len(layers), bt, pages, "q2")
        return pools[:3] + [None] + pools[4:]
    lens = _lens(case)
    Tp = -(-max(lens) // PAGE) * PAGE
    ko = torch.zeros((case["B"], Tp, case["HKV"], D), dtype=torch.float64, device="cuda")
    vo = torch.zeros_like(ko)
    for b, T in enumerate(lens):
        k, v = _dequant_kv(case, seed, b)
        coarse = _coarse("q2", k)[0]
        ko[b, :T] = coarse + _residual(k, coarse, torch.float8_e4m3fn).double()
        vo[b, :T] = v.half().double()
    return ko, vo
