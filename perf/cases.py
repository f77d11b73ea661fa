"""Performance cases of the weight-only quantized GEMM, through the package's public calls.

Families (`kind`), each over the sizes a serving engine meets:
  gemm    one projection, hq.gemm: int4 (zero point 8) or ternary weights, decode steps of a
          few rows up to prefill chunks;
  fused   projections sharing one input, hq.gemm_fused (QKV, gate || up);
  q4k     int4 with a scale and a bias per 32 weights, as Q4_K tensors import: hq.gemm(bias=,
          group=32);
  layer   the projections of one decoder layer on TQ1_0-style ternary weights (group 256),
          decoder.LayerProjections: mixer in, mixer out, gate || up, down;
  int8    fp32 activations on int8 weights, hq.gemm_w8a8;
  import  weights into the tile layout on the device: hq.repack_tq1_0_device and
          hq.repack_device (int4, ternary), once per tensor when a model is loaded.

Weights are bell-shaped int4 codes, ternary codes with half zeros, or TQ1_0 blocks; scales
|N(0, 0.02)| in fp16; activations N(0, 1) (int8: N(0, 0.3), whose quantiser clamps at 1).
"""
from __future__ import annotations

import torch

from nebula_amd import decoder, hq

INT4, TERNARY = hq.FORMAT_INT4, hq.FORMAT_TERNARY2
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
FORMATS = {"int4": INT4, "ternary": TERNARY}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One token of one stream through a 4096-wide projection: the shortest call.
        dict(name="decode_int4_m1_4096", kind="gemm", fmt="int4", dtype="f16", M=1, K=4096, Ns="4096", group=128),
        # A full decode batch through the 27B-class up projection: the weight stream.
        dict(name="decode_int4_m16_up", kind="gemm", fmt="int4", dtype="f16", M=16, K=5120, Ns="27648", group=128),
        # One token through a decoder layer's projections (four calls): the step of one chat.
        dict(name="layer_attention_m1", kind="layer", layer="attention", dtype="bf16", M=1),
        # A split-fuse step: 16 decode tokens and a 64-token prompt chunk through an SSM layer.
        dict(name="layer_ssm_m80", kind="layer", layer="ssm", dtype="f16", M=80),
        # An odd mixed batch through an 11008-wide projection, bf16.
        dict(name="mixed_int4_m37", kind="gemm", fmt="int4", dtype="bf16", M=37, K=4096, Ns="11008", group=128),
        # Q4_K weights (scale and bias per 32): a small decode batch and a prompt chunk.
        dict(name="q4k_m4", kind="q4k", dtype="bf16", M=4, K=4096, Ns="14336", group=32),
        dict(name="q4k_m384", kind="q4k", dtype="f16", M=384, K=5120, Ns="5120", group=32),
        # A ragged prompt chunk through the decoder's fused gate || up, bf16.
        dict(name="gate_up_ternary_m333", kind="fused", fmt="ternary", dtype="bf16", M=333, K=5120,
             Ns="17408,17408", group=256),
        # A 1024-token chunk through the fused QKV of a grouped-query model.
        dict(name="qkv_int4_m1024", kind="fused", fmt="int4", dtype="f16", M=1024, K=5120, Ns="5120,1024,1024",
             group=128),
        # A long prompt through the up projection: the largest call.
        dict(name="prefill_int4_m2048", kind="gemm", fmt="int4", dtype="f16", M=2048, K=5120, Ns="27648", group=128),
        # Eight streams on int8 weights.
        dict(name="int8_m8_up", kind="int8", M=8, K=5120, Ns="27648"),
        # A TQ1_0 tensor imported while a model is loaded.
        dict(name="import_tq1_0_down", kind="import", source="tq1_0", K=17408, Ns="5120"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: sizes spread over the logarithm of their range, ragged ones among them."""
    kind = rng.choice(["gemm", "gemm", "gemm", "fused", "q4k", "layer", "int8", "import"])
    dtype = rng.choice(["f16", "bf16"])
    K = 128 * _log_int(rng, 8, 216)
    N = _log_int(rng, 1024, 34816)
    if rng.random() < 0.7:
        N = (N + 127) // 128 * 128
    if kind == "layer":
        return dict(kind=kind, layer=rng.choice(["attention", "ssm"]), dtype=dtype, M=_log_int(rng, 1, 512))
    if kind == "int8":
        return dict(kind=kind, M=rng.randint(1, 16), K=K, Ns=str(N))
    if kind == "import":
        return dict(kind=kind, source=rng.choice(["tq1_0", "tq1_0", "int4", "ternary"]), K=(K + 255) // 256 * 256,
                    Ns=str(N))
    M = _log_int(rng, 1, 2048)
    # No more work than 2048 x 5120 x 27648, and at most about its weight bytes.
    while M * K * N > 2048 * 5120 * 27648:
        M = max(1, M // 2)
    while K * N > 2 * 5120 * 27648:
        N = max(1024, N // 2)
    if kind == "q4k":
        return dict(kind=kind, dtype=dtype, M=min(M, 1024), K=(K + 255) // 256 * 256, Ns=str(N), group=32)
    fmt = rng.choice(["int4", "ternary"])
    group = 256 if fmt == "ternary" and K % 256 == 0 else 128
    Ns = str(N)
    if kind == "fused":
        kv = max(16, N // 6)
        Ns = rng.choice([f"{N // 2},{N // 2}", f"{N - 2 * kv},{kv},{kv}"])
    return dict(kind=kind, fmt=fmt, dtype=dtype, M=M, K=K, Ns=Ns, group=group)


def _widths(case):
    return [int(n) for n in case["Ns"].split(",")]


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 2654435761 % (1 << 62) + 17)


def _randint_words(g, n):
    return torch.randint(-(1 << 31), 1 << 31, (n,), dtype=torch.int64, device="cuda", generator=g).to(torch.int32)


def _linear(g, fmt, K, N):
    """Linear weight words: int4 codes around 7.5 (the sum of two 3-bit values and a bit per
    nibble), ternary codes with P(0) = 1/2."""
    n = hq.linear_words(fmt, K, N)
    a, b = _randint_words(g, n), _randint_words(g, n)
    if fmt == INT4:
        return (a & 0x77777777) + (b & 0x77777777) + ((a >> 3) & 0x11111111)
    # Two bits c = t + 1 per weight: 1 where the low bit of a is set, else 0 or 2 by b's.
    one = a & 0x55555555
    return one | ((b & 0x55555555 & ~one) << 1)


def _scales(g, rows, N):
    return (torch.randn((rows, N), device="cuda", generator=g).abs() * 0.02).to(torch.float16)


def _acts(g, M, K, dtype):
    return torch.randn((M, K), device="cuda", generator=g).to(DTYPES[dtype])


LAYER_INPUTS = (("mixer_in", decoder.EMBEDDING), ("mixer_out", decoder.MIXER_IN),
                ("ffn_in", decoder.EMBEDDING), ("ffn_out", decoder.FFN))


def _inputs(case, seed):
    """The case's raw inputs (activations, linear weights, scales), from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "layer":
        groups = decoder.FUSED_GROUPS[case["layer"]] + decoder.FUSED_GROUPS["ffn"]
        weights = {}
        for name in [n for grp in groups for n in grp]:
            K, N = decoder.SHAPES[name]
            weights[name] = (_linear(g, TERNARY, K, N), _scales(g, K // decoder.TQ1_GROUP, N))
        return dict(weights=weights, x={n: _acts(g, case["M"], K, case["dtype"]) for n, K in LAYER_INPUTS},
                    groups=groups)
    K, Ns = case["K"], _widths(case)
    if kind == "int8":
        N = Ns[0]
        N16 = (N + 15) // 16 * 16
        # The tile layout of N16 columns; the columns past N hold zeros.
        w = torch.randint(-128, 128, (N16 // 16, K // 128, 4, 16, 2, 16), dtype=torch.int8, device="cuda", generator=g)
        if N16 > N:
            w[-1, :, :, N - N16:] = 0
        return dict(x=torch.randn((case["M"], K), device="cuda", generator=g) * 0.3, w=w,
                    s=torch.rand((N,), device="cuda", generator=g) * 0.02 + 0.001)
    if kind == "import":
        N = Ns[0]
        if case["source"] == "tq1_0":
            return dict(blocks=decoder.random_tq1_0(K, N, generator=g))
        return dict(lin=_linear(g, FORMATS[case["source"]], K, N))
    fmt = INT4 if kind == "q4k" else FORMATS[case["fmt"]]
    x = _acts(g, case["M"], K, case["dtype"])
    segs = []
    for N in Ns:
        lin, s = _linear(g, fmt, K, N), _scales(g, K // case["group"], N)
        b = None
        if kind == "q4k":  # -dmin * m: around the zero point, as real tensors have it
            b = -8.0 * s.float() * (0.75 + 0.5 * torch.rand(s.shape, device="cuda", generator=g))
        segs.append((lin, s, b, N))
    return dict(x=x, segs=segs)


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "layer":
        w = {}
        for name, (lin, s) in d["weights"].items():
            K, N = decoder.SHAPES[name]
            w[name] = decoder.TernaryProjection(K, N, hq.repack_device(TERNARY, lin, K, N), s)
        return dict(kind=kind, layer=decoder.LayerProjections(case["layer"], w), x=d["x"])
    K, Ns = case["K"], _widths(case)
    if kind == "int8":
        return dict(kind=kind, x=d["x"], w=d["w"].reshape(-1), s=d["s"], N=Ns[0])
    if kind == "import":
        return dict(kind=kind, source=case["source"], K=K, N=Ns[0], **d)
    fmt = INT4 if kind == "q4k" else FORMATS[case["fmt"]]
    segs = [(hq.repack_device(fmt, lin, K, N), s, N, b) for lin, s, b, N in d["segs"]]
    return dict(kind=kind, fmt=fmt, x=d["x"], segs=segs, group=case["group"])


# ---------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind == "layer":
        layer, x = state["layer"], state["x"]
        return layer.mixer_in(x["mixer_in"]) + [layer.mixer_out(x["mixer_out"])] + layer.ffn_in(x["ffn_in"]) + [
            layer.ffn_out(x["ffn_out"])]
    if kind == "int8":
        return hq.gemm_w8a8(state["x"], state["w"], state["s"], state["N"])
    if kind == "import":
        if state["source"] == "tq1_0":
            return list(hq.repack_tq1_0_device(state["blocks"], state["K"], state["N"]))
        return hq.repack_device(FORMATS[state["source"]], state["lin"], state["K"], state["N"])
    if kind == "fused":
        return hq.gemm_fused(state["fmt"], state["x"], state["segs"], state["group"])
    wp, s, n, b = state["segs"][0]
    return hq.gemm(state["fmt"], state["x"], wp, s, n, state["group"], bias=b)


def work(case):
    kind = case["kind"]
    if kind == "layer":
        M, nbytes, flops = case["M"], 0, 0
        for _, K in LAYER_INPUTS:
            nbytes += 2 * M * K
        for grp in decoder.FUSED_GROUPS[case["layer"]] + decoder.FUSED_GROUPS["ffn"]:
            for name in grp:
                K, N = decoder.SHAPES[name]
                nbytes += K * N // 4 + K // decoder.TQ1_GROUP * N * 2 + 2 * M * N
                flops += 2 * M * K * N
        return {"bytes": nbytes, "flops": flops}
    K, N = case["K"], sum(_widths(case))
    if kind == "int8":
        M = case["M"]
        return {"bytes": K * N + 4 * N + 4 * M * K + 4 * M * N, "flops": 2 * M * K * N}
    if kind == "import":
        if case["source"] == "tq1_0":
            return {"bytes": hq.tq1_0_bytes(K, N) + K * N // 4 + K // 256 * N * 2, "flops": 0}
        return {"bytes": 2 * (K * N // 2 if case["source"] == "int4" else K * N // 4), "flops": 0}
    M, g = case["M"], case["group"]
    int4 = kind == "q4k" or case["fmt"] == "int4"
    wbytes = K * N // 2 if int4 else K * N // 4
    sbytes = K // g * N * (6 if kind == "q4k" else 2)
    return {"bytes": wbytes + sbytes + 2 * M * K + 2 * M * N, "flops": 2 * M * K * N}


def tolerance(case):
    kind = case["kind"]
    if kind == "import":
        return "exact"
    if kind == "int8":  # exact integer sums, two fp32 roundings
        return {"rel": 1e-6}
    # The output's rounding, and from about 80 rows on that of each scaled weight to the activation type.
    return {"rel": 1.5e-3} if case["dtype"] == "f16" else {"rel": 1e-2}


# ---------------------------------------------------------------- the same results in 64 bits
def _unpack(lin, fmt, K, N):
    """Linear words -> integer codes [K, N]."""
    per, bits = (8, 4) if fmt == INT4 else (16, 2)
    sh = torch.arange(per, device="cuda", dtype=torch.int32).mul_(bits).view(1, per, 1)
    return ((lin.view(K // per, 1, N) >> sh) & ((1 << bits) - 1)).reshape(K, N)


def _dense(lin, fmt, K, N, s, b, group):
    q = _unpack(lin, fmt, K, N).double()
    s64 = s.double().repeat_interleave(group, dim=0)
    if fmt == TERNARY:
        return (q - 1.0) * s64
    return (q - 8.0) * s64 if b is None else q * s64 + b.double().repeat_interleave(group, dim=0)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "import":
        if case["source"] != "tq1_0":
            return None
        K, N = case["K"], _widths(case)[0]
        blocks = d["blocks"].view(N, K // 256, 56)
        return [None, blocks[:, :, :2].contiguous().view(torch.float16).view(N, K // 256).t().double()]
    if kind == "int8":
        K, N = case["K"], _widths(case)[0]
        # Tile [ct][kb][k-slice][column][chunk][16]: k = 128 kb + 64 chunk + 16 slice + i.
        w = d["w"].permute(1, 4, 2, 5, 0, 3).reshape(K, -1)[:, :N].double()
        xq = (d["x"] * 127.0).clamp(-128.0, 127.0).to(torch.int8).double()
        return (xq @ w) / 127.0 * d["s"].double()
    if kind == "layer":
        out = []
        for (name, _), grp in zip(LAYER_INPUTS, d["groups"]):
            x = d["x"][name].double()
            for proj in grp:
                K, N = decoder.SHAPES[proj]
                lin, s = d["weights"][proj]
                out.append(x @ _dense(lin, TERNARY, K, N, s, None, decoder.TQ1_GROUP))
        return out
    fmt = INT4 if kind == "q4k" else FORMATS[case["fmt"]]
    x = d["x"].double()
    ys = [x @ _dense(lin, fmt, case["K"], N, s, b, case["group"]) for lin, s, b, N in d["segs"]]
    return ys if kind == "fused" else ys[0]
