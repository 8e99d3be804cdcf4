"""The work this library is measured on: attention calls as a program makes them, from one
small decode step to the 4k GQA prefill, through transfer_station_amd's entry points on torch
tensors (bf16 inputs, fp32 output, caller-owned scratch, the default stream).

A case is a dict of the call's arguments: Hq, Hkv, Sq, Sk, D, causal, sigma_q (the standard
deviation of Q; K and V are N(0, 1)) and v, the form V arrives in:
  "row"   V [Hkv][Sk][D]
  "vt"    V^T [Hkv][D][Sk], kept that way by the caller (v_prepacked = 1)
  "pack"  V [Hkv][Sk][D], packed by pack_v_full on every pass and then used as V^T
A batch folds into the head counts, as the entry points have it.
"""
import math

import torch

import transfer_station_amd as ts

BK = 128  # any legal bk gives the same result at the same speed


def _case(Hq, Hkv, Sq, Sk, D, causal=0, v="row", sigma_q=1.0, name=None):
    c = {"Hq": Hq, "Hkv": Hkv, "Sq": Sq, "Sk": Sk, "D": D, "causal": causal, "v": v,
         "sigma_q": sigma_q}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # One sequence early in its generation: the smallest call, made once per layer and token.
        _case(32, 8, 1, 777, 128, name="decode_b1_777"),
        # One sequence over a long context: few kv heads, so the key range is split.
        _case(32, 8, 1, 32768, 128, name="decode_b1_32k"),
        # A full serving batch of 64 sequences (benchmark configuration 2), HBM-bound.
        _case(64 * 32, 64 * 8, 1, 4096, 128, name="decode_b64_4k"),
        # 16 sequences whose cache holds V^T, at a length that is no multiple of anything.
        _case(16 * 32, 16 * 8, 1, 4001, 128, v="vt", name="decode_vt_4001"),
        # Speculative decoding: 8 draft tokens of 4 sequences checked in one call.
        _case(4 * 64, 4 * 8, 8, 4001, 128, causal=1, name="verify_8x4001"),
        # A small encoder layer (configuration 1): latency, not throughput.
        _case(4, 4, 256, 256, 64, name="mha_256"),
        # The headline prefill (configuration 3 at 4k).
        _case(4 * 32, 4 * 8, 4096, 4096, 128, name="gqa_prefill_4k"),
        # One prompt of an ordinary length through a Qwen3-shaped layer, causal.
        _case(16, 8, 3000, 3000, 128, causal=1, name="qwen3_causal_3000"),
        # Ragged GQA with sharply peaked rows at head dim 64 (configuration 5).
        _case(2 * 24, 2 * 6, 1000, 4000, 64, sigma_q=4.0, name="ragged_d64"),
        # A 512-token chunk of a long prompt over the 8192 keys so far.
        _case(32, 8, 512, 8192, 128, causal=1, name="chunk_512x8192"),
        # The widest head dim the entry points take, causal.
        _case(64, 16, 2048, 2048, 256, causal=1, name="causal_d256_2k"),
        # A head dim that is no multiple of 8 over an odd key count, V packed first (the
        # --prepack-v flow of the command line).
        _case(24, 6, 1000, 2003, 100, v="pack", name="odd_d100_pack"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the same kinds: decode and short draft blocks, prefill with and without
    earlier keys, and shapes that miss the 16-byte vector layout."""
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "odd"])
        g = rng.choice([1, 2, 4, 8, 16])
        v = rng.choice(["row", "row", "vt"])
        if kind == "decode":
            Hkv = _log_int(rng, 1, 512)
            Sq = rng.choice([1, 1, 1, rng.randint(2, 8)])
            Sk = max(Sq, _log_int(rng, 64, 65536))
            D = rng.choice([64, 80, 96, 128, 128, 128, 192, 256])
            causal, flop_max, byte_max = int(Sq > 1), 1e11, 1.0e9
        elif kind == "prefill":
            Hkv = _log_int(rng, 1, 64)
            Sq = _log_int(rng, 64, 8192)
            Sk = Sq + rng.choice([0, 0, _log_int(rng, 16, 16384)])
            D = rng.choice([32, 40, 64, 64, 80, 96, 128, 128, 128, 192, 256])
            causal, flop_max, byte_max = rng.choice([0, 1]), 5e11, 4e8
        else:
            Hkv = _log_int(rng, 1, 32)
            Sq = rng.choice([1, _log_int(rng, 2, 2048)])
            Sk = Sq + _log_int(rng, 16, 8192)
            D = rng.choice([rng.randint(1, 256), rng.randint(33, 128)])
            v = rng.choice(["row", "vt", "pack"])
            causal, flop_max, byte_max = rng.choice([0, 1]), 2e10, 1e8
        c = _case(g * Hkv, Hkv, Sq, Sk, D, causal, v, rng.choice([1.0, 1.0, 4.0]))
        w = work(c)
        if w["flops"] <= flop_max and w["bytes"] <= byte_max:
            return c


def _pairs(c):
    """(query, key) pairs of one head that the mask admits."""
    Sq, Sk = c["Sq"], c["Sk"]
    if not c["causal"]:
        return Sq * Sk
    # row i sees max(0, Sk - Sq + i + 1) keys
    first = max(0, Sq - Sk)
    n, lo = Sq - first, Sk - Sq + first + 1
    return n * lo + n * (n - 1) // 2


def work(c):
    q = c["Hq"] * c["Sq"] * c["D"]
    kv = c["Hkv"] * c["Sk"] * c["D"]
    nbytes = 2 * q + 2 * 2 * kv + 4 * q + (2 * kv if c["v"] == "pack" else 0)
    return {"bytes": nbytes, "flops": 4 * c["D"] * c["Hq"] * _pairs(c)}


def _inputs(c, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def normal(heads, rows):
        return torch.randn(heads, rows, c["D"], generator=gen, device="cuda")

    q = normal(c["Hq"], c["Sq"]).mul_(c["sigma_q"]).bfloat16()
    k = normal(c["Hkv"], c["Sk"]).bfloat16()
    v = normal(c["Hkv"], c["Sk"]).bfloat16()
    return q, k, v


def prepare(c, seed):
    q, k, v = _inputs(c, seed)
    s = {"case": c, "q": q, "k": k, "v": v, "vt": None,
         "o": torch.empty(c["Hq"], c["Sq"], c["D"], dtype=torch.float32, device="cuda"),
         "scratch": torch.empty(ts.attn_flash_scratch_bytes(c["D"], BK), dtype=torch.uint8,
                                device="cuda")}
    if c["v"] == "vt":
        s["vt"] = v.transpose(1, 2).contiguous()
    elif c["v"] == "pack":
        s["vt"] = torch.empty(c["Hkv"], c["D"], c["Sk"], dtype=torch.bfloat16, device="cuda")
    return s


def run(s):
    c = s["case"]
    v = s["v"]
    if c["v"] == "pack":
        ts.pack_v_full(v.data_ptr(), s["vt"].data_ptr(), c["Hkv"], c["Sk"], c["D"])
    if c["v"] != "row":
        v = s["vt"]
    ts.attn_flash(s["q"].data_ptr(), s["k"].data_ptr(), v.data_ptr(), s["o"].data_ptr(), c["Hq"],
                  c["Hkv"], c["Sq"], c["Sk"], c["D"], c["causal"], BK, s["scratch"].data_ptr(),
                  0 if c["v"] == "row" else 1)
    return {"o": s["o"], "vt": s["vt"]} if c["v"] == "pack" else {"o": s["o"]}


def tolerance(c):
    # P enters the second product rounded to bf16 (up to 2^-9 of a weight); the sums are fp32.
    # Measured against exact() over the listed and 30 drawn calls: relative error up to 1.7e-3,
    # largest difference up to 3.7e-2 of the result's rms or of the value (causal rows that see a
    # few keys are much larger than the rms of the whole result). Stated: about four times that.
    return {"rel": 6e-3, "max": 0.15}


def exact(c, seed):
    q, k, v = _inputs(c, seed)
    Hq, Hkv, Sq, Sk, D = c["Hq"], c["Hkv"], c["Sq"], c["Sk"], c["D"]
    g = Hq // Hkv
    o = torch.zeros(Hq, Sq, D, dtype=torch.float64, device="cuda")
    rows = max(1, (1 << 25) // Sk)  # 256 MiB of scores at a time
    limit = (Sk - Sq + torch.arange(Sq, device="cuda")).repeat(g)  # last key of each row
    keys = torch.arange(Sk, device="cuda")
    for u in range(Hkv):
        qu = q[u * g:(u + 1) * g].reshape(g * Sq, D).double() / math.sqrt(D)
        ku, vu = k[u].double(), v[u].double()
        ou = o[u * g:(u + 1) * g].view(g * Sq, D)
        for r in range(0, g * Sq, rows):
            s = qu[r:r + rows] @ ku.t().contiguous()
            if c["causal"]:
                s.masked_fill_(keys[None, :] > limit[r:r + rows, None], -math.inf)
            p = (s - s.amax(1, keepdim=True).clamp_min(-1e300)).exp_()
            ou[r:r + rows] = (p @ vu) / p.sum(1, keepdim=True).clamp_min(1e-300)
    return {"o": o, "vt": v.transpose(1, 2).double()} if c["v"] == "pack" else {"o": o}
