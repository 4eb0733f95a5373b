"""The work that a user of this package has it do, as cases that can be prepared, run, timed and checked.

Every case is one attention call through a public entry point: ``sageattention.sageattn`` (the drop-in call, with
masks and ``return_lse``), ``sageattention.sageattn_varlen`` (packed batches) or ``cdna4_sage.attention`` (the kernel
route for calls below the router's size thresholds).  Sizes come from cdna4_sage.configs (the benchmark configurations
and the model shapes) and from the tests, with ragged lengths among them.
"""
import math
import os
import sys

import torch

_PACKAGES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rdna4-sageattention_amd")
if _PACKAGES not in sys.path:
    sys.path.insert(0, _PACKAGES)

import cdna4_sage  # noqa: E402
import sageattention  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _case(entry, B, H, Hkv, Sq, Skv, D, layout, dtype, causal=False, lse=False, mask="none", lens=""):
    """entry: "attention", "sageattn" or "varlen" (lens: the sequence lengths, "q/k" each, comma separated; B, Sq and
    Skv are then their count and totals).  mask: "none", "padding" (bool [B, 1, 1, Skv], the last keys of every batch
    entry hidden) or "bias" (additive [1, H, Sq, Skv] of the inputs' dtype)."""
    return {"entry": entry, "B": B, "H": H, "Hkv": Hkv, "Sq": Sq, "Skv": Skv, "D": D, "layout": layout,
            "dtype": dtype, "causal": causal, "lse": lse, "mask": mask, "lens": lens}


def _packed(H, Hkv, D, dtype, lens, causal):
    text = ",".join("%d/%d" % p for p in lens)
    return _case("varlen", len(lens), H, Hkv, sum(a for a, _ in lens), sum(b for _, b in lens), D, "NHD", dtype,
                 causal=causal, lens=text)


def listed():
    return [
        # the smallest call: one short sequence (configuration 1), where launches and the host's work count
        dict(_case("attention", 1, 8, 8, 1024, 1024, 64, "HND", "bf16"), name="small_self_d64"),
        # an image UNet's largest self-attention (SDXL 1024, level 1) with classifier-free guidance: token-major, fp16
        dict(_case("sageattn", 2, 10, 10, 4096, 4096, 64, "NHD", "f16"), name="image_self_d64"),
        # an image transformer's joint attention, the benchmark's default workload (configuration 2, Flux)
        dict(_case("sageattn", 1, 24, 24, 4608, 4608, 128, "HND", "bf16"), name="joint_d128"),
        # the other head dims of joint attention: Neta Lumina (96) and AuraFlow (256, ragged length, batch 2)
        dict(_case("sageattn", 1, 24, 24, 4352, 4352, 96, "HND", "bf16"), name="joint_d96"),
        dict(_case("sageattn", 2, 12, 12, 4360, 4360, 256, "HND", "f16"), name="joint_d256"),
        # video tokens attending the text prompt (Wan 1.3B 480p cross): many query rows, few keys
        dict(_case("attention", 1, 12, 12, 32760, 512, 128, "NHD", "f16"), name="cross_d128"),
        # a language model's prefill over its whole prompt, grouped heads, with the row logsumexp (configuration 5a)
        dict(_case("sageattn", 2, 32, 8, 8192, 8192, 128, "HND", "bf16", causal=True, lse=True), name="causal_gqa_lse"),
        # a chunk of a longer prompt against the keys so far: fewer queries than keys, ragged lengths, token-major
        dict(_case("sageattn", 1, 32, 8, 1500, 9001, 128, "NHD", "bf16", causal=True), name="prefill_chunk"),
        # a padded batch: every prompt's own number of visible keys
        dict(_case("sageattn", 2, 24, 24, 3000, 3000, 128, "HND", "bf16", mask="padding"), name="padding_mask"),
        # a learned or distance bias per head, added to the scores
        dict(_case("sageattn", 1, 16, 16, 3072, 3072, 64, "HND", "bf16", mask="bias"), name="head_bias"),
        # sequences of different lengths packed along the token axis
        dict(_packed(24, 24, 128, "bf16", [(4608, 4608), (1152, 1152), (2304, 2304), (640, 640), (3333, 3333),
                                           (4097, 4097)], False), name="packed_batch"),
        # the largest: a video transformer's self-attention (Wan 14B 480p), where the matrix products are everything
        dict(_case("sageattn", 1, 40, 40, 32760, 32760, 128, "NHD", "f16"), name="video_d128"),
    ]


_LARGEST = 4 * 40 * 32760 * 32760 * 128  # matrix operations of the largest listed case


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _routed(H, Sq, Skv, causal):
    """Whether the router sends a call of these sizes to the kernels (smaller ones are torch's own attention)."""
    return Skv >= 1024 and H * Sq * Skv // (2 if causal else 1) >= 64 * 2**20


def draw(rng):
    while True:
        kind = rng.choice(["self", "self", "self", "cross", "causal", "chunk", "lse", "padding", "bias", "varlen"])
        dtype = rng.choice(["bf16", "bf16", "f16"])
        layout = rng.choice(["HND", "NHD"])
        D = rng.choice([64, 128, 128, 96, 256])
        B = rng.choice([1, 1, 2])
        Hkv = rng.choice([4, 8, 10, 12, 16, 24, 32, 40])
        H = Hkv
        if kind == "self":
            S = _log_int(rng, 1024, 32760)
            c = _case("sageattn", B, H, Hkv, S, S, D, layout, dtype)
        elif kind == "cross":
            c = _case("attention", B, H, Hkv, _log_int(rng, 2048, 32760), _log_int(rng, 77, 1024), D, layout, dtype)
        elif kind in ("causal", "lse"):
            H = Hkv * rng.choice([1, 2, 4])
            # the logsumexp of head dims 96 and 256 is drawn at moderate sizes
            S = _log_int(rng, 2048, 4096 if kind == "lse" and D in (96, 256) else 16384)
            c = _case("sageattn", B, H, Hkv, S, S, D, layout, dtype, causal=kind == "causal" or rng.random() < 0.7,
                      lse=kind == "lse")
        elif kind == "chunk":
            H = Hkv * rng.choice([1, 4, 8])
            Skv = _log_int(rng, 4096, 32760)
            c = _case("sageattn", B, H, Hkv, _log_int(rng, 256, 4096), Skv, D, layout, dtype, causal=True)
        elif kind == "padding":
            S = _log_int(rng, 1024, 12000)
            c = _case("sageattn", B, H, Hkv, S, S, D, layout, dtype, mask="padding")
        elif kind == "bias":
            S = _log_int(rng, 1024, 5000)
            c = _case("sageattn", 1, H, Hkv, S, S, D, layout, dtype, mask="bias")
        else:
            lens = [_log_int(rng, 1024, 6000) for _ in range(rng.randint(2, 8))]
            c = _packed(H, Hkv, D, dtype, [(n, n) for n in lens], rng.random() < 0.5)
            if sum(_routed(H, n, n, c["causal"]) for n in lens) < len(lens) - 1:
                continue
        if c["entry"] == "sageattn" and not _routed(B * H, c["Sq"], c["Skv"], c["causal"]):
            if c["lse"]:
                continue
            c["entry"] = "attention"  # the kernel route, asked for
        if H <= 64 and _flops(c) <= _LARGEST // 4 and c["B"] * H * max(c["Sq"], c["Skv"]) * D * 2 < 1 << 30:
            return c


def _lens(case):
    if case["lens"]:
        return [tuple(int(x) for x in p.split("/")) for p in case["lens"].split(",")]
    return [(case["Sq"], case["Skv"])] * case["B"]


def _visible(case, b):
    """Keys that batch entry b's padding mask shows: between five eighths and all of them."""
    n = case["Skv"]
    return n - ((b * 5 + 3) * n // 16) % (3 * n // 8) // 5 * 5


def _pairs(case):
    """(query, key) pairs per head of every sequence together."""
    total = 0
    for b, (sq, sk) in enumerate(_lens(case)):
        if case["causal"]:
            total += sq * sk - sq * (sq - 1) // 2
        else:
            total += sq * (_visible(case, b) if case["mask"] == "padding" else sk)
    return total


def _flops(case):
    return (6 if case["lse"] else 4) * case["H"] * _pairs(case) * case["D"]


def work(case):
    """Q, K, V and the mask read once, the output (and the logsumexp) written once; the two matrix products over the
    visible pairs (and the logsumexp's own product of Q and K on the unquantized inputs)."""
    nb = 1 if case["lens"] else case["B"]
    q = nb * case["Sq"] * case["H"] * case["D"]
    kv = nb * case["Skv"] * case["Hkv"] * case["D"]
    nbytes = 2 * (2 * q + 2 * kv)
    if case["lse"]:
        nbytes += 4 * nb * case["Sq"] * case["H"]
    if case["mask"] == "padding":
        nbytes += nb * case["Skv"]
    if case["mask"] == "bias":
        nbytes += 2 * case["H"] * case["Sq"] * case["Skv"]
    return {"bytes": nbytes, "flops": _flops(case)}


def _inputs(case, seed):
    """q, k, v (and a mask) on the GPU.  Activations are normal; K has a few channels with an offset shared by its
    tokens, as the keys of these models have (cdna4_sage.configs, configuration 2)."""
    dev = torch.device("cuda", torch.cuda.current_device())
    dt = DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)
    B, H, Hkv, Sq, Skv, D = (case[n] for n in ("B", "H", "Hkv", "Sq", "Skv", "D"))
    if case["lens"]:
        shape_q, shape_k = (Sq, H, D), (Skv, Hkv, D)
    elif case["layout"] == "HND":
        shape_q, shape_k = (B, H, Sq, D), (B, Hkv, Skv, D)
    else:
        shape_q, shape_k = (B, Sq, H, D), (B, Skv, Hkv, D)
    q = torch.randn(shape_q, generator=g, device=dev, dtype=torch.float32).to(dt)
    offset = torch.zeros(D, device=dev)
    channels = torch.randperm(D, generator=g, device=dev)[:8]
    offset[channels] = torch.randn(8, generator=g, device=dev) * math.sqrt(3.0)
    k = (torch.randn(shape_k, generator=g, device=dev, dtype=torch.float32) + offset).to(dt)
    v = torch.randn(shape_k, generator=g, device=dev, dtype=torch.float32).to(dt)
    mask = None
    if case["mask"] == "padding":
        shown = torch.tensor([_visible(case, b) for b in range(B)], device=dev)
        mask = (torch.arange(Skv, device=dev)[None, :] < shown[:, None])[:, None, None, :].contiguous()
    elif case["mask"] == "bias":
        # a distance penalty with a slope per head, and some noise in the place of a learned table
        slope = torch.exp2(-8.0 * torch.arange(1, H + 1, device=dev) / H)[:, None, None]
        dist = (torch.arange(Sq, device=dev)[:, None] - torch.arange(Skv, device=dev)[None, :]).abs()
        mask = torch.empty((1, H, Sq, Skv), device=dev, dtype=dt)
        for h in range(H):
            noise = torch.randn((Sq, Skv), generator=g, device=dev, dtype=torch.float32)
            mask[0, h] = (0.25 * noise - slope[h] * dist).to(dt)
    return q, k, v, mask


def prepare(case, seed):
    q, k, v, mask = _inputs(case, seed)
    state = {"case": case, "q": q, "k": k, "v": v, "mask": mask}
    if case["lens"]:
        lens = _lens(case)
        for name, i in (("cu_q", 0), ("cu_k", 1)):
            ends = [0]
            for p in lens:
                ends.append(ends[-1] + p[i])
            state[name] = torch.tensor(ends, dtype=torch.int32, device=q.device)
            state["max_" + name[3]] = max(p[i] for p in lens)
    return state


def run(state):
    c, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if c["entry"] == "varlen":
        return sageattention.sageattn_varlen(q, k, v, state["cu_q"], state["cu_k"], state["max_q"], state["max_k"],
                                             is_causal=c["causal"])
    if c["entry"] == "attention":
        return cdna4_sage.attention(q, k, v, c["layout"], is_causal=c["causal"], attn_mask=state["mask"])
    if c["lse"]:
        return sageattention.sageattn(q, k, v, tensor_layout=c["layout"], is_causal=c["causal"], return_lse=True)
    if state["mask"] is not None:
        return sageattention.sageattn(q, k, v, tensor_layout=c["layout"], is_causal=c["causal"],
                                      attn_mask=state["mask"])
    return sageattention.sageattn(q, k, v, tensor_layout=c["layout"], is_causal=c["causal"])


def tolerance(case):
    """Probabilities and V are E4M3 (3 mantissa bits) and the outputs average values of random sign, so the rounding
    does not average out against the result: the kernels with their probabilities taken against another running max
    (other E4M3 roundings of the same values) differ by 3.5e-2 to 3.9e-2 on every listed shape, as they do from
    float64.  Sums in another order alone give up to 9e-4 (a bf16 step here and there)."""
    return {"rel": 0.06}


def _reference(q, k, v, causal, bias, shown, out, lse):
    """One head in float64: q [Sq, D], k / v [Skv, D]; fills out [Sq, D] (and lse [Sq])."""
    Sq, Skv = q.shape[0], k.shape[0]
    scale = q.shape[1] ** -0.5
    k, v = k.double(), v.double()
    kt = k.t().contiguous()
    rows = max(1, (1 << 27) // Skv)
    key = torch.arange(Skv, device=q.device)
    for r0 in range(0, Sq, rows):
        r1 = min(Sq, r0 + rows)
        s = torch.mm(q[r0:r1].double(), kt).mul_(scale)
        if causal:
            last = torch.arange(r0, r1, device=q.device) + (Skv - Sq)
            s.masked_fill_(key[None, :] > last[:, None], float("-inf"))
        if lse is not None:
            lse[r0:r1] = torch.logsumexp(s, dim=1)
        if bias is not None:
            s += bias[r0:r1].double()
        if shown is not None:
            s[:, shown:] = float("-inf")
        out[r0:r1] = torch.mm(torch.softmax(s, dim=1), v)


def exact(case, seed):
    q, k, v, mask = _inputs(case, seed)
    group = case["H"] // case["Hkv"]
    out = torch.empty(q.shape, device=q.device, dtype=torch.float64)
    lse = torch.empty((case["B"], case["H"], case["Sq"]), device=q.device, dtype=torch.float64) if case["lse"] else None
    q0 = k0 = 0
    for b, (sq, sk) in enumerate(_lens(case)):
        for h in range(case["H"]):
            hk = h // group
            if case["lens"]:
                views = q[q0:q0 + sq, h], k[k0:k0 + sk, hk], v[k0:k0 + sk, hk], out[q0:q0 + sq, h]
            elif case["layout"] == "HND":
                views = q[b, h], k[b, hk], v[b, hk], out[b, h]
            else:
                views = q[b, :, h], k[b, :, hk], v[b, :, hk], out[b, :, h]
            _reference(views[0], views[1], views[2], case["causal"], mask[0, h] if case["mask"] == "bias" else None,
                       _visible(case, b) if case["mask"] == "padding" else None, views[3],
                       None if lse is None else lse[b, h])
        q0, k0 = q0 + sq, k0 + sk
    return out if lse is None else (out, lse)
