"""The work that programs have this package do, as cases that can be timed and compared.

Every case goes through the package's public entry points as a program calls them, from the
smallest ring to the largest, in each direction (forward, backward, a whole training step, the
FP8 producer), each input type and each K/V layout.  A case is a dict of plain values:

  kind   "forward"    ring_flash_attn, one kernel for the whole sweep where the package has one
         "perstep"    ring_flash_attn(fused=False): attention per ring step, then the merges
         "backward"   ring_flash_attn_backward on the forward's saved out and LSE
         "train"      ring_flash_attn_func: forward and torch.autograd backward
         "quantize"   zig-zag shards of full q / k / v, then their e4m3 form and descales
  lens   lengths of the full sequences, one or several packed ones ("4856 9720 ...")
  cp, rank, h, h_kv, d, dtype ("bf16", "fp16", "e4m3")
  page   rows per page of a paged K/V cache, 0 for contiguous shards (forward)
  merge  "incremental" or "batched" (perstep)
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fa4-cp_amd"))

from fa4_ring import (LocalKVRing, PagedKVRing, RingConfig, quantize_ring, ring_flash_attn,  # noqa: E402
                      ring_flash_attn_backward, ring_flash_attn_func, zigzag_shard)
from fa4_ring.zigzag import zigzag_shard_varlen  # noqa: E402

# the packed benchmark's document lengths
PACKED = "4856 9720 8592 4864 1832 15456 2784 1576"


def case(name, kind, lens, cp, rank, h, h_kv, d, dtype, page=0, merge="incremental"):
    c = dict(kind=kind, lens=str(lens), cp=cp, rank=rank, h=h, h_kv=h_kv, d=d, dtype=dtype, page=page, merge=merge)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest ring in use (the CPU benchmark's shape): launches and host work count
        case("fwd_small", "forward", 2048, 4, 1, 8, 2, 128, "bf16"),
        # a prompt of ordinary length on the serving model's heads
        case("fwd_16k", "forward", 16384, 8, 3, 32, 8, 128, "bf16"),
        # the headline: one rank of a 131072-token ring
        case("fwd_131k", "forward", 131072, 8, 3, 32, 8, 128, "bf16"),
        # FP8 prefill of a length that fills no tile evenly, a late rank (front-half steps mostly)
        case("fwd_e4m3_30k", "forward", 30064, 8, 6, 32, 8, 128, "e4m3"),
        # the longest ring: FP8 at head dim 256
        case("fwd_e4m3_d256_262k", "forward", 262144, 8, 3, 16, 2, 256, "e4m3"),
        # packed documents of a real length mix
        case("fwd_packed_8", "forward", PACKED, 4, 3, 32, 8, 128, "bf16"),
        # many short packed sequences, fp16, one kv head per query head, head dim 64
        case("fwd_packed_short_fp16", "forward", " ".join(str(4 * (37 * i % 230 + 12)) for i in range(24)), 2, 1,
             16, 16, 64, "fp16"),
        # serving from a paged K/V cache
        case("fwd_paged_49k", "forward", 49152, 4, 2, 32, 8, 128, "bf16", page=256),
        # the reference's per-step form with the batched merge, head dim 256
        case("perstep_batched_d256", "perstep", 32768, 4, 2, 16, 2, 256, "bf16", merge="batched"),
        # a training step at an ordinary length: forward, backward, gradients in the input type
        case("train_8k", "train", 8192, 4, 1, 32, 8, 128, "bf16"),
        # the headline ring's backward
        case("bwd_131k", "backward", 131072, 8, 3, 32, 8, 128, "bf16"),
        # the step before an FP8 ring: shard full q / k / v and quantise every shard
        case("quantize_65k", "quantize", 65536, 8, 3, 32, 8, 128, "e4m3"),
    ]


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "forward", "train", "backward", "perstep", "quantize"])
    cp = rng.choice([2, 4, 8, 8, 16]) if kind == "forward" else rng.choice([2, 4, 8])
    rank = rng.randrange(cp)
    d = rng.choice([128, 128, 128, 64, 256])
    h, h_kv = rng.choice([(32, 8), (32, 8), (16, 2), (8, 2), (16, 16), (24, 8), (8, 1)])
    dtype = rng.choice(["bf16", "bf16", "fp16", "e4m3"] if kind in ("forward", "perstep") else ["bf16", "bf16", "fp16"])
    if dtype == "e4m3" and d == 64:
        d = 128
    if kind == "quantize":
        dtype = "e4m3"
    top = {"forward": 131072, "perstep": 65536, "train": 49152, "backward": 65536, "quantize": 131072}[kind]
    total = int(math.exp(rng.uniform(math.log(1024), math.log(top))))
    page = rng.choice([128, 256, 384]) if kind == "forward" and rng.random() < 0.2 else 0
    many = rng.choice([1, 1, 1, 3, 9, 30]) if kind != "quantize" else 1
    merge = rng.choice(["incremental", "batched"])
    weights = [math.exp(rng.gauss(0, 0.8)) for _ in range(many)]
    unit = 2 * cp  # every sequence is two chunks per rank; the chunks may have any length
    while True:
        lens = [max(1, round(total * w / sum(weights) / unit)) * unit for w in weights]
        c = case(None, kind, " ".join(map(str, lens)), cp, rank, h, h_kv, d, dtype, page, merge)
        if work(c)["flops"] <= 2e13:
            return c
        total = total * 3 // 4


def _lens(c):
    return [int(x) for x in c["lens"].split()]


def _bounds(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _inputs(c, seed):
    """Full q, k, v, dout in 16 bits on the GPU: unit normal activations, v with the per-channel
    offsets that a value projection gives it."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, d = sum(_lens(c)), c["d"]
    dt = torch.float16 if c["dtype"] == "fp16" else torch.bfloat16

    def make(heads, offset):
        x = torch.randn(n, heads, d, generator=g, device="cuda", dtype=torch.float32)
        if offset:
            x += offset * torch.randn(heads, d, generator=g, device="cuda", dtype=torch.float32)
        return x.to(dt)

    return make(c["h"], 0.0), make(c["h_kv"], 0.0), make(c["h_kv"], 0.5), make(c["h"], 0.0)


def _cu(c):
    """Local cu_seqlens (device int32) and the longest local sequence; None for one sequence."""
    lens = [n // c["cp"] for n in _lens(c)]
    if len(lens) == 1:
        return None, None
    return torch.tensor(_bounds(lens), dtype=torch.int32, device="cuda"), max(lens)


def prepare(c, seed):
    q, k, v, dout = _inputs(c, seed)
    cp, rank = c["cp"], c["rank"]
    full_cu = _bounds(_lens(c)) if len(_lens(c)) > 1 else None
    cfg = RingConfig(cp_size=cp, cp_rank=rank, merge_mode=c["merge"])
    state = dict(case=c, cfg=cfg)
    if c["kind"] == "quantize":
        state.update(q=q, k=k, v=v)
        return state
    cu, longest = _cu(c)
    state.update(cu=cu, longest=longest, descales=None)
    ring = LocalKVRing.from_full(k, v, cp, full_cu)
    local = (lambda x: zigzag_shard(x, rank, cp)) if full_cu is None else (
        lambda x: zigzag_shard_varlen(x, full_cu, rank, cp)[0])
    q = local(q)
    if c["dtype"] == "e4m3":
        q, ks, vs, state["descales"] = quantize_ring(q, ring.k, ring.v)
        ring = LocalKVRing(ks, vs)
    if c["page"]:
        # (the page order of a cache that has been in use for a while)
        ring = PagedKVRing.from_shards(ring.k, ring.v, c["page"], cu, spare_pages=3,
                                       generator=torch.Generator().manual_seed(seed), fill=0.0)
    state.update(q=q, ring=ring)
    if c["kind"] == "train":
        for x in (q, *ring.k, *ring.v):
            x.requires_grad_(True)
        state["dout"] = local(dout)
    elif c["kind"] == "backward":
        state["dout"] = local(dout)
        state["out"], state["lse"] = ring_flash_attn(q, ring.k[rank], ring.v[rank], cfg, group=ring, cu_seqlens=cu,
                                                     max_seqlen=longest, return_lse=True)
    return state


def run(s):
    c, cfg = s["case"], s["cfg"]
    cp, rank = c["cp"], c["rank"]
    if c["kind"] == "quantize":
        q = zigzag_shard(s["q"], rank, cp)
        ring = LocalKVRing.from_full(s["k"], s["v"], cp)
        q8, k8, v8, desc = quantize_ring(q, ring.k, ring.v)
        return dict(q=q8, k=k8, v=v8, qd=desc.q, kd=desc.k, vd=desc.v)
    ring = s["ring"]
    packed = dict(cu_seqlens=s["cu"], max_seqlen=s["longest"])
    if c["kind"] == "train":
        out = ring_flash_attn_func(s["q"], ring, cfg, **packed)
        grads = torch.autograd.grad(out, [s["q"], *ring.k, *ring.v], s["dout"])
        return dict(out=out.detach(), dq=grads[0], dk=grads[1:1 + cp], dv=grads[1 + cp:])
    if c["kind"] == "backward":
        dq, dk, dv = ring_flash_attn_backward(s["dout"], s["q"], ring.k[rank], ring.v[rank], s["out"], s["lse"], cfg,
                                              group=ring, **packed)
        return dict(dq=dq, dk=dk, dv=dv)
    lk, lv = (None, None) if c["page"] else ring.kv(rank)
    out, lse = ring_flash_attn(s["q"], lk, lv, cfg, group=ring, descales=s["descales"],
                               fused=False if c["kind"] == "perstep" else None, return_lse=True, **packed)
    return dict(out=out, lse=lse)


def work(c):
    """q, the k / v rows that the rank attends and the results, each once; the products of the
    attended (row, key) pairs: two of them forward, five backward."""
    cp, h, h_kv, d = c["cp"], c["h"], c["h_kv"], c["d"]
    esz = 1 if c["dtype"] == "e4m3" else 2
    pairs = keys = rows = 0
    for n in _lens(c):
        t = n // cp
        rows += t
        pairs += t * (t + 1) // 2 + (cp - 1) * (t // 2) * t
        keys += t + c["rank"] * (t // 2) + (cp - 1 - c["rank"]) * t
    q, kv, lse = rows * h * d, 2 * keys * h_kv * d, rows * h * 4
    if c["kind"] == "quantize":
        values = q + 2 * rows * cp * h_kv * d
        return dict(bytes=3 * values, flops=3 * values)
    forward = esz * (q + kv) + 2 * q + lse
    if c["kind"] in ("forward", "perstep"):
        return dict(bytes=forward, flops=4 * pairs * h * d)
    grad = 4 if c["kind"] == "backward" else 2
    grads = grad * (q + 2 * rows * cp * h_kv * d)
    if c["kind"] == "backward":
        return dict(bytes=esz * (3 * q + kv) + lse + grads, flops=10 * pairs * h * d)
    return dict(bytes=forward + 2 * q + grads, flops=14 * pairs * h * d)


def tolerance(c):
    # the quantiser's bytes and scales are the correctly rounded ones
    if c["kind"] == "quantize":
        return "exact"
    # Measured: the fused sweep against the per-step one (other sums, other roundings of the
    # partial results) 3.0e-3 in bf16, 3.4e-3 in e4m3 and 3.1e-4 in fp16; the gradients
    # against exact() up to 3.4e-3 in bf16, and 9.4e-3 for dq of the longest ring, whose delta
    # comes from the 16-bit out
    if c["kind"] in ("train", "backward"):
        return {"rel": 6e-3, "max": 0.5} if c["dtype"] == "fp16" else {"rel": 2e-2, "max": 0.5}
    return {"rel": 1.3e-3, "max": 0.05} if c["dtype"] == "fp16" else {"rel": 1.3e-2, "max": 0.1}


def _positions(n, cp, rank):
    """Rows of a full sequence of n that a rank holds, in its local order."""
    h = n // (2 * cp)
    a = torch.arange(h, device="cuda")
    return torch.cat([rank * h + a, (2 * cp - 1 - rank) * h + a])


def _attend(q, k, v, pos, scale, dout=None):
    """float64 causal attention of the rows q [T, H, D] at positions pos over the whole sequence
    k / v [N, H_kv, D]: (out, lse), and with dout the gradients (dq, dk, dv)."""
    (t, h, d), (n, h_kv, _) = q.shape, k.shape
    group = h // h_kv
    out, lse = torch.empty_like(q), torch.empty(t, h, dtype=torch.float64, device=q.device)
    dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    step = max(32, min(t, (1 << 27) // max(1, n)))
    for j in range(h):
        kj, vj = k[:, j // group].contiguous(), v[:, j // group].contiguous()
        kt, vt = kj.t().contiguous(), vj.t().contiguous()
        for a in range(0, t, step):
            p = pos[a:a + step]
            top = int(p.max()) + 1
            s = (q[a:a + step, j] * scale) @ kt[:, :top]
            low = int(p.min()) + 1
            if low < top:
                s[:, low:].masked_fill_(torch.arange(low, top, device=q.device)[None] > p[:, None], float("-inf"))
            m = s.amax(1, keepdim=True)
            s.sub_(m).exp_()
            l = s.sum(1, keepdim=True)
            s.div_(l)
            o = s @ vj[:top]
            out[a:a + step, j], lse[a:a + step, j] = o, (m + l.log())[:, 0]
            if dout is not None:
                g = dout[a:a + step, j].contiguous()
                dv[:top, j // group] += s.t().contiguous() @ g
                ds = s * (g @ vt[:, :top] - (g * o).sum(1, keepdim=True))
                dq[a:a + step, j] = ds @ kj[:top] * scale
                dk[:top, j // group] += ds.t().contiguous() @ q[a:a + step, j] * scale
    return out, lse, dq, dk, dv


def exact(c, seed):
    q, k, v, dout = _inputs(c, seed)
    cp, rank, d = c["cp"], c["rank"], c["d"]
    lens = _lens(c)
    cu = _bounds(lens)
    rows = [torch.cat([b + _positions(n, cp, r) for b, n in zip(cu, lens)]) for r in range(cp)]
    if c["dtype"] == "e4m3":
        def code(x):
            x, amax = x.double(), x.double().abs().amax()
            scale = torch.where(amax > 0, amax / 448, torch.ones_like(amax)).float()
            return (x / scale.double()).float().clamp(-448, 448).to(torch.float8_e4m3fn), scale

        def shards(x):
            return [code(x[r]) for r in rows]

        q8, k8, v8 = code(q[rows[rank]]), shards(k), shards(v)
        if c["kind"] == "quantize":
            return dict(q=q8[0], k=[x for x, _ in k8], v=[x for x, _ in v8], qd=q8[1], kd=[s for _, s in k8],
                        vd=[s for _, s in v8])
        ql = q8[0].double() * q8[1].double()
        k, v = k.double(), v.double()
        for r in range(cp):
            k[rows[r]] = k8[r][0].double() * k8[r][1].double()
            v[rows[r]] = v8[r][0].double() * v8[r][1].double()
    else:
        ql, k, v = q[rows[rank]].double(), k.double(), v.double()
    dl = dout[rows[rank]].double() if c["kind"] in ("train", "backward") else None
    parts, at = [], 0
    for b, n in zip(cu, lens):
        t = n // cp
        parts.append(_attend(ql[at:at + t], k[b:b + n], v[b:b + n], _positions(n, cp, rank), 1 / math.sqrt(d),
                             None if dl is None else dl[at:at + t]))
        at += t
    out, lse, dq, dk, dv = (torch.cat(x) for x in zip(*parts))
    if c["kind"] in ("forward", "perstep"):
        return dict(out=out, lse=lse)
    grads = dict(dq=dq, dk=[dk[r] for r in rows], dv=[dv[r] for r in rows])
    return grads if c["kind"] == "backward" else dict(out=out, **grads)
