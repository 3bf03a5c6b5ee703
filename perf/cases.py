"""The workloads this library is timed on: one decoded token (or one token of
every sequence of a batch) through the layers a program holds, by way of the
public binding, leap_amd.attention.

A case is a dict of plain values:
  kind       "step": HipAttention.step_async, one sequence, device buffers
             "batch": HipAttention.step_batched_async, positions on the device
             "host": HipAttention.step, host buffers (the engine's drop-in call)
             "block": HipAttention.block_async with fp32 weights
             "block_q8": the same with int8 weights, group_size values a scale
  heads, kv_heads, head_dim, theta   the model's head shape and RoPE base
  layers     layers the handle holds; a pass runs each of them once
  ctx        rows attended over, the new token's included (position ctx - 1);
             for a batch, the longest sequence's
  batch, shortest, len_seed   for a batch: sequences of shortest..ctx rows
             (the first has ctx), drawn with len_seed; shortest == ctx: equal
"""
import math
import random

import numpy as np
import torch

from leap_amd.attention import HipAttention

DEV = "cuda"

# (q heads, KV heads, head_dim, RoPE base, layers of the model)
TINY = (32, 4, 64, 10000.0, 22)
L32_3B = (24, 8, 128, 500000.0, 28)
L3_8B = (32, 8, 128, 500000.0, 32)
L2_7B = (32, 32, 128, 10000.0, 32)
L2_13B = (40, 40, 128, 10000.0, 40)
L3_70B = (64, 8, 128, 500000.0, 80)
L31_405B = (128, 8, 128, 500000.0, 126)


def _case(kind, model, layers, ctx, name=None, **more):
    c = {"kind": kind, "heads": model[0], "kv_heads": model[1], "head_dim": model[2], "theta": model[3],
         "layers": layers, "ctx": ctx, **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: every decode starts at short contexts, where a launch and one merge are all there is
        _case("step", TINY, 22, 256, "step-tinyllama-ctx256"),
        # the benchmark's headline: one token of one conversation at the model's native context
        _case("step", L3_8B, 32, 4096, "step-llama3-8b-ctx4096"),
        # long-context decode, one sequence: a gigabyte of cache a layer
        _case("step", L3_8B, 3, 131072, "step-llama3.1-8b-ctx131072"),
        # the engine's own call, host vectors in and out, at an ordinary odd context
        _case("host", L3_8B, 8, 1501, "host-llama3-8b-ctx1501"),
        # a server's full batch of conversations of all lengths
        _case("batch", L3_8B, 3, 8192, "batch64-llama3-8b-ragged8192", batch=64, shortest=512, len_seed=2),
        # a server at ordinary load: fewer and shorter conversations, odd lengths
        _case("batch", L3_8B, 12, 2011, "batch16-llama3-8b-ragged2011", batch=16, shortest=97, len_seed=5),
        # a pipeline stage of a large model, equal lengths
        _case("batch", L3_70B, 3, 8192, "batch16-llama3-70b-ctx8192", batch=16, shortest=8192, len_seed=0),
        # many short sequences of a small model, equal lengths (the same prompt answered many times)
        _case("batch", TINY, 22, 1000, "batch32-tinyllama-ctx1000", batch=32, shortest=1000, len_seed=0),
        # the attention sub-block with the engine's fp32 weights
        _case("block", L3_8B, 4, 4096, "block-llama3-8b-ctx4096"),
        # the same of a small model at an odd short context
        _case("block", TINY, 22, 499, "block-tinyllama-ctx499"),
        # the quantized engine's sub-block
        _case("block_q8", L3_8B, 10, 4096, "q8block-llama3-8b-ctx4096", group_size=64),
        # the same for the widest model without grouped heads, odd context
        _case("block_q8", L2_13B, 5, 777, "q8block-llama2-13b-ctx777", group_size=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "batch", "batch", "batch", "host", "block", "block", "block_q8", "block_q8"])
    if kind == "step" or kind == "host":
        model = rng.choice([TINY, L32_3B, L3_8B, L2_7B, L3_70B, L31_405B])
        ctx = _log_int(rng, 16, 131072 if kind == "step" and model[1] <= 8 else 16384)
        more = {}
    elif kind == "batch":
        model = rng.choice([TINY, L32_3B, L3_8B, L2_7B, L3_70B])
        batch = _log_int(rng, 2, 64)
        ctx = _log_int(rng, 64, 8192 if model[1] <= 8 else 2048)
        shortest = ctx if rng.random() < 0.3 else max(1, int(ctx * rng.uniform(0.03, 0.6)))
        more = {"batch": batch, "shortest": shortest, "len_seed": rng.randrange(1 << 16)}
    else:
        model = rng.choice([TINY, L32_3B, L3_8B, L2_7B, L2_13B, L3_70B])
        ctx = _log_int(rng, 16, 16384 if model[1] <= 8 else 4096)
        more = {"group_size": rng.choice([32, 64] if model[0] * model[2] == 5120 else [32, 64, 128])} \
            if kind == "block_q8" else {}
    case = _case(kind, model, 1, ctx, **more)
    if kind == "block_q8" and not _has_q8(case):
        case["group_size"] = 64
    # as many of the model's layers as keep a pass under 1.5 GB of traffic and its weights and cache under 24 GB
    case["layers"] = max(1, min(model[4], int(1.5e9 // work(case)["bytes"]), int(24e9 // _held(case)),
                                8 if kind == "host" else 32))
    return case


def _has_q8(c):
    # group sizes the int8 projections take, by model width
    return c["group_size"] in {2048: (32, 64, 128), 3072: (32, 64, 128), 4096: (32, 64, 128), 5120: (64, 128),
                               8192: (64, 128)}[c["heads"] * c["head_dim"]]


def _seq_len(c):
    return 1 << max(6, (c["ctx"] - 1).bit_length())


def _held(c):
    """Bytes of cache and weights of one layer."""
    dim, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    w = (2 * dim + 2 * kv) * dim * (4 if c["kind"] == "block" else 2) if c["kind"].startswith("block") else 0
    return c.get("batch", 1) * _seq_len(c) * kv * 8 + w


def lengths(c):
    """Rows of each sequence, the new token's included."""
    n = c.get("batch", 1)
    r = random.Random(c.get("len_seed", 0))
    return [c["ctx"]] + [r.randint(c.get("shortest", c["ctx"]), c["ctx"]) for _ in range(n - 1)]


def work(c):
    dim, kv, hd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["head_dim"]
    b = f = 0
    for t in lengths(c):
        # K and V rows, q in and the result out, the new k and v in and out, the table row
        b += 8 * t * kv + 8 * dim + 16 * kv + 4 * hd
        f += 4 * t * dim
    if c["kind"].startswith("block"):
        w = (2 * dim + 2 * kv) * dim
        b += 4 * w if c["kind"] == "block" else w + 4 * (w // c["group_size"])
        b += 4 * dim + 8 * dim  # the norm's weights, the residual stream in and out
        f += 2 * w
    return {"bytes": b * c["layers"], "flops": f * c["layers"]}


# ---- inputs ----------------------------------------------------------------

def _gen(seed, *what):
    s = seed & 0xFFFFFFFF
    for w in what:
        s = (s * 1000003 + w + 12345) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(s)


def _fill_cache(t, seed, seq, which):
    """Cache rows of one sequence, [layers][seq_len][kv_dim], in place: unit keys, as after RoPE, and values."""
    return t.normal_(generator=_gen(seed, 1, seq, which))


def _token(c, seed):
    """q, k and v of the new tokens, [layers][batch][...].  Queries of twice the keys' spread give scores with the
    few heavy rows that trained attention has."""
    n, L, hd = c.get("batch", 1), c["layers"], c["head_dim"]
    g = _gen(seed, 2)
    q = torch.randn(L, n, c["heads"] * hd, device=DEV, generator=g) * 2.0
    k = torch.randn(L, n, c["kv_heads"] * hd, device=DEV, generator=g)
    v = torch.randn(L, n, c["kv_heads"] * hd, device=DEV, generator=g)
    return q, k, v


def _stream_in(c, seed):
    """The residual stream ahead of each layer, [layers][dim]."""
    return torch.randn(c["layers"], c["heads"] * c["head_dim"], device=DEV, generator=_gen(seed, 3))


def _weights(c, seed, layer):
    """rms_att, Wq, Wk, Wv, Wo of a layer (fp32)."""
    dim, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    g = _gen(seed, 4, layer)
    rms = 1.0 + 0.1 * torch.randn(dim, device=DEV, generator=g)
    return [rms] + [torch.randn(rows, dim, device=DEV, generator=g) * dim ** -0.5 for rows in (dim, kv, kv, dim)]


def _quantized(w, gs):
    """int8 values and one scale per gs consecutive values of a row, as the quantized engine's files hold them."""
    g = w.reshape(-1, gs)
    s = g.abs().amax(dim=1) / 127.0
    return torch.round(g / s[:, None]).clamp(-127, 127).to(torch.int8).reshape(w.shape), s


class _DeviceArray:
    """A float32 array in device memory of a handle, for torch.as_tensor."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _caches(h, c):
    """The handle's key and value caches, [batch][layers][seq_len][kv_dim] (its sequences follow one another)."""
    shape = (c.get("batch", 1), c["layers"], _seq_len(c), c["kv_heads"] * c["head_dim"])
    return tuple(torch.as_tensor(_DeviceArray(h, p, shape), device=DEV) for p in h.kv_device_ptr(0, 0))


def prepare(c, seed):
    """A handle with its caches (and weights) filled, as a program holds it when a token comes, and the token's
    buffers."""
    n, L = c.get("batch", 1), c["layers"]
    h = HipAttention(c["heads"], c["kv_heads"], c["head_dim"], _seq_len(c), n_layers=L, rope_theta=c["theta"],
                     max_batch=n)
    rows, caches = lengths(c), _caches(h, c)
    for which, t in enumerate(caches):
        for i in range(n):
            _fill_cache(t[i], seed, i, which)
    st = {"h": h, "kind": c["kind"], "n": n, "pos": c["ctx"] - 1, "caches": caches}
    if min(rows) == c["ctx"]:
        st["new_rows"] = [t[:, :, c["ctx"] - 1] for t in caches]  # where the new tokens' k and v go
    else:
        st["at"] = torch.tensor([[(i * L + l) * _seq_len(c) + rows[i] - 1 for l in range(L)] for i in range(n)],
                                device=DEV).reshape(-1)
        st["new_rows"] = [torch.empty(n * L, t.shape[-1], device=DEV) for t in caches]
        st["rows_of"] = [t.view(-1, t.shape[-1]) for t in caches]
    if c["kind"].startswith("block"):
        for l in range(L):
            ws = _weights(c, seed, l)
            if c["kind"] == "block":
                h.set_layer_weights(l, *(w.cpu().numpy() for w in ws))
            else:
                qs = [tuple(a.cpu().numpy() for a in _quantized(w, c["group_size"])) for w in ws[1:]]
                h.set_layer_weights_q8(l, c["group_size"], ws[0].cpu().numpy(), *qs)
        st["x_in"] = _stream_in(c, seed)
        st["x"] = torch.empty_like(st["x_in"])
        st["calls"] = [st["x"][l].data_ptr() for l in range(L)]
        return st
    q, k, v = _token(c, seed)
    if c["kind"] == "host":
        st["calls"] = [tuple(a[l, 0].cpu().numpy() for a in (q, k, v)) for l in range(L)]
        return st
    out = torch.empty_like(q)
    st["bufs"], st["out"] = (q, k, v), out
    st["calls"] = [tuple(a[l].data_ptr() for a in (q, k, v, out)) for l in range(L)]
    if c["kind"] == "batch":
        st["positions"] = torch.tensor([t - 1 for t in rows], dtype=torch.int32, device=DEV)
        st["pos_ptr"], st["rows"] = st["positions"].data_ptr(), sum(rows)
    torch.cuda.synchronize()
    return st


def run(st):
    h, kind, pos = st["h"], st["kind"], st["pos"]
    if kind == "host":
        return [h.step(l, pos, q, k, v) for l, (q, k, v) in enumerate(st["calls"])], st["new_rows"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "step":
        for l, (q, k, v, out) in enumerate(st["calls"]):
            h.step_async(l, pos, q, k, v, out, stream)
        return st["out"], st["new_rows"]
    if kind == "batch":
        for l, (q, k, v, out) in enumerate(st["calls"]):
            h.step_batched_async(l, st["n"], st["pos_ptr"], pos, q, k, v, out, stream, total_rows=st["rows"])
        if "at" in st:  # the appended rows of sequences at unlike positions, gathered for the caller
            for t, to in zip(st["rows_of"], st["new_rows"]):
                torch.index_select(t, 0, st["at"], out=to)
        return st["out"], st["new_rows"]
    st["x"].copy_(st["x_in"])
    for l, x in enumerate(st["calls"]):
        h.block_async(l, pos, x, stream)
    return st["x"], st["new_rows"]


# ---- the same in 64 bits ----------------------------------------------------

def _rope(c, pos):
    """cos and sin of the pairs at a position.  The engine's table rounds the frequencies and angles to fp32, which
    is part of its definition (at position 131071 an angle's last bit is 0.008): base 500000 is a constant of its
    build, whose powers its compiler forms as exp(-i log(base)) with the exponent in fp32."""
    hd, base = c["head_dim"], c["theta"]
    i = np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)
    if base == 500000.0:
        freq = np.exp((-i * np.float32(math.log(base))).astype(np.float64)).astype(np.float32)
    else:
        freq = (1.0 / np.power(base, i.astype(np.float64))).astype(np.float32)
    a = torch.tensor((np.float32(pos) * freq).astype(np.float64), device=DEV)
    return torch.cos(a), torch.sin(a)


def _rotate(x, cs):
    p = x.reshape(-1, cs[0].numel(), 2)
    a, b = p[..., 0], p[..., 1]
    return torch.stack((a * cs[0] - b * cs[1], b * cs[0] + a * cs[1]), dim=-1).reshape(x.shape)


def _attend(c, q, kc, vc, k, v, pos):
    """One token: q [dim], cache rows kc and vc [>= pos][kv_dim], the token's k and v; 64 bits.  Returns the output
    and the rotated k."""
    hd, nkv = c["head_dim"], c["kv_heads"]
    cs = _rope(c, pos)
    q, k = _rotate(q, cs), _rotate(k, cs)
    keys = torch.cat((kc[:pos].double(), k[None])).reshape(-1, nkv, hd).permute(1, 2, 0).contiguous()
    vals = torch.cat((vc[:pos].double(), v[None])).reshape(-1, nkv, hd).permute(1, 0, 2).contiguous()
    p = torch.softmax(torch.matmul(q.reshape(nkv, -1, hd), keys) / math.sqrt(hd), dim=-1)
    return torch.matmul(p, vals).reshape(-1), k


def _project(c, w, x, rms=None):
    """W x, of rmsnorm(x) if rms is given; with both quantized per group in the int8 engine."""
    if rms is not None:
        x = rms.double() * x / torch.sqrt((x * x).mean() + 1e-5)
    if c["kind"] == "block":
        return w.double() @ x
    gs = c["group_size"]
    wq, ws = _quantized(w, gs)
    g = x.reshape(-1, gs)
    s = g.abs().amax(dim=1, keepdim=True) / 127.0
    u = g / torch.where(s > 0, s, torch.ones_like(s))
    xq = torch.sign(u) * torch.floor(u.abs() + 0.5)  # half away from zero
    return (wq.double() * ws.double().repeat_interleave(gs).reshape(w.shape)) @ (xq * s).reshape(-1)


def exact(c, seed):
    n, L, kv = c.get("batch", 1), c["layers"], c["kv_heads"] * c["head_dim"]
    rows = lengths(c)
    block = c["kind"].startswith("block")
    if block:
        x = _stream_in(c, seed).double()
    else:
        q, k, v = (a.double() for a in _token(c, seed))
    out = [[None] * n for _ in range(L)]
    new_rows = []
    for i in range(n):
        kc, vc = (_fill_cache(torch.empty(L, _seq_len(c), kv, device=DEV), seed, i, which) for which in (0, 1))
        ks, vs = [], []
        for l in range(L):
            if block:
                rms, wq, wk, wv, wo = _weights(c, seed, l)
                ql, kl, vl = (_project(c, w, x[l], rms) for w in (wq, wk, wv))
            else:
                ql, kl, vl = q[l, i], k[l, i], v[l, i]
            o, kr = _attend(c, ql, kc[l], vc[l], kl, vl, rows[i] - 1)
            out[l][i] = x[l] + _project(c, wo, o) if block else o
            ks.append(kr)
            vs.append(vl)
        new_rows.append((torch.stack(ks), torch.stack(vs)))
    new_rows = [torch.stack(t) for t in zip(*new_rows)]  # [batch][layers][kv_dim]
    if min(rows) < c["ctx"]:
        new_rows = [t.reshape(n * L, kv) for t in new_rows]
    if c["kind"] == "host":
        return [o[0].cpu().numpy() for o in out], new_rows
    if block:
        return torch.stack([o[0] for o in out]), new_rows
    return torch.stack([torch.stack(o) for o in out]), new_rows


def tolerance(c):
    # fp32 products and sums in any order: up to 6e-7 from 64 bits is measured (131072 rows).  In the int8 sub-block
    # a value that lies on a rounding boundary may move by one step, 1/127 of its group's largest: one such value
    # moves a projection's result by up to 9e-5.
    return {"rel": 4e-4 if c["kind"] == "block_q8" else 3e-6}
