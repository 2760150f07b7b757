"""Workloads of the KIVI cache library by which its speed is followed, through the Python binding
of its device entry points (the calls a serving loop makes).

Five paths, each over the sizes, head widths, groups and code widths it is used with:

  attn      one decode-attention call over a filled cache (``KiviCache.attention_device``)
  serve     one request: ``RuntimeKv`` made, prompt appended, `steps` decode steps, freed
  prefill   a cache made, the prompt appended in `pieces`, its content taken out as packed
            streams (handed to another worker) or as dense rows, freed
  sessions  one batched attention call over sessions that share a prefix
  codec     ``quantize_per_channel`` and ``quantize_per_token`` of device tensors, then the
            PyTorch-order codes and the dense reconstruction of both

Keys are N(0, 1) with 1% of each KV head's channels ten times larger, values N(0, 1): the
distribution the library's benchmark uses. `exact` restates the format in plain torch: codes,
scales and zeros by the format's own float32 rule (they are defined bit for bit), everything
computed from them in float64."""
import importlib.util
import math
import os

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """kivi-cache-rs_amd/kivi.py (the folder's name is no module name)."""
    spec = importlib.util.spec_from_file_location("kivi", os.path.join(_ROOT, "kivi-cache-rs_amd", "kivi.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


kivi = _package()


# ---------------------------------------------------------------- the cases


def _case(path, name, batch, kv, q, dim, tokens, bits, group, residual, **more):
    c = {"path": path, "batch": batch, "kv_heads": kv, "q_heads": q, "head_dim": dim,
         "tokens": tokens, "bits": bits, "group": group, "residual": residual}
    if name is not None:
        c["name"] = name
    c.update(more)
    return c


def listed():
    return [
        # one user's short chat, a layer of a small model without grouped heads: latency alone
        _case("attn", "attn one short sequence", 1, 8, 8, 128, 4097, 2, 32, 128),
        # a full batch of long chats, grouped heads: the library's benchmark workload
        _case("attn", "attn batch of long sequences", 16, 8, 32, 128, 32768, 2, 32, 128),
        # one very long document, eight query heads per KV head, wider codes
        _case("attn", "attn one 131072-token sequence", 1, 8, 64, 128, 131072, 4, 32, 128),
        # small-model heads, larger groups, a length that fills no block
        _case("attn", "attn head_dim 64, group 64", 5, 8, 32, 64, 12345, 2, 64, 128),
        # heads of 96 channels without grouping, a short window, a ragged length
        _case("attn", "attn head_dim 96", 3, 32, 32, 96, 5003, 4, 32, 64),
        # one request of a chat: prompt of 8192 tokens, 256 tokens out (two key flushes)
        _case("serve", "serve one request", 1, 8, 32, 128, 8192, 2, 32, 128, steps=256),
        # a small batch of short requests, seven query heads per KV head, 4-bit codes
        _case("serve", "serve a small batch", 4, 4, 28, 128, 777, 4, 32, 128, steps=100),
        # a batch of long prompts encoded and handed on as packed streams
        _case("prefill", "prefill a long batch, streams", 16, 8, 8, 128, 32768, 2, 32, 128, pieces=1, give="streams"),
        # a chunked prompt of ragged pieces whose dense reconstruction is wanted (8-bit)
        _case("prefill", "prefill in pieces, dense", 2, 8, 8, 96, 2999, 8, 32, 96, pieces=3, give="dense"),
        # 64 questions on one 65536-token document
        _case("sessions", "64 sessions on a long prefix", 1, 8, 32, 128, 65536, 2, 32, 128, sessions=64, suffix=96),
        # a handful of sessions on a shorter one, ragged questions, 8-bit codes
        _case("sessions", "5 sessions on a prefix", 1, 8, 16, 128, 10007, 8, 32, 128, sessions=5, suffix=150),
        # standalone tensors encoded, re-ordered for PyTorch and decoded
        _case("codec", "codec round trip", 4, 8, 8, 128, 8192, 4, 32, 32),
    ]


def _odd_log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: Elements of one key tensor: the largest listed case (16 x 8 heads x 32768 tokens x 128).
_MOST = 16 * 8 * 32768 * 128


def draw(rng):
    path = rng.choice(["attn", "attn", "serve", "prefill", "sessions", "codec"])
    bits = rng.choice([2, 2, 4, 8])
    dim = rng.choice([128] * 6 + [64, 64, 80, 96, 96, 256])
    groups = [g for g in (32, 32, 32, 32, 64, 16, 128) if dim % g == 0 and g * bits % 32 == 0]
    if not groups:  # 80 channels at two bits: groups of 16
        groups = [16]
    group = rng.choice(groups)
    residual = group * rng.choice([1, 2, 4]) if group < 128 else group
    kv = rng.choice([1, 2, 4, 8, 8, 8, 16, 32])
    gq = rng.choice([1, 1, 2, 3, 4, 4, 7, 8, 16] if kv <= 8 else [1, 1, 2])
    batch = _odd_log(rng, 1, 24)
    tokens = _odd_log(rng, 200, 131072)
    more = {}
    if path == "serve":
        tokens, more["steps"] = _odd_log(rng, 100, 16384), _odd_log(rng, 32, 300)
        batch = min(batch, 8)
    elif path == "prefill":
        more["pieces"], more["give"] = rng.choice([1, 1, 2, 5]), rng.choice(["streams", "dense"])
        gq = 1
    elif path == "sessions":
        batch, kv = 1, rng.choice([4, 8, 8])
        gq = rng.choice([1, 2, 4, 4, 7, 8])
        tokens = _odd_log(rng, 500, 65536)
        more["sessions"], more["suffix"] = _odd_log(rng, 2, 64), _odd_log(rng, 8, 300)
    elif path == "codec":
        gq = 1
        tokens = max(1, tokens // group) * group  # whole key groups
    while batch > 1 and batch * kv * tokens * dim > _MOST:
        batch -= 1
    case = _case(path, None, batch, kv, kv * gq, dim, tokens, bits, group, residual, **more)
    # no more than the largest listed cases move (a prefill) and compute (the 64 sessions)
    most = [work(c) for c in listed()]
    while any(work(case)[what] > max(m[what] for m in most) for what in ("bytes", "flops")):
        tokens = max(1, tokens // 2 // group) * group + (tokens % group if path != "codec" else 0)
        case["tokens"] = tokens
        if "steps" in case and tokens < 1000:
            case["steps"] = case["steps"] // 2 + 1
    return case


# ---------------------------------------------------------------- inputs


def _rng(seed, salt):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)


def _keys(c, seed, n, salt, batch=None):
    """[batch * kv_heads, n, head_dim]; 1% of each KV head's channels (at least one) x10, the same
    ones for every token."""
    units = (batch or c["batch"]) * c["kv_heads"]
    k = torch.randn(units, n, c["head_dim"], generator=_rng(seed, salt), device="cuda")
    many = max(1, round(c["head_dim"] / 100))
    hot = torch.rand(units, c["head_dim"], generator=_rng(seed, 1), device="cuda").topk(many, 1).indices
    factor = torch.ones(units, c["head_dim"], device="cuda").scatter_(1, hot, 10.0)
    return k.mul_(factor[:, None, :])


def _values(c, seed, n, salt, batch=None):
    units = (batch or c["batch"]) * c["kv_heads"]
    return torch.randn(units, n, c["head_dim"], generator=_rng(seed, salt), device="cuda")


def _queries(c, seed, n, salt):
    return torch.randn(n, c["batch"], c["q_heads"], c["head_dim"], generator=_rng(seed, salt), device="cuda")


def _suffix_lengths(c):
    """Ragged questions of up to `suffix` tokens; with `sessions` >= 32 all of that length (the
    batched benchmark's form)."""
    n, most = c["sessions"], c["suffix"]
    return [most] * n if n >= 32 else [max(1, most * (i + 1) // n - i % 3) for i in range(n)]


def _piece_sizes(c):
    n, pieces = c["tokens"], c["pieces"]
    edges = [round(n * (i + 1) / pieces + (3 if i + 1 < pieces else 0)) for i in range(pieces)]
    return [b - a for a, b in zip([0] + edges[:-1], edges)]


def _config(c):
    return kivi.KiviConfig(c["bits"], c["group"], c["residual"])


def _scale(c):
    return 1.0 / math.sqrt(c["head_dim"])


def _packed(c, tokens):
    """(packed key tokens, packed value tokens) of a cache that holds `tokens`."""
    r = c["residual"]
    return tokens // r * r, max(0, tokens - r)


def _stream():
    return torch.cuda.current_stream().cuda_stream


class _State:
    """What the program has in hand: tensors and handles by name."""

    def __init__(self, case, **held):
        self.case = case
        self.__dict__.update(held)


def _filled(c, seed):
    """A cache with the case's tokens in it."""
    cache = kivi.KiviCache(kivi.Backend.amd(), _config(c), c["batch"], c["kv_heads"], c["head_dim"])
    cache.reserve(c["tokens"])
    k, v = _keys(c, seed, c["tokens"], 2), _values(c, seed, c["tokens"], 3)
    cache.append_device(k.data_ptr(), k.numel(), v.data_ptr(), v.numel(), c["tokens"], _stream())
    torch.cuda.current_stream().synchronize()  # k and v are let go
    return cache


def prepare(case, seed):
    c, path = case, case["path"]
    amd = kivi.Backend.amd()
    units, dim = c["batch"] * c["kv_heads"], c["head_dim"]
    if path == "attn":
        q = _queries(c, seed, 1, 4)[0]
        return _State(c, cache=_filled(c, seed), q=q, out=torch.empty_like(q))
    if path == "serve":
        k, v = _keys(c, seed, c["tokens"], 2), _values(c, seed, c["tokens"], 3)
        # one row per step: [steps][units][dim]
        sk = _keys(c, seed, c["steps"], 5).transpose(0, 1).contiguous()
        sv = _values(c, seed, c["steps"], 6).transpose(0, 1).contiguous()
        q = _queries(c, seed, c["steps"], 4)
        return _State(c, amd=amd, k=k, v=v, sk=sk, sv=sv, q=q, out=torch.empty_like(q))
    if path == "prefill":
        n = c["tokens"]
        k, v = _keys(c, seed, n, 2), _values(c, seed, n, 3)
        pieces, at = [], 0
        for m in _piece_sizes(c):
            pieces.append((k[:, at:at + m].contiguous(), v[:, at:at + m].contiguous()))
            at += m
        if c["give"] == "dense":
            outs = [torch.empty(units, n, dim, device="cuda") for _ in range(2)]
        else:
            kq, vq = _packed(c, n)
            w = 32 // c["bits"]
            outs = [torch.empty(units * kq * dim // w, dtype=torch.int32, device="cuda"),
                    torch.empty(units, kq // c["group"], dim, 2, device="cuda"),
                    torch.empty(units * vq * dim // w, dtype=torch.int32, device="cuda"),
                    torch.empty(units, vq, dim // c["group"], 2, device="cuda")]
        return _State(c, amd=amd, pieces=pieces, outs=outs)
    if path == "sessions":
        prefix = _filled(c, seed).share_prefix()
        sessions = []
        for i, n in enumerate(_suffix_lengths(c)):
            s = prefix.session()
            k, v = _keys(c, seed, n, 100 + 2 * i), _values(c, seed, n, 101 + 2 * i)
            s.append_device(k.data_ptr(), k.numel(), v.data_ptr(), v.numel(), n, _stream())
            torch.cuda.current_stream().synchronize()  # k and v are let go
            sessions.append(s)
        q = _queries(c, seed, c["sessions"], 4)
        return _State(c, amd=amd, prefix=prefix, sessions=sessions, handles=kivi.session_handles(sessions),
                      q=q, out=torch.empty_like(q))
    if path == "codec":
        k, v = _keys(c, seed, c["tokens"], 2), _values(c, seed, c["tokens"], 3)
        words = k.numel() // (32 // c["bits"])
        return _State(c, amd=amd, k=k, v=v,
                      codes=[torch.empty(words, dtype=torch.int32, device="cuda") for _ in range(2)],
                      dense=[torch.empty_like(k), torch.empty_like(v)])
    raise ValueError(path)


# ---------------------------------------------------------------- one pass


def run(state):
    c, path, stream = state.case, state.case["path"], _stream()
    if path == "attn":
        state.cache.attention_device(state.q.data_ptr(), state.q.numel(), c["q_heads"], _scale(c),
                                     state.out.data_ptr(), state.out.numel(), stream)
        return state.out
    if path == "serve":
        rt = kivi.RuntimeKv(state.amd, _config(c), c["batch"], c["kv_heads"], c["head_dim"])
        cache = rt.cache()
        cache.reserve(c["tokens"] + c["steps"])
        cache.append_device(state.k.data_ptr(), state.k.numel(), state.v.data_ptr(), state.v.numel(),
                            c["tokens"], stream)
        n_kv, n_q, scale = state.sk[0].numel(), state.q[0].numel(), _scale(c)
        kp, vp, qp, op = (t.data_ptr() for t in (state.sk, state.sv, state.q, state.out))
        for i in range(c["steps"]):
            rt.decode_device(kp + 4 * i * n_kv, n_kv, vp + 4 * i * n_kv, n_kv, qp + 4 * i * n_q, n_q,
                             c["q_heads"], scale, op + 4 * i * n_q, n_q, stream)
        return state.out
    if path == "prefill":
        cache = kivi.KiviCache(state.amd, _config(c), c["batch"], c["kv_heads"], c["head_dim"])
        for k, v in state.pieces:
            cache.append_device(k.data_ptr(), k.numel(), v.data_ptr(), v.numel(), k.shape[1], stream)
        if c["give"] == "dense":
            k, v = state.outs
            cache.dequantize_device(k.data_ptr(), k.numel(), v.data_ptr(), v.numel(), stream)
        else:
            cache.export_streams_device([t.data_ptr() for t in state.outs], [t.numel() for t in state.outs], stream)
        return state.outs
    if path == "sessions":
        kivi.sessions_attention_device(state.amd, state.sessions, state.q.data_ptr(), state.q.numel(),
                                       c["q_heads"], _scale(c), state.out.data_ptr(), state.out.numel(),
                                       stream, handles=state.handles)
        return state.out
    if path == "codec":
        shape = (c["batch"], c["kv_heads"], c["tokens"], c["head_dim"], c["bits"], c["group"])
        for i, x in enumerate((state.k, state.v)):
            t = kivi.quantize_device(state.amd, i == 0, x.data_ptr(), x.numel(), *shape, stream)
            t.pytorch_codes_device(state.codes[i].data_ptr(), state.codes[i].numel(), stream)
            t.dequantize_device(state.dense[i].data_ptr(), state.dense[i].numel(), stream)
        return state.codes + state.dense
    raise ValueError(path)


# ---------------------------------------------------------------- what a pass cannot do without


def _cache_bytes(c, tokens, units=None):
    """Packed codes and (scale, zero) pairs plus the float32 rows of a cache of `tokens`."""
    units = c["batch"] * c["kv_heads"] if units is None else units
    kq, vq = _packed(c, tokens)
    d, g, b = c["head_dim"], c["group"], c["bits"]
    packed = (kq + vq) * (d * b / 8 + d / g * 8)
    return units * (packed + (2 * tokens - kq - vq) * d * 4)


def work(case):
    c, path, dim = case, case["path"], case["head_dim"]
    rows = c["batch"] * c["kv_heads"] * c["tokens"] * dim * 4.0  # one dense tensor of the case
    heads = c["batch"] * c["q_heads"]
    if path == "attn":
        return {"bytes": _cache_bytes(c, c["tokens"]) + 2 * heads * dim * 4, "flops": 4.0 * heads * dim * c["tokens"]}
    if path == "serve":
        spent, flops = 2 * rows + _cache_bytes(c, c["tokens"]), 0.0
        for i in range(1, c["steps"] + 1):
            spent += _cache_bytes(c, c["tokens"] + i) + 2 * heads * dim * 4
            flops += 4.0 * heads * dim * (c["tokens"] + i)
        return {"bytes": spent, "flops": flops}
    if path == "prefill":
        out = 2 * rows if c["give"] == "dense" else _cache_bytes(c, c["tokens"])
        return {"bytes": 2 * rows + out, "flops": 4.0 * rows / 4}
    if path == "sessions":
        extra = sum(_suffix_lengths(c))
        n = c["sessions"]
        return {"bytes": _cache_bytes(c, c["tokens"]) + 2 * extra * c["kv_heads"] * dim * 4 + 2 * n * heads * dim * 4,
                "flops": 4.0 * heads * dim * (n * c["tokens"] + extra)}
    words = 2 * (rows / 4) * c["bits"] / 8
    return {"bytes": 4 * rows + words, "flops": 8.0 * rows / 4}


def tolerance(case):
    # Codes, (scale, zero) pairs and dense rows are defined bit for bit; attention is a float32
    # softmax whose sums may be taken in any order (float64 against it: see `exact`).
    if case["path"] in ("prefill", "codec"):
        return "exact"
    return {"rel": 2e-5, "max": 2e-4}


# ---------------------------------------------------------------- the same in plain torch


def _coded(x, levels):
    """(codes, scale, zero) of groups along the last axis by the format's float32 rule:
    scale = span / levels, code = round-half-even((x - zero) / scale)."""
    zero, top = x.min(-1, keepdim=True).values, x.max(-1, keepdim=True).values
    scale = (top - zero) / torch.full_like(top, levels)  # by a tensor: torch takes a number's reciprocal
    safe = torch.where(scale == 0, torch.ones_like(scale), scale)
    return torch.where(scale == 0, torch.zeros_like(x), ((x - zero) / safe).round_().clamp_(0, levels)), scale, zero


def _decoded(x, levels):
    codes, scale, zero = _coded(x, levels)
    return codes.double() * scale.double() + zero.double()


def _key_rows(c, k):
    """Keys [n, d] of one unit, n whole groups, quantized per channel and reconstructed."""
    g = c["group"]
    return _decoded(k.view(-1, g, k.shape[-1]).transpose(1, 2).contiguous(), 2 ** c["bits"] - 1).transpose(1, 2).reshape(k.shape)


def _value_rows(c, v):
    return _decoded(v.view(v.shape[0], -1, c["group"]), 2 ** c["bits"] - 1).reshape(v.shape)


def _held(c, k, v):
    """What a cache holds of one unit's rows [n, d], as float64 rows."""
    kq, vq = _packed(c, k.shape[0])
    kd, vd = k.double(), v.double()
    if kq:
        kd[:kq] = _key_rows(c, k[:kq])
    if vq:
        vd[:vq] = _value_rows(c, v[:vq])
    return kd, vd


def _attend(q, k, v, scale):
    """q [heads, d] over rows k, v [n, d], in float64."""
    return torch.softmax((q.double() @ k.t()) * scale, dim=-1) @ v


def exact(case, seed):
    c, path = case, case["path"]
    units, kv, dim = c["batch"] * c["kv_heads"], c["kv_heads"], c["head_dim"]
    gq, scale = c["q_heads"] // c["kv_heads"], _scale(c)
    n = c["tokens"]
    k, v = _keys(c, seed, n, 2), _values(c, seed, n, 3)
    if path == "attn":
        q = _queries(c, seed, 1, 4)[0].view(units, gq, dim)
        return torch.stack([_attend(q[u], *_held(c, k[u], v[u]), scale) for u in range(units)]).view(c["batch"], -1, dim)
    if path == "serve":
        if units * c["steps"] * n > 32 * 300 * 8192:
            return None  # a float64 attention of the whole cache per step and unit
        sk, sv = _keys(c, seed, c["steps"], 5), _values(c, seed, c["steps"], 6)
        q = _queries(c, seed, c["steps"], 4)
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda").view(c["steps"], units, gq, dim)
        qv = q.view(c["steps"], units, gq, dim)
        for u in range(units):
            # every row as it is once packed; a step takes its float32 rows from the input
            ku, vu = torch.cat([k[u], sk[u]]), torch.cat([v[u], sv[u]])
            whole = ku.shape[0] // c["group"] * c["group"]
            kp, vp = _key_rows(c, ku[:whole]), _value_rows(c, vu)
            kf, vf = ku.double(), vu.double()
            for i in range(c["steps"]):
                m = n + i + 1
                kq, vq = _packed(c, m)
                out[i, u] = _attend(qv[i, u], torch.cat([kp[:kq], kf[kq:m]]), torch.cat([vp[:vq], vf[vq:m]]), scale)
        return out.view(q.shape)
    if path == "prefill":
        if c["give"] == "dense":
            both = [torch.empty(units, n, dim, dtype=torch.float64, device="cuda") for _ in range(2)]
            for u in range(units):
                both[0][u], both[1][u] = _held(c, k[u], v[u])
            return both
        levels, g = 2 ** c["bits"] - 1, c["group"]
        kq, vq = _packed(c, n)

        def pairs(x):
            zero, top = x.amin(-1).double(), x.amax(-1).double()
            return torch.stack([(top - zero) / levels, zero], -1)

        kp = torch.stack([pairs(k[u, :kq].view(-1, g, dim).transpose(1, 2)) for u in range(units)])
        vp = torch.stack([pairs(v[u, :vq].view(vq, -1, g)) for u in range(units)])
        return [None, kp, None, vp]
    if path == "sessions":
        q = _queries(c, seed, c["sessions"], 4).view(c["sessions"], units, gq, dim)
        out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        held = [_held(c, k[u], v[u]) for u in range(units)]
        for i, m in enumerate(_suffix_lengths(c)):
            sk, sv = _keys(c, seed, m, 100 + 2 * i).double(), _values(c, seed, m, 101 + 2 * i).double()
            for u in range(units):
                out[i, u] = _attend(q[i, u], torch.cat([held[u][0], sk[u]]), torch.cat([held[u][1], sv[u]]), scale)
        return out.view(c["sessions"], c["batch"], -1, dim)
    if path == "codec":
        both = [torch.empty(units, n, dim, dtype=torch.float64, device="cuda") for _ in range(2)]
        for u in range(units):
            both[0][u], both[1][u] = _key_rows(c, k[u]), _value_rows(c, v[u])
        return [None, None] + both
    raise ValueError(path)
