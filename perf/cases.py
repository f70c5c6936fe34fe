"""The measured workloads of this library: attention as training and serving programs call it.

Three families, each through the package's public entry points:

* dense: `tilelang_flash_attn_func` on [B, S, H, D] tensors, forward only (an encoder or
  an inference prompt) or forward and backward (a training step's attention layer);
* prefill: `tilelang_paged_forward` on a vLLM-style paged cache, whole prompts, chunks
  after a cached history, and batches that mix chunks with single decode tokens;
* decode: `tilelang_decode_forward`, one token per sequence, optionally after
  `reshape_and_cache` has appended that token's K and V rows.

`listed()` names twelve of them, `draw()` gives others from the same ranges.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "tilelang-fa-v100_amd"))
import tilelang_fa_v100 as fa  # noqa: E402

DEVICE = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def dense(name, batch, sq, sk, heads, kv_heads, dim, dtype, causal, left=-1, right=-1,
          backward=True):
    return dict(name=name, kind="dense", batch=batch, sq=sq, sk=sk, heads=heads,
                kv_heads=kv_heads, dim=dim, dtype=dtype, causal=causal, left=left, right=right,
                backward=backward)


def prefill(name, seqs, q_lo, q_hi, prefix_lo, prefix_hi, singles, heads, kv_heads, dim, page,
            dtype, lens_seed, table_keys=0):
    """`seqs` sequences with q_lo..q_hi new tokens after prefix_lo..prefix_hi cached keys,
    the last `singles` of them with one new token (decode steps in a prefill batch).
    table_keys: keys the block table has room for (0: just the longest sequence)."""
    return dict(name=name, kind="prefill", seqs=seqs, q_lo=q_lo, q_hi=q_hi, prefix_lo=prefix_lo,
                prefix_hi=prefix_hi, singles=singles, heads=heads, kv_heads=kv_heads, dim=dim,
                page=page, dtype=dtype, lens_seed=lens_seed, table_keys=table_keys)


def decode(name, seqs, len_lo, len_hi, heads, kv_heads, dim, page, dtype, lens_seed,
           table_keys=0, append=False):
    return dict(name=name, kind="decode", seqs=seqs, len_lo=len_lo, len_hi=len_hi, heads=heads,
                kv_heads=kv_heads, dim=dim, page=page, dtype=dtype, lens_seed=lens_seed,
                table_keys=table_keys, append=append)


def listed():
    return [
        # A short encoder block at inference: the smallest call, one launch.
        dense("encoder_512_d64", 1, 512, 512, 16, 16, 64, "fp16", False, backward=False),
        # The training step the repository's benchmark reports.
        dense("train_2k_d128", 4, 2048, 2048, 16, 16, 128, "fp16", True),
        # Long-sequence training, the largest case.
        dense("train_8k_d128", 2, 8192, 8192, 16, 16, 128, "fp16", True),
        # Training a grouped-query model on a packed length that fills no tile evenly.
        dense("train_gqa_2000_d128", 2, 2000, 2000, 32, 8, 128, "bf16", True),
        # Training with narrow heads.
        dense("train_2k_d64", 4, 2048, 2048, 16, 16, 64, "bf16", True),
        # Training with wide heads.
        dense("train_4k_d256", 2, 4096, 4096, 8, 8, 256, "fp16", True),
        # Training a sliding-window layer.
        dense("train_window_4k_d128", 2, 4096, 4096, 16, 16, 128, "bf16", True, 1024, 0),
        # Serving: a batch of whole prompts, scattered 16-key pages.
        prefill("prompts_8_d128", 8, 512, 4096, 0, 0, 0, 32, 8, 128, 16, "fp16", 3),
        # Serving: chunked prefill, 512 new tokens after cached histories.
        prefill("chunks_16_d128", 16, 512, 512, 0, 8192, 0, 64, 8, 128, 16, "bf16", 5),
        # Serving: continuous batching, two prompt chunks among 30 decoding sequences, the
        # block table as wide as the model's longest context.
        prefill("mixed_32_d128", 32, 256, 512, 512, 8192, 30, 32, 8, 128, 16, "bf16", 7,
                table_keys=16384),
        # Serving: a large decode batch of long, uneven contexts.
        decode("decode_64_d128", 64, 1024, 32768, 32, 8, 128, 16, "fp16", 4),
        # Serving: a decode step of a few sequences, cache append and attention, the block
        # table as wide as the model's longest context.
        decode("decode_step_4_d128", 4, 512, 8192, 32, 8, 128, 16, "bf16", 9,
               table_keys=32768, append=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    dtype = rng.choice(["fp16", "bf16"])
    kind = rng.choice(["dense", "dense", "dense", "prefill", "prefill", "decode", "decode"])
    if kind == "dense":
        heads = rng.choice([8, 12, 16, 24, 32])
        kv_heads = rng.choice([heads, heads, heads // 4])
        dim = rng.choice([64, 128, 128, 256])
        sq = _log_int(rng, 100, 8192)
        sk = sq if rng.random() < 0.8 else _log_int(rng, 100, 8192)
        causal = rng.random() < 0.7 and sk >= sq
        left = _log_int(rng, 128, 2048) if causal and sk == sq and rng.random() < 0.2 else -1
        c = dense("", rng.choice([1, 2, 3, 4, 8, 16]), sq, sk, heads, kv_heads, dim, dtype,
                  causal, left, 0 if left >= 0 else -1, rng.random() < 0.7)
    elif kind == "prefill":
        heads, kv_heads = rng.choice([(32, 8), (64, 8), (16, 2), (16, 16), (28, 4)])
        seqs = _log_int(rng, 1, 48)
        prefix_hi = rng.choice([0, _log_int(rng, 256, 32768)])
        lo = _log_int(rng, 16, 2048)
        longest = prefix_hi + 2 * lo
        c = prefill("", seqs, lo, 2 * lo, prefix_hi // 4, prefix_hi,
                    rng.randint(0, seqs - 1) if prefix_hi and rng.random() < 0.5 else 0,
                    heads, kv_heads, rng.choice([64, 128, 128, 256]), rng.choice([16, 16, 32, 64]),
                    dtype, rng.randrange(1 << 20), rng.choice([0, 2 * longest]))
    else:
        heads, kv_heads = rng.choice([(32, 8), (64, 8), (16, 2), (16, 16), (28, 4)])
        hi = _log_int(rng, 256, 32768)
        c = decode("", _log_int(rng, 1, 128), max(1, hi // 16), hi, heads, kv_heads,
                   rng.choice([64, 128, 128, 256, 512]), rng.choice([16, 16, 32, 64]), dtype,
                   rng.randrange(1 << 20), rng.choice([0, 2 * hi]), rng.random() < 0.5)
    c.pop("name")
    return c


def draw(rng):
    most = work(next(c for c in listed() if c["name"] == "train_8k_d128"))["flops"]
    wide = work(next(c for c in listed() if c["name"] == "decode_64_d128"))["bytes"]
    while True:
        c = _draw(rng)
        w = work(c)
        # Sizes whose cost stays below the largest listed case; a decode step that returns its
        # caches keeps them small.
        if w["flops"] <= most / 3 and w["bytes"] <= wide / (6 if c.get("append") else 1):
            return c


# ------------------------------------------------------------------ sizes

def _lens(case):
    """(new tokens, total keys) of every sequence of a paged case."""
    r = random.Random(case["lens_seed"])
    if case["kind"] == "decode":
        return [1] * case["seqs"], [r.randint(case["len_lo"], case["len_hi"])
                                    for _ in range(case["seqs"])]
    new, total = [], []
    for i in range(case["seqs"]):
        one = i >= case["seqs"] - case["singles"]
        n = 1 if one else r.randint(case["q_lo"], case["q_hi"])
        new.append(n)
        total.append(n + r.randint(case["prefix_lo"], case["prefix_hi"]))
    return new, total


def _dense_pairs(case):
    sq, sk = case["sq"], case["sk"]
    left = case["left"]
    right = 0 if case["causal"] else case["right"]
    off = sk - sq
    pairs = 0
    for i in range(sq):
        hi = sk if right < 0 else max(0, min(sk, i + off + right + 1))
        lo = 0 if left < 0 else min(sk, max(0, i + off - left))
        pairs += max(0, hi - lo)
    return pairs


def work(case):
    H, D = case["heads"], case["dim"]
    Hk = case["kv_heads"]
    if case["kind"] == "dense":
        B = case["batch"]
        flops = 4 * D * H * B * _dense_pairs(case)
        nbytes = 2 * D * B * (2 * case["sq"] * H + 2 * case["sk"] * Hk)
        if case["backward"]:
            # Five products for the forward's two; reads q, k, v, out, dout, writes dq, dk, dv.
            return {"bytes": nbytes + 2 * D * B * (4 * case["sq"] * H + 4 * case["sk"] * Hk),
                    "flops": 3.5 * flops}
        return {"bytes": nbytes, "flops": flops}
    new, total = _lens(case)
    pairs = sum(sum(t - n + i + 1 for i in range(n)) for n, t in zip(new, total))
    table = sum(4 * -(-t // case["page"]) + 4 for t in total)
    kv = 2 * 2 * D * Hk * sum(total)
    qo = 2 * 2 * D * H * sum(new)
    append = 2 * 2 * 2 * D * Hk * sum(new) if case.get("append") else 0
    lse = 4 * H * sum(new) if case["kind"] == "prefill" else 0
    return {"bytes": kv + qo + table + append + lse, "flops": 4 * D * H * pairs}


# ------------------------------------------------------------------ inputs

def _paged_state(case, g):
    new, total = _lens(case)
    page, Hk, D, H = case["page"], case["kv_heads"], case["dim"], case["heads"]
    dtype = DTYPES[case["dtype"]]
    pages = [-(-t // page) for t in total]
    # Pages are handed out from a shared pool in no order; the table's unused entries hold -1.
    perm = torch.randperm(sum(pages), generator=g, device=DEVICE).to(torch.int32)
    width = max(max(pages), -(-case["table_keys"] // page))
    table = torch.full((len(total), width), -1, dtype=torch.int32, device=DEVICE)
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        at += n

    def mk(*shape):
        return torch.randn(*shape, generator=g, device=DEVICE, dtype=dtype)

    st = {"case": case, "q": mk(sum(new), H, D), "k_cache": mk(sum(pages), page, Hk, D),
          "v_cache": mk(sum(pages), page, Hk, D), "block_table": table,
          "seq_lens": torch.tensor(total, dtype=torch.int32, device=DEVICE)}
    return st, new, total, mk


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    if case["kind"] == "dense":
        B, H, Hk, D = case["batch"], case["heads"], case["kv_heads"], case["dim"]
        dtype = DTYPES[case["dtype"]]

        def mk(s, h):
            return torch.randn(B, s, h, D, generator=g, device=DEVICE, dtype=dtype)

        st = {"case": case, "q": mk(case["sq"], H), "k": mk(case["sk"], Hk),
              "v": mk(case["sk"], Hk)}
        if case["backward"]:
            st["dout"] = mk(case["sq"], H)
            for n in ("q", "k", "v"):
                st[n].requires_grad_()
        return st
    st, new, total, mk = _paged_state(case, g)
    if case["kind"] == "prefill":
        starts = [0]
        for n in new:
            starts.append(starts[-1] + n)
        st["query_start_loc"] = torch.tensor(starts, dtype=torch.int32, device=DEVICE)
        st["prefix_kv_lens"] = torch.tensor([t - n for n, t in zip(new, total)],
                                            dtype=torch.int32, device=DEVICE)
    elif case["append"]:
        st["key"], st["value"] = mk(len(new), case["kv_heads"], case["dim"]), \
            mk(len(new), case["kv_heads"], case["dim"])
        last = st["seq_lens"].long() - 1
        row = torch.arange(len(total), device=DEVICE)
        st["slots"] = st["block_table"][row, last // case["page"]].long() * case["page"] \
            + last % case["page"]
    return st


def run(st):
    case = st["case"]
    if case["kind"] == "dense":
        q, k, v = st["q"], st["k"], st["v"]
        window = (case["left"], case["right"])
        if not case["backward"]:
            return fa.tilelang_flash_attn_func(q, k, v, causal=case["causal"],
                                               window_size=window)
        q.grad = k.grad = v.grad = None
        out = fa.tilelang_flash_attn_func(q, k, v, causal=case["causal"], window_size=window)
        out.backward(st["dout"])
        return {"out": out, "dq": q.grad, "dk": k.grad, "dv": v.grad}
    if case["kind"] == "prefill":
        out, lse = fa.tilelang_paged_forward(
            st["q"], st["k_cache"], st["v_cache"], st["block_table"], st["seq_lens"],
            st["query_start_loc"], st["prefix_kv_lens"], block_size=case["page"])
        return {"out": out, "lse": lse}
    if case["append"]:
        fa.reshape_and_cache(st["key"], st["value"], st["k_cache"], st["v_cache"], st["slots"])
    out = fa.tilelang_decode_forward(st["q"], st["k_cache"], st["v_cache"], st["block_table"],
                                     st["seq_lens"], block_size=case["page"])
    if case["append"]:
        return {"out": out, "k_cache": st["k_cache"], "v_cache": st["v_cache"]}
    return {"out": out}


# ------------------------------------------------------------------ what is right

def tolerance(case):
    # About four times the present kernels' distance from 64 bits (measured over the listed
    # cases and 14 drawn ones).  Relative: fp16 2.2e-4 .. 2.9e-4 for outputs and up to 3.1e-4
    # for gradients, bf16 up to 2.4e-3 and 2.5e-3; both are the rounding of the probabilities
    # and of the result itself to the type.  Largest: a causal row that sees a few keys, or a
    # gradient that cancels, sits far above the root mean square of a long sequence (fp16
    # 6.7e-3 and 2.5e-2 at 8192 keys, bf16 3.3e-2 and 1.1e-1 at 2000 to 8192).
    half = case["dtype"] == "fp16"
    if case["kind"] == "dense" and case["backward"]:
        return {"rel": 0.00125, "max": 0.1} if half else {"rel": 0.01, "max": 0.45}
    return {"rel": 0.0011, "max": 0.03} if half else {"rel": 0.0095, "max": 0.15}


def _exact_dense(case, st):
    with torch.no_grad():
        q, k, v = (st[n].double() for n in ("q", "k", "v"))
        B, Sq, H, D = q.shape
        Sk, G = k.shape[1], H // k.shape[2]
        scale = D ** -0.5
        right = 0 if case["causal"] else case["right"]
        i = torch.arange(Sq, device=q.device)[:, None] + (Sk - Sq)
        j = torch.arange(Sk, device=q.device)[None, :]
        hidden = torch.zeros(Sq, Sk, dtype=torch.bool, device=q.device)
        if right >= 0:
            hidden |= j > i + right
        if case["left"] >= 0:
            hidden |= j < i - case["left"]
        out = torch.zeros_like(q)
        if case["backward"]:
            do = st["dout"].double()
            dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for b in range(B):
            for h in range(H):
                qh, kh, vh = q[b, :, h], k[b, :, h // G], v[b, :, h // G]
                p = torch.softmax((qh @ kh.t() * scale).masked_fill_(hidden, -math.inf), -1)
                out[b, :, h] = o = p @ vh
                if case["backward"]:
                    doh = do[b, :, h]
                    dv[b, :, h // G] += p.t() @ doh
                    ds = doh @ vh.t()
                    ds -= (o * doh).sum(-1, keepdim=True)
                    ds.mul_(p).mul_(scale)
                    dq[b, :, h] = ds @ kh
                    dk[b, :, h // G] += ds.t() @ qh
        if case["backward"]:
            return {"out": out, "dq": dq, "dk": dk, "dv": dv}
        return out


def _exact_paged(case, st):
    new, total = _lens(case)
    H, D, Hk, page = case["heads"], case["dim"], case["kv_heads"], case["page"]
    G = H // Hk
    kc, vc = st["k_cache"], st["v_cache"]
    if case.get("append"):
        kc.view(-1, Hk, D)[st["slots"]] = st["key"]
        vc.view(-1, Hk, D)[st["slots"]] = st["value"]
    out = torch.zeros(st["q"].shape, dtype=torch.float64, device=DEVICE)
    lse = torch.zeros(H, sum(new), dtype=torch.float64, device=DEVICE)
    at = 0
    for b, (n, t) in enumerate(zip(new, total)):
        rows = st["block_table"][b, :-(-t // page)].long()
        k = kc[rows].reshape(-1, Hk, D)[:t].double()
        v = vc[rows].reshape(-1, Hk, D)[:t].double()
        i = torch.arange(n, device=DEVICE)[:, None] + (t - n)
        hidden = torch.arange(t, device=DEVICE)[None, :] > i
        for h in range(H):
            s = st["q"][at:at + n, h].double() @ k[:, h // G].t() * D ** -0.5
            s.masked_fill_(hidden, -math.inf)
            lse[h, at:at + n] = torch.logsumexp(s, -1)
            out[at:at + n, h] = torch.softmax(s, -1) @ v[:, h // G]
        at += n
    if case["kind"] == "prefill":
        return {"out": out, "lse": lse}
    if case["append"]:
        return {"out": out, "k_cache": kc.double(), "v_cache": vc.double()}
    return {"out": out}


def exact(case, seed):
    st = prepare(case, seed)
    return _exact_dense(case, st) if case["kind"] == "dense" else _exact_paged(case, st)
