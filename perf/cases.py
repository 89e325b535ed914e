"""The work that a user of this framework has it do, as cases that can be timed.

``listed()`` is a fixed selection, ``draw(rng)`` gives further cases of the same ranges.  The kinds:

attn      the dense fused-bias op: encoder self-attention or a decoder prompt (causal), forward alone or forward
          and backward
packed    the packed variable-length op on sequences laid back to back
sparse    the long-document ops: sliding window, blocks with leading global tokens, window with side tokens
decode    one decoding step's cross-attention of a batch over its encoder memories
encoder   a whole T5 encoder: a forward pass, or a training step's forward and backward on a right-padded batch

q, k and v have the layout that the attention modules hand over, (B, H, L, D) views of (B, L, H*D) projections, and
scores of deviation around 2; T5 scores carry no 1/sqrt(d).
"""
import math

import numpy as np
import torch

import turbot5_amd as t5
from turbot5_amd import ops

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# T5-small and T5-base encoders
SMALL = {"d_model": 512, "d_ff": 2048, "layers": 6, "H": 8, "D": 64}
BASE = {"d_model": 768, "d_ff": 3072, "layers": 12, "H": 12, "D": 64}


def listed():
    return [
        # a single short prompt through a small model's attention: launch and host latency are all there is
        dict(name="prompt_short", kind="attn", B=1, H=8, L=100, D=64, dtype="bf16", causal=False, train=False),
        # an encoder batch of ordinary length, T5-base heads
        dict(name="encoder_batch", kind="attn", B=16, H=12, L=1024, D=64, dtype="bf16", causal=False, train=False),
        # a serving batch of ragged requests, packed without padding
        dict(name="packed_ragged", kind="packed", n_seq=32, min_len=128, max_len=4096, H=12, D=64, dtype="bf16",
             causal=False, train=False),
        # one long document in each of the long-input attention types
        dict(name="local_long", kind="sparse", pattern="local", B=1, H=12, L=16384, D=64, dtype="bf16", block_len=128, aux=0),
        dict(name="block_pair_fp16", kind="sparse", pattern="block", B=2, H=12, L=7900, D=64, dtype="fp16", block_len=128,
             aux=64),
        dict(name="tglobal_long", kind="sparse", pattern="tglobal", B=1, H=12, L=16384, D=64, dtype="bf16", block_len=128,
             aux=16),
        # a decoding step of a full serving batch over long memories
        dict(name="decode_memory", kind="decode", B=64, H=12, N=8192, D=64, dtype="bf16", ragged=False),
        # training: attention forward and backward of an encoder batch
        dict(name="train_batch", kind="attn", B=16, H=12, L=1024, D=64, dtype="bf16", causal=False, train=True),
        # ... of a small model in full precision
        dict(name="train_small_fp32", kind="attn", B=4, H=8, L=512, D=64, dtype="fp32", causal=False, train=True),
        # ... of the decoder of a model with wide heads, odd length
        dict(name="train_causal_d128", kind="attn", B=2, H=8, L=1999, D=128, dtype="bf16", causal=True, train=True),
        # two documents of 8192 tokens through the T5-base encoder
        dict(name="encoder_8k", kind="encoder", **BASE, B=2, L=8192, min_len=8192, train=False),
        # a training step's forward and backward through the T5-small encoder, padded batch
        dict(name="encoder_train", kind="encoder", **SMALL, B=16, L=512, min_len=64, train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case.  Lengths and batches are logarithmic; the attended pairs of a dense case stay below those of
    four heads' worth of the largest listed one, so that no draw outgrows the encoder pass."""
    kind = rng.choice(["attn", "attn", "attn_train", "attn_train", "packed", "packed_train", "sparse", "sparse", "sparse",
                       "decode", "encoder", "encoder_train"])
    if kind in ("attn", "attn_train"):
        train = kind == "attn_train"
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        D = rng.choice([64, 64, 128]) if dtype != "fp32" else 64
        H = rng.choice([6, 8, 12, 16])
        L = _log_int(rng, 16, 2048 if dtype == "fp32" else 8192 if train else 16384)
        most = 2.0e8 if dtype == "fp32" else 8.0e8 if train else 3.2e9     # B * H * L * L
        B = _log_int(rng, 1, max(1, min(32, int(most / (H * L * L)))))
        return dict(kind="attn", B=B, H=H, L=L, D=D, dtype=dtype, causal=rng.random() < 0.4, train=train)
    if kind in ("packed", "packed_train"):
        train = kind == "packed_train"
        hi = _log_int(rng, 128, 2048 if train else 4096)
        return dict(kind="packed", n_seq=_log_int(rng, 2, 32), min_len=_log_int(rng, 16, hi), max_len=hi,
                    H=rng.choice([8, 12]), D=64, dtype=rng.choice(["bf16", "bf16", "fp16"]), causal=rng.random() < 0.4,
                    train=train)
    if kind == "sparse":
        pattern = rng.choice(["local", "block", "tglobal"])
        aux = {"local": 0, "block": rng.choice([32, 64]), "tglobal": rng.choice([16, 32])}[pattern]
        L = _log_int(rng, 1024, 32768)
        return dict(kind="sparse", pattern=pattern, B=_log_int(rng, 1, max(1, min(8, 32768 // L))), H=rng.choice([8, 12]), L=L,
                    D=64, dtype=rng.choice(["bf16", "bf16", "fp16"]), block_len=rng.choice([64, 128, 128, 256]), aux=aux)
    if kind == "decode":
        N = _log_int(rng, 512, 16384)
        return dict(kind="decode", B=_log_int(rng, 1, max(1, min(128, 64 * 8192 // N))), H=rng.choice([8, 12]), N=N, D=64,
                    dtype=rng.choice(["bf16", "bf16", "fp16"]), ragged=rng.random() < 0.5)
    train = kind == "encoder_train"
    size = SMALL if train else rng.choice([SMALL, BASE])
    L = _log_int(rng, 32, 1024 if train else 8192)
    B = _log_int(rng, 1, max(1, min(32, (4096 if train else 16384) // L)))
    return dict(kind="encoder", **size, B=B, L=L, min_len=rng.choice([L, max(1, L // 8)]), train=train)


def _lengths(seed, n, lo, hi):
    """n lengths over [lo, hi], the same ones for every seed in an order of its own: shapes belong to the case."""
    lens = np.random.default_rng(n * 1000003 + hi).integers(lo, hi + 1, size=n)
    lens[0] = hi      # the longest of the declared range is always met
    np.random.default_rng(seed).shuffle(lens)
    return [int(x) for x in lens]


def _rows(g, case, *shape):
    """A projection's output in the attention dtype."""
    return torch.randn(*shape, generator=g, device="cuda").mul_(0.5).to(DTYPES[case["dtype"]])


def _table(g, case):
    return torch.randn(32, case["H"], generator=g, device="cuda")


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, H, D = case["kind"], case["H"], case["D"]
    st = {"case": case}
    if kind == "attn":
        B, L = case["B"], case["L"]
        st["qkv"] = [_rows(g, case, B, L, H, D).transpose(1, 2) for _ in range(3)]
        st["table"] = _table(g, case)
        if case["train"]:
            st["dout"] = _rows(g, case, B, L, H, D).transpose(1, 2)
    elif kind == "packed":
        lens = _lengths(seed, case["n_seq"], case["min_len"], case["max_len"])
        total = sum(lens)
        st["cu"] = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device="cuda")
        st["max_len"] = max(lens)
        st["qkv"] = [_rows(g, case, total, H, D) for _ in range(3)]
        st["table"] = _table(g, case)
        if case["train"]:
            st["dout"] = _rows(g, case, total, H, D)
    elif kind == "sparse":
        B, L = case["B"], case["L"]
        st["qkv"] = [_rows(g, case, B, L, H, D).transpose(1, 2) for _ in range(3)]
        st["table"] = _table(g, case)
        if case["pattern"] == "tglobal":
            st["side"] = [_rows(g, case, B, L // case["aux"], H, D).transpose(1, 2) for _ in range(2)]
    elif kind == "decode":
        B, N = case["B"], case["N"]
        st["q"] = _rows(g, case, B, 1, H, D).transpose(1, 2)
        st["kv"] = [_rows(g, case, B, N, H, D).transpose(1, 2) for _ in range(2)]
        st["lens"] = None
        if case["ragged"]:
            st["lens"] = torch.tensor(_lengths(seed, B, max(1, N // 8), N), dtype=torch.int32, device="cuda")
    else:
        cfg = t5.T5Config(d_model=case["d_model"], d_kv=D, d_ff=case["d_ff"], num_layers=case["layers"], num_heads=H,
                          attention_type="flash", dropout_rate=0.0,
                          # training keeps fp32 weights and activations around the 16-bit attention
                          attention_dtype=torch.bfloat16 if case["train"] else None)
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.cuda.manual_seed(seed)
            with torch.device("cuda"):
                model = t5.T5EncoderModel(cfg)
        st["model"] = model.train() if case["train"] else model.eval().to(torch.bfloat16)
        B, L = case["B"], case["L"]
        st["ids"] = torch.randint(1, cfg.vocab_size, (B, L), generator=g, device="cuda")
        st["mask"] = None
        if case["min_len"] < L:
            lens = torch.tensor(_lengths(seed, B, case["min_len"], L), device="cuda")
            st["mask"] = (torch.arange(L, device="cuda")[None, :] < lens[:, None]).to(torch.long)
        if case["train"]:
            st["dout"] = torch.randn(B, L, cfg.d_model, generator=g, device="cuda")
    if case.get("train") and kind in ("attn", "packed"):
        for t in st["qkv"] + [st["table"]]:
            t.requires_grad_()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        o = t5.flash_attention_with_fusing_bias(*state["qkv"], state["table"], causal=case["causal"], sm_scale=1.0)
    elif kind == "packed":
        o = t5.flash_attention_with_fusing_bias_varlen(*state["qkv"], state["table"], state["cu"], state["cu"],
                                                       state["max_len"], state["max_len"], causal=case["causal"], sm_scale=1.0)
    elif kind == "sparse":
        if case["pattern"] == "local":
            return t5.local_attention_with_fusing_bias(*state["qkv"], state["table"], case["block_len"])
        if case["pattern"] == "block":
            return t5.block_attention_with_fusing_bias(*state["qkv"], state["table"], case["block_len"], case["aux"])
        return t5.transient_global_attention_with_fusing_bias(*state["qkv"], *state["side"], state["table"],
                                                              case["block_len"], case["aux"])
    elif kind == "decode":
        return t5.flash_decoding_attention(state["q"], *state["kv"], None, 1.0, key_lens=state["lens"])
    else:
        model = state["model"]
        if not case["train"]:
            with torch.no_grad():
                return model(state["ids"], state["mask"])
        model.zero_grad(set_to_none=True)
        hidden = model(state["ids"], state["mask"])
        hidden.backward(state["dout"])
        return {"hidden": hidden.detach(), "grads": [p.grad for p in model.parameters()]}
    if not case["train"]:
        return o
    return [o.detach(), *torch.autograd.grad(o, state["qkv"] + [state["table"]], state["dout"])]


def work(case):
    """Bytes: inputs and outputs once.  Operations: two per multiply-add of the products; backward of an attention has
    five products to the forward's two, a linear layer's backward two to the forward's one."""
    kind, H, D = case["kind"], case["H"], case["D"]
    e = 4 if case.get("dtype") == "fp32" else 2
    train = bool(case.get("train"))
    if kind in ("attn", "packed"):
        lens = [case["L"]] * case["B"] if kind == "attn" else _lengths(0, case["n_seq"], case["min_len"], case["max_len"])
        pairs = sum(L * (L + 1) / 2 if case["causal"] else L * L for L in lens) * H
        rows = sum(lens) * H
        return {"bytes": rows * D * e * (4 + (8 if train else 0)), "flops": 4.0 * pairs * D * (3.5 if train else 1.0)}
    if kind == "sparse":
        B, L, w, aux = case["B"], case["L"], case["block_len"], case["aux"]
        if case["pattern"] == "block":
            pairs = (L - aux) * (w + aux) + aux * L
            side = 0
        else:
            side = L // aux if case["pattern"] == "tglobal" else 0
            pairs = L * (2 * w - 1 + side)
        return {"bytes": B * H * D * e * (4.0 * L + 2.0 * side), "flops": 4.0 * B * H * D * pairs}
    if kind == "decode":
        B, N = case["B"], case["N"]
        keys = sum(_lengths(0, B, max(1, N // 8), N)) if case["ragged"] else B * N
        return {"bytes": keys * H * D * e * 2, "flops": 4.0 * keys * H * D}
    lens = _lengths(0, case["B"], case["min_len"], case["L"])
    tokens, squares = sum(lens), sum(L * L for L in lens)
    d, ff, n = case["d_model"], case["d_ff"], case["layers"]
    weights = n * (4 * d * H * D + 2 * d * ff)
    flops = 2.0 * tokens * weights * (3 if train else 1) + n * 4.0 * squares * H * D * (3.5 if train else 1)
    return {"bytes": 2.0 * (weights * (2 if train else 1) + tokens * d * (3 if train else 2)), "flops": flops}


def tolerance(case):
    """Largest relative error of another correct implementation: about four times what the path differs by from the
    same formulas in a wider type on the same inputs (fp32 against fp64: 2e-6 at most; 16-bit forward 3.5e-3, with
    gradients 3.2e-3 to 9.2e-3, the largest that of the table at head_dim 128; encoder pass 8e-3).  A training step
    through the encoder is up to 2.6e-2 from the formulas in 64 bits, since rounding moves activations across the
    ReLU's edge: two such steps, each as far from them on a side of its own, differ by 3.7e-2."""
    if case["kind"] == "encoder":
        return {"rel": 0.08, "max": 0.9} if case["train"] else {"rel": 0.02, "max": 0.3}
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 0.03, "max": 0.4} if case.get("train") else {"rel": 0.012, "max": 0.2}


# ---- the same formulas in 64 bits ----

def _bucket(rel, bidirectional):
    """T5's bucket of memory position - query position: 32 buckets, logarithmic from a quarter of them to distance
    128.  The logarithm is T5's own in 32 bits, which is what fixes where the buckets begin."""
    n = 16 if bidirectional else 32
    first = (rel > 0).long() * n if bidirectional else torch.zeros_like(rel)
    dist = rel.abs() if bidirectional else (-rel).clamp(min=0)
    half = n // 2
    far = half + (torch.log(dist.float() / half) / math.log(128 / half) * (n - half)).long()
    return first + torch.where(dist < half, dist, far.clamp(max=n - 1))


def _softmax(s):
    """Over the last dimension; a row without a visible key gives zeros."""
    return torch.softmax(s, -1).nan_to_num(0.0)


def _dense(q, k, v, table, causal, dout=None):
    """Attention of one sequence over (H, L, D) rows, a few query rows at a time: o, and with ``dout`` the gradients of
    q, k, v and the table."""
    H, L, _ = q.shape
    N = k.shape[1]
    kT, vT = k.transpose(1, 2).contiguous(), v.transpose(1, 2).contiguous()
    o = torch.empty_like(q)
    grads = [torch.zeros_like(t) for t in (q, k, v)] + [torch.zeros_like(table)] if dout is not None else None
    step = max(1, min(L, (1 << 26) // (H * N)))
    for r in range(0, L, step):
        rows = slice(r, min(L, r + step))
        rel = torch.arange(N, device=q.device)[None, :] - torch.arange(rows.start, rows.stop, device=q.device)[:, None]
        bucket = _bucket(rel, not causal)
        s = q[:, rows] @ kT + table[bucket].permute(2, 0, 1)
        if causal:
            s.masked_fill_(rel > 0, -math.inf)
        p = _softmax(s)
        o[:, rows] = p @ v
        if dout is None:
            continue
        g = dout[:, rows]
        ds = p * (g @ vT - (g * o[:, rows]).sum(-1, keepdim=True))
        grads[0][:, rows] = ds @ k
        grads[1] += ds.transpose(1, 2).contiguous() @ q[:, rows]
        grads[2] += p.transpose(1, 2).contiguous() @ g
        for b in range(table.shape[0]):
            grads[3][b] += (ds * (bucket == b)).sum((1, 2))
    return (o, *grads) if dout is not None else o


def _sparse(case, st):
    q, k, v = (t.double() for t in st["qkv"])
    table = st["table"].double()
    L, w, aux, dev = case["L"], case["block_len"], case["aux"], q.device
    o = torch.empty_like(q)
    pos = torch.arange(L, device=dev)
    for lo in range(0, L, w):
        i = pos[lo:lo + w, None]
        if case["pattern"] == "block":
            # columns: the leading global tokens, then the own block; the last block is filled up with zero keys, and
            # the first one does not see its last columns
            pad = (0, 0, 0, lo + w - min(L, lo + w))
            kk, vv = (torch.cat([t[:, :, :aux], torch.nn.functional.pad(t[:, :, lo:lo + w], pad)], 2) for t in (k, v))
            col = torch.arange(w + aux, device=dev)[None, :]
            rel, seen = col - aux - (i - lo), (col < w) | (lo > 0)
        else:
            a, b = max(0, lo - w + 1), min(L, lo + 2 * w - 1)
            kk, vv = k[:, :, a:b], v[:, :, a:b]
            rel = pos[None, a:b] - i
            seen = rel.abs() < w
            if case["pattern"] == "tglobal":
                side = st["side"][0].shape[2]
                kk, vv = (torch.cat([t, x.double()], 2) for t, x in zip((kk, vv), st["side"]))
                srel = torch.arange(side, device=dev)[None, :] - (i // aux).clamp(max=side - 1)
                rel, seen = torch.cat([rel, srel], 1), torch.cat([seen, torch.ones_like(srel, dtype=torch.bool)], 1)
        s = q[:, :, lo:lo + w] @ kk.transpose(2, 3).contiguous() + table[_bucket(rel, True)].permute(2, 0, 1)
        o[:, :, lo:lo + w] = _softmax(s.masked_fill(~seen, -math.inf)) @ vv
    if case["pattern"] == "block":
        for b in range(case["B"]):
            rel = pos[None, :] - pos[:aux, None]
            s = q[b, :, :aux] @ k[b].transpose(1, 2).contiguous() + table[_bucket(rel, True)].permute(2, 0, 1)
            o[b, :, :aux] = torch.softmax(s, -1) @ v[b]
    return o


def _encoder(case, st):
    w = {n: p.detach().double().requires_grad_(case["train"]) for n, p in st["model"].named_parameters()}
    B, L, H = case["B"], case["L"], case["H"]
    lens = st["mask"].sum(1).tolist() if st["mask"] is not None else [L] * B

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w[name]

    def attend(q, k, v, table):
        if not case["train"]:
            return _dense(q, k, v, table, False)
        p = torch.arange(q.shape[1], device=q.device)
        s = q @ k.transpose(1, 2).contiguous() + table[_bucket(p[None, :] - p[:, None], True)].permute(2, 0, 1)
        return torch.softmax(s, -1) @ v

    table = w["encoder.block.0.layer.0.SelfAttention.relative_attention_bias.weight"]
    xs = []
    for b, n in enumerate(lens):
        x = w["shared.weight"][st["ids"][b, :n]]
        for j in range(case["layers"]):
            at, ff = f"encoder.block.{j}.layer.0.", f"encoder.block.{j}.layer.1."
            y = norm(x, at + "layer_norm.weight")
            q, k, v = ((y @ w[at + f"SelfAttention.{c}.weight"].T).view(n, H, -1).transpose(0, 1).contiguous() for c in "qkv")
            x = x + attend(q, k, v, table).transpose(0, 1).reshape(n, -1) @ w[at + "SelfAttention.o.weight"].T
            y = norm(x, ff + "layer_norm.weight")
            x = x + torch.relu(y @ w[ff + "DenseReluDense.wi.weight"].T) @ w[ff + "DenseReluDense.wo.weight"].T
        # positions behind a sequence's end are zero
        xs.append(torch.nn.functional.pad(norm(x, "encoder.final_layer_norm.weight"), (0, 0, 0, L - n)))
    hidden = torch.stack(xs)
    if not case["train"]:
        return hidden
    hidden.backward(st["dout"].double())
    return {"hidden": hidden.detach(), "grads": [w[n].grad for n, _ in st["model"].named_parameters()]}


def exact(case, seed):
    """What ``run`` returns for these inputs, from the formulas in 64 bits."""
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "encoder":
        with torch.set_grad_enabled(case["train"]):
            return _encoder(case, st)
    with torch.no_grad():
        if kind == "sparse":
            return _sparse(case, st)
        if kind == "decode":
            q, (k, v) = st["q"].double(), st["kv"]
            lens = st["lens"].tolist() if st["lens"] is not None else [case["N"]] * case["B"]
            out = [torch.softmax(q[b] @ k[b, :, :n].double().transpose(1, 2).contiguous(), -1) @ v[b, :, :n].double()
                   for b, n in enumerate(lens)]
            return torch.stack(out)
        rows = [t.detach().double() for t in st["qkv"]] + ([st["dout"].double()] if case["train"] else [])
        table = st["table"].detach().double()
        if kind == "attn":
            each = [[t[b] for t in rows] for b in range(case["B"])]
        else:
            cu = st["cu"].tolist()
            each = [[t[a:b].transpose(0, 1) for t in rows] for a, b in zip(cu, cu[1:])]
        outs = [_dense(*(t.contiguous() for t in r[:3]), table, case["causal"], *(t.contiguous() for t in r[3:])) for r in each]

        def join(ts):
            return torch.stack(ts) if kind == "attn" else torch.cat([t.transpose(0, 1) for t in ts])

        if not case["train"]:
            return join(outs)
        return [*(join([o[i] for o in outs]) for i in range(4)), sum(o[4] for o in outs)]
