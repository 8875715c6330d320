"""The work a user of this framework has it do, as measurable cases.

Each case is one call (or the few calls that belong together) of a public entry point, at
LLaDA-8B widths unless it says otherwise (d_model 4096, 32 heads of 128, MLP 12288, vocabulary
126464), on synthetic inputs made from a seed: N(0, 1) hidden states, N(0, 0.02) weights, caches
with the spread of projected hidden states, masked blocks of 32 rows at each sequence's frontier
and tracked rows drawn from its decoded slots.

kinds
  projection  fdl.ops.qkv_rope_cache: Q/K/V projection, RoPE and the write of K/V into the cache
  attention   fdl.ops.block_attention over a ragged batch, then what a layer does with the
              importance (the head reduction, or at a step's last layer the ranking)
  verify      the Flash-Verify pair: packed projection, fdl.ops.verify_attention
  head        fdl.ops.softmax_confidence over LM-head logits
  block       one transformer block through flash_fused_elastic_cache, the call a model makes
  model       a whole forward of fdl.model.LLaDAModelLM to the logits of the masked rows
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

PKG = Path(__file__).resolve().parent.parent / "flash-dllm_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

from fdl import lib, ops  # noqa: E402
from fdl.model import LLaDAConfig, LLaDALlamaBlock, LLaDAModelLM  # noqa: E402
from fdl.schedule import SeqRows, make_plan  # noqa: E402
from flash_cache_hip import flash_fused_elastic_cache  # noqa: E402

HEAD_DIM = 128
BLOCK = 32          # rows of a masked block
PAGE = 32           # slots of a cache page
THETA = 500000.0
EPS = 1e-5
VOCAB = 126464
MLP_PER_D = 3       # mlp width / d_model
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEV = "cuda:0"
SCALE = 1.0 / math.sqrt(HEAD_DIM)


def listed():
    return [
        # one sequence being decoded: the 32 masked rows and 8 tracked ones (latency; the
        # weights are all there is to read)
        dict(name="projection_one_sequence", kind="projection", heads=32, rows=40, slots=384),
        # the decode step of a batch of eight: 32 masked and 32 tracked rows each
        dict(name="projection_batch", kind="projection", heads=32, rows=512, slots=7168),
        # a mixed batch: a few new prompts recompute every row, the rest decode
        dict(name="projection_recompute", kind="projection", heads=32, rows=6842, slots=32768),
        # the attention of that decode step at the step's last layer, softmax importance ranked
        dict(name="attention_batch_ranked", kind="attention", heads=32, seqs=8, keys_lo=768,
             keys_hi=768, rows_lo=64, rows_hi=64, full=0, shape=1, importance="softmax", rank=True),
        # a serving batch: 32 sequences of 512-1536 keys in permuted pages, 1-96 rows each, a
        # fifth of them recomputed in full
        dict(name="attention_mixed", kind="attention", heads=32, seqs=32, keys_lo=512,
             keys_hi=1536, rows_lo=1, rows_hi=96, full=6, shape=3, importance="raw", rank=False),
        # the first step of eight prompts: every row of 768 keys
        dict(name="attention_recompute", kind="attention", heads=32, seqs=8, keys_lo=768,
             keys_hi=768, rows_lo=1, rows_hi=1, full=8, shape=1, importance="none", rank=False),
        # the verify forward of sixteen sequences
        dict(name="verify_batch", kind="verify", heads=32, seqs=16, keys=1024, max_s=16),
        # the confidences of the masked rows of a batch of eight
        dict(name="confidence_batch", kind="head", rows=256, vocab=VOCAB, token=False),
        # a transformer block while one sequence is decoded, and while eight are
        dict(name="block_one_sequence", kind="block", heads=32, seqs=1, keys_lo=384, keys_hi=384,
             rows_lo=64, rows_hi=64, full=0, shape=1),
        dict(name="block_batch", kind="block", heads=32, seqs=8, keys_lo=768, keys_hi=768,
             rows_lo=64, rows_hi=64, full=0, shape=1),
        # a block in the first step of a few prompts of uneven length
        dict(name="block_recompute", kind="block", heads=32, seqs=3, keys_lo=320, keys_hi=900,
             rows_lo=1, rows_hi=1, full=3, shape=5),
        # a whole forward: embedding, four blocks, final norm and LM head
        dict(name="model_batch", kind="model", heads=32, layers=4, seqs=8, keys_lo=512,
             keys_hi=1024, rows_lo=33, rows_hi=96, full=0, shape=2),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["projection", "projection", "attention", "attention", "verify", "head",
                       "block", "block"])
    heads = rng.choice([32, 32, 32, 16])
    if kind == "projection":
        rows = _log(rng, 1, 6842)
        return dict(kind=kind, heads=heads, rows=rows, slots=(max(rows, 320) // 32 + 3) * 64)
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 1, 512), vocab=rng.choice([VOCAB, VOCAB, 32000]),
                    token=rng.random() < 0.4)
    if kind == "verify":
        return dict(kind=kind, heads=heads, seqs=_log(rng, 1, 24), keys=_log(rng, 160, 1536),
                    max_s=rng.randint(1, 16))
    if kind == "attention":
        seqs = _log(rng, 1, 32)
        full = rng.choice([0, 0, seqs // 4, max(1, seqs // 2)]) if seqs <= 16 else rng.choice([0, 4])
        importance = rng.choice(["raw", "raw", "softmax", "none"])
        lo = _log(rng, 128, 900)
        return dict(kind=kind, heads=heads, seqs=seqs, keys_lo=lo, keys_hi=rng.randint(lo, 1536),
                    rows_lo=rng.randint(1, 40), rows_hi=rng.randint(40, 120), full=full,
                    shape=rng.randrange(1 << 20), importance=importance, rank=importance != "none" and rng.random() < 0.3)
    seqs = _log(rng, 1, 12)
    lo = _log(rng, 160, 800)
    return dict(kind=kind, heads=heads, seqs=seqs, keys_lo=lo, keys_hi=rng.randint(lo, 1024),
                rows_lo=rng.randint(1, 33), rows_hi=rng.randint(33, 100),
                full=rng.choice([0, 0, 1, min(2, seqs)]), shape=rng.randrange(1 << 20))


# ------------------------------------------------------------------------------------ inputs

def _randn(gen, *shape, std=1.0, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=gen)


def _rope(n):
    """float32 sin, cos [n, 128] of positions 0 .. n - 1, halves repeated."""
    inv = 1.0 / THETA ** (torch.arange(0, HEAD_DIM, 2, device=DEV, dtype=F64) / HEAD_DIM)
    f = torch.outer(torch.arange(n, device=DEV, dtype=F64), inv)
    f = torch.cat((f, f), dim=-1)
    return f.sin().to(F32), f.cos().to(F32)


def _batch(case, rng):
    """The sequences of a batch: per sequence its key count, its query positions (masked block
    first, then tracked rows; every position where it is recomputed in full), the number of
    masked rows and the frontier; the page table of permuted pages; packed rows. The lengths
    belong to the case ("shape"), the pages and the tracked positions to the seed."""
    n, full = case["seqs"], case["full"]
    shape = np.random.default_rng(case["shape"])
    ks = shape.integers(case["keys_lo"], case["keys_hi"] + 1, n)
    is_full = np.zeros(n, bool)
    is_full[shape.permutation(n)[:full]] = True
    per = -(-ks // PAGE)
    table = np.zeros((n, int(per.max())), np.int32)
    perm, at = rng.permutation(int(per.sum())), 0
    for b in range(n):
        table[b, :per[b]] = np.sort(perm[at:at + per[b]])
        at += per[b]
    pos, masked, frontier = [], [], []
    for b in range(n):
        k = int(ks[b])
        if is_full[b]:
            f = int(shape.integers(k // 2, k - BLOCK + 1))
            p = np.concatenate([np.arange(f, f + BLOCK), np.arange(f), np.arange(f + BLOCK, k)])
            m = BLOCK
        else:
            q = int(shape.integers(case["rows_lo"], case["rows_hi"] + 1))
            m = min(q, BLOCK)
            f = int(shape.integers(96, k - BLOCK + 1))
            p = np.concatenate([np.arange(f, f + m), rng.choice(f, q - m, replace=False)])
        pos.append(p)
        masked.append(m)
        frontier.append(f)
    # packed as a step packs them: every sequence's masked rows, then every tracked row
    row, rows_m, rows_t = 0, [], []
    for b in range(n):
        rows_m.append(np.arange(row, row + masked[b]))
        row += masked[b]
    n_masked = row
    for b in range(n):
        rows_t.append(np.arange(row, row + len(pos[b]) - masked[b]))
        row += len(pos[b]) - masked[b]
    packed = np.concatenate([pos[b][:masked[b]] for b in range(n)] +
                            [pos[b][masked[b]:] for b in range(n)])
    owner = np.concatenate([np.full(masked[b], b) for b in range(n)] +
                           [np.full(len(pos[b]) - masked[b], b) for b in range(n)])
    slots = table[owner, packed // PAGE].astype(np.int64) * PAGE + packed % PAGE
    rows = [np.concatenate([rows_m[b], rows_t[b]]) for b in range(n)]
    return dict(ks=ks, rows=rows, masked=masked, frontier=frontier, table=table, pos=packed,
                slots=slots, n_rows=row, n_masked=n_masked, n_slots=int(per.sum()) * PAGE)


def _key_slots(bt, b):
    p = np.arange(int(bt["ks"][b]))
    return torch.from_numpy(bt["table"][b, p // PAGE].astype(np.int64) * PAGE + p % PAGE).to(DEV)


def _plan(bt, importance):
    seqs = [SeqRows(batch=b, k_end=int(bt["ks"][b]), rows=r, n_imp=bt["masked"][b] if importance else 0)
            for b, r in enumerate(bt["rows"])]
    return make_plan(seqs, bt["table"], device=DEV)


def _weights(gen, d, mlp, n):
    names = ("q_proj", "k_proj", "v_proj", "attn_out", "ff_proj", "up_proj", "ff_out")
    shapes = ((d, d),) * 4 + ((mlp, d), (mlp, d), (d, mlp))
    return [{k: _randn(gen, *s, std=0.02) for k, s in zip(names, shapes)} for _ in range(n)]


def _inputs(case, seed):
    """Every input of a case, on the GPU, from the seed alone."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "head":
        x = _randn(gen, case["rows"], case["vocab"], std=2.0)
        # about half of the rows know their token
        top = torch.from_numpy(rng.integers(0, case["vocab"], case["rows"])).to(DEV)
        lift = torch.from_numpy(rng.uniform(-8.0, 24.0, case["rows"])).to(DEV)
        x[torch.arange(case["rows"], device=DEV), top] += lift.clamp_min(0.0).to(BF16)
        return dict(x=x, token=top if case["token"] else None)
    d = case["heads"] * HEAD_DIM
    s = dict(d=d)
    if kind in ("projection", "verify"):
        s["w"] = [_randn(gen, d, d, std=0.02) for _ in range(3)]
    if kind == "projection":
        n = case["slots"]
        s["slot"] = torch.from_numpy(rng.permutation(n)[:case["rows"]].astype(np.int64)).to(DEV)
        s["sin"], s["cos"] = _rope(n)
        s["x"] = _randn(gen, case["rows"], d)
        s["k"], s["v"] = _randn(gen, n, d, std=1.28), _randn(gen, n, d, std=1.28)
    elif kind == "verify":
        nb, keys = case["seqs"], case["keys"]
        two = 2 * BLOCK
        key_pos, vb, meta, slots, k0 = [], [], [], [], 0
        for b in range(nb):
            S = int(rng.integers(1, case["max_s"] + 1))
            T = two - 2 * S
            nd = int(rng.integers(T, keys - S + 1))  # decoded slots before the candidates
            order = rng.permutation(nd)
            kp = np.concatenate([order[:nd - T], np.arange(nd + S, keys)]) + b * keys
            cand = np.arange(nd, nd + S) + b * keys
            slots.append(np.concatenate([order[nd - T:] + b * keys, cand, cand]))
            vb.append([k0, k0 + len(kp), two * b, two * (b + 1)])
            meta.append([T, S])
            key_pos.append(kp)
            k0 += len(kp)
        s["keys"] = torch.from_numpy(np.concatenate(key_pos).astype(np.int64)).to(DEV)
        s["vb"], s["meta"] = np.array(vb, np.int32), np.array(meta, np.int32)
        s["slot"] = torch.from_numpy(np.concatenate(slots).astype(np.int64)).to(DEV)
        sin, cos = _rope(keys)
        s["sin"], s["cos"] = sin.repeat(nb, 1), cos.repeat(nb, 1)
        s["x"] = _randn(gen, two * nb, d)
        s["k"], s["v"] = _randn(gen, nb * keys, d, std=1.28), _randn(gen, nb * keys, d, std=1.28)
    else:
        bt = s["bt"] = _batch(case, rng)
        n = bt["n_slots"]
        if kind == "attention":
            s["q"] = _randn(gen, bt["n_rows"], d, std=1.28)
            s["k"], s["v"] = _randn(gen, n, d, std=1.28), _randn(gen, n, d, std=1.28)
            # the scores that earlier layers have left
            s["scores"] = _randn(gen, n, dtype=F32)
        else:
            layers = case.get("layers", 1)
            s["w"] = _weights(gen, d, MLP_PER_D * d, layers)
            s["kv"] = [(_randn(gen, n, d, std=1.28), _randn(gen, n, d, std=1.28))
                       for _ in range(layers)]
            s["sin"], s["cos"] = _rope(int(bt["ks"].max()))
            s["pos"] = torch.from_numpy(bt["pos"].astype(np.int64)).to(DEV)
            s["slot"] = torch.from_numpy(bt["slots"]).to(DEV)
            if kind == "block":
                s["x"] = _randn(gen, bt["n_rows"], d)
            else:
                s["wte"] = _randn(gen, VOCAB, d, std=0.02)
                s["head"] = _randn(gen, VOCAB, d, std=0.02)
                s["ids"] = torch.from_numpy(rng.integers(0, VOCAB, bt["n_rows"])).to(DEV)
    return s


# ------------------------------------------------------------------------- prepare, run

def _fill(block, w):
    for name, t in w.items():
        getattr(block, name).weight.data.copy_(t)


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    s["kind"], s["case"] = kind, case
    if kind == "head":
        return s
    d, heads = s["d"], case["heads"]
    if kind in ("projection", "verify"):
        s["q"] = torch.empty_like(s["x"])
    if kind == "verify":
        s["k1"], s["v1"], s["att"] = (torch.empty_like(s["x"]) for _ in range(3))
        s["vb"], s["meta"] = torch.from_numpy(s["vb"]).to(DEV), torch.from_numpy(s["meta"]).to(DEV)
    if kind == "attention":
        bt = s["bt"]
        s["plan"] = _plan(bt, case["importance"] != "none")
        s["att"] = torch.empty_like(s["q"])
        s["imp"] = torch.empty((heads, bt["n_slots"]), dtype=F32, device=DEV)
        s["out_scores"] = torch.empty_like(s["scores"])
        if case["rank"]:
            order = [bt["table"][b, np.arange(f) // PAGE].astype(np.int64) * PAGE +
                     np.arange(f) % PAGE for b, f in enumerate(bt["frontier"])]
            starts = np.cumsum([0] + [len(o) for o in order[:-1]])
            s["order"] = torch.from_numpy(np.concatenate(order)).to(DEV)
            s["seg"] = torch.from_numpy(np.array([[a, len(o)] for a, o in zip(starts, order)],
                                                 np.int32)).to(DEV)
            s["seg_keys"] = torch.from_numpy(np.array([[b, int(k)] for b, k in enumerate(bt["ks"])],
                                                      np.int32)).to(DEV)
            s["max_len"] = max(len(o) for o in order)
            s["topk"] = torch.empty((case["seqs"], BLOCK), dtype=torch.int64, device=DEV)
    if kind in ("block", "model"):
        bt = s["bt"]
        cfg = LLaDAConfig(d_model=d, n_heads=heads, n_layers=case.get("layers", 30),
                          mlp_hidden_size=MLP_PER_D * d, vocab_size=VOCAB, rope_theta=THETA,
                          rms_norm_eps=EPS)
        plan = _plan(bt, True)
        plan.kv_slot = s["slot"]
        s["scores"] = torch.zeros(bt["n_slots"], dtype=F32, device=DEV)
        none = torch.zeros((0, 4), dtype=torch.int64)
        s["positions"] = [s["pos"], torch.empty(0, dtype=torch.int32, device=DEV),
                          [s["sin"], s["cos"]], plan, s["scores"], []]
        s["lengths"] = [[-1] * case["seqs"], None, none, none, none, list(range(case["seqs"])),
                        case["seqs"], bt["table"].shape[1] * PAGE, BLOCK, 32, None, False]
        if kind == "block":
            with torch.device(DEV):
                block = LLaDALlamaBlock(cfg, 5, flash_fused_elastic_cache, DEV, BF16)
            s["blocks"] = [block]
        else:
            with torch.device(DEV):
                s["model"] = LLaDAModelLM(cfg, flash_fused_elastic_cache, device=DEV, dtype=BF16)
            s["model"].requires_grad_(False)
            t = s["model"].model.transformer
            t.wte.weight.data.copy_(s.pop("wte"))
            t.ff_out.weight.data.copy_(s.pop("head"))
            s["blocks"] = list(t.blocks)
            s["ids"] = s["ids"][None]
            s["logit_rows"] = torch.arange(bt["n_masked"], device=DEV)
        for blk, w, (k, v) in zip(s["blocks"], s.pop("w"), s.pop("kv")):
            blk.requires_grad_(False)
            _fill(blk, w)
            blk.k_cache, blk.v_cache = k, v
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "head":
        prob, arg = ops.softmax_confidence(s["x"], s["token"])
        return dict(prob=prob, arg=arg)
    heads = case["heads"]
    if kind == "projection":
        ops.qkv_rope_cache(s["x"], *s["w"], s["sin"], s["cos"], s["slot"], s["q"], s["k"], s["v"],
                           heads)
        return dict(q=s["q"], k=s["k"], v=s["v"])
    if kind == "verify":
        ops.qkv_rope_cache(s["x"], *s["w"], s["sin"], s["cos"], s["slot"], s["q"], s["k1"],
                           s["v1"], heads, kv_packed=True)
        ops.verify_attention(s["q"], s["k1"], s["v1"], s["k"], s["v"], s["keys"], s["vb"],
                             s["meta"], 2 * BLOCK, s["att"], heads, SCALE)
        return dict(q=s["q"], k=s["k1"], v=s["v1"], att=s["att"])
    if kind == "attention":
        imp = case["importance"]
        mode = {"none": lib.IMP_NONE, "raw": lib.IMP_RAW_LOGIT, "softmax": lib.IMP_SOFTMAX_COLSUM}
        ops.block_attention(s["q"], s["k"], s["v"], s["plan"], s["att"], heads, SCALE, mode[imp],
                            None if imp == "none" else s["imp"])
        if imp == "none":
            return dict(att=s["att"])
        scale = 1.0 / (BLOCK * heads)
        scores = s["out_scores"].copy_(s["scores"])  # accumulated in place over the layers
        if case["rank"]:
            ops.importance_rank(scores, s["order"], s["seg"], s["max_len"], s["topk"], BLOCK,
                                imp_part=s["imp"], scale=scale, plan=s["plan"],
                                seg_keys=s["seg_keys"])
            return dict(att=s["att"], scores=scores, order=s["order"], topk=s["topk"])
        ops.importance_accumulate(s["imp"], s["plan"], scale, scores)
        return dict(att=s["att"], scores=scores)
    s["scores"].zero_()
    if kind == "block":
        x = s["blocks"][0].attention(s["x"], 5, positions=s["positions"], lengths=s["lengths"])
    else:
        x = s["model"](s["ids"], use_cache=True, lengths=s["lengths"], positions=s["positions"],
                       logit_rows=s["logit_rows"]).logits
    out = dict(out=x, scores=s["scores"])
    for i, b in enumerate(s["blocks"]):
        out["k%d" % i], out["v%d" % i] = b.k_cache, b.v_cache
    return out


# ------------------------------------------------------------------- work and tolerance

def work(case):
    kind = case["kind"]
    if kind == "head":
        n = case["rows"] * case["vocab"]
        return dict(bytes=2 * n + 16 * case["rows"], flops=3 * n)
    d, heads = case["heads"] * HEAD_DIM, case["heads"]
    proj = lambda q: (6 * d * d + q * d * 2 * 4 + q * HEAD_DIM * 8 + q * 8, 6 * q * d * d)  # noqa: E731
    if kind == "projection":
        b, f = proj(case["rows"])
        return dict(bytes=b, flops=f)
    if kind == "verify":
        q = 2 * BLOCK * case["seqs"]
        b, f = proj(q)
        s = (case["max_s"] + 1) / 2
        cached = case["keys"] - (2 * BLOCK - s)  # cache keys of a block, on average
        b += case["seqs"] * cached * (4 * d + 8) + 8 * q * d
        return dict(bytes=b, flops=f + 4 * q * (cached + 2 * BLOCK) * d)
    bt = _batch(case, np.random.default_rng(0))
    q, ks = bt["n_rows"], bt["ks"].astype(np.float64)
    qs = np.array([len(r) for r in bt["rows"]], np.float64)
    att_b = float(4 * q * d + 4 * d * ks.sum())
    att_f = float((4 * qs * ks * d).sum())
    if kind == "attention":
        scores = 0 if case["importance"] == "none" else 8 * ks.sum()
        return dict(bytes=float(att_b + scores), flops=att_f)
    b, f = proj(q)
    mlp = MLP_PER_D * d
    b += att_b + 8 * ks.sum() + 2 * (d * d + 3 * d * mlp) + 4 * q * d
    f += att_f + 2 * q * (d * d + 3 * d * mlp)
    n = case.get("layers", 1)
    b, f = n * b, n * f
    if kind == "model":
        b += 2 * VOCAB * d + 2 * q * d + 2 * bt["n_masked"] * VOCAB
        f += 2 * bt["n_masked"] * VOCAB * d
    return dict(bytes=float(b), flops=float(f))


def tolerance(case):
    kind = case["kind"]
    if kind == "head":
        return dict(rel=1e-14, differ=0.0)  # 64-bit sums of up to 126464 terms
    if kind == "projection":
        return dict(rel=7e-3)  # bf16 results of 32-bit sums
    if kind == "attention":
        # bf16 probabilities and results; ranks of scores that are equal to 32 bits may swap
        return dict(rel=1e-2, differ=0.01)
    if kind == "verify":
        return dict(rel=1.5e-2)  # attention over rounded queries, keys and values
    # a chain of bf16 results: one block; four blocks and the head
    return dict(rel=2e-2 if kind == "block" else 6e-2)


# ------------------------------------------------------------------------------- exact

def _rotate64(y, sin, cos, heads):
    y = y.view(y.shape[0], heads, 2, HEAD_DIM // 2)
    sin, cos = sin.double()[:, None], cos.double()[:, None]
    lo, hi = y[:, :, 0], y[:, :, 1]
    h = HEAD_DIM // 2
    return torch.stack((lo * cos[..., :h] - hi * sin[..., :h], hi * cos[..., h:] + lo * sin[..., h:]),
                       2).reshape(y.shape[0], heads * HEAD_DIM)


def _project64(x, w, sin, cos, heads):
    wq, wk, wv = w
    return (_rotate64(x @ wq.double().t(), sin, cos, heads),
            _rotate64(x @ wk.double().t(), sin, cos, heads), x @ wv.double().t())


def _heads64(t, heads):
    return t.double().view(t.shape[0], heads, HEAD_DIM).transpose(0, 1).contiguous()


def _attend64(q, k, v, heads, visible=None):
    """softmax(q k^T / sqrt(128)) v per head; also the logits."""
    s = torch.matmul(_heads64(q, heads), _heads64(k, heads).transpose(1, 2).contiguous())
    z = s * SCALE
    if visible is not None:
        z = z.masked_fill(~visible, -math.inf)
    p = torch.softmax(z, -1)
    return torch.matmul(p, _heads64(v, heads)).transpose(0, 1).reshape(q.shape), s, p


def _batch64(bt, q, k, v, heads, importance):
    """Attention of every sequence of the batch and its importance per slot."""
    att = torch.empty(q.shape, dtype=F64, device=DEV)
    imp = torch.zeros(bt["n_slots"], dtype=F64, device=DEV)
    for b, r in enumerate(bt["rows"]):
        rows, keys = torch.from_numpy(r).to(DEV), _key_slots(bt, b)
        att[rows], s, p = _attend64(q[rows], k[keys], v[keys], heads)
        if importance != "none":
            t = (s if importance == "raw" else p)[:, :bt["masked"][b]]
            imp[keys] += t.sum((0, 1)) / (BLOCK * heads)
    return att, imp


def _norm64(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _block64(s, w, kv, x, heads):
    """One block on float64 hidden states; the caches it leaves, its importance."""
    k, v = kv[0].double(), kv[1].double()
    names = ("q_proj", "k_proj", "v_proj")
    q, kn, vn = _project64(_norm64(x), [w[n] for n in names], s["sin"][s["pos"]],
                           s["cos"][s["pos"]], heads)
    k[s["slot"]], v[s["slot"]] = kn, vn
    att, imp = _batch64(s["bt"], q, k, v, heads, "raw")
    x = x + att @ w["attn_out"].double().t()
    y = _norm64(x)
    g = y @ w["ff_proj"].double().t()
    g = g * torch.sigmoid(g) * (y @ w["up_proj"].double().t())
    return x + g @ w["ff_out"].double().t(), k, v, imp


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "head":
        prob, arg = [], []
        for r in range(case["rows"]):
            x = s["x"][r].double()
            m = x.max()
            at = (x == m).nonzero()[0, 0]
            e = (x - m).exp().sum()
            top = m if s["token"] is None else x[s["token"][r]]
            prob.append((top - m).exp() / e)
            arg.append(at)
        return dict(prob=torch.stack(prob), arg=torch.stack(arg))
    heads = case["heads"]
    if kind in ("projection", "verify"):
        q, kn, vn = _project64(s["x"].double(), s["w"], s["sin"][s["slot"]], s["cos"][s["slot"]],
                               heads)
    if kind == "projection":
        k, v = s["k"].double(), s["v"].double()
        k[s["slot"]], v[s["slot"]] = kn, vn
        return dict(q=q, k=k, v=v)
    if kind == "verify":
        att = torch.empty_like(q)
        for (k0, k1, q0, q1), (T, S) in zip(s["vb"].tolist(), s["meta"].tolist()):
            n = q1 - q0
            # fill rows do not see the drafts; draft i sees drafts <= i and masks > i; mask i
            # sees drafts < i and masks >= i
            vis = torch.ones(n, n, dtype=torch.bool, device=DEV)
            i = torch.arange(S, device=DEV)
            vis[:T, T:T + S] = False
            vis[T:T + S, T:T + S] = i[:, None] >= i[None]
            vis[T:T + S, T + S:] = i[:, None] < i[None]
            vis[T + S:, T:T + S] = i[:, None] > i[None]
            vis[T + S:, T + S:] = i[:, None] <= i[None]
            keys = s["keys"][k0:k1]
            see = torch.cat((torch.ones(n, k1 - k0, dtype=torch.bool, device=DEV), vis), 1)
            att[q0:q1] = _attend64(q[q0:q1], torch.cat((s["k"][keys].double(), kn[q0:q1])),
                                   torch.cat((s["v"][keys].double(), vn[q0:q1])), heads, see)[0]
        return dict(q=q, k=kn, v=vn, att=att)
    bt = s["bt"]
    if kind == "attention":
        att, imp = _batch64(bt, s["q"], s["k"], s["v"], heads, case["importance"])
        if case["importance"] == "none":
            return dict(att=att)
        scores = s["scores"].double() + imp
        if not case["rank"]:
            return dict(att=att, scores=scores)
        order, topk = [], torch.full((case["seqs"], BLOCK), -1, dtype=torch.int64, device=DEV)
        for b, f in enumerate(bt["frontier"]):
            sl = _key_slots(bt, b)[:f]
            sl = sl[torch.argsort(scores[sl])]
            order.append(sl)
            top = sl.flip(0)[:BLOCK]
            topk[b, :len(top)] = top
        return dict(att=att, scores=scores, order=torch.cat(order), topk=topk)
    x = s["x"].double() if kind == "block" else s["wte"][s["ids"]].double()
    scores = torch.zeros(bt["n_slots"], dtype=F64, device=DEV)
    out = {}
    for i, (w, kv) in enumerate(zip(s["w"], s["kv"])):
        x, out["k%d" % i], out["v%d" % i], imp = _block64(s, w, kv, x, heads)
        if kind == "block" or i > 1:  # the first two blocks of a model feed no importance
            scores += imp
    if kind == "block":
        out["out"] = x[None]
    else:
        y = _norm64(x[:bt["n_masked"]])
        out["out"] = (y @ s["head"].double().t())[None]
    out["scores"] = scores
    return out
