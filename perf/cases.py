"""The work this framework is measured on: what a QLoRA fine-tuning program of the Qwen2.5-1.5B
shapes has it do through its public entry points, from a single token to the largest packed batches.

    linear  a LoRA'd NF4 linear as a module (w4linear.QLoRALinear): the forward, and in training
            the gradients of x, A and B
    mlp     the MLP of a layer: gate|up with SwiGLU, down, and in training both backward GEMMs;
            reading NF4, or fp16 copies dequantised first (w16)
    proj    the attention projections of a layer with two LoRA adapters and the rotary embedding on
            weights dequantised ahead: downs, q|k|v, o, and their backward
    attn    causal attention of a packed batch, forward and backward to d(q|k|v)
    head    the LM head over the vocabulary: loss, statistics, d(hidden)
    nf4     a weight quantised to NF4 and dequantised again (loading a model)
    step    a whole training step (model.QwenQLoRAStep): the loss, the statistics, the head's
            gradient and the LoRA gradients
"""

import math

import torch

from decentrik_prime_amd import k_attn, k_head, k_rope, model, quant, w4linear

HIDDEN, INTER, KV = 1536, 8960, 256      # Qwen2.5-1.5B, as in stack.NF4LinearStack
NQ, NKV, HD = 12, 2, 128
VOCAB = 151936
LORA_SCALE, DROP = 2.0, 0.05
KEEP_SCALE = 1.0 / float(torch.tensor(1.0 - DROP, dtype=torch.float32))
DEV = "cuda"
F16, F32, F64 = torch.float16, torch.float32, torch.float64


def listed():
    return [
        # a short prompt through one adapted projection: latency and launches
        dict(name="linear_17", kind="linear", m=17, n=HIDDEN, k=HIDDEN, rank=16, train=True),
        # the reference's usual packed batch is 850 to 900 tokens
        dict(name="linear_853", kind="linear", m=853, n=HIDDEN, k=HIDDEN, rank=16, train=True),
        # sixteen sequences of 512 tokens through an adapted projection
        dict(name="linear_8192", kind="linear", m=8192, n=HIDDEN, k=HIDDEN, rank=16, train=True),
        # a single token in evaluation: the packed weights are all there is to read
        dict(name="mlp_1", kind="mlp", m=1, hidden=HIDDEN, inter=INTER, train=False, w16=False),
        # the usual packed batch through an MLP that keeps nothing but NF4 weights
        dict(name="mlp_853", kind="mlp", m=853, hidden=HIDDEN, inter=INTER, train=True, w16=False),
        # a large batch, with the reference's fp16 workspace
        dict(name="mlp_4096_w16", kind="mlp", m=4096, hidden=HIDDEN, inter=INTER, train=True, w16=True),
        # four sequences of 512 tokens through the attention projections
        dict(name="proj_2048", kind="proj", m=2048, nq=NQ, nkv=NKV, rank=16),
        # a ragged batch of chat-sized examples
        dict(name="attn_ragged", kind="attn", lens="200,512,37,411,1,318", nq=NQ, nkv=NKV),
        # one long document
        dict(name="attn_8192", kind="attn", lens="8192", nq=NQ, nkv=NKV),
        # the whole vocabulary on the usual packed batch, a part of whose tokens has labels
        dict(name="head_853", kind="head", n=853, n_lab=701, vocab=VOCAB, hidden=HIDDEN),
        # loading one gate projection
        dict(name="nf4_gate", kind="nf4", rows=INTER, cols=HIDDEN),
        # a training step on four sequences of 512 tokens, two of the layers
        dict(name="step_4x512", kind="step", lens="512,512,512,512", layers=2, vocab=VOCAB),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_lens(rng, most):
    total = _log_int(rng, 16, most)
    lens = [_log_int(rng, max(8, total // 4), total)]
    total -= lens[0]
    while total > 0:
        lens.append(total if len(lens) == 23 else _log_int(rng, 1, total))
        total -= lens[-1]
    rng.shuffle(lens)
    return ",".join(str(n) for n in lens)


def draw(rng):
    kind = rng.choice(("linear", "linear", "mlp", "mlp", "proj", "attn", "attn", "head", "nf4", "step"))
    if kind == "linear":
        n, k = rng.choice(((HIDDEN, HIDDEN), (KV, HIDDEN), (HIDDEN, INTER), (INTER, HIDDEN), (1024, 1024)))
        return dict(kind=kind, m=_log_int(rng, 1, 8192 if n * k <= HIDDEN * HIDDEN else 2048), n=n, k=k,
                    rank=rng.choice((16, 16, 32, 64)), train=rng.random() < 0.7)
    if kind == "mlp":
        hidden, inter = rng.choice(((HIDDEN, INTER), (HIDDEN, INTER), (1024, 4096)))
        return dict(kind=kind, m=_log_int(rng, 1, 4096), hidden=hidden, inter=inter,
                    train=rng.random() < 0.6, w16=rng.random() < 0.4)
    if kind == "proj":
        nq, nkv = rng.choice(((NQ, NKV), (NQ, NKV), (8, 4)))
        return dict(kind=kind, m=_log_int(rng, 16, 4096), nq=nq, nkv=nkv, rank=rng.choice((16, 16, 32)))
    if kind == "attn":
        nq, nkv = rng.choice(((NQ, NKV), (NQ, NKV), (4, 4), (8, 4)))
        return dict(kind=kind, lens=_draw_lens(rng, 8192), nq=nq, nkv=nkv)
    if kind == "head":
        n = _log_int(rng, 8, 1024)
        return dict(kind=kind, n=n, n_lab=rng.randint(n // 2, n), vocab=64 * _log_int(rng, 64, VOCAB // 64),
                    hidden=rng.choice((HIDDEN, HIDDEN, 1024)))
    if kind == "nf4":
        rows, cols = rng.choice(((HIDDEN, HIDDEN), (KV, HIDDEN), (HIDDEN, INTER), (INTER, HIDDEN)))
        return dict(kind=kind, rows=64 * _log_int(rng, 1, rows // 64), cols=cols)
    return dict(kind=kind, lens=_draw_lens(rng, 2048), layers=rng.randint(1, 2),
                vocab=64 * _log_int(rng, 64, VOCAB // 64))


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


# ---- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * scale


def _mask(g, *shape):
    return (torch.rand(*shape, generator=g, device=DEV) >= DROP).to(torch.uint8)


def _nf4_weight(g, rows, cols):
    """W ~ N(0, 0.02) in double-quantised NF4, as a checkpoint holds it."""
    code2, nf4 = w4linear.default_tables(DEV)
    w = _randn(g, rows, cols, scale=0.02).view(-1, 64)
    absmax = w.abs().amax(1)
    mid = (nf4[1:] + nf4[:-1]) / 2
    code = torch.bucketize(w / absmax[:, None], mid).to(torch.uint8).view(-1, 2)
    packed = (code[:, 0] << 4) | code[:, 1]
    offset = absmax.mean()
    rest = (absmax - offset).view(-1, 256)
    scale2 = rest.abs().amax(1)
    qabs = torch.bucketize(rest / scale2[:, None], (code2[1:] + code2[:-1]) / 2).to(torch.uint8)
    return w4linear.W4(packed.contiguous(), qabs.reshape(-1).contiguous(), scale2.contiguous(),
                       offset.expand(scale2.numel()).contiguous(), code2, nf4, rows, cols)


def _lora(g, rank, cols, rows):
    return (((torch.rand(rank, cols, generator=g, device=DEV) * 2 - 1) / math.sqrt(cols)).half(),
            _randn(g, rows, rank, scale=0.02).half())


def _positions(m):
    return (torch.arange(m, device=DEV) % 512).to(torch.int32)


def _rope_tables(positions):
    inv = 1.0 / (1.0e6 ** (torch.arange(0, HD, 2, device=DEV, dtype=F64) / HD))
    a = torch.arange(positions, device=DEV, dtype=F64)[:, None] * inv[None, :]
    a = torch.cat((a, a), 1)
    return a.cos().float().contiguous(), a.sin().float().contiguous()


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        layer = w4linear.QLoRALinear(_nf4_weight(g, n, k), rank=case["rank"], alpha=2 * case["rank"],
                                     dropout=DROP, bias=_randn(g, n, scale=0.02).half())
        a, b = _lora(g, case["rank"], k, n)
        layer.lora_A.data.copy_(a)
        layer.lora_B.data.copy_(b)
        return dict(case=case, layer=layer.train(case["train"]),
                    x=_randn(g, m, k).half().requires_grad_(case["train"]),
                    mask=_mask(g, m, k) if case["train"] else None, dy=_randn(g, m, n, scale=1e-2).half())
    if kind == "mlp":
        m, d, inter = case["m"], case["hidden"], case["inter"]
        wgu, wd = _nf4_weight(g, 2 * inter, d), _nf4_weight(g, d, inter)
        slots = [torch.empty(w.rows, w.cols, dtype=F16, device=DEV) if case["w16"] else None for w in (wgu, wd)]
        return dict(case=case, wgu=wgu, wd=wd, slots=slots, x=_randn(g, m, d).half(),
                    dh=_randn(g, m, d, scale=1e-2).half())
    if kind == "proj":
        m, nq, nkv, r = case["m"], case["nq"], case["nkv"], case["rank"]
        qd, kvd = nq * HD, nkv * HD
        s = dict(case=case, wqkv=_nf4_weight(g, qd + 2 * kvd, qd), wo=_nf4_weight(g, qd, qd))
        s["wqkv16"], s["wo16"] = s["wqkv"].dequantize(), s["wo"].dequantize()
        s["bias"] = _randn(g, qd + 2 * kvd, scale=0.02).half()
        s["Aq"], s["Bq"] = _lora(g, r, qd, qd)
        s["Av"], s["Bv"] = _lora(g, r, qd, kvd)
        s["mq"], s["mv"] = _mask(g, m, qd), _mask(g, m, qd)
        s["y"], s["att"] = _randn(g, m, qd).half(), _randn(g, m, qd, scale=0.3).half()
        s["dqkv"], s["dh"] = (_randn(g, m, qd + 2 * kvd, scale=1e-2).half(), _randn(g, m, qd, scale=1e-2).half())
        s["pos"] = _positions(m)
        s["cos"], s["sin"] = _rope_tables(512)
        return s
    if kind == "attn":
        lens, nq, nkv = _lens(case), case["nq"], case["nkv"]
        n = sum(lens)
        pos = torch.cat([torch.arange(k, device=DEV) for k in lens]).to(torch.int32)
        cos, sin = _rope_tables(max(lens))
        return dict(case=case, meta=k_attn.meta_for(lens, DEV), qkv=_randn(g, n, (nq + 2 * nkv) * HD).half(),
                    dout=_randn(g, n, nq * HD, scale=1e-2).half(), pos=pos, cos=cos, sin=sin,
                    dqkv=torch.empty(n, (nq + 2 * nkv) * HD, dtype=F16, device=DEV))
    if kind == "head":
        n, n_lab, v, d = case["n"], case["n_lab"], case["vocab"], case["hidden"]
        emb = _randn(g, v, d, scale=0.02).half()
        perm = torch.randperm(n, generator=g, device=DEV)
        tgt = torch.randint(0, v, (n,), generator=g, device=DEV).to(torch.int32)
        # hidden states that point towards their targets by differing amounts: some tokens are
        # predicted well and some are not
        yf = _randn(g, n, d)
        yf[perm] += emb[tgt.long()].float() * (15 * torch.rand(n, 1, generator=g, device=DEV))
        tgt[n_lab:] = -1
        return dict(case=case, yf=yf.half(), source=k_head.ResidentEmbedding(emb), tgt=tgt,
                    perm=perm.to(torch.int32), e_target=emb.index_select(0, tgt[:n_lab].long()).contiguous())
    if kind == "nf4":
        return dict(case=case, w=_randn(g, case["rows"], case["cols"], scale=0.02).half())
    return dict(case=case, step=model.QwenQLoRAStep(_lens(case), n_layers=case["layers"], vocab=case["vocab"],
                                                    seed=int(seed)))


# ---- the passes

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        layer, x = s["layer"], s["x"]
        if not case["train"]:
            with torch.no_grad():
                return dict(y=layer(x))
        y = layer(x, s["mask"])
        dx, da, db = torch.autograd.grad(y, (x, layer.lora_A, layer.lora_B), s["dy"])
        return dict(y=y, dx=dx, dA=da, dB=db)
    if kind == "mlp":
        w16 = [w.dequantize(out=slot) if slot is not None else None
               for w, slot in zip((s["wgu"], s["wd"]), s["slots"])]
        act, gu = w4linear.gateup_swiglu_forward(s["x"], s["wgu"], save_gu=case["train"], w16=w16[0])
        y = w4linear.linear_forward(act, s["wd"], w16=w16[1])
        if not case["train"]:
            return dict(act=act, y=y)
        w4linear.down_swiglu_backward(s["dh"], s["wd"], gu, w16=w16[1])
        dx = w4linear.linear_backward_dx(gu, s["wgu"], out_dtype=F16, w16=w16[0])
        return dict(act=act, y=y, dgu=gu, dx=dx)
    if kind == "proj":
        nq, nkv = case["nq"], case["nkv"]
        qd, kvd = nq * HD, nkv * HD
        y, dqkv, mq, mv = s["y"], s["dqkv"], s["mq"], s["mv"]
        zq, zv = w4linear.lora_down_multi(y, [(s["Aq"], mq, KEEP_SCALE), (s["Av"], mv, KEEP_SCALE)])
        qkv = w4linear.linear_forward_rope(
            y, s["wqkv"], s["bias"], [(zq, s["Bq"], 0, qd, LORA_SCALE),
                                      (zv, s["Bv"], qd + kvd, qd + 2 * kvd, LORA_SCALE)],
            s["pos"], s["cos"], s["sin"], qd + kvd, w16=s["wqkv16"])
        o = w4linear.linear_forward(s["att"], s["wo"], w16=s["wo16"])
        datt = w4linear.linear_backward_dx(s["dh"], s["wo"], out_dtype=F16, w16=s["wo16"])
        sums = w4linear.lora_dz_multi(y, [(dqkv[:, :qd], zq, s["Bq"], LORA_SCALE, mq, KEEP_SCALE),
                                          (dqkv[:, qd + kvd:], zv, s["Bv"], LORA_SCALE, mv, KEEP_SCALE)])
        (daq, dbq, dzq), (dav, dbv, dzv) = sums.grads
        dy = w4linear.linear_backward_dx_lora(dqkv, s["wqkv"], [(dzq, s["Aq"], mq, KEEP_SCALE),
                                                                (dzv, s["Av"], mv, KEEP_SCALE)],
                                              w16=s["wqkv16"], sums=sums)
        return dict(qkv=qkv, o=o, datt=datt, dy=dy, dAq=daq, dBq=dbq, dAv=dav, dBv=dbv)
    if kind == "attn":
        nq, nkv, meta = case["nq"], case["nkv"], s["meta"]
        out, lse = k_attn.attention_forward(s["qkv"], meta, nq, nkv, HD)
        dq, dk, dv = k_attn.attention_backward(s["qkv"], out, lse, s["dout"], meta, nq, nkv, HD)
        k_rope.qkv_epilogue_backward(dq, dk, dv, s["pos"], s["cos"], s["sin"], s["dqkv"], nq, nkv, HD, nq // nkv)
        return dict(out=out, lse=lse, dq=dq, dk=dk, dv=dv, dqkv=s["dqkv"])
    if kind == "head":
        loss, stats, dy = k_head.streamed_head(s["yf"], s["source"], s["tgt"], s["perm"], case["n_lab"],
                                               s["e_target"], 1024.0)
        return dict(loss=loss, stats=stats, dy=dy)
    if kind == "nf4":
        q = quant.quantize_4bit(s["w"])
        w = w4linear.W4.from_params(q)
        return dict(packed=w.packed, qabs=w.qabs, scale2=w.scale2, offset=w.offset2[:1], w=w.dequantize())
    st = s["step"]
    loss, stats, dy = st.forward()
    grads = st.backward(dy)
    return dict(loss=loss, stats=stats, dy=dy, grads=list(grads))


# ---- what a pass cannot do without

def _nf4_bytes(n):
    return n // 2 + n // 64 + n // 2048


def _linear_flops(m, n, k, r, train):
    f = 2 * m * n * k + 2 * m * r * (n + k)
    return f + (2 * m * n * k + 4 * m * r * (n + k) if train else 0)


def _attn_flops(lens, nq):
    return sum(2 * HD * n * (n + 1) for n in lens) * nq * 3.5


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k, r, t = (case[x] for x in ("m", "n", "k", "rank", "train"))
        b = _nf4_bytes(n * k) + 2 * m * (n + k) + 4 * r * (n + k)
        if t:
            b += 2 * m * (n + k) + m * k + 4 * r * (n + k)
        return dict(bytes=b, flops=_linear_flops(m, n, k, r, t))
    if kind == "mlp":
        m, d, i, t = (case[x] for x in ("m", "hidden", "inter", "train"))
        b = _nf4_bytes(3 * d * i) + 2 * m * (2 * d + i)
        if t:
            b += 2 * m * (2 * d + 2 * i)
        return dict(bytes=b, flops=6 * m * d * i * (2 if t else 1))
    if kind == "proj":
        m, nq, nkv, r = (case[x] for x in ("m", "nq", "nkv", "rank"))
        d, kvd = nq * HD, nkv * HD
        b = 2 * d * (2 * d + 2 * kvd) + 2 * m * (2 * d + 2 * (d + 2 * kvd) + 3 * d) + 2 * m * d + 4 * m * d
        b += 4 * r * (3 * d + kvd) + 2 * r * (3 * d + kvd)
        return dict(bytes=b, flops=4 * m * d * (2 * d + 2 * kvd) + 6 * m * r * (3 * d + kvd))
    if kind == "attn":
        lens, nq, nkv = _lens(case), case["nq"], case["nkv"]
        n = sum(lens)
        b = n * HD * (2 * 2 * (nq + 2 * nkv) + 2 * 2 * nq + 3 * 4 * nq) + 4 * n * nq
        return dict(bytes=b, flops=_attn_flops(lens, nq))
    if kind == "head":
        n, n_lab, v, d = (case[x] for x in ("n", "n_lab", "vocab", "hidden"))
        return dict(bytes=2 * v * d + 4 * n * d + 2 * n_lab * d + 16 * n, flops=2 * v * d * (n + n_lab))
    if kind == "nf4":
        n = case["rows"] * case["cols"]
        return dict(bytes=4 * n + _nf4_bytes(n), flops=8 * n)
    lens, layers = _lens(case), case["layers"]
    m = sum(lens)
    weights = HIDDEN * (2 * HIDDEN + 2 * KV + 3 * INTER)
    f = layers * (4 * m * weights + 6 * m * 16 * (3 * HIDDEN + KV) + _attn_flops(lens, NQ))
    b = layers * (_nf4_bytes(weights) + 4 * 16 * (3 * HIDDEN + KV) + 2 * m * HIDDEN) + 2 * case["vocab"] * HIDDEN
    return dict(bytes=b + 6 * m * HIDDEN, flops=f + 4 * m * case["vocab"] * HIDDEN)


def tolerance(case):
    """About four times what each case differs from exact() by: one fp16 rounding is 2.1e-4 to 2.9e-4
    in the 2-norm, and a case rounds once to three times on the way to an output (measured: linear,
    proj, attn 2.1e-4 to 3.7e-4, mlp 4.4e-4, head 2.1e-4; two layers of a step 2e-3)."""
    kind = case["kind"]
    if kind == "nf4":
        return "exact"
    return {"rel": {"linear": 1.5e-3, "mlp": 1.8e-3, "proj": 1.5e-3, "attn": 1.4e-3, "head": 1e-3, "step": 8e-3}[kind]}


# ---- the same in 64 bits

def _deq(w):
    """The fp16 values that a double-quantised NF4 weight stands for."""
    absmax = w.code2[w.qabs.long()] * w.scale2.repeat_interleave(256) + w.offset2.repeat_interleave(256)
    codes = torch.stack((w.packed >> 4, w.packed & 15), 1).view(-1, 64).long()
    return (w.nf4[codes] * absmax[:, None]).half().double().view(w.rows, w.cols)


def _silu_grads(g, u, da):
    sig = torch.sigmoid(g)
    return da * u * sig * (1 + g * (1 - sig)), da * g * sig


def _rotate(x, c, s, back=False):
    h = HD // 2
    x1, x2 = x[..., :h], x[..., h:]
    c, s = c[:, None, :h], s[:, None, :h]
    if back:
        return torch.cat((x1 * c + x2 * s, x2 * c - x1 * s), -1)
    return torch.cat((x1 * c - x2 * s, x2 * c + x1 * s), -1)


def _exact_attn(case, s):
    lens, nq, nkv = _lens(case), case["nq"], case["nkv"]
    n, g = sum(lens), nq // nkv
    qkv = s["qkv"].double().view(n, nq + 2 * nkv, HD)
    dout = s["dout"].double().view(n, nq, HD)
    out, lse = torch.empty(n, nq, HD, dtype=F64, device=DEV), torch.empty(nq, n, dtype=F64, device=DEV)
    dq, dk, dv = (torch.empty(n, nq, HD, dtype=F64, device=DEV) for _ in range(3))
    s0 = 0
    for k in lens:
        at = slice(s0, s0 + k)
        above = torch.ones(k, k, dtype=torch.bool, device=DEV).triu_(1)
        for h in range(nq):
            q, ky, v = qkv[at, h], qkv[at, nq + h // g], qkv[at, nq + nkv + h // g]
            p = (q @ ky.T) / math.sqrt(HD)
            p.masked_fill_(above, float("-inf"))
            l = torch.logsumexp(p, 1)
            p.sub_(l[:, None]).exp_()
            o, do = p @ v, dout[at, h]
            out[at, h], lse[h, at], dv[at, h] = o, l / math.log(2), p.T @ do
            p.mul_(do @ v.T - (o * do).sum(1, keepdim=True)).div_(math.sqrt(HD))
            dq[at, h], dk[at, h] = p @ ky, p.T @ q
        s0 += k
    c, sn = s["cos"].double()[s["pos"].long()], s["sin"].double()[s["pos"].long()]
    dqkv = torch.cat((_rotate(dq, c, sn, True), _rotate(dk.view(n, nkv, g, HD).sum(2), c, sn, True),
                      dv.view(n, nkv, g, HD).sum(2)), 1)
    return dict(out=out.view(n, -1), lse=lse, dq=dq.view(n, -1), dk=dk.view(n, -1), dv=dv.view(n, -1),
                dqkv=dqkv.reshape(n, -1))


def _exact_head(yf, emb, tgt, perm, n_lab, scale):
    """Rows in blocks, so that the whole vocabulary's logits fit."""
    n, e = yf.shape[0], emb.double()
    ys = yf.double()[perm]
    stats, dy = torch.zeros(n, 4, dtype=F64, device=DEV), torch.zeros_like(ys)
    for r0 in range(0, n, 512):
        r = slice(r0, min(r0 + 512, n))
        x = ys[r] @ e.T
        lse = torch.logsumexp(x, 1)
        t = tgt[r].long()
        has = (t >= 0).double()
        hit = (x.argmax(1) == t).double() * has
        xt = x.gather(1, t.clamp(min=0)[:, None])[:, 0]
        x.sub_(lse[:, None])
        p = x.exp()
        ent = -(p * x).sum(1)
        d = (p @ e - e[t.clamp(min=0)]) * has[:, None]
        stats[r] = torch.stack(((lse - xt) * has, ent, hit, lse), 1)
        dy[perm[r]] = d * scale
    return stats[:, 0].sum(), stats, dy


def _exact_step(st, case):
    lens, n, dt = _lens(case), st.m, F64
    c, sn = st.cos.to(dt)[st.pos.long()], st.sin.to(dt)[st.pos.long()]
    x, leaves = st.x0.to(dt), []

    def rms(h, w):
        return w.to(dt) * (h * torch.rsqrt((h * h).mean(-1, keepdim=True) + st.eps))

    for i in range(case["layers"]):
        w, lo = st.layers[i], st.lora[i]
        a = {k: lo[k].to(dt).requires_grad_(True) for k in ("Aq", "Bq", "Av", "Bv")}
        leaves += [a[k] for k in ("Aq", "Bq", "Av", "Bv")]
        y = rms(x, st.w_in[i])
        xq, xv = y * (lo["mq"] != 0) * st.keep_scale, y * (lo["mv"] != 0) * st.keep_scale
        qkv = y @ _deq(w["qkv"]).T + lo["bias"].to(dt)
        q = qkv[:, :HIDDEN] + st.s * ((xq @ a["Aq"].T) @ a["Bq"].T)
        v = qkv[:, HIDDEN + KV:] + st.s * ((xv @ a["Av"].T) @ a["Bv"].T)
        q = _rotate(q.view(n, NQ, HD), c, sn)
        k = _rotate(qkv[:, HIDDEN:HIDDEN + KV].view(n, NKV, HD), c, sn)
        v, outs, s0 = v.view(n, NKV, HD), [], 0
        for ln in lens:
            at = slice(s0, s0 + ln)
            above = torch.ones(ln, ln, dtype=torch.bool, device=DEV).triu_(1)
            heads = []
            for h in range(NQ):
                p = (q[at, h] @ k[at, h * NKV // NQ].T) / math.sqrt(HD)
                heads.append(torch.softmax(p.masked_fill(above, float("-inf")), 1) @ v[at, h * NKV // NQ])
            outs.append(torch.cat(heads, 1))
            s0 += ln
        hid = x + torch.cat(outs) @ _deq(w["o"]).T
        gu = rms(hid, st.w_post[i]) @ _deq(w["gu"]).T
        act = torch.nn.functional.silu(gu[:, :INTER]) * gu[:, INTER:]
        x = hid + act @ _deq(w["d"]).T
    yf = rms(x, st.w_final)
    loss, stats, dy = _exact_head(yf.detach(), st.emb, st.tgt_sorted, st.perm.long(), st.n_lab, 1.0)
    grads = torch.autograd.grad(yf, leaves, dy)
    return dict(loss=loss, stats=stats, dy=dy * st.head_grad_scale,
                grads=[tuple(grads[4 * i:4 * i + 4]) for i in range(case["layers"])])


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "linear":
            layer, x, dy = s["layer"], s["x"].double(), s["dy"].double()
            w, a, b = _deq(layer.w), layer.lora_A.double(), layer.lora_B.double()
            keep = s["mask"].double() * layer.keep_scale if case["train"] else 1.0
            xd = x * keep
            z = xd @ a.T
            y = x @ w.T + layer.bias.double() + layer.scale * (z @ b.T)
            if not case["train"]:
                return dict(y=y)
            dz = layer.scale * (dy @ b)
            return dict(y=y, dx=dy @ w + keep * (dz @ a), dA=dz.T @ xd, dB=layer.scale * (dy.T @ z))
        if kind == "mlp":
            i, x = case["inter"], s["x"].double()
            wgu, wd = _deq(s["wgu"]), _deq(s["wd"])
            gu = x @ wgu.T
            g, u = gu[:, :i], gu[:, i:]
            act = torch.nn.functional.silu(g) * u
            y = act @ wd.T
            if not case["train"]:
                return dict(act=act, y=y)
            dgu = torch.cat(_silu_grads(g, u, s["dh"].double() @ wd), 1)
            return dict(act=act, y=y, dgu=dgu, dx=dgu @ wgu)
        if kind == "proj":
            qd, kvd, m = case["nq"] * HD, case["nkv"] * HD, case["m"]
            y, dqkv, wqkv, wo = s["y"].double(), s["dqkv"].double(), _deq(s["wqkv"]), _deq(s["wo"])
            kq, kv = s["mq"].double() * KEEP_SCALE, s["mv"].double() * KEEP_SCALE
            aq, bq, av, bv = (s[k].double() for k in ("Aq", "Bq", "Av", "Bv"))
            zq, zv = (y * kq) @ aq.T, (y * kv) @ av.T
            qkv = y @ wqkv.T + s["bias"].double()
            qkv[:, :qd] += LORA_SCALE * (zq @ bq.T)
            qkv[:, qd + kvd:] += LORA_SCALE * (zv @ bv.T)
            c, sn = s["cos"].double()[s["pos"].long()], s["sin"].double()[s["pos"].long()]
            qkv[:, :qd + kvd] = _rotate(qkv[:, :qd + kvd].view(m, -1, HD), c, sn).reshape(m, -1)
            gq, gv = dqkv[:, :qd], dqkv[:, qd + kvd:]
            dzq, dzv = LORA_SCALE * (gq @ bq), LORA_SCALE * (gv @ bv)
            return dict(qkv=qkv, o=s["att"].double() @ wo.T, datt=s["dh"].double() @ wo,
                        dy=dqkv @ wqkv + kq * (dzq @ aq) + kv * (dzv @ av),
                        dAq=dzq.T @ (y * kq), dBq=LORA_SCALE * (gq.T @ zq),
                        dAv=dzv.T @ (y * kv), dBv=LORA_SCALE * (gv.T @ zv))
        if kind == "attn":
            return _exact_attn(case, s)
        if kind == "head":
            loss, stats, dy = _exact_head(s["yf"], s["source"].emb, s["tgt"], s["perm"].long(), case["n_lab"], 1024.0)
            return dict(loss=loss, stats=stats, dy=dy)
        if kind == "nf4":
            absmax = s["w"].double().view(-1, 64).abs().amax(1)
            offset = absmax.mean().float()
            scale2 = (absmax.float() - offset).view(-1, 256).abs().amax(1)
            return dict(packed=None, qabs=None, scale2=scale2.double(), offset=offset.double().view(1), w=None)
    return _exact_step(s["step"], case)
