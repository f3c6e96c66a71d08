"""The framework's work as its users run it: decode attention over a quantized KV cache, with the step's K/V stored first
where a decoder stores it, and prefill.  Each case is one decode step over a number of attention layers (each layer
called in turn, as a decoder must: a layer's query depends on the layer before it) or one prefill call.  Everything
goes through the KVStore binding; inputs are on the GPU and the calls go to the current stream.

Fields of a case
  kind    "decode", or "prefill"
  spec    the store's formats (the MK_KV grammar), win its q8 window, page 0 (contiguous) or positions per page
  layers  attention layers of the step
  lens    context lengths of the sequences after the step's rows, comma separated (prefill: the one length after the chunk)
  T       query tokens per sequence of a decode step (1, or 1 + drafts in a speculative verify); prefill: the chunk's tokens
  mode    decode:  "attend" (rows already stored), "slot" (append, then attend), "fused" (append_attend), "gated" (attend
          with the output gate), "prep" (append_prep + attend_prep: raw projections), "all" (attend, every layer in one call)
          prefill: "plain", or "prep" (raw projections, output gate)
  f16     the appended K/V rows are fp16 (else fp32)
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen38-megakernel_amd"))

import qkv  # noqa: E402

HD, NKV, NH, GQA, BUCKET, CHUNK = 256, 4, 24, 6, 640, 4096
PRESET_F = "K*=5r,V*=6"


def listed():
    return [
        # one attention layer over a 4,096-position q8 context: the smallest call, launches and latency
        dict(name="attend_4k_q8", kind="decode", spec="", win=0, page=0, layers=1, lens="4096", T=1, mode="attend", f16=1),
        # a whole decode step of 16 layers in a short chat, from the raw projections to the gated output
        dict(name="step_1k_prep", kind="decode", spec=PRESET_F, win=2048, page=0, layers=16, lens="1025", T=1, mode="prep", f16=0),
        # a decode step of 16 layers at a usual document length, storing the step's rows in the attention launch
        dict(name="step_9k_fused", kind="decode", spec=PRESET_F, win=2048, page=0, layers=16, lens="9001", T=1, mode="fused", f16=1),
        # the headline workload: 16 layers' attention at 101,600 positions
        dict(name="attend_101k_f", kind="decode", spec=PRESET_F, win=2048, page=0, layers=16, lens="101600", T=1, mode="attend", f16=1),
        # a verify of 3 drafts over 40,013 positions in the reference's preset E
        dict(name="verify4_40k_e", kind="decode", spec="K*=6r,V*=4r", win=2048, page=0, layers=8, lens="40013", T=4, mode="slot", f16=1),
        # a verify of 7 drafts at 38,000 positions, all q8, 16 layers replayed in one call
        dict(name="verify8_38k_q8", kind="decode", spec="", win=0, page=0, layers=16, lens="38000", T=8, mode="all", f16=1),
        # a verify of 7 drafts at the headline length, rows stored first
        dict(name="verify8_101k_f", kind="decode", spec=PRESET_F, win=2048, page=0, layers=8, lens="101600", T=8, mode="slot", f16=1),
        # 8 short conversations decoded together on a shared page pool, with the output gate
        dict(name="batch8_short", kind="decode", spec="K*=5r,V*=5", win=2048, page=64, layers=16,
             lens="417,700,1281,1999,2048,3333,5120,7777", T=1, mode="gated", f16=1),
        # 4 long sequences of mixed lengths decoded together on a shared page pool
        dict(name="batch4_long", kind="decode", spec=PRESET_F, win=2048, page=256, layers=4, lens="23000,23000,60000,262144", T=1,
             mode="attend", f16=1),
        # a short prompt into an all-q8 store
        dict(name="prefill_1k_q8", kind="prefill", spec="", win=0, page=0, layers=4, lens="1111", T=1111, mode="plain", f16=0),
        # one chunk of a chunked prefill late in a long document, from the raw projections
        dict(name="prefill_chunk_60k", kind="prefill", spec=PRESET_F, win=2048, page=256, layers=2, lens="60621", T=433, mode="prep", f16=0),
        # a whole 16,384-position prompt
        dict(name="prefill_16k_f", kind="prefill", spec=PRESET_F, win=2048, page=0, layers=1, lens="16384", T=16384, mode="plain", f16=1),
    ]


FORMATS = [(PRESET_F, 2048), (PRESET_F, 2048), ("K*=5r,V*=5", 2048), ("K*=6r,V*=4r", 2048), ("K*=6,V*=5", 2048), ("", 0), ("", 0),
           ("K*=4,V*=4", 0), ("K*=7,V*=6", 1024), ("K*=5r,V*=8", 512), ("K*=4,V*=7", 640)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _row_bytes(bits):
    return 32 * bits + 16


def _kv_bytes(spec, win, L, layers):
    """Bytes of the rows that `layers` layers' attention reads over L positions (4 kv heads, K and V, with scales)."""
    kb, vb, _, _ = qkv.parse_spec(spec, layers)
    ws = qkv.window_start(L, win) if win else L
    return sum(NKV * (ws * (_row_bytes(k) + _row_bytes(v)) + (L - ws) * 2 * _row_bytes(8)) for k, v in zip(kb, vb))


def draw(rng):
    spec, win = rng.choice(FORMATS)
    if rng.random() < 0.35:
        c = dict(kind="prefill", spec=spec, win=win, page=rng.choice([0, 0, 96, 256]), mode=rng.choice(["plain", "plain", "prep"]))
        T, pos = _log(rng, 16, 8192), rng.choice([0, 0, _log(rng, 100, 60000)])
        if pos and win:  # a chunk within one bucket: the window it reads stays in the ring when the chunk is stored again
            T = min(T, BUCKET - pos % BUCKET)
        while T * (pos + T / 2) > 1.3e8:  # (the listed 16,384-position prompt)
            T //= 2
        one = T * (pos + T / 2)
        c.update(layers=rng.randint(1, 4) if one < 3e7 else 1, lens=str(pos + T), T=T, f16=0 if c["mode"] == "prep" else rng.randint(0, 1))
        return c
    n = rng.choice([1, 1, 1, 2, 3, 4, 8])
    T = rng.choice([1, 1, 1, 1, 2, 3, 4, 5, 6, 8, 8])
    mode = rng.choice(["attend", "slot", "fused", "gated", "prep", "all"])
    lens = [max(T, _log(rng, 100, 200000 if n == 1 else 160000 // n)) for _ in range(n)]
    lens = [L + T if (L - T) // BUCKET != (L - 1) // BUCKET else L for L in lens]  # the T rows share one bucket
    layers = 16
    while layers > 1 and sum(_kv_bytes(spec, win, L, layers) for L in lens) * (1 + T / 4) > 2.4e9:
        layers -= 1
    return dict(kind="decode", spec=spec, win=win, page=rng.choice([0, 0, 256]) if n == 1 else rng.choice([32, 64, 256]),
                layers=rng.randint(max(1, layers // 2), layers), lens=",".join(map(str, lens)), T=T, mode=mode,
                f16=0 if mode == "prep" else rng.randint(0, 1))


# ------------------------------------------------------------------------------------------------ inputs
def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + what) % (1 << 62))
    return g


def _outliers():
    """4 K channels per kv head are 12 times as large as the others."""
    s = torch.ones(NKV, HD, device="cuda")
    for h in range(NKV):
        r = torch.Generator()
        r.manual_seed(1000 + h)
        s[h, torch.randperm(HD, generator=r)[:4].cuda()] = 12.0
    return s


def _rows(g, n, nl, f16, scale):
    k = torch.randn(n, nl, NKV, HD, device="cuda", generator=g) * scale
    v = torch.randn(n, nl, NKV, HD, device="cuda", generator=g)
    return (k.half(), v.half()) if f16 else (k, v)


def _history(case, seed, s, n):
    """The K/V rows of positions 0 .. n-1 of sequence s, a chunk at a time (fp16)."""
    g, scale = _gen(seed, 10 + s), _outliers()
    for p in range(0, n, CHUNK):
        yield p, *_rows(g, min(CHUNK, n - p), case["layers"], True, scale)


def _step(case, seed):
    """What the step brings: new K/V rows, queries, gates and norm weights (as the case's mode takes them)."""
    nl, T, ns, mode = case["layers"], case["T"], len(_lens(case)), case["mode"]
    g, d = _gen(seed, 1), {}
    if case["kind"] == "prefill" or mode in ("slot", "fused", "prep"):
        # per sequence: [T][layers][4][256]
        rows = [_rows(g, T, nl, case["f16"], _outliers()) for _ in range(ns)]
        d["k"], d["v"] = torch.stack([r[0] for r in rows]), torch.stack([r[1] for r in rows])
    shape = (nl, T, NH) if case["kind"] == "prefill" else (nl, ns, T, NH)
    d["q"] = torch.randn(*shape, 2 * HD if mode == "prep" else HD, device="cuda", generator=g)
    if mode == "gated":
        d["gate"] = torch.randn(*shape, HD, device="cuda", generator=g)
    if mode == "prep":
        d["kw"] = 1 + 0.2 * torch.randn(nl, HD, device="cuda", generator=g)
        d["qw"] = 1 + 0.2 * torch.randn(nl, HD, device="cuda", generator=g)
    return d


def prepare(case, seed):
    nl, T, lens, mode = case["layers"], case["T"], _lens(case), case["mode"]
    page, ctx = case["page"], max(lens)
    if page:
        npg = [-(-L // page) for L in lens]
        st = qkv.KVStore(case["spec"], win=case["win"], n_layers=nl, n_seq=len(lens), ctx=ctx, page=page, n_pages=sum(npg))
        r = torch.Generator()
        r.manual_seed(5)
        perm, o = torch.randperm(sum(npg), generator=r).tolist(), 0
        for s, n in enumerate(npg):
            st.set_pages(s, perm[o:o + n])
            o += n
    else:
        st = qkv.KVStore(case["spec"], win=case["win"], n_layers=nl, n_seq=len(lens), ctx=ctx)
    stores = case["kind"] == "prefill" or mode in ("slot", "fused", "prep")
    for s, L in enumerate(lens):
        for p, k, v in _history(case, seed, s, L - T if stores else L):
            st.append(s, 0, nl, p, k.shape[0], k.data_ptr(), v.data_ptr(), 1, torch.cuda.current_stream().cuda_stream)
    d = _step(case, seed)
    d.update(case=dict(case), st=st, lens=lens, seqs=list(range(len(lens))))
    if case["kind"] == "decode" and "k" in d:
        # one block per layer, as a layer's projection leaves its rows: [layers][sequences][T][1][4][256]
        d["k"], d["v"] = (x.permute(2, 0, 1, 3, 4).contiguous() for x in (d["k"], d["v"]))
    q = d["q"]
    d["out"] = torch.empty(*q.shape[:-1], HD, device="cuda")
    if mode == "prep":
        st.set_rope()
    return d


# ------------------------------------------------------------------------------------------------ a pass
def run(d):
    c, st, out, q = d["case"], d["st"], d["out"], d["q"]
    nl, T, mode, lens, seqs, f16 = c["layers"], c["T"], c["mode"], d["lens"], d["seqs"], c["f16"]
    stream = torch.cuda.current_stream().cuda_stream
    qp, op = q.data_ptr(), out.data_ptr()
    if c["kind"] == "prefill":
        k, v, pos = d["k"].data_ptr(), d["v"].data_ptr(), lens[0] - T
        if pos == 0:
            st.rewind(0, 0)  # a new prompt on the lane
        if mode == "prep":
            st.prefill_prep(0, 0, nl, pos, T, k, v, d["kw"].data_ptr(), qp, d["qw"].data_ptr(), op, stream=stream)
        else:
            st.prefill(0, 0, nl, pos, T, k, v, f16, qp, op, stream)
        return out
    if mode == "all":
        st.attend(0, nl, seqs, lens, T, qp, op, stream)
        return out
    ql, ol = q[0].numel() * 4, out[0].numel() * 4
    if mode in ("slot", "fused", "prep"):
        kp, vp = d["k"].data_ptr(), d["v"].data_ptr()
        one = T * NKV * HD * (2 if f16 else 4)  # one sequence's rows of one layer
        kl = one * len(seqs)
    for l in range(nl):
        if mode == "attend":
            st.attend(l, 1, seqs, lens, T, qp + l * ql, op + l * ol, stream)
        elif mode == "gated":
            st.attend_gated(l, 1, seqs, lens, T, qp + l * ql, d["gate"].data_ptr() + l * ql, op + l * ol, stream=stream)
        elif mode == "fused":
            st.append_attend(l, 1, seqs, lens, T, kp + l * kl, vp + l * kl, f16, qp + l * ql, op + l * ol, stream)
        elif mode == "slot":
            for s in seqs:
                st.append(s, l, 1, lens[s] - T, T, kp + l * kl + s * one, vp + l * kl + s * one, f16, stream)
            st.attend(l, 1, seqs, lens, T, qp + l * ql, op + l * ol, stream)
        else:
            for s in seqs:
                st.append_prep(s, l, 1, lens[s] - T, T, kp + l * kl + s * one, vp + l * kl + s * one, d["kw"].data_ptr() + l * HD * 4, stream)
            st.attend_prep(l, 1, seqs, lens, T, qp + l * ql, d["qw"].data_ptr() + l * HD * 4, op + l * ol, stream=stream)
    return out


def work(case):
    nl, T, lens = case["layers"], case["T"], _lens(case)
    kv = sum(_kv_bytes(case["spec"], case["win"], L, nl) for L in lens)
    io = nl * len(lens) * T * NH * HD * 4 * (3 if case["mode"] in ("prep", "gated") else 2)
    new = nl * len(lens) * T * NKV * HD * 2 * (2 if case["f16"] else 4) if case["kind"] == "prefill" or case["mode"] in ("slot", "fused", "prep") else 0
    if case["kind"] == "prefill":  # causal: query i of the chunk sees pos + i + 1 keys
        pairs = T * (lens[0] - T) + T * (T + 1) / 2
    else:
        pairs = sum(T * L - T * (T - 1) / 2 for L in lens)
    return {"bytes": kv + io + new, "flops": nl * 4 * HD * NH * pairs}


def tolerance(case):
    # fp16 operands (queries, dequantized K and V, probabilities), fp32 sums: measured against exact() 4e-4 to 1.3e-3
    return {"rel": 4e-3, "max": 4e-2}


# ------------------------------------------------------------------------------------------------ 64 bits
def _fwht(x):
    """256-point Walsh-Hadamard transform of the last dim, index bits ascending, over 16 (any dtype)."""
    shape = x.shape
    for b in range(8):
        y = x.reshape(-1, HD >> (b + 1), 2, 1 << b)
        x = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], 2)
    return x.reshape(shape) * 0.0625


def _q8(x):
    """fp32 rows -> the stored q8 values d q (exact in fp32)."""
    b = x.reshape(-1, 8, 32)
    am = b.abs().amax(-1, keepdim=True)
    q = torch.where(am > 0, torch.round(b * (127.0 / am)), torch.zeros_like(b))
    return (q * (am / 127.0).half().float()).reshape(x.shape)


def _qn(x, bits):
    """fp32 rows -> the stored values of the 4..7-bit format."""
    h = 1 << (bits - 1)
    b = x.reshape(-1, 8, 32)
    hi, lo = b.amax(-1, keepdim=True), b.amin(-1, keepdim=True)
    d = torch.where(hi >= -lo, hi, lo) / -h
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    n = (b.double() * inv.double() + (h + 0.5)).float().trunc().clamp(max=2 * h - 1)
    return ((n - h) * d.half().float()).reshape(x.shape)


def _stored(x, bits, rot):
    """fp32 rows [..][256] -> (main row, q8 window row) values."""
    if rot:
        x = _fwht(x)
    return (_q8(x) if bits == 8 else _qn(x, bits)), _q8(x)


def _rope(p0, n):
    p = torch.arange(p0, p0 + n, dtype=torch.float64, device="cuda")[:, None]
    th = p * 1e7 ** (-2.0 * torch.arange(32, dtype=torch.float64, device="cuda") / 64.0)
    return th.cos().float().double(), th.sin().float().double()


def _prep(x, w, cs):
    """RMSNorm and RoPE of rows x [n][heads][256] (fp64) at the n positions of cs."""
    x = x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w
    c, s = cs[0][:, None], cs[1][:, None]
    a, b = x[..., :32], x[..., 32:64]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 64:]], -1)


def exact(case, seed):
    """softmax(q K / 16) V in fp64 on the values the store holds: window positions from their q8 rows, the others from the
    packed rows."""
    nl, T, lens, mode, win = case["layers"], case["T"], _lens(case), case["mode"], case["win"]
    kb, vb, kr, vr = qkv.parse_spec(case["spec"], nl)
    d = _step(case, seed)
    pre, out = case["kind"] == "prefill", None
    q = d["q"][:, None] if pre else d["q"]  # [layers][sequences][T][24][..]
    out = torch.empty(*q.shape[:-1], HD, device="cuda", dtype=torch.float64)
    for s, L in enumerate(lens):
        n0 = L - T if "k" in d else L
        # the stored values [side][layer] -> main and q8 rows [4][L][256], fp32
        main = [[torch.empty(NKV, L, HD, device="cuda") for _ in range(nl)] for _ in range(2)]
        ring = [[torch.empty(NKV, L, HD, device="cuda") if win and (vb if w else kb)[l] != 8 else None for l in range(nl)] for w in range(2)]

        def put(p, w, l, x):  # x [n][4][256] fp32
            m, r = _stored(x, (vb if w else kb)[l], (vr if w else kr)[l])
            main[w][l][:, p:p + x.shape[0]] = m.transpose(0, 1)
            if ring[w][l] is not None:
                ring[w][l][:, p:p + x.shape[0]] = r.transpose(0, 1)

        for p, k, v in _history(case, seed, s, n0):
            for l in range(nl):
                put(p, 0, l, k[:, l].float())
                put(p, 1, l, v[:, l].float())
        cs = _rope(L - T, T)
        for l in range(nl):
            if "k" in d:
                k, v = d["k"][s][:, l].double(), d["v"][s][:, l]
                put(n0, 0, l, (_prep(k, d["kw"][l].double(), cs) if mode == "prep" else k).float())
                put(n0, 1, l, v.float())
            qs = q[l, s, :, :, :HD].double()
            if mode == "prep":
                qs = _prep(qs, d["qw"][l].double(), cs)
            if kr[l]:
                qs = _fwht(qs)
            qs = qs / 16
            # the rows of one 640-position bucket see one window start
            a = 0
            while a < T:
                b = min(T, a + BUCKET - (L - T + a) % BUCKET)
                n = L - T + b
                ws = qkv.window_start(n, win) if win else n
                lim = torch.arange(n - (b - a), n, device="cuda")[:, None, None]
                dead = torch.arange(n, device="cuda")[None, None, :] > lim
                for g in range(NKV):
                    K, V = (torch.cat([main[w][l][g, :ws], (main if ring[w][l] is None else ring)[w][l][g, ws:n]]).double() for w in (0, 1))
                    x = qs[a:b, GQA * g:GQA * (g + 1)].reshape(-1, HD)
                    S = (x @ K.T).reshape(b - a, GQA, n).masked_fill_(dead, -math.inf)
                    y = (torch.softmax(S, -1).reshape(-1, n) @ V).reshape(b - a, GQA, HD)
                    out[l, s, a:b, GQA * g:GQA * (g + 1)] = _fwht(y) if vr[l] else y
                a = b
        del main, ring
    if mode == "gated":
        out = out * torch.sigmoid(d["gate"].double())
    if mode == "prep":
        out = out * torch.sigmoid(q[..., HD:].double())
    return out[:, 0] if pre else out
