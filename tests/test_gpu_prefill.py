"""Prefill (mk_kv_prefill, mk_kv_prefill_prep) on the GPU: the chunk's causal attention over the mixed store within
2e-3 of the exact attention, bitwise independence from how the prompt is chunked, the stored rows bit-exact, decode
continuing after it, and the raw-projection form against the oracle's prep, gate and o_proj units."""
import numpy as np
import pytest

from kvcase import HD, NH, NKV, check_rows, expected_attention, rel_err, synth_kv

pytestmark = pytest.mark.gpu


def run_prefill(qkv, torch, spec, win, K, V, Q, chunks, ctx):
    """Prefill K/V [P][nl][4][256] with queries Q [nl][P][24][256] in the given chunks -> (store, out [nl][P][24][256])."""
    P, nl = K.shape[0], K.shape[1]
    st = qkv.KVStore(spec, win=win, n_layers=nl, ctx=ctx)
    outs, p = [], 0
    for c in chunks:
        k = torch.from_numpy(np.ascontiguousarray(K[p:p + c])).cuda()
        v = torch.from_numpy(np.ascontiguousarray(V[p:p + c])).cuda()
        q = torch.from_numpy(np.ascontiguousarray(Q[:, p:p + c])).cuda()
        o = torch.empty_like(q)
        print(f"prefill spec={spec!r} win={win} pos={p} T={c}", flush=True)
        st.prefill(0, 0, nl, p, c, k.data_ptr(), v.data_ptr(), 0, q.data_ptr(), o.data_ptr())
        torch.cuda.synchronize()
        outs.append(o.cpu().numpy())
        p += c
    return st, np.concatenate(outs, axis=1)


def pieces(P):
    a, out = 0, []
    while a < P:
        b = min(P, (a // 640 + 1) * 640)
        out.append((a, b))
        a = b
    return out


@pytest.mark.parametrize("spec,win", [("K*=5r,V*=6", 512), ("", 0), ("K*=4,V*=5r", 1280)])
def test_prefill_parity_and_chunking(qkv, oracle, torch_gpu, spec, win):
    torch = torch_gpu
    rng = np.random.default_rng(41)
    P, nl = 2100, 2
    K, V = synth_kv(rng, P, nl, outliers=True)
    Q = rng.standard_normal((nl, P, NH, HD)).astype(np.float32)
    st, out = run_prefill(qkv, torch, spec, win, K, V, Q, [700, 1400], 4096)
    check_rows(oracle, st, K, V, ring_from=max(0, P - qkv.ring_rows(win)))
    for l in range(nl):
        kb, vb, kr, vr = st.kbits[l], st.vbits[l], st.krot[l], st.vrot[l]
        for a, b in pieces(P)[::2]:
            ws = qkv.window_start(b, win)
            ref = expected_attention(oracle, Q[l, a:b], K[:b, l], V[:b, l], b - a, kr, vr, kb, vb, ws, win > 0 and kb != 8,
                                     win > 0 and vb != 8)
            assert rel_err(out[l, a:b], ref) <= 2e-3, (l, a, b)
    st.close()
    for chunks in ([2100], [1, 639, 3, 1457]):
        st2, out2 = run_prefill(qkv, torch, spec, win, K, V, Q, chunks, 4096)
        assert np.array_equal(out2, out), chunks
        st2.close()


def test_prefill_two_segments_then_decode(qkv, oracle, torch_gpu):
    """A 9,000-position context (the last pieces over two key segments of 4,864 positions, the combine folding both),
    then a decode step on the same store."""
    torch = torch_gpu
    rng = np.random.default_rng(42)
    P, nl, win, spec = 9000, 1, 2048, "K*=5r,V*=6"
    K, V = synth_kv(rng, P + 1, nl, outliers=True)
    Q = rng.standard_normal((nl, P, NH, HD)).astype(np.float32)
    st, out = run_prefill(qkv, torch, spec, win, K[:P], V[:P], Q, [5000, 4000], 10240)
    kb, vb, kr, vr = st.kbits[0], st.vbits[0], st.krot[0], st.vrot[0]
    a, b = pieces(P)[-1]
    ref = expected_attention(oracle, Q[0, a:b], K[:b, 0], V[:b, 0], b - a, kr, vr, kb, vb, qkv.window_start(b, win), True, True)
    assert rel_err(out[0, a:b], ref) <= 2e-3
    st2, out2 = run_prefill(qkv, torch, spec, win, K[:P], V[:P], Q, [8200, 800], 10240)
    assert np.array_equal(out2, out)
    st2.close()
    # decode position P
    k = torch.from_numpy(np.ascontiguousarray(K[P:P + 1])).cuda()
    v = torch.from_numpy(np.ascontiguousarray(V[P:P + 1])).cuda()
    st.append(0, 0, 1, P, 1, k.data_ptr(), v.data_ptr(), 0)
    qd = rng.standard_normal((1, 1, 1, NH, HD)).astype(np.float32)
    q = torch.from_numpy(qd).cuda()
    o = torch.empty_like(q)
    st.attend(0, 1, [0], [P + 1], 1, q.data_ptr(), o.data_ptr())
    torch.cuda.synchronize()
    ref = expected_attention(oracle, qd[0, 0], K[:P + 1, 0], V[:P + 1, 0], 1, kr, vr, kb, vb, qkv.window_start(P + 1, win), True, True)
    assert rel_err(o.cpu().numpy()[0, 0], ref) <= 2e-3
    st.close()


def test_prefill_prep(qkv, oracle, torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(43)
    P, nl, win, spec = 1000, 2, 512, "K*=5r,V*=5r"
    K, V = synth_kv(rng, P, nl)
    K *= 4.0
    QG = rng.standard_normal((nl, P, NH, 2 * HD)).astype(np.float32)
    KW = (1 + 0.2 * rng.standard_normal((nl, HD))).astype(np.float32)
    QW = (1 + 0.2 * rng.standard_normal((nl, HD))).astype(np.float32)
    table = oracle.rope_rows(0, P)
    Kp = np.empty_like(K)
    for t in range(P):
        for l in range(nl):
            for g in range(NKV):
                Kp[t, l, g] = oracle.qk_prep(K[t, l, g], KW[l], table[t])
    Qp = np.empty((nl, P, NH, HD), np.float32)
    for l in range(nl):
        for t in range(P):
            for h in range(NH):
                Qp[l, t, h] = oracle.qk_prep(QG[l, t, h, :HD], QW[l], table[t])
    st = qkv.KVStore(spec, win=win, n_layers=nl, ctx=1024)
    k, v, kw, qw, qg = (torch.from_numpy(a).cuda() for a in (K, V, KW, QW, QG))
    o = torch.empty((nl, P, NH, HD), device="cuda")
    xa = torch.zeros((nl, P, 192, 16), dtype=torch.int8, device="cuda")
    xb = torch.zeros_like(xa)
    m = torch.zeros((nl, P, 192, 4), dtype=torch.int16, device="cuda")
    st.prefill_prep(0, 0, nl, 0, P, k.data_ptr(), v.data_ptr(), kw.data_ptr(), qg.data_ptr(), qw.data_ptr(), o.data_ptr(), xa.data_ptr(),
                    xb.data_ptr(), m.data_ptr())
    torch.cuda.synchronize()
    check_rows(oracle, st, Kp, V, ring_from=max(0, P - qkv.ring_rows(win)))
    ref_st, y = run_prefill(qkv, torch, spec, win, Kp, V, Qp, [P], 1024)
    ref_st.close()
    o = o.cpu().numpy()
    og = oracle.gate(y, QG[..., HD:]).reshape(o.shape)
    assert np.abs(o - og).max() <= 1e-6 * np.abs(og).max()
    xa, xb, m = xa.cpu().numpy(), xb.cpu().numpy(), m.cpu().numpy().view(np.uint16)
    for l in range(nl):
        for t in range(0, P, 37):
            ea, eb, em = oracle.q32_row(o[l, t])
            assert np.array_equal(xa[l, t], ea) and np.array_equal(xb[l, t], eb) and np.array_equal(m[l, t], em), (l, t)
    st.close()


def test_prefill_errors(qkv, torch_gpu):
    torch = torch_gpu
    st = qkv.KVStore("", n_layers=1, ctx=256)
    x = torch.zeros((8, 1, NKV, HD), device="cuda")
    q = torch.zeros((1, 8, NH, HD), device="cuda")
    o = torch.empty_like(q)
    with pytest.raises(qkv.KVError):
        st.prefill(0, 0, 1, 16, 8, x.data_ptr(), x.data_ptr(), 0, q.data_ptr(), o.data_ptr())  # gap: nothing stored yet
    with pytest.raises(qkv.KVError):
        st.prefill(0, 0, 1, 250, 8, x.data_ptr(), x.data_ptr(), 0, q.data_ptr(), o.data_ptr())  # beyond ctx
    st.prefill(0, 0, 1, 0, 8, x.data_ptr(), x.data_ptr(), 0, q.data_ptr(), o.data_ptr())
    torch.cuda.synchronize()
    assert np.all(np.isfinite(o.cpu().numpy()))
    st.close()


@pytest.mark.parametrize("page", [256, 32, 96])
def test_prefill_paged_equals_contiguous(qkv, torch_gpu, page):
    """Prefill on a shared page pool with a permuted page table gives the contiguous store's outputs bit for bit.  The
    kernel's copy side follows its tiles from page to page: 32-position pages change page at every tile, and 96-position
    pages put the second key segment's start (position 1,024 of the last pieces) inside a page."""
    torch = torch_gpu
    rng = np.random.default_rng(44)
    P, nl, win, spec = 1500, 1, 512, "K*=5r,V*=6"
    K, V = synth_kv(rng, P, nl, outliers=True)
    Q = rng.standard_normal((nl, P, NH, HD)).astype(np.float32)
    st, ref = run_prefill(qkv, torch, spec, win, K, V, Q, [900, 600], 2048)
    st.close()
    npg = -(-2048 // page)
    paged = qkv.KVStore(spec, win=win, n_layers=nl, n_seq=2, ctx=2048, page=page, n_pages=2 * npg)
    perm = np.random.default_rng(7).permutation(2 * npg)
    paged.set_pages(1, perm[:npg])
    outs, p = [], 0
    for c in (900, 600):
        k = torch.from_numpy(np.ascontiguousarray(K[p:p + c])).cuda()
        v = torch.from_numpy(np.ascontiguousarray(V[p:p + c])).cuda()
        q = torch.from_numpy(np.ascontiguousarray(Q[:, p:p + c])).cuda()
        o = torch.empty_like(q)
        paged.prefill(1, 0, nl, p, c, k.data_ptr(), v.data_ptr(), 0, q.data_ptr(), o.data_ptr())
        torch.cuda.synchronize()
        outs.append(o.cpu().numpy())
        p += c
    assert np.array_equal(np.concatenate(outs, axis=1), ref)
    paged.close()


@pytest.mark.parametrize("spec,win,win_all", [("K*=6r,V*=7", 640, 0), ("", 1024, 1)])
def test_prefill_after_appends(qkv, oracle, torch_gpu, spec, win, win_all):
    """Rows stored by decode-style appends, then a prefill chunk from that position (one-token piece included), then the
    exact attention of the chunk's rows; q8 sides with their own ring (win_all) as well."""
    torch = torch_gpu
    rng = np.random.default_rng(45)
    nl, P0, P = 1, 1279, 2000
    K, V = synth_kv(rng, P, nl, outliers=True)
    Q = rng.standard_normal((nl, P - P0, NH, HD)).astype(np.float32)
    st = qkv.KVStore(spec, win=win, n_layers=nl, ctx=2048, win_all=win_all)
    for p0, c in ((0, 1000), (1000, 279)):
        k = torch.from_numpy(np.ascontiguousarray(K[p0:p0 + c])).cuda()
        v = torch.from_numpy(np.ascontiguousarray(V[p0:p0 + c])).cuda()
        st.append(0, 0, nl, p0, c, k.data_ptr(), v.data_ptr(), 0)
    k = torch.from_numpy(np.ascontiguousarray(K[P0:])).cuda()
    v = torch.from_numpy(np.ascontiguousarray(V[P0:])).cuda()
    q = torch.from_numpy(Q).cuda()
    o = torch.empty_like(q)
    st.prefill(0, 0, nl, P0, P - P0, k.data_ptr(), v.data_ptr(), 0, q.data_ptr(), o.data_ptr())
    torch.cuda.synchronize()
    out = o.cpu().numpy()
    kb, vb, kr, vr = st.kbits[0], st.vbits[0], st.krot[0], st.vrot[0]
    ring_k = win > 0 and (kb != 8 or win_all)
    ring_v = win > 0 and (vb != 8 or win_all)
    for a, b in ((P0, 1280), (1280, 1920), (1920, P)):
        ref = expected_attention(oracle, Q[0, a - P0:b - P0], K[:b, 0], V[:b, 0], b - a, kr, vr, kb, vb, qkv.window_start(b, win),
                                 ring_k, ring_v)
        assert rel_err(out[0, a - P0:b - P0], ref) <= 2e-3, (a, b)
    st.close()


def fill(torch, st, P, nl, seed, chunk=4096):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    for p in range(0, P, chunk):
        c = min(chunk, P - p)
        k, v = (torch.randn(c, nl, NKV, HD, device="cuda", dtype=torch.float16, generator=g) for _ in range(2))
        st.append(0, 0, nl, p, c, k.data_ptr(), v.data_ptr(), 1)
    torch.cuda.synchronize()


@pytest.mark.parametrize("L0,T,spec,win", [(20700, 400, "K*=5r,V*=6", 2048), (41000, 300, "K*=6r,V*=4r", 1024), (170000, 70, "", 0)])
def test_prefill_far_into_a_context(qkv, torch_gpu, L0, T, spec, win):
    """Chunks far into a context: four key segments per row past 20,480 positions, eight past 40,960 (both across the
    boundary of the rule and of a 640-position bucket), and a context whose fp16 tiles exceed the scratch for all four kv
    heads at once.  Bitwise the same in one chunk and in three, and each row within the two forms' tolerances (2e-3 each
    of the exact attention) of the decode attention at its length."""
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(L0)
    k, v = (torch.randn(T, 1, NKV, HD, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(1, T, NH, HD, device="cuda", generator=g)
    outs = []
    for chunks in ([T], [T // 3, 1, T - T // 3 - 1]):
        st = qkv.KVStore(spec, win=win, n_layers=1, ctx=L0 + T)
        fill(torch, st, L0, 1, L0 + 1)
        o, p = torch.full_like(q, float("nan")), 0
        for c in chunks:
            oc = torch.empty(1, c, NH, HD, device="cuda")
            st.prefill(0, 0, 1, L0 + p, c, k[p:].data_ptr(), v[p:].data_ptr(), 0, q[0, p:].data_ptr(), oc.data_ptr())
            torch.cuda.synchronize()
            o[:, p:p + c] = oc
            p += c
        outs.append(o)
        if len(outs) == 1:
            st.close()
    assert torch.equal(outs[0], outs[1])
    d = torch.empty(1, 1, 1, NH, HD, device="cuda")
    for t in (T - 1, T - 30, T - 59):  # (rows of the last bucket: the ring still holds their windows)
        st.attend(0, 1, [0], [L0 + t + 1], 1, q[0, t].data_ptr(), d.data_ptr())
        torch.cuda.synchronize()
        assert rel_err(outs[0][0, t].cpu().numpy(), d[0, 0, 0].cpu().numpy()) <= 2 * 2e-3, t
    st.close()


def test_prefill_more_layers_than_the_scratch_holds(qkv, torch_gpu):
    """17 layers at 9,740 positions: their fp16 tiles exceed the scratch, so each launch holds one layer and one piece and
    writes all its tiles (window tiles included).  Bitwise the layers' own calls, which keep theirs."""
    torch = torch_gpu
    nl, L0, T = 17, 9610, 130  # (one bucket: the ring still holds its window when a layer is stored again)
    st = qkv.KVStore("K*=5r,V*=6", win=2048, n_layers=nl, ctx=L0 + T)
    fill(torch, st, L0, nl, 7)
    g = torch.Generator(device="cuda")
    g.manual_seed(8)
    k, v = (torch.randn(T, nl, NKV, HD, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(nl, T, NH, HD, device="cuda", generator=g)
    o = torch.full_like(q, float("nan"))
    st.prefill(0, 0, nl, L0, T, k.data_ptr(), v.data_ptr(), 0, q.data_ptr(), o.data_ptr())
    torch.cuda.synchronize()
    for l in (0, 9, 16):
        kl, vl, ol = k[:, l].contiguous(), v[:, l].contiguous(), torch.empty_like(q[l])
        st.prefill(0, l, 1, L0, T, kl.data_ptr(), vl.data_ptr(), 0, q[l].contiguous().data_ptr(), ol.data_ptr())
        torch.cuda.synchronize()
        assert torch.equal(ol, o[l]), l
    st.close()


@pytest.mark.parametrize("P,cut", [(1280, 1279), (1281, 5), (650, 640), (1, 0)])
def test_prefill_rows_written_without_the_merge(qkv, oracle, torch_gpu, P, cut):
    # pieces of one key segment (up to 1,280 positions) write their output rows in the attention kernel, later ones through
    # partials: the bucket's last row and the next one's first, one row alone, rotated and plain V, gate and units.  Every
    # chunking the same bits; the last row against the decode step's, each side within 1e-3 of the exact attention
    torch = torch_gpu
    rng = np.random.default_rng(P)
    nl, spec = 2, "K0=5r,V0=6r,K1=6,V1=5"
    K, V = synth_kv(rng, P, nl, outliers=False)
    k, v = torch.from_numpy(K).cuda(), torch.from_numpy(V).cuda()
    qg = torch.from_numpy(rng.standard_normal((nl, P, NH, 2 * HD)).astype(np.float32)).cuda()
    kn, qn = (torch.from_numpy((1 + 0.1 * rng.standard_normal((nl, HD))).astype(np.float32)).cuda() for _ in range(2))

    def run(chunks):
        st = qkv.KVStore(spec, win=640, n_layers=nl, ctx=1400)
        outs, xas, p = [], [], 0
        for c in chunks:
            if not c:
                continue
            kc, vc, qc = k[p:p + c].contiguous(), v[p:p + c].contiguous(), qg[:, p:p + c].contiguous()
            o = torch.full((nl, c, NH, HD), float("nan"), device="cuda")
            xa = torch.zeros((nl, c, 192, 16), dtype=torch.int8, device="cuda")
            xb, meta = torch.zeros_like(xa), torch.zeros((nl, c, 192, 4), dtype=torch.int16, device="cuda")
            st.prefill_prep(0, 0, nl, p, c, kc.data_ptr(), vc.data_ptr(), kn.data_ptr(), qc.data_ptr(), qn.data_ptr(), o.data_ptr(),
                            xa.data_ptr(), xb.data_ptr(), meta.data_ptr())
            torch.cuda.synchronize()
            outs.append(o)
            xas.append(torch.cat([xa.flatten(2).int(), xb.flatten(2).int(), meta.flatten(2).int()], dim=2))
            p += c
        return st, torch.cat(outs, 1), torch.cat(xas, 1)

    st, one, units = run([P])
    st2, two, units2 = run([cut, P - cut])
    assert torch.isfinite(one).all() and torch.equal(one, two) and torch.equal(units, units2)
    for l in range(nl):
        for t in (0, P // 2, P - 1):
            ea, eb, em = oracle.q32_row(one[l, t].cpu().numpy())
            got = units[l, t].cpu().numpy()
            assert np.array_equal(got[:3072], ea.reshape(-1)) and np.array_equal(got[3072:6144], eb.reshape(-1))
            assert np.array_equal(got[6144:].astype(np.int16).view(np.uint16), em.reshape(-1))
    dec = torch.empty((nl, 1, 1, NH, HD), device="cuda")
    last = qg[:, P - 1:].contiguous()
    st.attend_prep(0, nl, [0], [P], 1, last.data_ptr(), qn.data_ptr(), dec.data_ptr())
    torch.cuda.synchronize()
    assert rel_err(one[:, P - 1].cpu().numpy(), dec[:, 0, 0].cpu().numpy()) <= 2e-3
    st.close()
    st2.close()


@pytest.mark.parametrize("spec,win,pos", [("K0=5r,V0=6,K1=6,V1=5r", 2048, 2500), ("", 0, 700)])
def test_prefill_in_less_workspace(qkv, torch_gpu, spec, win, pos):
    """The shapes that a bound on the workspace leaves, on the way down: four pieces per launch, one piece and one layer, one
    layer's tiles at a time, two kv heads', one's (test_host_prefill.py follows their launches).  The same bits in all:
    several groups of a call that starts past a window, and window tiles past the end of their ring (182 tiles, 5,824
    positions).  Less than that is refused, and nothing is stored."""
    torch = torch_gpu
    nl, T = 2, 4000
    g = torch.Generator(device="cuda")
    g.manual_seed(pos)
    k, v = (torch.randn(T, nl, NKV, HD, device="cuda", generator=g) for _ in range(2))
    qg = torch.randn(nl, T, NH, 2 * HD, device="cuda", generator=g)
    kn, qn = (1 + 0.1 * torch.randn(nl, HD, device="cuda", generator=g) for _ in range(2))
    outs = []
    for room in (0, 140, 90, 45, 24, 10):
        st = qkv.KVStore(spec, win=win, n_layers=nl, ctx=pos + T)
        fill(torch, st, pos, nl, 3)
        st.set_rope()
        st.config("prefill_scratch", room << 20)
        o = torch.full((nl, T, NH, HD), float("nan"), device="cuda")
        args = (0, 0, nl, pos, T, k.data_ptr(), v.data_ptr(), kn.data_ptr(), qg.data_ptr(), qn.data_ptr(), o.data_ptr())
        if room == 10:
            with pytest.raises(qkv.KVError, match="no device memory"):
                st.prefill_prep(*args)
            assert st.digest(0)[1] == pos
        else:
            st.prefill_prep(*args)
            torch.cuda.synchronize()
            outs.append(o)
            assert torch.isfinite(o).all() and torch.equal(o, outs[0]), room
        st.close()


@pytest.mark.parametrize("spec,win,T,prep", [("", 0, 342, False), ("K*=5r,V*=6r", 2048, 683, False), ("K*=6,V*=5", 640, 683, True)])
def test_prefill_queries_beside_the_tiles(qkv, torch_gpu, spec, win, T, prep):
    # launches of up to 64 workgroups (128 with prep or rotated K) take queries prepared with the tiles, larger ones prepare
    # their own: the call of one token less is the last of the first kind (4 x 16 workgroups; 4 x (30 + 2)).  The same bits
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(T)
    k, v = (torch.randn(T, 1, NKV, HD, device="cuda", generator=g) for _ in range(2))
    q = torch.randn(1, T, NH, (2 if prep else 1) * HD, device="cuda", generator=g)
    kn, qn = (1 + 0.1 * torch.randn(1, HD, device="cuda", generator=g) for _ in range(2))
    outs = []
    for chunks in ([T], [T - 1, 1]):
        st = qkv.KVStore(spec, win=win, n_layers=1, ctx=T)
        st.set_rope()
        o, p = torch.full((1, T, NH, HD), float("nan"), device="cuda"), 0
        for c in chunks:
            oc, qc = torch.empty(1, c, NH, HD, device="cuda"), q[:, p:p + c].contiguous()
            if prep:
                st.prefill_prep(0, 0, 1, p, c, k[p:].data_ptr(), v[p:].data_ptr(), kn.data_ptr(), qc.data_ptr(), qn.data_ptr(), oc.data_ptr())
            else:
                st.prefill(0, 0, 1, p, c, k[p:].data_ptr(), v[p:].data_ptr(), 0, qc.data_ptr(), oc.data_ptr())
            torch.cuda.synchronize()
            o[:, p:p + c] = oc
            p += c
        outs.append(o)
        st.close()
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])
