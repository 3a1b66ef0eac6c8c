"""Performance cases of the quantized path, through its public entry points.

The shapes are the ones this repository's engine, tests and benchmark use:
hidden 3840, MLP 15360, vocabulary 262144; five of six layers attend a
1024-slot ring (16 query and 8 KV heads of 256), every sixth attends the whole
prompt (16 query heads and one k == v head of 512). Weights are Gaussian
matrices through the library's own quantizer, so codes and scales have the
distribution a checkpoint gives. ``exact`` quantizes the same matrices with
plain torch and computes everything after that in 64 bits.

Kinds (``case["kind"]``):

- ``gemv``: decode projections of several layers, recorded in one graph.
- ``token``: one decode token through the engine mirror (``forward``).
- ``verify``: several draft tokens through the projections of a layer.
- ``attn``: decode attention (with this token's K/V) of several layers.
- ``w4a16``: a prefill GEMM on int4 weights.
- ``w8a8`` / ``w4a8``: activation quantizer and int8 GEMM.
- ``pre_attn``: causal attention of a prefill chunk.
- ``chunk``: one 128-token prefill chunk through the layer graph.
- ``quant``: quantizing a matrix at load.
"""
import importlib
import math

import torch

PKG = "gemma4-12b-snapdragonx2elite_amd"
ops = importlib.import_module(PKG + ".ops")
E = importlib.import_module(PKG + ".vk_engine")
_lib = importlib.import_module(PKG + "._lib")

H, I, V, BLK = 3840, 15360, 262144, 32
SLIDING = dict(nH=16, nkv=8, hd=256, window=1024)
GLOBAL = dict(nH=16, nkv=1, hd=512, window=0)
LAYER_SCALE = 0.75
F16, F32, F64 = torch.float16, torch.float32, torch.float64


def listed():
    return [
        # the k == v projections of the eight global layers, fp32 activations as the reference engine keeps them:
        # the smallest matrices of a token, where launch and ramp are most of the time
        dict(name="gemv_kv512_f32", kind="gemv", N=512, K=H, layers=8, half=False, e4m3=False),
        # the vocabulary projection of every decoded token, with the engine's GEMV_FP8 scales
        dict(name="gemv_lm_head_e4m3", kind="gemv", N=V, K=H, layers=1, half=True, e4m3=True),
        # a decoded token: one period of the layer pattern (five sliding layers, one global) and the vocabulary
        # projection, at a position past the ring
        dict(name="token_6_layers", kind="token", layers=6, pos=2500, stride=4096, half=True, e4m3=False),
        # speculative decoding: eight draft tokens through all projections of two layers
        dict(name="verify_8_tokens", kind="verify", M=8, q=4096, kv=2048, layers=2, exact=False, e4m3=False),
        # decode attention of the global layers far into a long context
        dict(name="attn_global_8k", kind="attn", nH=16, nkv=1, hd=512, window=0, stride=8192, pos=8100, layers=4),
        # four prefill chunks at once through the up (or gate) projection
        dict(name="w4a16_m512", kind="w4a16", M=512, N=I, K=H),
        # the ragged end of a prompt through the down projection
        dict(name="w4a16_down_m77", kind="w4a16", M=77, N=H, K=I),
        # the int8 prefill route on a long batch of rows
        dict(name="w8a8_m2048", kind="w8a8", M=2048, N=I, K=H, packed=True),
        # int8 activations on int4 weights, at the prefill chunk the reference measures it on
        dict(name="w4a8_m128", kind="w4a8", M=128, N=I, K=H),
        # a chunk of a long prompt in a global layer
        dict(name="pre_attn_global_8k", kind="pre_attn", M=128, nH=16, nkv=1, hd=512, window=0, stride=8192, p0=8000),
        # the last chunk of a 4096-token prompt through one period of the layer pattern
        dict(name="chunk_6_layers", kind="chunk", layers=6, p0=3968, stride=4096),
        # model load: int4 codes, both scale formats and the folded int8 weights of one MLP matrix
        dict(name="quant_mlp", kind="quant", N=I, K=H, fp8=True, i8=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "token", "verify", "attn", "w4a16", "w4a16", "w8a8", "w4a8", "pre_attn", "chunk",
                       "quant"])
    k32 = lambda lo, hi: max(1, _log(rng, lo, hi) // 32) * 32   # noqa: E731
    k64 = lambda lo, hi: max(1, _log(rng, lo, hi) // 64) * 64   # noqa: E731
    if kind == "gemv":
        N, K = _log(rng, 256, 65536), k32(1024, I)
        return dict(kind=kind, N=N, K=K, layers=max(1, min(8, int(2e8 / (N * K)))), half=rng.random() < 0.6,
                    e4m3=rng.random() < 0.4)
    if kind == "token":
        return dict(kind=kind, layers=rng.choice([2, 3, 6]), pos=_log(rng, 16, 4000), stride=4096,
                    half=rng.random() < 0.7, e4m3=rng.random() < 0.4)
    if kind == "verify":
        kv, q = rng.choice([(2048, 4096), (512, 8192)])
        return dict(kind=kind, M=rng.randint(2, 16), q=q, kv=kv, layers=rng.randint(1, 3), exact=rng.random() < 0.3,
                    e4m3=rng.random() < 0.4)
    if kind == "attn":
        a = rng.choice([SLIDING, GLOBAL])
        stride = a["window"] or rng.choice([2048, 4096, 8192])
        return dict(kind=kind, stride=stride, pos=rng.randint(1, stride - 1), layers=rng.randint(1, 6), **a)
    if kind == "w4a16":
        N, K = rng.choice([(I, H), (H, I), (4096, H), (H, 4096), (8192, H), (_log(rng, 500, 16000), k32(1000, 8000))])
        return dict(kind=kind, M=_log(rng, 17, 1024), N=N, K=K)
    if kind in ("w8a8", "w4a8"):
        N, K = rng.choice([(I, H), (H, I), (4096, H), (H, 4096), (_log(rng, 500, 16000), k64(1000, 8000))])
        c = dict(kind=kind, M=_log(rng, 17, 2048 if kind == "w8a8" else 1024), N=N, K=K)
        return dict(c, packed=rng.random() < 0.7) if kind == "w8a8" else c
    if kind == "pre_attn":
        a = rng.choice([SLIDING, GLOBAL])
        stride = a["window"] or rng.choice([2048, 4096, 8192])
        M = rng.randint(9, 128)
        return dict(kind=kind, M=M, stride=stride, p0=rng.randint(0, (stride if not a["window"] else 4096) - M), **a)
    if kind == "chunk":
        return dict(kind=kind, layers=rng.choice([2, 3, 6]), p0=rng.randint(0, 3968), stride=4096)
    return dict(kind=kind, N=_log(rng, 300, 20000), K=k32(1000, I), fp8=rng.random() < 0.5, i8=rng.random() < 0.5)


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _weight(gen, N, K):
    return torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5


def _norms(gen, n, lo=0.5):
    return torch.rand(n, device="cuda", generator=gen) + lo


def _layers(case):
    """Attention kind of each layer: the last one is global, as every sixth is."""
    n = case["layers"]
    return [GLOBAL if li == n - 1 else SLIDING for li in range(n)]


def _rope_tab(n, hd, base=10000.0):
    ang = torch.arange(n, device="cuda", dtype=F64)[:, None] / base ** (torch.arange(0, hd, 2, device="cuda",
                                                                                      dtype=F64) / hd)[None]
    ang = torch.cat([ang, ang], 1)
    return torch.cos(ang).to(F32).contiguous(), torch.sin(ang).to(F32).contiguous()


def _layer_inputs(gen, a, stride):
    """One layer's matrices (name -> fp32 W), norm weights and fp16 caches."""
    nq, nk, hd = a["nH"] * a["hd"], a["nkv"] * a["hd"], a["hd"]
    shapes = dict(q=(nq, H), k=(nk, H), o=(H, nq), g=(I, H), u=(I, H), d=(H, I))
    if a["window"]:
        shapes["v"] = (nk, H)
    mats = {m: _weight(gen, *s) for m, s in shapes.items()}
    norms = {m: _norms(gen, n) for m, n in dict(inw=H, paw=H, pfw=H, ofw=H, knw=hd).items()}
    for m in ("paw", "ofw"):   # a block adds a fraction of the residual stream
        norms[m] *= 0.3
    # unscaled scores: the q-norm weights carry the 1 / sqrt(hd)
    norms["qnw"] = _norms(gen, hd) * hd ** -0.5
    st = a["window"] or stride
    kc, vc = (torch.randn(a["nkv"] * st * hd, device="cuda", generator=gen).to(F16) for _ in range(2))
    return mats, norms, kc, vc, st


def _own(state):
    """The engine keeps what its graphs use for the process; here the state owns it."""
    state["keep"] = list(E.KEEP)
    E.KEEP.clear()
    return state


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _gen(seed))


def run(state):
    return state["run"](state)


def _graph(body):
    g = ops.Graph()
    with g.capture():
        body()
    return g


def _launch(state):
    state["graph"].launch(torch.cuda.current_stream())
    return state["out"]


def _scales(e4m3, wq, sc16, sc32, N, K):
    if not e4m3:
        return sc16, 1.0, _lib.SCALE_F16
    sc8, inv = ops.scales_e4m3(sc32, N, K)
    return sc8, inv, _lib.SCALE_E4M3


def _gemv_inputs(case, gen):
    N, K = case["N"], case["K"]
    return [(_weight(gen, N, K), torch.randn(K, device="cuda", generator=gen).to(F16 if case["half"] else F32))
            for _ in range(case["layers"])]


def _prepare_gemv(case, gen):
    N, K = case["N"], case["K"]
    mats = []
    for W, x in _gemv_inputs(case, gen):
        q = ops.quantize(W)
        mats.append((q[0], *_scales(case["e4m3"], *q, N, K), x))
    y = torch.empty(case["layers"], N, device="cuda")
    ws = ops.default_workspace(N, K)

    def body():
        for i, (wq, sc, inv, fmt, x) in enumerate(mats):
            ops.gemv(x, wq, sc, N, K, scale_fmt=fmt, inv=inv, y=y[i], ws=ws)

    return dict(run=_launch, graph=_graph(body), out=y, hold=(mats, ws))


def _verify_shapes(case):
    return dict(q=(case["q"], H), k=(case["kv"], H), o=(H, case["q"]), g=(I, H), u=(I, H), d=(H, I))


def _verify_inputs(case, gen):
    out = []
    for _ in range(case["layers"]):
        for N, K in _verify_shapes(case).values():
            out.append((_weight(gen, N, K), torch.randn(case["M"], K, device="cuda", generator=gen).to(F16)))
    return out


def _prepare_verify(case, gen):
    M, mats = case["M"], []
    for W, x in _verify_inputs(case, gen):
        N, K = W.shape
        q = ops.quantize(W)
        mats.append((N, K, q[0], *_scales(case["e4m3"], *q, N, K), x, torch.empty(M, N, device="cuda", dtype=F16)))
    need = max(ops.gemv_multi_workspace_bytes(M, m[0], m[1]) for m in mats)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")

    def body():
        for N, K, wq, sc, inv, fmt, x, y in mats:
            ops.gemv_multi(x, wq, sc, N, K, scale_fmt=fmt, inv=inv, y=y, exact=case["exact"], ws=ws)

    return dict(run=_launch, graph=_graph(body), out=[m[-1] for m in mats], hold=(mats, ws))


def _attn_inputs(case, gen):
    nH, nkv, hd, st = case["nH"], case["nkv"], case["hd"], case["stride"]
    nq, nk = nH * hd, nkv * hd
    cos, sin = _rope_tab(case["pos"] + 1, hd)
    out = []
    for _ in range(case["layers"]):
        qkv = torch.randn(nq + nk * (2 if case["window"] else 1), device="cuda", generator=gen)
        kc, vc = (torch.randn(nkv * st * hd, device="cuda", generator=gen).to(F16) for _ in range(2))
        out.append((qkv, _norms(gen, hd), _norms(gen, hd) * hd ** -0.5, kc, vc))
    return out, cos[case["pos"]].contiguous(), sin[case["pos"]].contiguous()


def _prepare_attn(case, gen):
    nH, nkv, hd, st, win = (case[k] for k in ("nH", "nkv", "hd", "stride", "window"))
    nq, nk = nH * hd, nkv * hd
    ins, cos, sin = _attn_inputs(case, gen)
    dyn = torch.tensor([case["pos"], case["pos"] + 1, 0, 0], dtype=torch.int32, device="cuda")
    out = torch.empty(case["layers"], nq, device="cuda", dtype=F16)
    ws = ops.attn_workspace(nH, hd, st)

    def body():
        for i, (qkv, knw, qnw, kc, vc) in enumerate(ins):
            ops.prepkv_attn(qkv, knw, qnw, cos, sin, kc, vc, out[i], nH=nH, nkv=nkv, hd=hd, stride=st, window=win,
                            qoff=0, koff=nq, voff=nq + nk if win else nq, keqv=not win, grp=nH // nkv, dyn=dyn, ws=ws)

    return dict(run=_launch, graph=_graph(body), out=[out, *(t for x in ins for t in x[3:])],
                hold=(ins, cos, sin, dyn, ws))


def _gemm_inputs(case, gen):
    return _weight(gen, case["N"], case["K"]), torch.randn(case["M"], case["K"], device="cuda", generator=gen).to(F16)


def _prepare_w4a16(case, gen):
    W, X = _gemm_inputs(case, gen)
    M, N, K = case["M"], case["N"], case["K"]
    wq, sc16, _ = ops.quantize(W)
    need = ops.gemm_workspace_bytes(M, N, K)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda") if need else None
    return dict(run=lambda s: ops.gemm_w4a16(s["X"], s["wq"], s["sc"], N, Y=s["Y"], ws=s["ws"]), X=X, wq=wq, sc=sc16,
                ws=ws, Y=torch.empty(M, N, dtype=F16, device="cuda"))


def _run_w8a8(s):
    ops.quant_act_i8(s["X"], s["A"], s["sa"])
    if s["packed"]:
        return ops.gemm_w8a8_packed(s["A"], s["W8"], s["sa"], s["sw"], s["N"], Y=s["Y"])
    return ops.gemm_w8a8(s["A"], s["W8"], s["sa"], s["sw"], Y=s["Y"])


def _run_w4a8(s):
    ops.quant_act_i8(s["X"], s["A"], s["sa"])
    return ops.gemm_w4a8(s["A"], s["wq"], s["ratio"], s["sa"], s["sw"], s["N"], Y=s["Y"])


def _int8_state(case, X, **kw):
    M, N, K = case["M"], case["N"], case["K"]
    return dict(X=X, N=N, A=torch.empty(M, K, dtype=torch.int8, device="cuda"), sa=torch.empty(M, device="cuda"),
                Y=torch.empty(M, N, dtype=F16, device="cuda"), **kw)


def _prepare_w8a8(case, gen):
    W, X = _gemm_inputs(case, gen)
    wq, _, sc32 = ops.quantize(W)
    W8, _, sw16 = ops.w8_fold(wq, sc32, case["N"], case["K"])
    return _int8_state(case, X, run=_run_w8a8, packed=case["packed"], sw=sw16,
                       W8=ops.w8_pack(W8) if case["packed"] else W8)


def _prepare_w4a8(case, gen):
    W, X = _gemm_inputs(case, gen)
    wq, _, sc32 = ops.quantize(W)
    _, sw32, sw16 = ops.w8_fold(wq, sc32, case["N"], case["K"])
    return _int8_state(case, X, run=_run_w4a8, wq=wq, ratio=ops.w4a8_ratio(sc32, sw32, case["N"], case["K"]), sw=sw16)


def _pre_attn_inputs(case, gen):
    nH, nkv, hd, st, M = (case[k] for k in ("nH", "nkv", "hd", "stride", "M"))
    q = torch.randn(M, nH * hd, device="cuda", generator=gen).to(F16)
    qnw = _norms(gen, hd) * hd ** -0.5
    kc, vc = (torch.randn(nkv * st * hd, device="cuda", generator=gen).to(F16) for _ in range(2))
    cos, sin = (t[case["p0"]:].contiguous() for t in _rope_tab(case["p0"] + M, hd))
    return q, qnw, cos, sin, kc, vc


def _prepare_pre_attn(case, gen):
    nH, nkv, hd, st, M, win = (case[k] for k in ("nH", "nkv", "hd", "stride", "M", "window"))
    ins = _pre_attn_inputs(case, gen)
    kw = dict(M=M, ldq=nH * hd, nH=nH, nkv=nkv, hd=hd, stride=st, window=win, max_keys=win or st,
              dyn=torch.tensor([case["p0"], M, 0, 0], dtype=torch.int32, device="cuda"),
              ws=ops.pre_attn_workspace(M, nH, nkv, hd, win or st))
    out = torch.empty(M, nH * hd, dtype=F16, device="cuda")
    return dict(run=lambda s: ops.pre_attn(*s["ins"], s["out"], **s["kw"]), ins=ins, kw=kw, out=out)


def _run_quant(s):
    q = E.quant(s["W"], fp8=s["fp8"], prefill_i8=s["i8"])
    return [b.t for b in (q.bw, q.bs16, q.bs, q.w8, q.sw8) if b is not None] + [q.inv]


def _prepare_quant(case, gen):
    return dict(run=_run_quant, W=_weight(gen, case["N"], case["K"]), fp8=case["fp8"], i8=case["i8"])


def _scale_word(v):
    return int(torch.tensor([v], dtype=F32).view(torch.int32).item())


def _qw(W, fp8):
    return E.quant(W, pf=False, fp8=fp8, prefill_i8=False), tuple(W.shape)


def _token_inputs(case, gen):
    """Token id, embedding rows, layers, final norm, vocabulary matrix."""
    tid = int(torch.randint(0, V, (1,), device="cuda", generator=gen).item())
    emb = torch.randn(V, H, device="cuda", generator=gen)
    layers = [(a, _layer_inputs(gen, a, case["stride"])) for a in _layers(case)]
    return tid, emb, layers, _norms(gen, H), _weight(gen, V, H)


def _prepare_token(case, gen):
    tid, emb, ins, finw, lm = _token_inputs(case, gen)
    xdt = F16 if case["half"] else F32
    buf = lambda t: E.Buf(tensor=t)   # noqa: E731
    fb = lambda n: E.Buf(n * 4)   # noqa: E731
    B = {k: fb(n) for k, n in dict(h=H, normed=H, normed2=H, o=H, down=H, normed_f=H, attn=8192, gate=I, up=I, act=I,
                                   logits=V, qkv=16384).items()}
    dyn, duh, dui = E.buf_u32([0, 0, 0, 0]), [H], [I]
    max_pos = case["stride"]
    tabs = {hd: _rope_tab(max_pos, hd) for hd in (256, 512)}
    rows = {hd: (fb(hd), fb(hd)) for hd in (256, 512)}
    layers, caches = [], []
    for a, (mats, nw, kc, vc, st) in ins:
        hd, nkv, win, nH = a["hd"], a["nkv"], a["window"], a["nH"]
        nq, nk = nH * hd, nkv * hd
        W = {m: _qw(t, case["e4m3"]) for m, t in mats.items()}
        mats.clear()
        n = {k: buf(t) for k, t in nw.items()}
        cb, sb = rows[hd]
        kcb, vcb = buf(kc), buf(vc)
        caches += [kc, vc]
        P = [nkv, hd, nq, nq + nk if win else nq, 0 if win else 1, st, win, 0]
        A = [nH, nkv, hd, st, win, 0, nH // nkv, 0]
        L = dict(
            d_in=E.normbg(B["h"], n["inw"], B["normed"], duh, out_dtype=xdt),
            d_q=E.gemv_ds(W["q"], B["normed"], B["qkv"], 0, x_dtype=xdt),
            d_k=E.gemv_ds(W["k"], B["normed"], B["qkv"], nq * 4, x_dtype=xdt),
            d_v=E.gemv_ds(W["v"], B["normed"], B["qkv"], (nq + nk) * 4, x_dtype=xdt) if win else None,
            d_prep=E.prepkv_ds(B["qkv"], n["knw"], cb, sb, kcb, vcb, P, dyn),
            d_attn=E.attn_ds(B["qkv"], n["qnw"], cb, sb, kcb, vcb, B["attn"], A, dyn, out_dtype=xdt),
            d_o=E.gemv_ds(W["o"], B["attn"], B["o"], 0, x_dtype=xdt),
            d_na=E.normadd_ds(B["o"], n["paw"], B["h"], duh),
            d_pfn=E.normbg(B["h"], n["pfw"], B["normed2"], duh, out_dtype=xdt),
            d_g=E.gemv_ds(W["g"], B["normed2"], B["gate"], 0, x_dtype=xdt),
            d_u=E.gemv_ds(W["u"], B["normed2"], B["up"], 0, x_dtype=xdt),
            d_gm=E.gelumul_ds(B["gate"], B["up"], B["act"], dui, out_dtype=xdt),
            d_d=E.gemv_ds(W["d"], B["act"], B["down"], 0, x_dtype=xdt),
            d_nas=E.normadd_ds(B["down"], n["ofw"], B["h"], [H, _scale_word(LAYER_SCALE)]))
        L["d_gu"] = E.gate_up_ds(W["g"], W["u"], B["normed2"], B["act"], x_dtype=xdt, act_dtype=xdt)
        layers.append(L)
    d_fin = E.normbg(B["h"], buf(finw), B["normed_f"], duh, out_dtype=xdt)
    d_lm = E.gemv_ds(_qw(lm, case["e4m3"]), B["normed_f"], B["logits"], 0, x_dtype=xdt)
    del lm
    step = torch.zeros(2, dtype=torch.int32, pin_memory=True)
    d_tok = E.token_inputs_ds(step, buf(emb), B["h"], dyn,
                              [(buf(tabs[hd][0]), buf(tabs[hd][1]), hd, *rows[hd]) for hd in tabs], vocab=V, H=H,
                              max_pos=max_pos)
    g = E.record_decode(layers, d_fin, d_lm, d_tok=d_tok)
    logits = B["logits"].view(F32, V)

    def one(s):
        E.forward(g, step, tid, case["pos"], vocab=V, max_pos=max_pos, timeout_ms=20000)
        return s["out"]

    return _own(dict(run=one, graph=g, out=[logits, *caches], hold=(layers, B, step, d_tok, rows, tabs)))


def _chunk_inputs(case, gen):
    h0 = torch.randn(E.MC, H, device="cuda", generator=gen)
    return h0, [(a, _layer_inputs(gen, a, case["stride"])) for a in _layers(case)]


def _prepare_chunk(case, gen):
    h0, ins = _chunk_inputs(case, gen)
    M, p0 = E.MC, case["p0"]
    buf = lambda t: E.Buf(tensor=t)   # noqa: E731
    fb = lambda n: E.Buf(n * 2)   # noqa: E731
    h = torch.empty_like(h0)
    X, Np, T, QKV, At, G, U, AC = buf(h), fb(M * H), fb(M * H), fb(M * 8704), fb(M * 8192), fb(M * I), fb(M * I), \
        fb(M * I)
    rope = {hd: tuple(buf(t[p0:].contiguous()) for t in _rope_tab(p0 + M, hd)) for hd in (256, 512)}
    dyn = E.buf_u32([p0, M, 0, 0])
    gk = dict(x_dtype=F16, y_dtype=F16)
    layers, caches = [], []
    for a, (mats, nw, kc, vc, st) in ins:
        hd, nkv, win, nH = a["hd"], a["nkv"], a["window"], a["nH"]
        nq, nk = nH * hd, nkv * hd
        ld = nq + nk * (2 if win else 1)
        W = {m: _qw(t, False) for m, t in mats.items()}
        mats.clear()
        n = {k: buf(t) for k, t in nw.items()}
        cb, sb = rope[hd]
        kcb, vcb = buf(kc), buf(vc)
        caches += [kc, vc]
        L = dict(
            p_in=E.pre_norm_ds(X, n["inw"], Np, [H], out_dtype=F16),
            p_qkv=E.gemm_cat_ds([W[m] for m in ("q", "k", "v") if m in W], Np, QKV, **gk),
            p_prep=E.pre_prepkv_ds(QKV, QKV, n["knw"], cb, sb, kcb, vcb, [nkv, hd, nk, 0, st, win, 0, 0], dyn,
                                   kv_dtype=F16, ld=ld, koff=nq, voff=nq + nk if win else nq),
            p_attn=E.pre_attn_ds(QKV, n["qnw"], cb, sb, kcb, vcb, At, [nH, nq, hd, st, win, nH // nkv, 0, 0], dyn, nkv,
                                 q_dtype=F16, out_dtype=F16, ldq=ld),
            p_o=E.gemm_ds(W["o"], At, T, **gk),
            p_na=E.pre_na_ds(T, n["paw"], X, [H], x_dtype=F16),
            p_pfn=E.pre_norm_ds(X, n["pfw"], Np, [H], out_dtype=F16),
            p_gu=E.pre_gate_up_ds(W["g"], W["u"], Np, AC),
            p_d=E.gemm_ds(W["d"], AC, T, **gk),
            p_nas=E.pre_na_ds(T, n["ofw"], X, [H, _scale_word(LAYER_SCALE)], x_dtype=F16))
        layers.append(L)
    g = E.record_prefill(layers, gemm_norms=True)

    def one(s):
        with torch.cuda.stream(g.stream):
            h.copy_(h0)
        E.submit(g, timeout_ms=20000)
        return s["out"]

    return _own(dict(run=one, graph=g, out=[h, *caches], hold=(layers, h0, X, Np, T, QKV, At, G, U, AC, rope, dyn)))


# ---- what a pass cannot do without ------------------------------------------
def _w_bytes(N, K, sb=2):
    return N * K // 2 + N * (K // BLK) * sb


def _layer_mats(a):
    nq, nk = a["nH"] * a["hd"], a["nkv"] * a["hd"]
    return [(nq, H), (nk, H)] + ([(nk, H)] if a["window"] else []) + [(H, nq), (I, H), (I, H), (H, I)]


def _keys(pos, window):
    return min(pos + 1, window) if window else pos + 1


def _chunk_scores(p0, M, window):
    return sum(_keys(p0 + m, window) for m in range(M))


def work(case):
    c, k = case, case["kind"]
    sb = 1 if c.get("e4m3") else 2
    if k == "gemv":
        N, K, L = c["N"], c["K"], c["layers"]
        return dict(bytes=L * (_w_bytes(N, K, sb) + K * (2 if c["half"] else 4) + 4 * N), flops=2 * L * N * K)
    if k == "verify":
        s, M, L = _verify_shapes(c).values(), c["M"], c["layers"]
        return dict(bytes=L * sum(_w_bytes(N, K, sb) + 2 * M * (N + K) for N, K in s),
                    flops=2 * M * L * sum(N * K for N, K in s))
    if k == "token":
        b = f = 0
        for a in _layers(c):
            T = _keys(c["pos"], a["window"])
            b += sum(_w_bytes(N, K, sb) for N, K in _layer_mats(a)) + 4 * T * a["nkv"] * a["hd"]
            f += sum(2 * N * K for N, K in _layer_mats(a)) + 4 * T * a["nH"] * a["hd"]
        return dict(bytes=b + _w_bytes(V, H, sb) + 4 * V, flops=f + 2 * V * H)
    if k == "attn":
        T, hd = _keys(c["pos"], c["window"]), c["hd"]
        return dict(bytes=c["layers"] * (4 * T * c["nkv"] * hd + 6 * c["nH"] * hd),
                    flops=4 * c["layers"] * T * c["nH"] * hd)
    if k == "w4a16":
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=_w_bytes(N, K) + 2 * M * (N + K), flops=2 * M * N * K)
    if k in ("w8a8", "w4a8"):
        M, N, K = c["M"], c["N"], c["K"]
        return dict(bytes=(N * K if k == "w8a8" else _w_bytes(N, K)) + 2 * M * (N + K), flops=2 * M * N * K)
    if k == "pre_attn":
        M, hd, nH = c["M"], c["hd"], c["nH"]
        return dict(bytes=4 * M * nH * hd + 4 * c["nkv"] * hd * _keys(c["p0"] + M - 1, c["window"]),
                    flops=4 * nH * hd * _chunk_scores(c["p0"], M, c["window"]))
    if k == "chunk":
        M, b, f = E.MC, 8 * E.MC * H, 0
        for a in _layers(c):
            b += sum(_w_bytes(N, K) for N, K in _layer_mats(a)) + 4 * a["nkv"] * a["hd"] * _keys(c["p0"] + M, a["window"])
            f += sum(2 * M * N * K for N, K in _layer_mats(a)) \
                + 4 * a["nH"] * a["hd"] * _chunk_scores(c["p0"], M, a["window"])
        return dict(bytes=b, flops=f)
    N, K = c["N"], c["K"]
    return dict(bytes=4 * N * K + _w_bytes(N, K) + (N * (K // BLK) if c["fp8"] else 0) + (N * K + 2 * N if c["i8"] else 0),
                flops=0)


def tolerance(case):
    return TOLERANCE[case["kind"]](case)


# About four times the distance of these outputs from the 64-bit results.
TOLERANCE = {
    # fp32 sums of exact products: 1.3e-7; with fp16 x the offset of the codes is taken off per block: 9.4e-6
    "gemv": lambda c: {"rel": 4e-5 if c["half"] else 1e-6},
    # fp16 outputs: 2.1e-4 (attention and the products of fp16-rounded weights up to 2.8e-4)
    "verify": lambda c: {"rel": 9e-4},
    "attn": lambda c: {"rel": 9e-4},
    "w4a16": lambda c: {"rel": 1.2e-3},
    "pre_attn": lambda c: {"rel": 1.2e-3},
    # integer sums and a fixed order of roundings
    "w8a8": lambda c: "exact",
    "w4a8": lambda c: "exact",
    "quant": lambda c: "exact",
    # fp16 GEMV and GEMM inputs and fp16 caches, carried through the layers: 6.5e-4 and 1.0e-3
    "token": lambda c: {"rel": 2.6e-3},
    "chunk": lambda c: {"rel": 4e-3},
}


# ---- the same in 64 bits, without this repository's code ----------------------
def _div(a, b):
    """The correctly rounded fp32 quotient of fp32 values."""
    return (a.to(F64) / (b.to(F64) if torch.is_tensor(b) else b)).to(F32)


def _block_scales(W):
    return torch.clamp(_div(W.view(W.shape[0], -1, BLK).abs().amax(2), 7.0), min=1e-8)


def _codes(W):
    """Signed int4 codes and fp32 block scales of the format."""
    sc = _block_scales(W)
    return torch.clamp(torch.round(_div(W.view(*sc.shape, BLK), sc[:, :, None])), -8, 7), sc


def _lift(sc):
    shift = math.floor(math.log2(256.0 / float(sc.max())))
    return torch.clamp(sc * 2.0 ** shift, 0.0, 448.0).to(torch.float8_e4m3fn), 2.0 ** -shift


def _mul(x, W, e4m3=False):
    """x @ W^T with W the matrix before quantization, by row blocks."""
    shift = None
    if e4m3:   # the lift is one per matrix
        sc = _block_scales(W)
        shift = math.floor(math.log2(256.0 / float(sc.max())))
    out = []
    for r in range(0, W.shape[0], 16384):
        q, sc = _codes(W[r:r + 16384])
        if e4m3:
            s = torch.clamp(sc * 2.0 ** shift, 0.0, 448.0).to(torch.float8_e4m3fn).to(F64) * 2.0 ** -shift
        else:
            s = sc.to(F16).to(F64)
        out.append(x @ (q.to(F64) * s[:, :, None]).view(q.shape[0], -1).T)
    return torch.cat(out, -1)


def _rms(x, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)
    return y if w is None else y * w.to(F64)


def _rope(x, cos, sin):
    hf = x.shape[-1] // 2
    return x * cos.to(F64) + torch.cat([-x[..., hf:], x[..., :hf]], -1) * sin.to(F64)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _attend(q, kc, vc, a, st, p0):
    """q [M][nH][hd] after norm and RoPE over caches [nkv][st][hd] (fp64)."""
    M, win = q.shape[0], a["window"]
    pos = p0 + torch.arange(M, device="cuda")
    s = torch.arange(st, device="cuda")
    live = s[None] < torch.clamp(pos + 1, max=win or st)[:, None]
    if win:
        base = p0 + M - 1
        live &= (base - (base + win - s) % win)[None] <= pos[:, None]
    grp = a["nH"] // a["nkv"]
    out = []
    for h in range(a["nH"]):
        sc = (q[:, h] @ kc[h // grp].T).masked_fill(~live, -math.inf)
        out.append(torch.softmax(sc, -1) @ vc[h // grp])
    return torch.stack(out, 1).reshape(M, -1)


def _into_caches(k, v, nw, cos, sin, kc, vc, a, st, p0):
    """k, v [M][nk] normed (and k rotated) into the fp64 caches."""
    M, nkv, hd = k.shape[0], a["nkv"], a["hd"]
    kn = _rope(_rms(k.view(M, nkv, hd), nw), cos[:, None], sin[:, None])
    vn = _rms(v.view(M, nkv, hd))
    kc, vc = (t.to(F64).view(nkv, st, hd).clone() for t in (kc, vc))
    slots = (p0 + torch.arange(M, device="cuda")) % (a["window"] or 1 << 30)
    kc[:, slots], vc[:, slots] = kn.transpose(0, 1), vn.transpose(0, 1)
    return kc, vc


def _layer_exact(h, a, ins, cos, sin, p0, e4m3):
    mats, nw, kc, vc, st = ins
    M, hd = h.shape[0], a["hd"]
    mul = lambda x, m: _mul(x, mats[m], e4m3)   # noqa: E731
    x = _rms(h, nw["inw"])
    q, k = mul(x, "q"), mul(x, "k")
    v = mul(x, "v") if "v" in mats else k
    kc, vc = _into_caches(k, v, nw["knw"], cos, sin, kc, vc, a, st, p0)
    q = _rope(_rms(q.view(M, a["nH"], hd), nw["qnw"]), cos[:, None], sin[:, None])
    h = h + _rms(mul(_attend(q, kc, vc, a, st, p0), "o"), nw["paw"])
    x = _rms(h, nw["pfw"])
    h = (h + _rms(mul(_gelu(mul(x, "g")) * mul(x, "u"), "d"), nw["ofw"])) * LAYER_SCALE
    return h, kc.view(-1), vc.view(-1)


def _stack_exact(h, ins, p0, e4m3):
    caches, M = [], h.shape[0]
    rope = {hd: tuple(t[p0:] for t in _rope_tab(p0 + M, hd)) for hd in (256, 512)}
    for a, layer in ins:
        h, kc, vc = _layer_exact(h, a, layer, *rope[a["hd"]], p0, e4m3)
        caches += [kc, vc]
    return h, caches


def _panel(t):
    """[N][blocks] in the device order of 64-row panels (padding rows zero)."""
    N, n = t.shape
    p = torch.zeros(-(-N // 64) * 64, n, dtype=t.dtype, device=t.device)
    p[:N] = t
    return p.view(-1, 64, n).transpose(1, 2).reshape(-1)


def exact(case, seed):
    gen, k = _gen(seed), case["kind"]
    if k == "gemv":
        return torch.stack([_mul(x.to(F64), W, case["e4m3"]) for W, x in _gemv_inputs(case, gen)])
    if k == "verify":
        return [_mul(x.to(F64), W, case["e4m3"]) for W, x in _verify_inputs(case, gen)]
    if k == "attn":
        ins, cos, sin = _attn_inputs(case, gen)
        nq, nk, st, pos = case["nH"] * case["hd"], case["nkv"] * case["hd"], case["stride"], case["pos"]
        outs, caches = [], []
        for qkv, knw, qnw, kc, vc in ins:
            x = qkv.to(F64)
            kk = x[None, nq:nq + nk]
            v = x[None, nq + nk:] if case["window"] else kk
            kc, vc = _into_caches(kk, v, knw, cos[None], sin[None], kc, vc, case, st, pos)
            q = _rope(_rms(x[:nq].view(1, case["nH"], case["hd"]), qnw), cos, sin)
            outs.append(_attend(q, kc, vc, case, st, pos)[0])
            caches += [kc.view(-1), vc.view(-1)]
        return [torch.stack(outs), *caches]
    if k == "w4a16":
        W, X = _gemm_inputs(case, gen)
        return _mul(X.to(F64), W)
    if k in ("w8a8", "w4a8"):
        W, X = _gemm_inputs(case, gen)
        q, sc = _codes(W)
        deq = (q * sc[:, :, None]).view(W.shape)
        sw = torch.clamp(_div(deq.abs().amax(1), 127.0), min=1e-12)
        if k == "w8a8":
            B = torch.round(_div(deq, sw[:, None]))
        else:
            B = torch.round(q * _div(sc, sw[:, None]).to(F16).to(F32)[:, :, None]).view(W.shape)
        B = torch.clamp(B, -127, 127)
        sa = torch.clamp(_div(X.to(F32).abs().amax(1), 127.0), min=1e-12)
        A = torch.clamp(torch.round(_div(X.to(F32), sa[:, None])), -127, 127)
        return A.to(F64) @ B.to(F64).T * sa.to(F64)[:, None] * sw.to(F16).to(F64)[None]
    if k == "pre_attn":
        q, qnw, cos, sin, kc, vc = _pre_attn_inputs(case, gen)
        st, hd = case["stride"], case["hd"]
        q = _rope(_rms(q.to(F64).view(case["M"], case["nH"], hd), qnw), cos[:, None], sin[:, None])
        kc, vc = (t.to(F64).view(case["nkv"], st, hd) for t in (kc, vc))
        return _attend(q, kc, vc, case, st, case["p0"])
    if k == "token":
        tid, emb, ins, finw, lm = _token_inputs(case, gen)
        h, caches = _stack_exact(emb[tid:tid + 1].to(F64), ins, case["pos"], case["e4m3"])
        return [_mul(_rms(h, finw), lm, case["e4m3"])[0], *caches]
    if k == "chunk":
        h0, ins = _chunk_inputs(case, gen)
        h, caches = _stack_exact(h0.to(F64), ins, case["p0"], False)
        return [h, *caches]
    W = _prepare_quant(case, gen)["W"]   # codes, e4m3 bytes and int8 weights are whole numbers; the scales are not
    q, sc = _codes(W)
    sc16 = _panel(torch.clamp(W.to(F64).view(W.shape[0], -1, BLK).abs().amax(2) / 7.0, min=1e-8))
    sw = torch.clamp((q.to(F64) * sc.to(F64)[:, :, None]).abs().amax((1, 2)) / 127.0, min=1e-12)
    return [None, sc16, None if case["fp8"] else sc16] + ([None, sw] if case["i8"] else []) \
        + [_lift(sc)[1] if case["fp8"] else 1.0]
