"""The work that programs give this framework, as cases to be timed: a lone quantised mat-vec, the mixture-of-experts half of
a verify window, whole verify windows and decode rounds of a small decoder, the two heads (greedy and sampled), and the
mixture-of-experts layer over prompt chunks. Every case goes through the library's public C ABI.

A case is a dict of plain values; `kind` names the path, the rest its sizes. Weights are synthetic: experts IQ3_S-encoded
from N(0, 0.02), a handful of distinct matrices copied to every expert's own address, dense matrices split Q8_0 of Gaussian
values, caches and activations N(0, 1)."""
import ctypes as C
import importlib
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.getcwd()
PKG_DIR = os.path.join(ROOT, "qwen3.8-flash-next-2x-p100_amd")
DEV = "cuda:0"
HIDDEN, HEAD, NQ, NKV = 2048, 256, 16, 2   # the model shape of the benchmark's decoder
BLOCK = {"iq3_s": (256, 110, 21), "q8_0": (32, 34, 8), "q4_k": (256, 144, 12), "q5_k": (256, 176, 13), "iq4_xs": (256, 136, 23)}   # values, bytes, ggml id


def _package():
    """the package (its directory's name is no identifier) and its loaded library"""
    name = "fnx_mi355x_pkg"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(PKG_DIR, "__init__.py"), submodule_search_locations=[PKG_DIR])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one quantised matrix over one token, the smallest call a program makes: bound by the launches
        {"name": "matvec-1row", "kind": "matvec", "rows": 4096, "cols": 2048, "T": 1},
        # the greedy end of a verify window of sixteen rows: picks, acceptance, prompt lookup over a long context
        {"name": "head-greedy", "kind": "head", "T": 16, "vocab": 151936, "ctx": 38862},
        # the sampled end of a window of one token and four drafts: norm, output head, penalised candidates, acceptance on the host
        {"name": "head-sampled", "kind": "sampled", "T": 5, "vocab": 151936, "pens": 600},
        # a layer's experts in plain decoding with one draft: two rows, each with experts of its own; a bf16 router as files have it
        {"name": "window-2rows", "kind": "window", "T": 2, "ff": 512, "nexp": 512, "topk": 10, "router": "bf16", "type": "iq3_s"},
        # the same under a full speculative window, the benchmark's headline
        {"name": "window-16rows", "kind": "window", "T": 16, "ff": 512, "nexp": 512, "topk": 10, "router": "f32", "type": "iq3_s"},
        # a layer whose experts a file keeps in another type (mixed quantisations are usual), an odd window
        {"name": "window-q4k-7rows", "kind": "window", "T": 7, "ff": 512, "nexp": 512, "topk": 10, "router": "f32", "type": "q4_k"},
        # a whole verify window and the draft layer over it, deep in a long context
        {"name": "verify-16rows-32k", "kind": "verify", "T": 16, "pos": 32752, "layers": 4, "vocab": 151936},
        # a generating session in mid-document: decode rounds that the host only enqueues, a chain of three drafts each
        {"name": "rounds-chain3", "kind": "rounds", "rounds": 8, "pos": 12000, "chain": 3, "layers": 4, "vocab": 151936},
        # a short follow-up prompt: an odd chunk of a few dozen rows
        {"name": "chunk-77", "kind": "chunk", "C": 77, "ff": 512, "nexp": 512, "topk": 10, "popularity": "uniform", "family": "f16"},
        # the ordinary prompt chunk, experts as unequally popular as they are in earnest
        {"name": "chunk-512", "kind": "chunk", "C": 512, "ff": 512, "nexp": 512, "topk": 10, "popularity": "zipf", "family": "f16"},
        # a long prompt in one large chunk: arithmetic rather than weights
        {"name": "chunk-4096", "kind": "chunk", "C": 4096, "ff": 512, "nexp": 512, "topk": 10, "popularity": "zipf", "family": "f16"},
        # the prompt path's other family, activations in q8_1, a ragged chunk
        {"name": "chunk-q8-300", "kind": "chunk", "C": 300, "ff": 512, "nexp": 512, "topk": 10, "popularity": "zipf", "family": "q8_1"},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["matvec", "head", "sampled", "window", "window", "verify", "rounds", "chunk", "chunk", "chunk"])
    if kind == "matvec":
        return {"kind": kind, "rows": 16 * log(32, 1024), "cols": rng.choice([512, 1024, 2048]), "T": rng.randint(1, 16)}
    if kind == "head":
        return {"kind": kind, "T": rng.randint(1, 16), "vocab": log(32000, 262144), "ctx": log(64, 131072)}
    if kind == "sampled":
        return {"kind": kind, "T": rng.randint(1, 16), "vocab": log(32000, 262144), "pens": rng.choice([0, log(1, 2000)])}
    if kind == "window":
        return {"kind": kind, "T": rng.randint(1, 16), "ff": rng.choice([256, 512, 1024]), "nexp": rng.choice([64, 128, 256, 512]),
                "topk": rng.choice([4, 6, 8, 10]), "router": rng.choice(["f32", "bf16"]),
                "type": rng.choice(["iq3_s", "iq3_s", "iq3_s", "iq3_s", "q4_k", "q5_k", "iq4_xs", "q8_0"])}
    if kind == "verify":
        return {"kind": kind, "T": rng.randint(1, 16), "pos": log(64, 32000), "layers": rng.randint(1, 4), "vocab": 16 * log(2000, 9496)}
    if kind == "rounds":
        return {"kind": kind, "rounds": rng.randint(2, 5), "pos": log(64, 12000), "chain": rng.randint(1, 3), "layers": rng.randint(1, 4),
                "vocab": 16 * log(2000, 9496)}
    family = rng.choice(["f16", "f16", "f16", "q8_1"])
    return {"kind": kind, "C": log(17, 4096), "ff": rng.choice([256, 512, 512, 1024] if family == "f16" else [512, 512, 1024]),
            "nexp": rng.choice([128, 256, 512]), "topk": rng.choice([4, 8, 10]), "popularity": rng.choice(["uniform", "zipf"]), "family": family}


# ---------------------------------------------------------------- making the inputs
class _Make:
    """tensors from one seed on the device, and the library's descriptors over them (the tensors stay alive in `keep`)"""

    def __init__(self, seed):
        self.pkg = _package()
        self.lib = self.pkg.lib()
        self.st = self.pkg.stream_ptr()
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)
        self.keep = []
        self.bank = {}

    def ok(self, status):
        self.pkg.check(status)

    def hold(self, t):
        self.keep.append(t)
        return t

    def randn(self, *shape, scale=1.0):
        t = torch.randn(shape, device=DEV, generator=self.g)
        return self.hold(t.mul_(scale) if scale != 1.0 else t)

    def ints(self, lo, hi, *shape):
        return self.hold(torch.randint(lo, hi, shape, dtype=torch.int32, device=DEV, generator=self.g))

    def zeros(self, shape, dtype=torch.float32):
        return self.hold(torch.zeros(shape, dtype=dtype, device=DEV))

    def norm_weights(self, n):
        return self.hold(1.0 + 0.1 * torch.randn(n, device=DEV, generator=self.g))

    def q8s(self, rows, cols, scale):
        """a dense matrix as split Q8_0, re-laid in tiles as at load: Gaussian values, a scale a block of 32"""
        q = torch.zeros((rows, cols), dtype=torch.int8, device=DEV)
        d = self.zeros((rows, cols // 32), torch.float16)
        for r0 in range(0, rows, 16384):
            w = torch.randn((min(16384, rows - r0), cols // 32, 32), device=DEV, generator=self.g) * scale
            dd = (w.abs().amax(dim=2) / 127.0).to(torch.float16)
            d[r0:r0 + w.shape[0]] = dd
            q[r0:r0 + w.shape[0]] = (w / dd.to(torch.float32).unsqueeze(2)).round_().clamp_(-127, 127).to(torch.int8).view(w.shape[0], cols)
        t = self.zeros(self.lib.fnx_q8s_tile_bytes(rows, cols), torch.int8)
        self.ok(self.lib.fnx_q8s_tile(q.data_ptr(), t.data_ptr(), rows, cols, self.st))
        torch.cuda.synchronize()
        return self.pkg.Q8S(t.data_ptr(), d.data_ptr(), rows, cols, 1)

    def experts(self, kind, nmat, rows, cols):
        """nmat matrices of rows x cols as a file holds them: bytes"""
        values, size, _ = BLOCK[kind]
        if kind == "iq3_s":
            if (rows, cols) not in self.bank:
                enc = importlib.import_module(self.pkg.__name__ + ".iq3s_encode")
                w = torch.randn((8, rows * cols), device=DEV, generator=self.g) * 0.02
                self.bank[(rows, cols)] = enc.encode_iq3s(w).view(8, -1)
            pick = torch.randint(0, 8, (nmat,), device=DEV, generator=self.g)
            return self.hold(self.bank[(rows, cols)][pick].reshape(-1))
        b = torch.randint(0, 256, (nmat * rows * cols // values, size), dtype=torch.uint8, device=DEV, generator=self.g)
        d = (torch.rand(b.shape[0], device=DEV, generator=self.g) + 0.5) * {"q8_0": 2.7e-4, "q4_k": 1e-4, "q5_k": 5e-5, "iq4_xs": 2.5e-5}[kind]
        b[:, 0:2] = d.to(torch.float16).view(torch.uint8).view(-1, 2)
        if kind in ("q4_k", "q5_k"):   # the minimum's scale: values around zero
            b[:, 2:4] = (d * (7.5 if kind == "q4_k" else 15.5)).to(torch.float16).view(torch.uint8).view(-1, 2)
        return self.hold(b.reshape(-1))

    def matrix(self, kind, nmat, rows, cols, layout):
        """(descriptor, bytes between matrices); layout: IQ3_S re-laid at load as "unit64" or "tile16" """
        values, size, ggml = BLOCK[kind]
        w = self.experts(kind, nmat, rows, cols)
        row_bytes = cols // values * size
        if kind != "iq3_s":
            return self.pkg.DW(w.data_ptr(), ggml, cols, rows, row_bytes, None), rows * row_bytes
        self.ok(self.lib.fnx_iq3s_repack(w.data_ptr(), w.data_ptr(), nmat * rows * cols, self.st))
        if layout == "unit64":
            return self.pkg.dw(w, cols, rows, packed=True), rows * row_bytes
        t = self.zeros(self.lib.fnx_iq3s_tile16_bytes(rows, cols, nmat), torch.uint8)
        self.ok(self.lib.fnx_iq3s_tile16(w.data_ptr(), t.data_ptr(), rows, cols, nmat, self.st))
        return self.pkg.dw(t, cols, rows, tile16=True), self.lib.fnx_iq3s_tile16_bytes(rows, cols, 1)

    def moe(self, ff, nexp, topk, kind="iq3_s", layout="unit64", down_layout=None, router="f32", popularity="uniform"):
        n, down_layout = HIDDEN, down_layout or layout
        r = torch.randn((nexp + 1, n), device=DEV, generator=self.g) * 0.02
        if popularity == "zipf":   # a constant input feature and a column of the router set how often an expert is picked
            pop = 1.0 / torch.arange(1, nexp + 1, device=DEV, dtype=torch.float64) ** 1.1
            r[:nexp, 0] = torch.log(pop / pop.sum()).to(torch.float32)[torch.randperm(nexp, device=DEV, generator=self.g)]
            r[nexp, 0] = 0.0
        r = self.hold(r.to(torch.bfloat16) if router == "bf16" else r)
        gu, gs = self.matrix(kind, nexp, 2 * ff, n, layout)
        dn, ds = self.matrix(kind, nexp, n, ff, down_layout)
        sg, _ = self.matrix(kind, 1, 2 * ff, n, layout)
        sd, _ = self.matrix(kind, 1, n, ff, down_layout)
        return self.pkg.MoeLayer(n, ff, nexp, topk, r.data_ptr(), int(router == "bf16"), gu, gs, dn, ds, sg, sd)

    def moe_ws(self, T, ff, nexp, topk):
        P = T * topk
        b = dict(xq=self.zeros(T * (HIDDEN // 32) * 36, torch.uint8), logits=self.zeros((T, nexp + 1)), topi=self.zeros((T, topk), torch.int32),
                 topw=self.zeros((T, topk)), jobs_gu=self.zeros((P + 1) * 136, torch.uint8), jobs_dn=self.zeros((P + 1) * 136, torch.uint8),
                 njobs=self.zeros(2, torch.int32), gu=self.zeros((P + T, 2 * ff)), part=self.zeros((P + T, HIDDEN)),
                 sync=self.zeros(self.pkg.MOE_SYNC_WORDS, torch.int32))
        order = ("xq", "logits", "topi", "topw", "jobs_gu", "jobs_dn", "njobs", "gu", "part", "sync")
        return b, self.pkg.MoeWs(*(b[k].data_ptr() for k in order))

    def decoder(self, layers, vocab, max_ctx, filled):
        """a decoder of the benchmark's shape with its draft layer, caches filled up to a position"""
        n, pkg, sw = HIDDEN, self.pkg, 1.0 / math.sqrt(HIDDEN)

        def layer():
            w = [self.norm_weights(n), self.norm_weights(HEAD), self.norm_weights(HEAD), self.norm_weights(n)]
            q = [self.q8s(NQ * 2 * HEAD, n, sw), self.q8s(NKV * HEAD, n, sw), self.q8s(NKV * HEAD, n, sw), self.q8s(n, NQ * HEAD, 1.0 / math.sqrt(NQ * HEAD))]
            moe = self.moe(512, 512, 10)
            kv = []
            for _ in range(2):   # (the V cache keeps eight positions of a dimension together: any order of Gaussian cells is as good)
                c = self.zeros((max_ctx, NKV, HEAD), torch.float16)
                c[:filled].normal_(generator=self.g)
                kv.append(c)
            return pkg.DecLayer(*[t.data_ptr() for t in w], *q, moe, kv[0].data_ptr(), kv[1].data_ptr()), kv

        arr, caches = (pkg.DecLayer * layers)(), []
        for i in range(layers):
            arr[i], kv = layer()
            caches += kv
        emb = self.hold(torch.randn((vocab, n), device=DEV, generator=self.g).to(torch.float16))
        D = pkg.Decoder(n, NQ, NKV, layers, vocab, max_ctx, 1e-6, pkg.Rope(1e7, 0, 0.0, 0.0, 1.0, 1.0), C.cast(arr, C.c_void_p),
                        self.norm_weights(n).data_ptr(), self.q8s(vocab, n, sw), emb.data_ptr())
        ml, kv = layer()
        M = pkg.Mtp(self.norm_weights(n).data_ptr(), self.norm_weights(n).data_ptr(), self.norm_weights(n).data_ptr(), self.q8s(n, n, sw),
                    self.q8s(n, n, sw), self.q8s(vocab, n, sw), ml)
        self.keep.append(arr)
        return D, M, caches + kv

    def dec_ws(self, vocab, max_ctx):
        T, n = 16, HIDDEN
        b = dict(x=self.zeros((T, n)), xn=self.zeros((T, n)), qg=self.zeros((T, NQ * 512)), k=self.zeros((T, NKV * 256)), v=self.zeros((T, NKV * 256)),
                 att=self.zeros((T, NQ * 256)), o=self.zeros((T, n)), attn_scratch=self.zeros(self.lib.fnx_attn_scratch_floats(NQ, T, max_ctx)),
                 xq=self.zeros(T * (max(n, NQ * HEAD) // 32) * 36, torch.uint8), hidden=self.zeros((T, n)), logits=self.zeros((T, vocab)),
                 best_v=self.zeros(T), best_i=self.zeros(T, torch.int32), keys=self.zeros(self.pkg.ARGMAX_WORDS, torch.int64),
                 err=self.zeros(1, torch.int32))
        _, moe = self.moe_ws(T, 512, 512, 10)
        order = ("x", "xn", "qg", "k", "v", "att", "o", "attn_scratch", "xq", "hidden", "logits", "best_v", "best_i", "keys", "err")
        return b, self.pkg.DecWs(*(b[k].data_ptr() for k in order), moe)


# ---------------------------------------------------------------- a lone mat-vec
def _matvec_prepare(c, m):
    T, rows, cols = c["T"], c["rows"], c["cols"]
    job = np.zeros(34, dtype=np.int32)
    job[1] = T
    job[2:2 + T] = job[18:18 + T] = np.arange(T)
    W, _ = m.matrix("iq3_s", 1, rows, cols, "unit64")
    return dict(W=W, x=m.randn(T, cols), xq=m.zeros(T * (cols // 32) * 36, torch.uint8), job=m.hold(torch.from_numpy(job).to(DEV)), out=m.zeros((T, rows)))


def _matvec_run(c, s):
    m, lib = s["m"], s["m"].lib
    m.ok(lib.fnx_quantize_q8_1(s["x"].data_ptr(), s["xq"].data_ptr(), c["cols"], c["T"], m.st))
    m.ok(lib.fnx_mmvq(C.byref(s["W"]), 0, s["job"].data_ptr(), None, 1, s["xq"].data_ptr(), s["out"].data_ptr(), c["rows"], m.st))
    return {"y": s["out"]}


# ---------------------------------------------------------------- the greedy head: argmax, acceptance, prompt lookup
def _head_prepare(c, m):
    T, V, n_ctx = c["T"], c["vocab"], c["ctx"]
    logits = m.randn(T, V)
    ctx = torch.randint(0, V, (n_ctx,), dtype=torch.int32, device=DEV, generator=m.g)
    if n_ctx >= 64:   # text repeats itself: the context ends inside a copy of an earlier span
        src = int(torch.randint(0, n_ctx // 2, (1,), device=DEV, generator=m.g))
        ctx[n_ctx - 12:] = ctx[src:src + 12].clone()
    else:
        src = 0
    m.hold(ctx)
    rows = m.zeros(16, torch.int32)
    rows[0] = ctx[n_ctx - 1]
    rows[1:T] = ctx[src + 12:src + 12 + T - 1]
    keep = torch.rand(T, device=DEV, generator=m.g) < 0.7
    for j in range(T - 1):   # most of the drafts are what the model picks
        if bool(keep[j]):
            logits[j, int(rows[j + 1])] = logits[j].max() + 1.0
    return dict(logits=logits, ctx=ctx, rows=rows, d1=m.hold(rows[1:2].clone() if T > 1 else ctx[src + 12:src + 13].clone()), bv=m.zeros(T), bi=m.zeros(T, torch.int32),
                keys=m.zeros(m.pkg.ARGMAX_WORDS, torch.int64), err=m.zeros(1, torch.int32), acc=m.zeros(1, torch.int32),
                drafts=m.zeros(15, torch.int32), n=m.zeros(1, torch.int32), match=m.zeros(1, torch.int32))


def _head_run(c, s):
    m, lib = s["m"], s["m"].lib
    m.ok(lib.fnx_argmax(s["logits"].data_ptr(), c["vocab"], c["T"], 0, s["bv"].data_ptr(), s["bi"].data_ptr(), s["keys"].data_ptr(), s["err"].data_ptr(), m.st))
    m.ok(lib.fnx_accept_greedy_dev(s["rows"].data_ptr(), s["bi"].data_ptr(), c["T"], s["acc"].data_ptr(), m.st))
    m.ok(lib.fnx_lookup_drafts_dev(s["ctx"].data_ptr(), c["ctx"], 3, 15, s["d1"].data_ptr(), s["drafts"].data_ptr(), s["n"].data_ptr(), s["match"].data_ptr(), m.st))
    return {k: s[k] for k in ("bv", "bi", "acc", "drafts", "n", "match", "err")}


# ---------------------------------------------------------------- the sampled head: norm, projection, candidates, acceptance on the host
def _sampled_prepare(c, m):
    T, V, K = c["T"], c["vocab"], c["pens"]
    s = dict(x=m.randn(T, HIDDEN), w=m.norm_weights(HIDDEN), xq=m.zeros(T * (HIDDEN // 32) * 36, torch.uint8), head=m.q8s(V, HIDDEN, 2.5 / math.sqrt(HIDDEN)),
             logits=m.zeros((T, V)), cv=m.zeros((T, 64)), ci=m.zeros((T, 64), torch.int32), err=m.zeros(1, torch.int32),
             pen_n=m.hold(torch.full((T,), K, dtype=torch.int32, device=DEV)), par=m.hold(torch.tensor([1.1, 0.05, 0.1] * T, device=DEV)),
             pen_tok=m.hold(torch.argsort(torch.rand((T, V), device=DEV, generator=m.g), dim=1)[:, :max(K, 1)].to(torch.int32).contiguous()),
             pen_cnt=m.ints(1, 5, T, max(K, 1)), sampling=m.pkg.Sampling(0.8, 0.95, 0.02, 40),
             hv=torch.zeros((T, 64), pin_memory=True), hi=torch.zeros((T, 64), dtype=torch.int32, pin_memory=True),
             rows=np.zeros(16, dtype=np.int32), tokens=np.zeros(17, dtype=np.int32), u=torch.rand(64, dtype=torch.float64, device=DEV, generator=m.g).cpu().numpy())
    s["m"] = m
    _candidates(c, s)
    torch.cuda.synchronize()
    likely = s["ci"].cpu().numpy()
    for j in range(1, T):   # a draft model mostly proposes what the model itself ranks first
        s["rows"][j] = likely[j - 1, 0 if s["u"][40 + j] < 0.8 else 3]
    return s


def _candidates(c, s):
    m, lib = s["m"], s["m"].lib
    T, V = c["T"], c["vocab"]
    m.ok(lib.fnx_add_norm_q8(s["x"].data_ptr(), None, s["w"].data_ptr(), None, s["xq"].data_ptr(), T, HIDDEN, 1e-6, m.st))
    m.ok(lib.fnx_q8s_gemv(C.byref(s["head"]), s["xq"].data_ptr(), s["logits"].data_ptr(), V, T, m.st))
    m.ok(lib.fnx_top_tokens(s["logits"].data_ptr(), V, T, 0, s["pen_tok"].data_ptr(), s["pen_cnt"].data_ptr(), s["pen_n"].data_ptr(), max(c["pens"], 1),
                            s["par"].data_ptr(), None, None, None, None, s["cv"].data_ptr(), s["ci"].data_ptr(), s["err"].data_ptr(), m.st))


def _sampled_run(c, s):
    m, used = s["m"], C.c_int(0)
    _candidates(c, s)
    s["hv"].copy_(s["cv"], non_blocking=True)
    s["hi"].copy_(s["ci"], non_blocking=True)
    torch.cuda.current_stream().synchronize()   # the acceptance draws on the host
    n = m.lib.fnx_accept_sampled(s["hv"].data_ptr(), s["hi"].data_ptr(), 64, c["T"], s["rows"].ctypes.data, C.byref(s["sampling"]), None, None, None, 0,
                                 s["u"].ctypes.data, 64, s["tokens"].ctypes.data, C.byref(used))
    if n < 0:
        m.ok(1)
    return {"logits": s["logits"], "candidates": s["cv"], "ids": s["ci"], "err": s["err"], "emitted": n, "tokens": s["tokens"]}


# ---------------------------------------------------------------- a verify window's mixture-of-experts half
def _window_prepare(c, m):
    L = m.moe(c["ff"], c["nexp"], c["topk"], kind=c["type"], router=c["router"])
    b, ws = m.moe_ws(c["T"], c["ff"], c["nexp"], c["topk"])
    return dict(L=L, b=b, ws=ws, x=m.randn(c["T"], HIDDEN), out=m.zeros((c["T"], HIDDEN)))


def _window_run(c, s):
    m = s["m"]
    m.ok(m.lib.fnx_moe_verify_layer(C.byref(s["L"]), s["x"].data_ptr(), c["T"], s["out"].data_ptr(), C.byref(s["ws"]), m.st))
    return {"out": s["out"], "logits": s["b"]["logits"], "topi": s["b"]["topi"], "topw": s["b"]["topw"]}


# ---------------------------------------------------------------- a whole verify window, acceptance and the draft layer
def _verify_prepare(c, m):
    max_ctx = (c["pos"] + c["T"] + 1023) // 1024 * 1024
    D, M, caches = m.decoder(c["layers"], c["vocab"], max_ctx, c["pos"])
    b, ws = m.dec_ws(c["vocab"], max_ctx)
    b2, ws2 = m.dec_ws(c["vocab"], max_ctx)   # the draft layer's own, so that the window's logits outlive it
    return dict(D=D, M=M, caches=caches, b=b, ws=ws, b2=b2, ws2=ws2, tokens=m.ints(0, c["vocab"], c["T"]), acc=m.zeros(1, torch.int32),
                pos=m.hold(torch.full((1,), c["pos"], dtype=torch.int32, device=DEV)))


def _verify_run(c, s):
    m, lib, T = s["m"], s["m"].lib, c["T"]
    m.ok(lib.fnx_decoder_verify(C.byref(s["D"]), s["tokens"].data_ptr(), T, s["pos"].data_ptr(), C.byref(s["ws"]), m.st))
    m.ok(lib.fnx_accept_greedy_dev(s["tokens"].data_ptr(), s["b"]["best_i"].data_ptr(), T, s["acc"].data_ptr(), m.st))
    m.ok(lib.fnx_mtp_draft(C.byref(s["D"]), C.byref(s["M"]), s["b"]["hidden"].data_ptr(), s["tokens"].data_ptr(), T, s["pos"].data_ptr(), C.byref(s["ws2"]), m.st))
    out = {k: s["b"][k] for k in ("hidden", "logits", "best_i", "err")}
    out.update({"draft_" + k: s["b2"][k] for k in ("hidden", "logits", "best_i", "err")})
    out.update(accepted=s["acc"], caches=s["caches"])
    return out


# ---------------------------------------------------------------- decode rounds
def _rounds_prepare(c, m):
    pkg, cap = m.pkg, (c["pos"] + 17 * c["rounds"] + 64 + 1023) // 1024 * 1024
    D, M, caches = m.decoder(c["layers"], c["vocab"], cap, c["pos"])
    b, ws = m.dec_ws(c["vocab"], cap)
    ctx = m.ints(0, c["vocab"], cap + 64)
    start = torch.zeros(pkg.RS_WORDS, dtype=torch.int32)
    start[pkg.RS_NCTX], start[pkg.RS_POS], start[pkg.RS_ROWS] = c["pos"] + 1, c["pos"], 1
    first = torch.zeros(16, dtype=torch.int32, device=DEV)
    first[0] = ctx[c["pos"]]
    s = dict(D=D, M=M, caches=caches, b=b, ws=ws, ctx=ctx, prompt=m.hold(ctx.clone()), start=m.hold(start.to(DEV)), first=m.hold(first),
             state=m.zeros(pkg.RS_WORDS, torch.int32), rows=m.zeros(16, torch.int32), log=m.zeros((c["rounds"], 2), torch.int32),
             scratch=m.zeros(16, torch.int32), src=m.zeros(HIDDEN))
    s["R"] = pkg.Round(s["state"].data_ptr(), s["rows"].data_ptr(), ctx.data_ptr(), cap + 64, s["log"].data_ptr(), c["rounds"], 1, 3, 15, s["scratch"].data_ptr(),
                       c["chain"], s["src"].data_ptr())
    return s


def _rounds_run(c, s):
    m = s["m"]
    s["state"].copy_(s["start"])   # the session begins at the end of its prompt
    s["rows"].copy_(s["first"])
    s["ctx"].copy_(s["prompt"])
    for _ in range(c["rounds"]):
        m.ok(m.lib.fnx_decode_round(C.byref(s["D"]), C.byref(s["M"]), C.byref(s["R"]), C.byref(s["ws"]), m.st))
    return {"state": s["state"], "rows": s["rows"], "ctx": s["ctx"], "log": s["log"], "caches": s["caches"], "err": s["b"]["err"]}


# ---------------------------------------------------------------- the mixture-of-experts layer over a prompt chunk
def _chunk_prepare(c, m):
    n, rows, ff, nexp, topk = HIDDEN, c["C"], c["ff"], c["nexp"], c["topk"]
    # the prompt path's own layout, except where its f16 family takes the down matrices in the decode path's
    L = m.moe(ff, nexp, topk, layout="tile16", down_layout="tile16" if c["family"] == "q8_1" or ff == 512 else "unit64", popularity=c["popularity"])
    x = m.randn(rows, n)
    x[:, 0] = 1.0   # the constant feature behind the experts' popularity
    P, S = rows * topk, (rows + 63) // 64
    J = P // 64 + nexp
    b = dict(logits=m.zeros((rows, nexp + 1)), topi=m.zeros((rows, topk), torch.int32), topw=m.zeros((rows, topk)), cnt=m.zeros(nexp, torch.int32),
             jbase=m.zeros(nexp, torch.int32), jobs_gu=m.zeros((J + S, 130), torch.int32), jobs_dn=m.zeros((J + S, 130), torch.int32),
             njobs=m.zeros(2, torch.int32), xh=m.zeros((rows, n), torch.float16), gu=m.zeros((P + rows, 2 * ff)), h16=m.zeros((P + rows, ff), torch.float16),
             part=m.zeros((P + rows, n)))
    order = ("logits", "topi", "topw", "cnt", "jbase", "jobs_gu", "jobs_dn", "njobs", "xh", "gu", "h16", "part")
    s = dict(L=L, x=x, b=b, J=J, S=S, P=P, ws=m.pkg.PfWs(*(b[k].data_ptr() for k in order)), out=m.zeros((rows, n)))
    if c["family"] == "q8_1":   # the shared expert's jobs are the same for every chunk of this many rows: made once
        s["xq"] = m.zeros(rows * (n // 32) * 36, torch.uint8)
        gu, dn = np.zeros((S, 130), dtype=np.int32), np.zeros((S, 130), dtype=np.int32)
        for j in range(S):
            t = np.arange(64 * j, min(64 * j + 64, rows))
            gu[j, 1] = dn[j, 1] = len(t)
            gu[j, 2:2 + len(t)] = t
            gu[j, 66:66 + len(t)] = dn[j, 2:2 + len(t)] = dn[j, 66:66 + len(t)] = P + t
        s["sh_gu"], s["sh_dn"] = m.hold(torch.from_numpy(gu).to(DEV)), m.hold(torch.from_numpy(dn).to(DEV))
        s["nsh"] = m.hold(torch.full((1,), S, dtype=torch.int32, device=DEV))
    return s


def _chunk_run(c, s):
    m, lib, L, b = s["m"], s["m"].lib, s["L"], s["b"]
    if c["family"] == "f16":
        m.ok(lib.fnx_moe_prefill_layer(C.byref(L), s["x"].data_ptr(), c["C"], s["out"].data_ptr(), C.byref(s["ws"]), m.st))
    else:
        p = {k: t.data_ptr() for k, t in b.items()}
        n, rows, nexp, topk, J, P, x = HIDDEN, c["C"], c["nexp"], c["topk"], s["J"], s["P"], s["x"].data_ptr()
        xq = s["xq"].data_ptr()
        m.ok(lib.fnx_gemv_f32(L.router, x, p["logits"], nexp + 1, n, rows, m.st))
        m.ok(lib.fnx_pf_route(p["logits"], nexp + 1, rows, nexp, topk, p["topi"], p["topw"], p["cnt"], p["jbase"], p["jobs_gu"], p["jobs_dn"], J, p["njobs"], m.st))
        m.ok(lib.fnx_quantize_q8_1(x, xq, n, rows, m.st))
        m.ok(lib.fnx_moe_gate_up_big(C.byref(L.gu), L.gu_stride, p["jobs_gu"], p["njobs"], J, xq, p["gu"], m.st))
        m.ok(lib.fnx_moe_gate_up_big(C.byref(L.sh_gu), 0, s["sh_gu"].data_ptr(), s["nsh"].data_ptr(), s["S"], xq, p["gu"], m.st))
        m.ok(lib.fnx_moe_down_big(C.byref(L.down), L.down_stride, p["jobs_dn"], p["njobs"], J, p["gu"], p["part"], m.st))
        m.ok(lib.fnx_moe_down_big(C.byref(L.sh_down), 0, s["sh_dn"].data_ptr(), s["nsh"].data_ptr(), s["S"], p["gu"], p["part"], m.st))
        m.ok(lib.fnx_moe_combine(p["part"], p["topw"], p["part"] + P * n * 4, p["logits"] + nexp * 4, nexp + 1, s["out"].data_ptr(), rows, n, topk, m.st))
    return {"out": s["out"], "logits": b["logits"], "topi": b["topi"], "topw": b["topw"]}


_PREPARE = {"matvec": _matvec_prepare, "head": _head_prepare, "sampled": _sampled_prepare, "window": _window_prepare, "verify": _verify_prepare,
            "rounds": _rounds_prepare, "chunk": _chunk_prepare}
_RUN = {"matvec": _matvec_run, "head": _head_run, "sampled": _sampled_run, "window": _window_run, "verify": _verify_run, "rounds": _rounds_run,
        "chunk": _chunk_run}


def prepare(case, seed):
    m = _Make(seed)
    s = _PREPARE[case["kind"]](case, m)
    m.bank.clear()
    s.update(m=m, case=dict(case))
    torch.cuda.synchronize()
    return s


def run(state):
    c = state["case"]
    return _RUN[c["kind"]](c, state)


# ---------------------------------------------------------------- what a pass cannot do without
def _expert_bytes(kind, ff):
    values, size, _ = BLOCK[kind]
    return 3 * ff * HIDDEN // values * size


def _distinct(nexp, topk, rows, popularity):
    """experts that at least one of `rows` rows picks, on average: an expert's logit is its bias plus Gaussian noise, a row
    picks the topk greatest, so an expert is picked where its logit lies above the level that topk of them exceed"""
    if popularity == "uniform":
        p = np.full(nexp, topk / nexp)
    else:
        w = 1.0 / np.arange(1, nexp + 1) ** 1.1
        bias, sigma = np.log(w / w.sum()), 0.02 * math.sqrt(HIDDEN)
        above = lambda level: np.array([0.5 * math.erfc((level - v) / (sigma * math.sqrt(2.0))) for v in bias])
        lo, hi = -40.0, 40.0
        for _ in range(60):
            mid = 0.5 * (lo + hi)
            lo, hi = (mid, hi) if above(mid).sum() > topk else (lo, mid)
        p = above(lo)
    return float((1.0 - (1.0 - p) ** rows).sum())


def _moe_work(rows, ff, nexp, topk, kind="iq3_s", router=4, popularity="uniform"):
    u = _distinct(nexp, topk, rows, popularity) + 1
    return (u * _expert_bytes(kind, ff) + (nexp + 1) * HIDDEN * router + 2 * rows * HIDDEN * 4,
            2.0 * rows * (topk + 1) * 3 * ff * HIDDEN + 2.0 * rows * (nexp + 1) * HIDDEN)


def _decoder_work(rows, ctx, layers, vocab):
    """(bytes, flops) of a window through `layers` layers (experts included) and one output head"""
    dense = NQ * 2 * HEAD * HIDDEN + 2 * NKV * HEAD * HIDDEN + HIDDEN * NQ * HEAD
    mb, mf = _moe_work(rows, 512, 512, 10)
    return (layers * (dense * 34 / 32 + mb + 2 * ctx * NKV * HEAD * 2) + vocab * HIDDEN * 34 / 32 + rows * vocab * 4,
            layers * (2.0 * rows * dense + mf + 4.0 * rows * NQ * HEAD * ctx) + 2.0 * rows * vocab * HIDDEN)


def work(case):
    c, kind = case, case["kind"]
    if kind == "matvec":
        b, f = c["rows"] * c["cols"] * 110 / 256 + c["T"] * (c["cols"] + c["rows"]) * 4, 2.0 * c["T"] * c["rows"] * c["cols"]
    elif kind == "head":
        b, f = c["T"] * c["vocab"] * 4 + c["ctx"] * 4, c["T"] * c["vocab"]
    elif kind == "sampled":
        b, f = c["vocab"] * HIDDEN * 34 / 32 + c["T"] * (c["vocab"] + HIDDEN + 2 * c["pens"] + 128) * 4, 2.0 * c["T"] * c["vocab"] * HIDDEN
    elif kind == "window":
        b, f = _moe_work(c["T"], c["ff"], c["nexp"], c["topk"], c["type"], 2 if c["router"] == "bf16" else 4)
    elif kind == "verify":   # the model's layers and its head, the draft layer and its head, the draft layer's two input projections
        b, f = _decoder_work(c["T"], c["pos"] + c["T"], c["layers"], c["vocab"])
        b1, f1 = _decoder_work(c["T"], c["pos"] + c["T"], 1, c["vocab"])
        b, f = b + b1 + 2 * HIDDEN * HIDDEN * 34 / 32, f + f1 + 4.0 * c["T"] * HIDDEN * HIDDEN
    elif kind == "rounds":   # nothing here predicts the next token: a window is the last token and the chain's drafts, one is kept
        rows = 1 + c["chain"]
        b, f = _decoder_work(rows, c["pos"] + rows, c["layers"], c["vocab"])
        b1, f1 = _decoder_work(1, c["pos"] + rows, 1, c["vocab"])
        extra = 2 * HIDDEN * HIDDEN
        b, f = c["rounds"] * (b + c["chain"] * (b1 + extra * 34 / 32)), c["rounds"] * (f + c["chain"] * (f1 + 2.0 * extra))
    else:
        b, f = _moe_work(c["C"], c["ff"], c["nexp"], c["topk"], popularity=c["popularity"])
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    return {
        # 32-bit sums of the same terms in another order (measured between two layouts' kernels: 1.2e-7, 5.9e-7)
        "matvec": {"rel": 5e-7, "max": 3e-6},
        # comparisons and whole numbers
        "head": "exact",
        # the norm's sum in another order moves a q8_1 code of the head's input (1/127 of its block's range) now and then
        "sampled": {"rel": 1e-3, "max": 0.02, "differ": 0.01},
        # a last-bit difference in h moves one of its q8_1 codes by a step now and then: 1e-4 of a single row's output
        "window": {"rel": 5e-4, "max": 0.02, "differ": 0.001},
        # the same through every layer, whose steps add up (measured against the sums in another order: 2.5e-3 of the rows, 5.5e-3 of the logits)
        "verify": {"rel": 2e-2, "max": 0.8, "differ": 0.01},
        "rounds": {"rel": 2e-2, "max": 0.8, "differ": 0.01},
        # f16 operands, 32-bit sums in another order: h rounds to the neighbouring half now and then (measured between two layouts'
        # kernels: 1.8e-5, 6e-4); q8_1 activations: 4e-6, 5e-5 and a code's step now and then
        "chunk": {"rel": 1e-4, "max": 3e-3, "differ": 0.001} if case.get("family") == "f16" else {"rel": 1e-4, "max": 5e-3, "differ": 0.001},
    }[case["kind"]]
