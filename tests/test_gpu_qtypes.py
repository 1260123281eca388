"""The other expert types the operators take (kernels.cu:2454-2471: Q4_0, Q8_0, IQ4_NL, Q4_K, Q5_K here) through
fnx_mmvq / fnx_moe_gate_up / fnx_moe_down against the CPU oracle. Bar: relative L2 <= 1e-6 (the same per-sub-block terms,
the same order of sums; what is left is the compiler's choice among equal-valued float forms)."""
import ctypes as C

import numpy as np
import pytest

import fnx_gpu
import oracle_lib as ol
import qtype_blocks as qb
from fnx_gpu import JOB_DTYPE

pytestmark = pytest.mark.gpu
TYPES = [qb.Q4_0, qb.Q5_1, qb.Q8_0, qb.IQ4_NL, qb.IQ4_XS, qb.Q4_K, qb.Q5_K]


def rel_l2(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b.astype(np.float64)) / max(np.linalg.norm(b.astype(np.float64)), 1e-30))


@pytest.fixture(scope="module")
def dev():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU"
    return fnx_gpu.Dev()


def make_jobs(rng, nexp, njobs, nrows_y):
    jobs = np.zeros(njobs, dtype=JOB_DTYPE)
    out_row = 0
    for j in range(njobs):
        n = int(rng.integers(1, 17)) if j else 16
        jobs["w"][j] = int(rng.integers(0, nexp))
        jobs["n"][j] = n
        jobs["y"][j, :n] = rng.integers(0, nrows_y, n)
        jobs["out"][j, :n] = np.arange(out_row, out_row + n)
        out_row += n
    return jobs, out_row


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("nrows,ncols", [(64, 512), (30, 2048), (8, 4096)])
def test_mmvq_other_types(dev, oracle, qtype, nrows, ncols):
    print(f"case mmvq type={qtype} {nrows} x {ncols}", flush=True)
    rng = np.random.default_rng(1000 * qtype + nrows)
    values, nbytes = qb.SHAPE[qtype]
    nexp, row_bytes = 3, ncols // values * nbytes
    w = qb.random_blocks(rng, qtype, nexp * nrows * ncols // values)
    x = rng.standard_normal((20, ncols)).astype(np.float32)
    yq = oracle.quantize_q8_1(x)
    jobs, out_rows = make_jobs(rng, nexp, 5, 20)
    want = np.zeros((out_rows, nrows), np.float32)
    oracle.lib.fnx_o_mmvq_type(qtype, ol.ptr(w), nrows * row_bytes, nrows, ncols, ol.ptr(np.ascontiguousarray(jobs)), len(jobs), ol.ptr(yq), ol.ptr(want),
                               nrows, 8)
    t = dev.torch
    dw_, dj, dy = dev.up(w), dev.up(jobs.view(np.uint8).reshape(-1)), dev.up(yq)
    out = dev.zeros((out_rows, nrows), t.float32)
    W = dev.pkg.DW(dw_.data_ptr(), qtype, ncols, nrows, row_bytes, None)
    nj = dev.up(np.array([len(jobs)], dtype=np.int32))
    dev.ok(dev.lib.fnx_mmvq(C.byref(W), nrows * row_bytes, dj.data_ptr(), nj.data_ptr(), len(jobs), dy.data_ptr(), out.data_ptr(), nrows, dev.st()))
    dev.sync()
    err = rel_l2(out.cpu().numpy(), want)
    assert err <= 1e-6, err
    # against the decoded weights and the real activations: the q8_1 path's own error band (dense.cuh:258-259: ~6e-3)
    wd = qb.np_dequant(qtype, w).reshape(nexp, nrows, ncols).astype(np.float64)
    exact = np.concatenate([x[jobs["y"][j, :jobs["n"][j]]].astype(np.float64) @ wd[jobs["w"][j]].T for j in range(len(jobs))])
    assert rel_l2(out.cpu().numpy(), exact) <= 3e-2


def test_gate_up_and_down_with_q4_k_experts(dev, oracle):
    # the operators of a window's MoE half, one by one, on Q4_K experts: gate|up, SwiGLU -> q8_1 in the library's buffer, down
    rng = np.random.default_rng(4242)
    qtype, n, ff, nexp, T, topk = qb.Q4_K, 512, 256, 4, 3, 2
    values, nbytes = qb.SHAPE[qtype]
    gu_w = qb.random_blocks(rng, qtype, nexp * 2 * ff * n // values)
    dn_w = qb.random_blocks(rng, qtype, nexp * n * ff // values)
    x = rng.standard_normal((T, n)).astype(np.float32)
    xq = oracle.quantize_q8_1(x)
    topi = np.array([[0, 2], [2, 1], [3, 0]], np.int32)
    gu_jobs, dn_jobs = oracle.jobs(topi)
    P = T * topk
    print("case gate|up, down on Q4_K experts", flush=True)
    gu_rb, dn_rb = n // values * nbytes, ff // values * nbytes
    want_gu = np.zeros((P, 2 * ff), np.float32)
    oracle.lib.fnx_o_mmvq_type(qtype, ol.ptr(gu_w), 2 * ff * gu_rb, 2 * ff, n, ol.ptr(np.ascontiguousarray(gu_jobs)), len(gu_jobs), ol.ptr(xq), ol.ptr(want_gu),
                               2 * ff, 8)
    hq = oracle.swiglu_stacked_q8_1(want_gu, ff)
    want_part = np.zeros((P, n), np.float32)
    oracle.lib.fnx_o_mmvq_type(qtype, ol.ptr(dn_w), n * dn_rb, n, ff, ol.ptr(np.ascontiguousarray(dn_jobs)), len(dn_jobs), ol.ptr(hq), ol.ptr(want_part), n, 8)
    t = dev.torch
    dgu, ddn, dxq = dev.up(gu_w), dev.up(dn_w), dev.up(xq)
    jg, jd = dev.up(gu_jobs.view(np.uint8).reshape(-1)), dev.up(dn_jobs.view(np.uint8).reshape(-1))
    nj = dev.up(np.array([len(gu_jobs)], dtype=np.int32))
    gu, part = dev.zeros((P, 2 * ff), t.float32), dev.zeros((P, n), t.float32)
    A = dev.pkg.DW(dgu.data_ptr(), qtype, n, 2 * ff, gu_rb, None)
    B = dev.pkg.DW(ddn.data_ptr(), qtype, ff, n, dn_rb, None)
    dev.ok(dev.lib.fnx_moe_gate_up(C.byref(A), 2 * ff * gu_rb, jg.data_ptr(), nj.data_ptr(), P, dxq.data_ptr(), gu.data_ptr(), topk, dev.st()))
    dev.ok(dev.lib.fnx_moe_down(C.byref(B), n * dn_rb, jd.data_ptr(), nj.data_ptr(), P, gu.data_ptr(), part.data_ptr(), dev.st()))
    dev.sync()
    assert rel_l2(gu.cpu().numpy(), want_gu) <= 1e-6
    assert rel_l2(part.cpu().numpy(), want_part) <= 1e-3   # SwiGLU's expf moves an int8 code by one step now and then


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("ff,T,nexp,topk", [(256, 1, 5, 2), (512, 16, 6, 3), (1024, 16, 3, 2), (1024, 2, 3, 1)])
def test_window_over_other_types(dev, oracle, qtype, ff, T, nexp, topk):
    """fnx_moe_verify_layer with all four matrices of one type (one launch, hidden 2048) against the oracle's operators in the
    reference's order (engine.cu:1569-1757): the smallest and the largest window, every expert width (two wave passes a
    trip at 1024), a window of few rows whose trips are dealt over a block's waves. The operators' bar: the same terms in
    the same order of sums, so 1e-6."""
    print(f"case window type={qtype} ff={ff} T={T} nexp={nexp} topk={topk}", flush=True)
    rng = np.random.default_rng(100 * qtype + ff + T)
    n, P, t, pkg = 2048, T * topk, dev.torch, dev.pkg
    values, nbytes = qb.SHAPE[qtype]
    rb = lambda cols: cols // values * nbytes
    gu_w, dn_w, sgu, sdn = (qb.random_blocks(rng, qtype, m * r * c // values) for m, r, c in ((nexp, 2 * ff, n), (nexp, n, ff), (1, 2 * ff, n), (1, n, ff)))
    W = (rng.standard_normal((nexp + 1, n)) * 0.02).astype(np.float32)
    bf16 = T == 2   # a window's router may be bf16 bits: the same values, kept in the upper halves
    if bf16:
        W = (W.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    x = rng.standard_normal((T, n)).astype(np.float32)
    up = dev.up
    d = [up(a) for a in (gu_w, dn_w, sgu, sdn)]
    dW = up((W.view(np.uint32) >> 16).astype(np.uint16)) if bf16 else up(W)
    mat = lambda i, cols, rows: pkg.DW(d[i].data_ptr(), qtype, cols, rows, rb(cols), None)
    L = pkg.MoeLayer(n, ff, nexp, topk, dW.data_ptr(), int(bf16), mat(0, n, 2 * ff), 2 * ff * rb(n), mat(1, ff, n), n * rb(ff), mat(2, n, 2 * ff), mat(3, ff, n))
    w = dict(xq=dev.zeros(T * (n // 32) * 36, t.uint8), logits=dev.zeros((T, nexp + 1), t.float32), topi=dev.zeros((T, topk), t.int32),
             topw=dev.zeros((T, topk), t.float32), jobs_gu=dev.zeros((P + 1) * 136, t.uint8), jobs_dn=dev.zeros((P + 1) * 136, t.uint8),
             njobs=dev.zeros(2, t.int32), gu=dev.zeros((P + T, 2 * ff), t.float32), part=dev.zeros((P + T, n), t.float32),
             sync=dev.zeros(pkg.MOE_SYNC_WORDS, t.int32))
    ws = pkg.MoeWs(*(w[k].data_ptr() for k in ("xq", "logits", "topi", "topw", "jobs_gu", "jobs_dn", "njobs", "gu", "part", "sync")))
    dx, out = up(x), dev.zeros((T, n), t.float32)
    dev.ok(dev.lib.fnx_moe_verify_layer(C.byref(L), dx.data_ptr(), T, out.data_ptr(), C.byref(ws), dev.st()))
    dev.sync()
    assert not w["sync"].cpu().numpy().any(), "every wait ended and the counters are back at zero"
    logits = oracle.gemv_f32(W, x)
    topi, topw = oracle.topk_logits(logits, nexp, topk)
    jg, jd = (np.ascontiguousarray(j) for j in oracle.jobs(topi))
    xq, mm, ptr = oracle.quantize_q8_1(x), oracle.lib.fnx_o_mmvq_type, ol.ptr
    gu, part = np.zeros((P + T, 2 * ff), np.float32), np.zeros((P + T, n), np.float32)
    sh = np.zeros(1, dtype=JOB_DTYPE)
    sh["n"][0] = T
    sh["y"][0, :T], sh["out"][0, :T] = np.arange(T), P + np.arange(T)
    mm(qtype, ptr(gu_w), 2 * ff * rb(n), 2 * ff, n, ptr(jg), len(jg), ptr(xq), ptr(gu), 2 * ff, 8)
    mm(qtype, ptr(sgu), 0, 2 * ff, n, ptr(sh), 1, ptr(xq), ptr(gu), 2 * ff, 8)
    hq = oracle.swiglu_stacked_q8_1(gu, ff)
    sh["y"][0, :T] = P + np.arange(T)
    mm(qtype, ptr(dn_w), n * rb(ff), n, ff, ptr(jd), len(jd), ptr(hq), ptr(part), n, 8)
    mm(qtype, ptr(sdn), 0, n, ff, ptr(sh), 1, ptr(hq), ptr(part), n, 8)
    want = oracle.moe_combine(part[:P], topw, part[P:], logits[:, nexp])
    assert np.array_equal(w["logits"].cpu().numpy().view(np.uint32), logits.view(np.uint32)) and np.array_equal(w["topi"].cpu().numpy(), topi)
    assert int(w["njobs"][0].item()) == len(jg)
    assert rel_l2(out.cpu().numpy(), want) <= 1e-6


def typed_layer(dev, oracle, qtype, ff, T, nexp, topk, seed, shared_q8=False, tables=False):
    """a layer of one type's experts (hidden 2048) on the device with a workspace of its own, the rows of x, and what the oracle's
    operators make of them. shared_q8: the shared expert as split Q8_0; tables: the experts through pointer tables, in a
    shuffled memory order, the bases null"""
    rng = np.random.default_rng(seed)
    n, P, t, pkg = 2048, T * topk, dev.torch, dev.pkg
    values, nbytes = qb.SHAPE[qtype]
    rb = lambda cols: cols // values * nbytes
    gu_w, dn_w, sgu, sdn = (qb.random_blocks(rng, qtype, m * r * c // values) for m, r, c in ((nexp, 2 * ff, n), (nexp, n, ff), (1, 2 * ff, n), (1, n, ff)))
    W = (rng.standard_normal((nexp + 1, n)) * 0.02).astype(np.float32)
    x = rng.standard_normal((T, n)).astype(np.float32)
    keep, up, size = [], dev.up, {0: 2 * ff * rb(n), 1: n * rb(ff)}

    def hold(a):
        keep.append(a)
        return a.data_ptr()

    def experts(i, w, cols, rows):
        if not tables:
            return pkg.DW(hold(up(w)), qtype, cols, rows, rb(cols), None)
        perm = rng.permutation(nexp)   # expert e's matrix lies at place perm[e]
        at = np.empty((nexp, size[i]), np.uint8)
        at[perm] = np.ascontiguousarray(w).view(np.uint8).reshape(nexp, size[i])
        base = hold(up(at))
        return pkg.DW(None, qtype, cols, rows, rb(cols), hold(up((base + perm.astype(np.int64) * size[i]).astype(np.int64))))

    one = lambda w, cols, rows: pkg.DW(hold(up(w)), qtype, cols, rows, rb(cols), None)
    L = pkg.MoeLayer(n, ff, nexp, topk, hold(up(W)), 0, experts(0, gu_w, n, 2 * ff), 0 if tables else size[0], experts(1, dn_w, ff, n),
                     0 if tables else size[1], one(sgu, n, 2 * ff), one(sdn, ff, n))
    q8 = []
    if shared_q8:
        for rows, cols in ((2 * ff, n), (n, ff)):
            w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
            q, d = np.zeros((rows, cols), dtype=np.int8), np.zeros((rows, cols // 32), dtype=np.uint16)
            oracle.lib.fnx_o_quantize_q8_0_split(ol.ptr(w), rows, cols, ol.ptr(q), ol.ptr(d))
            q8.append((q, d, rows, cols))
        L.sh_gu_q8, L.sh_down_q8 = (pkg.Q8S(hold(up(q)), hold(up(d)), rows, cols) for q, d, rows, cols in q8)
        L.sh_gu.p = L.sh_down.p = None   # not to be read
    w = dict(xq=dev.zeros(T * (n // 32) * 36, t.uint8), logits=dev.zeros((T, nexp + 1), t.float32), topi=dev.zeros((T, topk), t.int32),
             topw=dev.zeros((T, topk), t.float32), jobs_gu=dev.zeros((P + 1) * 136, t.uint8), jobs_dn=dev.zeros((P + 1) * 136, t.uint8),
             njobs=dev.zeros(2, t.int32), gu=dev.zeros((P + T, 2 * ff), t.float32), part=dev.zeros((P + T, n), t.float32),
             sync=dev.zeros(pkg.MOE_SYNC_WORDS, t.int32))
    ws = pkg.MoeWs(*(w[k].data_ptr() for k in ("xq", "logits", "topi", "topw", "jobs_gu", "jobs_dn", "njobs", "gu", "part", "sync")))
    # the oracle's operators in the reference's order (engine.cu:1569-1757)
    logits = oracle.gemv_f32(W, x)
    topi, topw = oracle.topk_logits(logits, nexp, topk)
    jg, jd = (np.ascontiguousarray(j) for j in oracle.jobs(topi))
    xq, mm, ptr = oracle.quantize_q8_1(x), oracle.lib.fnx_o_mmvq_type, ol.ptr
    gu, part = np.zeros((P + T, 2 * ff), np.float32), np.zeros((P + T, n), np.float32)
    sh = np.zeros(1, dtype=JOB_DTYPE)
    sh["n"][0] = T
    sh["y"][0, :T], sh["out"][0, :T] = np.arange(T), P + np.arange(T)
    mm(qtype, ptr(gu_w), size[0], 2 * ff, n, ptr(jg), len(jg), ptr(xq), ptr(gu), 2 * ff, 8)
    if shared_q8:
        oracle.lib.fnx_o_q8s_gemv(ptr(q8[0][0]), ptr(q8[0][1]), 2 * ff, n, ptr(xq), ptr(gu[P:]), 2 * ff, T)
    else:
        mm(qtype, ptr(sgu), 0, 2 * ff, n, ptr(sh), 1, ptr(xq), ptr(gu), 2 * ff, 8)
    hq = oracle.swiglu_stacked_q8_1(gu, ff)
    mm(qtype, ptr(dn_w), size[1], n, ff, ptr(jd), len(jd), ptr(hq), ptr(part), n, 8)
    if shared_q8:
        hs = np.ascontiguousarray(np.ascontiguousarray(hq).reshape(P + T, -1)[P:])
        oracle.lib.fnx_o_q8s_gemv(ptr(q8[1][0]), ptr(q8[1][1]), n, ff, ptr(hs), ptr(part[P:]), n, T)
    else:
        sh["y"][0, :T] = P + np.arange(T)
        mm(qtype, ptr(sdn), 0, n, ff, ptr(sh), 1, ptr(hq), ptr(part), n, 8)
    want = dict(out=oracle.moe_combine(part[:P], topw, part[P:], logits[:, nexp]), logits=logits, topi=topi, njobs=len(jg))
    return L, ws, w, x, keep, want


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("ff,T,nexp,topk,tables,shared_q8", [(1024, 16, 5, 3, True, False), (1024, 16, 4, 1, False, True), (512, 2, 8, 4, True, True),
                                                            (256, 1, 5, 2, False, True)])
def test_window_over_other_types_in_other_forms(dev, oracle, qtype, ff, T, nexp, topk, tables, shared_q8):
    """experts from pointer tables and a split-Q8_0 shared expert (the trips then start at the picks): at width 1024 with
    sixteen rows, where a wave makes its units two at a time, and in windows of few rows, whose trips are dealt over the waves"""
    print(f"case window forms type={qtype} ff={ff} T={T} topk={topk} tables={tables} q8={shared_q8}", flush=True)
    L, ws, w, x, keep, want = typed_layer(dev, oracle, qtype, ff, T, nexp, topk, 70 * qtype + ff + T, shared_q8=shared_q8, tables=tables)
    dx, out = dev.up(x), dev.zeros((T, 2048), dev.torch.float32)
    dev.ok(dev.lib.fnx_moe_verify_layer(C.byref(L), dx.data_ptr(), T, out.data_ptr(), C.byref(ws), dev.st()))
    dev.sync()
    assert not w["sync"].cpu().numpy().any(), "every wait ended and the counters are back at zero"
    assert np.array_equal(w["logits"].cpu().numpy().view(np.uint32), want["logits"].view(np.uint32)) and np.array_equal(w["topi"].cpu().numpy(), want["topi"])
    assert int(w["njobs"][0].item()) == want["njobs"]
    assert rel_l2(out.cpu().numpy(), want["out"]) <= 1e-6


# rows whose blocks are no power of two (on 256 CUs 28, 20, 80, 24, 36 and 40 a row): units of the down matrices that do not divide among them, at
# width 1024 four units a wave in two passes, a unit that two waves make, items of the shared expert dealt apart from the picks'
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("ff,T,nexp,topk,tables,shared_q8", [(512, 9, 12, 10, False, False), (1024, 11, 8, 4, True, False), (1024, 3, 12, 9, False, True),
                                                            (256, 10, 14, 8, True, True), (512, 7, 12, 9, False, False), (1024, 6, 9, 6, False, False)])
def test_window_over_other_types_over_all_blocks(dev, oracle, qtype, ff, T, nexp, topk, tables, shared_q8):
    print(f"case window over all blocks type={qtype} ff={ff} T={T} topk={topk} tables={tables} q8={shared_q8}", flush=True)
    L, ws, w, x, keep, want = typed_layer(dev, oracle, qtype, ff, T, nexp, topk, 75 * qtype + ff + T, shared_q8=shared_q8, tables=tables)
    dx, out = dev.up(x), dev.zeros((T, 2048), dev.torch.float32)
    for _ in range(2):   # the second over the workspace as the first left it
        out.fill_(7.5)
        dev.ok(dev.lib.fnx_moe_verify_layer(C.byref(L), dx.data_ptr(), T, out.data_ptr(), C.byref(ws), dev.st()))
        dev.sync()
        assert not w["sync"].cpu().numpy().any(), "every wait ended and the counters are back at zero"
        assert np.array_equal(w["logits"].cpu().numpy().view(np.uint32), want["logits"].view(np.uint32)) and np.array_equal(w["topi"].cpu().numpy(), want["topi"])
        assert int(w["njobs"][0].item()) == want["njobs"]
        assert rel_l2(out.cpu().numpy(), want["out"]) <= 1e-6
