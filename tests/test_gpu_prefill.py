"""Parity of the prompt path (prefill routing, matrix-core expert products, the chunk layer) with the CPU oracle,
through the C ABI.

Bar: bit-exact for picks, counts, job bases and job lists (integers), and for f32 -> f16 conversion; relative L2 <= 1e-3
for the matrix-core products (f16 operands identical to the oracle's, only the fp32 summation order differs: ~1e-6
measured); SwiGLU f16 codes within one step in a small share of places (device expf).
"""
import ctypes as C

import numpy as np
import pytest

import fnx_gpu
from fnx_gpu import random_iq3s

pytestmark = pytest.mark.gpu

REL_L2 = 1e-3
PF = 64


def rel_l2(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b.astype(np.float64)) / max(np.linalg.norm(b.astype(np.float64)), 1e-30))


@pytest.fixture(scope="module")
def dev():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU"
    return fnx_gpu.Dev()


def zipf_logits(rng, Cn, nexp, s=1.1, scale=3.0):
    """router logits whose picks follow a Zipf popularity over a random permutation of the experts"""
    pop = 1.0 / np.arange(1, nexp + 1) ** s
    bias = np.log(pop / pop.sum())[rng.permutation(nexp)]
    lg = rng.standard_normal((Cn, nexp + 1)).astype(np.float32) * scale
    lg[:, :nexp] += bias.astype(np.float32) * 2
    return lg


@pytest.mark.parametrize("Cn,nexp,topk,zipf", [(512, 512, 10, True), (512, 512, 10, False), (70, 8, 2, False), (1, 64, 4, False),
                                              (300, 1000, 8, True)])
def test_pf_route_bit_exact(dev, oracle, Cn, nexp, topk, zipf):
    print(f"case pf_route C={Cn} nexp={nexp} topk={topk} zipf={zipf}", flush=True)
    rng = np.random.default_rng(700 + Cn + nexp)
    logits = zipf_logits(rng, Cn, nexp) if zipf else rng.standard_normal((Cn, nexp + 1)).astype(np.float32)
    if Cn > 2:
        logits[2, :topk + 3] = logits[2].max() + 1.0   # a run of ties: the lower indexes win
    r = dev.pf_route(logits, nexp, topk)
    topi, topw = oracle.topk_logits(logits, nexp, topk)
    assert np.array_equal(r["topi"], topi)
    assert np.allclose(r["topw"], topw, rtol=2e-6, atol=0)
    gu, dn, cnt = oracle.pf_jobs(topi, nexp, PF)
    assert np.array_equal(r["cnt"], cnt)
    assert r["njobs"] == len(gu)
    assert np.array_equal(r["jbase"], np.concatenate([[0], np.cumsum((cnt + PF - 1) // PF)[:-1]]))
    for got, want in ((r["gu"], gu), (r["dn"], dn)):
        assert np.array_equal(got[:, :2], want[:, :2])
        for g, w in zip(got, want):
            n = w[1]
            assert np.array_equal(g[2:2 + n], w[2:2 + n]) and np.array_equal(g[2 + PF:2 + PF + n], w[2 + PF:2 + PF + n])


@pytest.mark.parametrize("Cn,nexp,topk", [(1, 1, 1), (63, 2, 1), (1025, 3, 1), (2731, 33, 3), (4100, 512, 10)])
def test_pf_jobs_of_busy_experts(dev, oracle, Cn, nexp, topk):
    """every row picks expert 0: one expert's pairs over many jobs and through every wave's list, wave spans of whole and of
    broken sixty-fours, an odd last expert"""
    print(f"case pf_jobs C={Cn} nexp={nexp} topk={topk}", flush=True)
    logits = np.random.default_rng(730 + Cn).standard_normal((Cn, nexp + 1)).astype(np.float32)
    logits[:, 0] = 9.0
    r = dev.pf_route(logits, nexp, topk)
    topi, _ = oracle.topk_logits(logits, nexp, topk)
    assert np.array_equal(r["topi"], topi)
    gu, dn, cnt = oracle.pf_jobs(topi, nexp, PF)
    assert np.array_equal(r["cnt"], cnt) and r["njobs"] == len(gu)
    assert np.array_equal(r["jbase"], np.concatenate([[0], np.cumsum((cnt + PF - 1) // PF)[:-1]]))
    for got, want in ((r["gu"], gu), (r["dn"], dn)):
        assert np.array_equal(got[:, :2], want[:, :2])
        for g, w in zip(got, want):
            n = w[1]
            assert np.array_equal(g[2:2 + n], w[2:2 + n]) and np.array_equal(g[2 + PF:2 + PF + n], w[2 + PF:2 + PF + n])


def test_pf_route_with_fewer_finite_logits_than_picks(dev, oracle):
    from test_oracle_routing import scarce_logits
    Cn, nexp, topk = 70, 512, 10
    print(f"case pf_route scarce C={Cn} nexp={nexp} topk={topk}", flush=True)
    logits = scarce_logits(np.random.default_rng(705), Cn, nexp)
    r = dev.pf_route(logits, nexp, topk)
    topi, topw = oracle.topk_logits(logits, nexp, topk)
    assert np.array_equal(r["topi"], topi)
    assert all(len(set(row.tolist())) == topk for row in r["topi"])
    assert np.all(np.isfinite(r["topw"])) and np.allclose(r["topw"], topw, rtol=2e-6, atol=0)
    gu, dn, cnt = oracle.pf_jobs(topi, nexp, PF)
    assert np.array_equal(r["cnt"], cnt) and r["njobs"] == len(gu)


@pytest.mark.parametrize("nexp,topk", [(3, 3), (64, 64), (65, 10), (513, 10), (1024, 64)])
def test_pf_route_ties_and_signed_zeros(dev, oracle, nexp, topk):
    """values from a handful (both zeros, both infinities' neighbours among them): ties within a lane's entries and across lanes"""
    print(f"case pf_route ties nexp={nexp} topk={topk}", flush=True)
    rng = np.random.default_rng(706 + nexp)
    values = np.array([0.0, -0.0, 1.0, -1.0, 0.5, 1e-40, -1e-40, -88.0, np.finfo(np.float32).min], dtype=np.float32)
    logits = values[rng.integers(0, len(values), (37, nexp + 1))]
    r = dev.pf_route(logits, nexp, topk)
    topi, topw = oracle.topk_logits(logits, nexp, topk)
    assert np.array_equal(r["topi"], topi)
    assert np.allclose(r["topw"], topw, rtol=2e-6, atol=0)


def test_f32_f16_bit_exact(dev, oracle):
    rng = np.random.default_rng(710)
    x = (rng.standard_normal((33, 257)) * 10.0 ** rng.integers(-8, 4, (33, 257))).astype(np.float32)
    assert np.array_equal(dev.f32_f16(x).view(np.uint16), oracle.f32_f16(x).view(np.uint16))


def test_swiglu_h16(dev, oracle):
    rng = np.random.default_rng(711)
    gu = (rng.standard_normal((50, 1024)) * 3).astype(np.float32)
    got, want = dev.swiglu_h16(gu, 512).view(np.uint16).astype(np.int32), oracle.swiglu_h16(gu, 512).view(np.uint16).astype(np.int32)
    diff = np.abs(got - want)
    assert diff.max() <= 1 and np.count_nonzero(diff) <= 1e-3 * diff.size


def h16_close(a, b):
    """two kernels' h = f16(silu(gate) * up) from the same f16 operands added up in different orders: nearly every value the
    same f16, the rest a rounding step apart"""
    differ = int((a.view(np.uint16) != b.view(np.uint16)).sum())
    print(f"{differ} of {a.size} f16 values of h differ", flush=True)
    assert differ <= a.size // 100 and rel_l2(a.astype(np.float32), b.astype(np.float32)) <= 1e-4


def make_jobs(rng, nexp, rows_avail, sizes):
    jobs = np.zeros((len(sizes), 2 + 2 * PF), dtype=np.int32)
    at = 0
    for j, n in enumerate(sizes):
        jobs[j, 0], jobs[j, 1] = rng.integers(0, nexp), n
        jobs[j, 2:2 + n] = rng.choice(rows_avail, size=n, replace=False)
        jobs[j, 2 + PF:2 + PF + n] = np.arange(at, at + n)
        at += n
    return jobs, at


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("nrows,ncols,down", [(1024, 2048, False), (2048, 512, True), (64, 256, False), (512, 1024, True)])
def test_moe_mma_matches_oracle(dev, oracle, nrows, ncols, down, packed):
    print(f"case moe_mma nrows={nrows} ncols={ncols} down={down} packed={packed}", flush=True)
    if packed and (nrows * ncols) % 2048:
        pytest.skip("unit64 takes whole units of 2048 weights")
    rng = np.random.default_rng(720 + nrows + ncols)
    nexp = 3
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((200, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, 200, [64, 1, 17, 16, 33, 48, 5])
    want = oracle.moe_mma(w, stride, nrows, ncols, jobs, PF, x16, total)
    # the arrays hold more jobs than the count says: the rest must not run (their entries are zero: n = 0)
    got = dev.moe_mma(w, stride, nrows, ncols, jobs, x16, total, packed=packed, down=down, cap=len(jobs) + 5)
    assert rel_l2(got, want) <= REL_L2
    assert rel_l2(got, want) <= 1e-5, "f16 operands are the oracle's: only the summation order may differ"


@pytest.mark.parametrize("nrows,nexp,sizes", [(2048, 40, [64, 1, 17, 0, 16, 33, 48, 5, 64, 64, 2, 0, 31, 64, 49, 15] * 6), (64, 3, [64, 1, 17, 16, 33, 48, 5]),
                                              (32, 2, [3]), (2048, 2, [64])])
def test_moe_mma_wave_form_tile16_rows_of_512(dev, oracle, nrows, nexp, sizes):
    # the down projection over tile16 matrices of 512 columns (k_moe_mma_wave16): blocks that end inside a job and blocks
    # that hold several, jobs without tokens, fewer items than blocks
    print(f"case moe_mma wave form nrows={nrows} nexp={nexp} jobs={len(sizes)}", flush=True)
    ncols = 512
    rng = np.random.default_rng(733 + nrows + len(sizes))
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    rows = max(200, sum(sizes))
    x16 = rng.standard_normal((rows, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    got = dev.moe_mma(w, stride, nrows, ncols, jobs, x16, total, packed=True, down=True, cap=len(jobs) + 5, tile16=True)
    other = dev.moe_mma(w, stride, nrows, ncols, jobs, x16, total, packed=True, down=True, cap=len(jobs) + 5)   # the same form over unit64
    assert rel_l2(got, other) <= 1e-6, "the same f16 products: only the summation order differs"
    assert np.array_equal(got == 0, other == 0)   # (rows no job writes stay as they were)
    if len(sizes) <= 8:
        want = oracle.moe_mma(w, stride, nrows, ncols, jobs, PF, x16, total)
        assert rel_l2(got, want) <= 1e-5, "f16 operands are the oracle's: only the summation order may differ"


@pytest.mark.parametrize("nrows,ncols,sizes", [
    (2048, 256, [64, 1, 17, 0, 16, 33, 48, 5, 64, 49] * 4), (32, 256, [3]), (64, 256, [9, 64, 31]),    # half a super-step a row: a job's whole tile in LDS
    (2048, 512, [64, 1, 17, 0, 16, 33, 48, 5, 64, 49] * 4), (96, 512, [16, 2, 64]),                    # one super-step, the same form
    (2048, 1024, [64, 1, 17, 0, 16, 33, 48, 5, 64, 49] * 4), (32, 1024, [5]), (96, 1024, [7, 40, 64]), # two, pairs of tiles: light lists, heavy units
    (1024, 2048, [2, 3, 1] * 100), (64, 4096, [64, 12, 20, 16]), (64, 6144, [3, 33]),                  # a unit a row, two and three
    (64, 768, [64, 1, 17, 33]), (32, 1536, [9, 48]), (64, 1280, [5, 64])])                             # rows that no wave form takes
def test_moe_mma_over_unit64_rows(dev, oracle, nrows, ncols, sizes):
    """every form that unit64 rows of a width go to: against the oracle, and a row's bits do not depend on what else the list holds"""
    print(f"case moe_mma unit64 nrows={nrows} ncols={ncols} jobs={len(sizes)}", flush=True)
    rng = np.random.default_rng(751 + nrows + ncols + len(sizes))
    nexp = 3
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((200, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, 200, sizes)

    def out_of(some):
        return dev.moe_mma(w, stride, nrows, ncols, some, x16, total + 2, packed=True, down=True, cap=len(some) + 3)

    got = out_of(jobs)
    assert not np.any(got[total:]), "rows no job writes stay as they were"
    few = jobs if len(jobs) <= 12 else jobs[:10]
    n = sum(sizes[:len(few)])
    want = oracle.moe_mma(w, stride, nrows, ncols, few, PF, x16, total + 2)
    assert rel_l2(got[:n], want[:n]) <= 1e-5, "f16 operands are the oracle's: only the summation order may differ"
    for j in {0, len(jobs) // 2, len(jobs) - 1}:
        at = jobs[j][2 + PF:2 + PF + int(jobs[j][1])]
        assert np.array_equal(got[at].view(np.uint32), out_of(jobs[j:j + 1])[at].view(np.uint32)), f"job {j} of {jobs[j][1]} rows"


@pytest.mark.parametrize("nrows,ncols", [(64, 256), (96, 512), (32, 1024), (64, 2048)])
def test_moe_mma_over_unit64_rows_and_unaligned_activations(dev, oracle, nrows, ncols):
    """rows of x that begin four bytes past a multiple of sixteen: the form without 16-byte loads into LDS, as for raw blocks"""
    print(f"case moe_mma unit64 unaligned nrows={nrows} ncols={ncols}", flush=True)
    rng = np.random.default_rng(752 + nrows + ncols)
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, 3 * nrows * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((80, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, 3, 80, [5, 64, 17, 1, 40])
    want = oracle.moe_mma(w, stride, nrows, ncols, jobs, PF, x16, total)
    dw_, dj = dev.up(w), dev.up(jobs)
    dx = dev.up(np.concatenate([np.zeros(2, np.float16), x16.reshape(-1)]))
    assert dx.data_ptr() % 16 == 0
    dev.ok(dev.lib.fnx_iq3s_repack(dw_.data_ptr(), dw_.data_ptr(), w.size // 110 * 256, dev.st()))
    W, nj, out = dev.pkg.dw(dw_, ncols, nrows, packed=True), dev.up(np.array([len(jobs)], np.int32)), dev.zeros((total, nrows), dev.torch.float32)
    dev.ok(dev.lib.fnx_moe_down_mma(C.byref(W), stride, dj.data_ptr(), nj.data_ptr(), len(jobs), dx.data_ptr() + 4, out.data_ptr(), dev.st()))
    dev.sync()
    assert rel_l2(out.cpu().numpy(), want) <= 1e-5, "f16 operands are the oracle's: only the summation order may differ"


# Lists of several jobs a block: phases of up to four token tiles, with jobs that fill one alone, jobs without tokens between them, and
# (18 tiles a job) second units of two tiles, where most waves have none.
@pytest.mark.parametrize("nrows,ncols,tile16", [(288, 512, True), (288, 512, False), (96, 256, False), (2048, 512, True)])
def test_moe_mma_phases_of_several_jobs_a_block(dev, oracle, nrows, ncols, tile16):
    """a row's bits do not depend on the jobs that share its phase: a long list against the same jobs in lists of one a block at most"""
    print(f"case moe_mma phases nrows={nrows} ncols={ncols} tile16={tile16}", flush=True)
    sizes = ([1, 16, 17, 0, 2, 64, 3, 3, 33, 0, 0, 5, 48, 9, 1, 32, 15, 31, 2, 8] * 60)[:1190 if nrows < 2048 else 610]
    rng = np.random.default_rng(757 + nrows + ncols)
    nexp, stride = 5, nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((400, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, 400, sizes)

    def out_of(some):
        return dev.moe_mma(w, stride, nrows, ncols, some, x16, total, packed=True, down=True, cap=len(some), tile16=tile16)

    got = out_of(jobs)
    few = 60
    for j0 in (0, len(jobs) // 2, len(jobs) - few):
        at = np.concatenate([j[2 + PF:2 + PF + int(j[1])] for j in jobs[j0:j0 + few]])
        assert np.array_equal(got[at].view(np.uint32), out_of(jobs[j0:j0 + few])[at].view(np.uint32)), f"jobs {j0} .. {j0 + few}"
    n = sum(sizes[:8])
    assert rel_l2(got[:n], oracle.moe_mma(w, stride, nrows, ncols, jobs[:8], PF, x16, total)[:n]) <= 1e-5, "f16 operands are the oracle's"


# More than 524,288 columns of all rows (on 256 CUs): a thread of the combine takes four columns, unless the rows are no whole
# 16-byte pieces or a buffer is not aligned to them (`off`: by how many floats part, sh and out are shifted).
@pytest.mark.parametrize("T,n,topk,off", [(257, 2048, 10, (0, 0, 0)), (300, 2048, 1, (0, 0, 0)), (410, 1300, 3, (0, 0, 0)), (140, 3844, 16, (0, 0, 0)), (1100, 512, 8, (0, 0, 0)),
                                          (300, 2050, 10, (0, 0, 0)), (300, 2047, 9, (0, 0, 0)), (257, 2048, 8, (1, 0, 0)), (257, 2048, 7, (0, 2, 0)), (257, 2048, 10, (0, 0, 1)),
                                          (256, 2048, 10, (0, 0, 0))])
def test_combine_of_many_rows_equals_few(dev, oracle, T, n, topk, off):
    """a row's bits do not depend on how many rows a call brings: against the same rows 64 a call (one column a thread), and the oracle"""
    print(f"case combine T={T} n={n} topk={topk} off={off}", flush=True)
    rng = np.random.default_rng(790 + T + n + topk)
    part, sh = rng.standard_normal((T * topk, n)).astype(np.float32), rng.standard_normal((T, n)).astype(np.float32)
    topw, logit = rng.random((T, topk)).astype(np.float32), rng.standard_normal((T, 1)).astype(np.float32)
    t = dev.torch
    flat = lambda a, o: t.cat((t.zeros(o, device="cuda:0"), dev.up(a).flatten()))
    dp, ds, dt, dl = flat(part, off[0]), flat(sh, off[1]), dev.up(topw), dev.up(logit)
    out, few = t.full((off[2] + T * n + 4,), float("nan"), device="cuda:0"), t.zeros((T, n), device="cuda:0")
    dev.ok(dev.lib.fnx_moe_combine(dp.data_ptr() + 4 * off[0], dt.data_ptr(), ds.data_ptr() + 4 * off[1], dl.data_ptr(), 1, out.data_ptr() + 4 * off[2], T, n, topk, dev.st()))
    for t0 in range(0, T, 64):
        k = min(64, T - t0)
        dev.ok(dev.lib.fnx_moe_combine(dp.data_ptr() + 4 * (off[0] + t0 * topk * n), dt.data_ptr() + 4 * t0 * topk, ds.data_ptr() + 4 * (off[1] + t0 * n), dl.data_ptr() + 4 * t0, 1,
                                       few.data_ptr() + 4 * t0 * n, k, n, topk, dev.st()))
    dev.sync()
    got = out.cpu().numpy()
    assert np.isnan(got[:off[2]]).all() and np.isnan(got[off[2] + T * n:]).all(), "nothing beside the rows"
    got = got[off[2]:off[2] + T * n].reshape(T, n)
    assert np.array_equal(got.view(np.uint32), few.cpu().numpy().view(np.uint32))
    assert rel_l2(got, oracle.moe_combine(part, topw, sh, logit[:, 0])) <= 1e-6   # the sigmoid's expf is the device's


@pytest.mark.parametrize("n", [1, 17, 33, 64])
def test_moe_mma_wave_form_output_rows_past_32_bit_offsets(dev, n):
    # a job with an output row past 3.5 GiB stores by whole addresses: the same bits as by buffer offsets, in both orders of rows
    print(f"case moe_mma wave form far rows n={n}", flush=True)
    import ctypes as C
    t, nrows, ncols = dev.torch, 2048, 512
    far = 0xE0000000 // (nrows * 4)
    rng = np.random.default_rng(760 + n)
    w = dev.up(random_iq3s(rng, nrows * ncols // 256, dmax=2e-2))
    dev.ok(dev.lib.fnx_iq3s_repack(w.data_ptr(), w.data_ptr(), nrows * ncols, dev.st()))
    d16 = dev.zeros(dev.lib.fnx_iq3s_tile16_bytes(nrows, ncols, 1), t.uint8)
    dev.ok(dev.lib.fnx_iq3s_tile16(w.data_ptr(), d16.data_ptr(), nrows, ncols, 1, dev.st()))
    W = dev.pkg.dw(d16, ncols, nrows, tile16=True)
    x = dev.up(rng.standard_normal((n, ncols)).astype(np.float16).view(np.int16))
    out = t.empty((far + 80, nrows), dtype=t.float32, device="cuda:0")
    nj, got = dev.up(np.array([1], dtype=np.int32)), []
    for last in (n - 1, far - 1, far, far + 79):   # the last token's row
        job = np.zeros((1, 2 + 2 * PF), dtype=np.int32)
        job[0, 1], job[0, 2:2 + n] = n, np.arange(n)
        job[0, 2 + PF:2 + PF + n] = np.arange(n)
        job[0, 2 + PF + n - 1] = last
        rows = t.from_numpy(job[0, 2 + PF:2 + PF + n].astype(np.int64)).to(out.device)
        out[rows] = float("nan")
        dj = dev.up(job)
        dev.ok(dev.lib.fnx_moe_down_mma(C.byref(W), 0, dj.data_ptr(), nj.data_ptr(), 1, x.data_ptr(), out.data_ptr(), dev.st()))
        dev.sync()
        got.append(out[rows].cpu().numpy())
    assert np.isfinite(got[0]).all()
    for g in got[1:]:
        assert np.array_equal(g, got[0])


@pytest.mark.parametrize("ffs,ncols,nexp,sizes", [(512, 2048, 24, [64, 1, 17, 0, 16, 33, 48, 5, 64, 64, 2, 0, 31, 64, 49, 15] * 3), (128, 512, 3, [64, 1, 17, 16, 33, 48, 5]),
                                                  (256, 1024, 2, [3]), (640, 2048, 2, [64, 9]), (128, 2560, 2, [5, 64, 20, 16])])
def test_moe_gate_up_h16_one_launch_equals_two(dev, oracle, ffs, ncols, nexp, sizes):
    # h = silu(gate) * up straight from the matrix-core launch (the wave form over tile16) against fnx_moe_gate_up_mma over
    # the unit64 copy followed by fnx_swiglu_h16, whatever the mix of job sizes, with rows no job writes left alone
    # (640: a job's last unit is short of pairs; 2560 columns: five activation tiles a row, so small jobs go as heavy units)
    tile16 = True
    print(f"case moe_gate_up_h16 ffs={ffs} ncols={ncols} nexp={nexp} jobs={len(sizes)}", flush=True)
    nrows = 2 * ffs
    rng = np.random.default_rng(741 + ffs + len(sizes))
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    rows = max(200, sum(sizes))
    x16 = rng.standard_normal((rows, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    one, two = dev.moe_mma(w, stride, nrows, ncols, jobs, x16, total + 3, packed=True, cap=len(jobs) + 5, tile16=tile16, h16=True)
    assert np.all(np.isfinite(two.astype(np.float32)))
    # the same f16 operands on both sides; the two kernels add a row's products in different orders, which now and then moves
    # an f16 value of h by one step
    h16_close(one, two)
    assert np.any(one[:total] != 0) and not np.any(one[total:])
    if len(sizes) <= 8:   # against the oracle: its products, its SwiGLU
        gu = oracle.moe_mma(w, stride, nrows, ncols, jobs, PF, x16, total + 3)
        want = oracle.swiglu_h16(gu, ffs)
        assert rel_l2(one.astype(np.float32), want.astype(np.float32)) <= 1e-3


@pytest.mark.parametrize("ffs,ncols,sizes", [
    (512, 2048, [1, 2, 3] * 140),                                              # some 400 jobs of two tokens: phases of many jobs
    (32, 512, [16, 8, 8, 15, 2, 16, 0, 1, 1, 14, 9, 7, 0, 16] * 20),           # two pairs a job: phases that end at sixteen tokens and just past them
    (16, 512, [1] * 600 + [16, 1]),                                            # a pair a job: phases of sixteen jobs
    (256, 2048, [9, 3, 12, 7] * 32), (1024, 2048, [16] * 60), (512, 2048, [9] * 125),   # stretches of whole eights
    (512, 2048, [16] * 80), (512, 1536, [5] * 40), (80, 1024, [16, 3] * 50),   # ten pairs a block, five, ten pairs a job
    (512, 2048, [20] * 3 + [9] * 50), (512, 2048, [64] * 40 + [12] * 60), (256, 1024, [64] * 300 + [10, 2] * 40),   # beside heavy units: some blocks, several a block
    (32, 512, [3, 16, 1, 40, 0, 17, 64, 33] * 270)])                           # more jobs than are ranked
def test_moe_gate_up_h16_lists_give_the_bits_of_their_jobs_alone(dev, ffs, ncols, sizes):
    """however a list's work is dealt to the blocks (a wave a tile or a pair of tiles, jobs staged together, ranked or in the
    list's order), a row's h is the same bits: every job of the list is compared with the same job in a list of a few, some of them with the job alone"""
    print(f"case moe_gate_up_h16 bits ffs={ffs} ncols={ncols} jobs={len(sizes)}", flush=True)
    assert len(sizes) <= 2048 or ffs == 32, "the kernel ranks up to 2,048 jobs"
    rng = np.random.default_rng(743 + ffs + len(sizes))
    nexp, nrows, rows = 3, 2 * ffs, 200
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((rows, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, rows, sizes)

    def h_of(some):
        return dev.moe_mma(w, stride, nrows, ncols, some, x16, total + 3, packed=True, tile16=True, h16=True)[0]

    got = h_of(jobs)
    assert np.all(np.any(got[:total] != 0, axis=1)) and not np.any(got[total:])
    few = np.zeros_like(got)
    for part in np.array_split(np.arange(len(jobs)), max(2, min(len(jobs) // 4, 60))):
        lo, hi = sum(sizes[:part[0]]), sum(sizes[:part[-1] + 1])
        few[lo:hi] = h_of(jobs[part])[lo:hi]
    assert np.array_equal(got.view(np.uint16), few.view(np.uint16)), f"rows {np.flatnonzero(np.any(got != few, axis=1))[:8]}"
    for j in [0, 1, 2, len(jobs) // 2, len(jobs) - 2, len(jobs) - 1]:
        at = jobs[j][2 + PF:2 + PF + int(jobs[j][1])]
        assert np.array_equal(got[at].view(np.uint16), h_of(jobs[j:j + 1])[at].view(np.uint16)), f"job {j} of {jobs[j][1]} rows"


@pytest.mark.parametrize("sizes", [[5, 64, 17], [3] * 1100 + [40]])
def test_moe_gate_up_h16_reads_no_job_past_the_count(dev, sizes):
    """the capacity bounds the count that the device word gives: the job array may end with the last job that counts"""
    import ctypes as C
    print(f"case moe_gate_up_h16 short array jobs={len(sizes)}", flush=True)
    rng = np.random.default_rng(744)
    ffs, ncols, nexp, rows, t = 32, 512, 3, 200, dev.torch
    w = random_iq3s(rng, nexp * 2 * ffs * ncols // 256, dmax=2e-2)
    x16 = rng.standard_normal((rows, ncols)).astype(np.float16)
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    want = dev.moe_mma(w, 2 * ffs * ncols // 256 * 110, 2 * ffs, ncols, jobs, x16, total, packed=True, tile16=True, h16=True)[0]
    u64, tiles = dev.up(w), dev.zeros(dev.lib.fnx_iq3s_tile16_bytes(2 * ffs, ncols, nexp), t.uint8)
    dev.ok(dev.lib.fnx_iq3s_repack(u64.data_ptr(), u64.data_ptr(), w.size // 110 * 256, dev.st()))
    dev.ok(dev.lib.fnx_iq3s_tile16(u64.data_ptr(), tiles.data_ptr(), 2 * ffs, ncols, nexp, dev.st()))
    W, dj, dx, got = dev.pkg.dw(tiles, ncols, 2 * ffs, tile16=True), dev.up(jobs), dev.up(x16), dev.zeros((total, ffs), t.float16)
    count = dev.up(np.array([len(sizes)], dtype=np.int32))
    dev.ok(dev.lib.fnx_moe_gate_up_h16_mma(C.byref(W), dev.lib.fnx_iq3s_tile16_bytes(2 * ffs, ncols, 1), dj.data_ptr(), count.data_ptr(), 4096, dx.data_ptr(),
                                           got.data_ptr(), dev.st()))
    dev.sync()
    assert np.array_equal(got.cpu().numpy().view(np.uint16), want.view(np.uint16)) and np.all(np.any(want != 0, axis=1))


def split_in_16s(jobs):
    """jobs of up to 64 rows as the jobs of up to 16 rows they consist of (the oracle's mmvq takes those)"""
    out = []
    for jb in jobs:
        n = int(jb[1])
        for t0 in range(0, n, 16):
            k = min(16, n - t0)
            j = np.zeros(1, dtype=fnx_gpu.JOB_DTYPE)
            j["w"], j["n"] = jb[0], k
            j["y"][0, :k], j["out"][0, :k] = jb[2 + t0:2 + t0 + k], jb[2 + PF + t0:2 + PF + t0 + k]
            out.append(j)
    return np.concatenate(out) if out else np.zeros(0, dtype=fnx_gpu.JOB_DTYPE)


@pytest.mark.parametrize("nrows,ncols,nexp,sizes", [(1024, 2048, 24, [64, 1, 17, 0, 16, 33, 48, 5, 64, 64, 2, 0, 31, 64, 49, 15] * 3), (64, 512, 3, [64, 1, 17, 16, 33, 48, 5]),
                                                  (32, 1024, 2, [3]), (2048, 512, 2, [64, 9, 0, 0, 40])])
def test_moe_big_jobs_over_q8_1_match_the_oracle(dev, oracle, nrows, ncols, nexp, sizes):
    """kernels.hpp:324-325: the prompt path's jobs with mmvq's terms. gate|up form: q8_1 rows in, the oracle's mmvq over the same
    jobs cut into sixteens; down form (where the matrix's columns allow rows [gate | up]): h = silu(gate) * up quantised on
    the way, against the oracle's SwiGLU -> q8_1 -> mmvq. The integer sums are exact; a row's sub-block terms are added in
    another order than the oracle's."""
    print(f"case moe_big nrows={nrows} ncols={ncols} nexp={nexp} jobs={len(sizes)}", flush=True)
    rng = np.random.default_rng(771 + nrows + len(sizes))
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    rows = max(200, sum(sizes))
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    small = split_in_16s(jobs)
    x = rng.standard_normal((rows, ncols)).astype(np.float32)
    xq = oracle.quantize_q8_1(x)
    want = oracle.mmvq(w, stride, nrows, ncols, small, xq, total + 3)
    got = dev.moe_big(w, stride, nrows, ncols, jobs, xq, total + 3, cap=len(jobs) + 5)
    assert rel_l2(got, want) <= 1e-5
    assert np.any(got[:total] != 0) and not np.any(got[total:])
    # the down form: the same matrix read as rows of ncols = ffs, fed rows [gate | up]
    gu = (rng.standard_normal((rows, 2 * ncols)) * 2).astype(np.float32)
    hq = oracle.swiglu_stacked_q8_1(gu, ncols)
    want = oracle.mmvq(w, stride, nrows, ncols, small, hq, total + 3)
    got = dev.moe_big(w, stride, nrows, ncols, jobs, gu, total + 3, down=True, cap=len(jobs) + 5)
    assert rel_l2(got, want) <= 1e-5
    assert not np.any(got[total:])


@pytest.mark.parametrize("nrows,ncols,sizes", [(1024, 2048, [64, 1, 17, 0, 16, 33, 48, 5, 32, 31] * 5), (2048, 512, [64, 1, 17, 0, 33, 48, 16, 5, 50, 49] * 2),
                                            (528, 1024, [64, 1, 17, 0, 33, 48, 16, 5, 50, 0] * 7), (16, 512, [64, 63, 33, 2] * 400),
                                            (1024, 2048, [64] * 17), (2048, 512, [40] * 13), (1024, 2048, [1] * 5), (1024, 2048, [64, 2] * 20),
                                            (48, 512, [64, 1, 33, 0, 17] * 819)])
def test_moe_big_lists_give_the_bits_of_their_jobs_alone(dev, nrows, ncols, sizes):
    """a long list's jobs go as units of one or two token tiles, runs of their rounds dealt to the blocks (a last round of a unit's
    tiles may be short), a short list's as units of one: a token's sums are the same bits. Every job of the list is compared
    with the same job in a list of a few, its first and last jobs with those jobs alone. (Jobs to a block, rounds to a block, a
    few tiles more than a wave each, 4,095 jobs: the plan's forms and their ends.)"""
    print(f"case moe_big bits nrows={nrows} ncols={ncols} jobs={len(sizes)}", flush=True)
    rng = np.random.default_rng(97 + nrows)
    nexp = 3
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    rows = 200
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    gu = (rng.standard_normal((rows, 2 * ncols)) * 2).astype(np.float32)
    xq = dev.quantize_q8_1(gu[:, :ncols])
    pieces = max(2, min(len(jobs) // 4, 60))
    for down, y in ((False, xq), (True, gu)):
        got = dev.moe_big(w, stride, nrows, ncols, jobs, y, total + 3, down=down, cap=min(len(jobs) + 5, 4096))
        assert np.all(np.any(got[:total] != 0, axis=1)) and not np.any(got[total:])
        few = np.zeros_like(got)
        for part in np.array_split(np.arange(len(jobs)), pieces):
            lo, hi = sum(sizes[:part[0]]), sum(sizes[:part[-1] + 1])
            few[lo:hi] = dev.moe_big(w, stride, nrows, ncols, jobs[part], y, total + 3, down=down)[lo:hi]
        assert np.array_equal(got.view(np.uint32), few.view(np.uint32)), f"rows {np.flatnonzero(np.any(got != few, axis=1))[:8]}, down={down}"
        for j in [*range(min(10, len(jobs))), len(jobs) - 2, len(jobs) - 1]:
            n = int(jobs[j][1])
            one = dev.moe_big(w, stride, nrows, ncols, jobs[j:j + 1], y, total + 3, down=down, cap=1)
            at = jobs[j][2 + PF:2 + PF + n]
            assert np.array_equal(got[at].view(np.uint32), one[at].view(np.uint32)), f"job {j} of {n} rows, down={down}"


@pytest.mark.parametrize("sizes,cap", [([5, 64, 17], 4096), ([3] * 1100 + [40], 4096), ([], 4096)])
def test_moe_big_reads_no_job_past_the_count(dev, sizes, cap):
    """njobs_cap bounds the count that the device word gives: the array itself may end with the last job that counts"""
    print(f"case moe_big short array jobs={len(sizes)} cap={cap}", flush=True)
    rng = np.random.default_rng(98)
    nrows, ncols, nexp, rows = 64, 512, 3, 200
    stride = nrows * ncols // 256 * 110
    w = random_iq3s(rng, nexp * nrows * ncols // 256, dmax=2e-2)
    jobs, total = make_jobs(rng, nexp, rows, sizes)
    if not sizes:   # one job that does not count
        jobs = make_jobs(rng, nexp, rows, [7])[0]
    gu = (rng.standard_normal((rows, 2 * ncols)) * 2).astype(np.float32)
    for down, y in ((False, dev.quantize_q8_1(gu[:, :ncols])), (True, gu)):
        got = dev.moe_big(w, stride, nrows, ncols, jobs, y, total + 3, down=down, cap=cap, short=True, count=len(sizes))
        want = dev.moe_big(w, stride, nrows, ncols, jobs, y, total + 3, down=down, cap=len(jobs), count=len(sizes))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)) and bool(np.any(want[:total] != 0)) == bool(sizes)


def test_moe_mma_weights_equal_the_oracles_f16(dev, oracle):
    # x = unit vectors: the product returns single weights, so every dequantised f16 value is checked bit for bit,
    # subnormal ones included (tiny d)
    rng = np.random.default_rng(730)
    nrows, ncols = 32, 256
    for dmax in (2e-2, 3e-6):
        w = random_iq3s(rng, nrows * ncols // 256, dmax=dmax)
        want = oracle.iq3s_dequant_f16(w).reshape(nrows, ncols)
        x16 = np.eye(ncols, dtype=np.float16)
        jobs = np.zeros((4, 2 + 2 * PF), dtype=np.int32)
        for j in range(4):
            jobs[j, 1] = 64
            jobs[j, 2:2 + 64] = np.arange(64 * j, 64 * j + 64)
            jobs[j, 2 + PF:] = np.arange(64 * j, 64 * j + 64)
        for packed in (False, True):
            got = dev.moe_mma(w, 0, nrows, ncols, jobs, x16, ncols, packed=packed)
            assert np.array_equal(got.T.astype(np.float16).view(np.uint16), want.view(np.uint16))
            assert np.array_equal(got.T, want.astype(np.float32))


@pytest.mark.parametrize("n,ff,nexp,topk,Cn", [(2048, 512, 32, 4, 100), (2048, 512, 512, 10, 64), (256, 256, 8, 2, 70)])
def test_prefill_layer_matches_oracle(dev, oracle, n, ff, nexp, topk, Cn):
    print(f"case prefill_layer n={n} ff={ff} nexp={nexp} topk={topk} C={Cn}", flush=True)
    rng = np.random.default_rng(740 + nexp + Cn)   # d small enough that h = silu(g) u stays inside f16's range
    nb = lambda rows, cols: rows * cols // 256
    gu = random_iq3s(rng, nexp * nb(2 * ff, n), dmax=1e-3)
    down = random_iq3s(rng, nexp * nb(n, ff), dmax=1e-3)
    sh_gu, sh_down = random_iq3s(rng, nb(2 * ff, n), dmax=1e-3), random_iq3s(rng, nb(n, ff), dmax=1e-3)
    router = (rng.standard_normal((nexp + 1, n)) * 0.05).astype(np.float32)
    x = rng.standard_normal((Cn, n)).astype(np.float32)
    want = oracle.moe_prefill_layer(n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, x)
    packed = (2 * ff * n) % 2048 == 0 and (n * ff) % 2048 == 0
    L = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=packed)
    for rep in range(2):   # a second chunk through the same workspace
        r = L.run(x)
        assert np.array_equal(r["logits"].view(np.uint32), want["logits"].view(np.uint32))
        assert np.array_equal(r["topi"], want["topi"])
        assert int(r["njobs"][0]) == want["njobs"] and int(r["njobs"][1]) == (Cn + PF - 1) // PF
        assert np.all(np.isfinite(want["out"]))
        assert rel_l2(r["out"], want["out"]) <= REL_L2


@pytest.mark.parametrize("n,ff,nexp,topk,Cn", [(2048, 512, 48, 10, 300), (1024, 256, 8, 2, 70)])
def test_prefill_layer_tile16_equals_unit64(dev, oracle, n, ff, nexp, topk, Cn):
    """the gate|up matrices (and the down matrices, where ff comes in 512s) in the prompt path's own layout: the same f16
    weights and activations as the unit64 layout's kernels; h and the
    chunk's result agree to float rounding (and with the oracle's within the bar either way)"""
    print(f"case prefill_layer tile16 n={n} ff={ff} nexp={nexp} topk={topk} C={Cn}", flush=True)
    rng = np.random.default_rng(760 + nexp)
    nb = lambda rows, cols: rows * cols // 256
    gu = random_iq3s(rng, nexp * nb(2 * ff, n), dmax=1e-3)
    down = random_iq3s(rng, nexp * nb(n, ff), dmax=1e-3)
    sh_gu, sh_down = random_iq3s(rng, nb(2 * ff, n), dmax=1e-3), random_iq3s(rng, nb(n, ff), dmax=1e-3)
    router = (rng.standard_normal((nexp + 1, n)) * 0.05).astype(np.float32)
    x = rng.standard_normal((Cn, n)).astype(np.float32)
    a = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=True).run(x)
    b = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=True, tile16=True).run(x)
    assert np.array_equal(a["topi"], b["topi"])
    h16_close(a["h16"], b["h16"])
    assert rel_l2(b["out"], a["out"]) <= 1e-5
    want = oracle.moe_prefill_layer(n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, x)
    assert rel_l2(b["out"], want["out"]) <= REL_L2


@pytest.mark.parametrize("tile16,Cn", [(False, 8192), (True, 8192), (True, 2048), (True, 16384)])
def test_prefill_layer_large_chunk_equals_small_chunks(dev, tile16, Cn):
    """A size-independent property at a size the oracle does not reach: a row's result does not depend on what else is in
    its chunk, so 8,192 rows in one call (more tasks than one pass of a block's task list holds, every kernel form's loop
    over list passes, a thousand jobs and more split over the wave form's blocks) must equal the same rows in 16 calls of
    512, bit for bit, in either layout. (2,048 rows: a few hundred jobs, ranked, their heavy units several to a block; 16,384:
    more jobs than the wave form ranks, the shared expert's in a list of their own.)"""
    n, ff, nexp, topk, small = 2048, 512, 64, 10, 512
    print(f"case prefill_layer large n={n} ff={ff} nexp={nexp} topk={topk} C={Cn} tile16={tile16}", flush=True)
    rng = np.random.default_rng(777)
    nb = lambda rows, cols: rows * cols // 256
    gu = random_iq3s(rng, nexp * nb(2 * ff, n), dmax=1e-3)
    down = random_iq3s(rng, nexp * nb(n, ff), dmax=1e-3)
    sh_gu, sh_down = random_iq3s(rng, nb(2 * ff, n), dmax=1e-3), random_iq3s(rng, nb(n, ff), dmax=1e-3)
    router = (rng.standard_normal((nexp + 1, n)) * 0.05).astype(np.float32)
    x = rng.standard_normal((Cn, n)).astype(np.float32)
    r = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=True, tile16=tile16).run(x)
    big = r["out"]
    assert Cn != 16384 or int(r["njobs"].sum()) > 2048, "more jobs than are ranked"
    del r
    L = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, small, packed=True, tile16=tile16)
    assert np.all(np.isfinite(big))
    for c0 in range(0, Cn, small):
        part = L.run(x[c0:c0 + small])["out"]
        assert int(np.count_nonzero(part.view(np.uint32) != big[c0:c0 + small].view(np.uint32))) == 0, f"rows {c0}.."


def test_prefill_layer_two_chunks_in_flight(dev):
    """A layer's chunks are independent, and a call's state is all in its workspace: chunks dealt to two streams with a
    workspace each must leave the bits that the same chunks leave one after the other on one stream."""
    import ctypes as C
    n, ff, nexp, topk, Cn, chunks = 2048, 512, 64, 10, 512, 6
    print(f"case prefill_layer two streams n={n} ff={ff} nexp={nexp} topk={topk} C={Cn}", flush=True)
    rng = np.random.default_rng(778)
    nb = lambda rows, cols: rows * cols // 256
    gu = random_iq3s(rng, nexp * nb(2 * ff, n), dmax=1e-3)
    down = random_iq3s(rng, nexp * nb(n, ff), dmax=1e-3)
    sh_gu, sh_down = random_iq3s(rng, nb(2 * ff, n), dmax=1e-3), random_iq3s(rng, nb(n, ff), dmax=1e-3)
    router = (rng.standard_normal((nexp + 1, n)) * 0.05).astype(np.float32)
    x = rng.standard_normal((chunks, Cn, n)).astype(np.float32)
    A = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=True, tile16=True)
    B = fnx_gpu.PfLayerDev(dev, n, ff, nexp, topk, router, gu, down, sh_gu, sh_down, Cn, packed=True, tile16=True)
    want = [A.run(x[c])["out"] for c in range(chunks)]
    t = dev.torch
    dx = dev.up(x)
    outs = dev.zeros((chunks, Cn, n), t.float32)
    streams = [t.cuda.Stream(), t.cuda.Stream()]
    t.cuda.synchronize()
    for rep in range(3):
        outs.zero_()
        t.cuda.synchronize()
        for c in range(chunks):
            L, s = ((A, streams[0]), (B, streams[1]))[c & 1]
            dev.ok(dev.lib.fnx_moe_prefill_layer(C.byref(L.L), dx[c].data_ptr(), Cn, outs[c].data_ptr(), C.byref(L.ws), s.cuda_stream))
        t.cuda.synchronize()
        got = outs.cpu().numpy()
        for c in range(chunks):
            assert int(np.count_nonzero(got[c].view(np.uint32) != want[c].view(np.uint32))) == 0, f"round {rep}, chunk {c}"
