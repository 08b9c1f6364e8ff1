"""GPU parity of the steps either side of the routed block: fmt 0 (f32) experts on the f32
matrix cores (the shared experts, src/model/kimi_k3.cpp:192-209), the router
(cpu_route, src/gpu/metal_ops.cpp:213-231), dense linears (QuantMat::gemm,
src/quant/weight.cpp:47-64; K3's latent down / up, src/model/kimi_k3.cpp:2003-2006,
2074-2090), RMSNorm (quant::rmsnorm, src/quant/quant.cpp:384-398) and a K3-shaped chain of
them around moe_block, against the CPU oracle (pinned to the reference build by the CPU
suite).

Bars: f32 arithmetic in another summation order, 2e-5 relative (max|y - ref| / max|ref|);
linears on int4 / MXFP4 weights take their input rows as two bf16 terms (2^-17), 1e-4.
Router: the device's dot products and expf may move a score by a few ulp, so picks must
agree wherever the host's k-th and (k+1)-th choices are more than 1e-5 (relative) apart,
and the weights of agreeing tokens within 1e-5.
"""
import sys

import numpy as np
import pytest
import torch

import npref
from cases import expert_arrays, random_case

pytestmark = pytest.mark.gpu

TOL_F32 = 2e-5


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def run_block(hip, c):
    keep = []

    def L(xs):
        if xs is None:
            return None
        out = []
        for x in xs:
            t = None if x is None else dev(x)
            keep.append(t)
            out.append(None if t is None else t.data_ptr())
        return out
    lists = [L(c.g), L(c.u), L(c.d), L(c.gs), L(c.us), L(c.ds)]
    out = dev(c.out)
    hip.moe_block_dev(c.nb, c.D, c.I, c.fmt, *lists, dev(c.xg), c.xoff, c.nr, c.rows, c.rw, out,
                      c.S, c.act, c.a, c.b)
    torch.cuda.synchronize()
    return out.cpu().numpy()


F32_CASES = [
    # D, I, nr, S, act, a, b
    (512, 256, [1, 2, 3], 6, 1, 7.0, 0.0),          # decode rows, ClampSwiGLU
    (7168, 2048, [1], 1, 2, 4.0, 25.0),             # K3 shared expert (SiTU), one token
    (6144, 2048, [3], 3, 1, 7.0, 0.0),              # GLM shared expert shape
    (1024, 512, [40, 5, 70], 80, 0, 0.0, 0.0),      # prefill rows: 16-, 32- and 64-row items
    (32, 16, [1], 1, 0, 0.0, 0.0),                  # one K block, one tile
    (4128, 272, [17, 16], 40, 1, 7.0, 0.0),         # K of unequal wave ranges, 8-column tiles
    (4160, 3600, [2], 2, 2, 4.0, 25.0),             # 16-column dual tiles, 16 waves
    (96, 2064, [64, 64, 33], 70, 2, 4.0, 25.0),     # 64-row blocks, 4 weight tiles, ragged columns
    (1056, 2064, [130, 64, 40], 150, 1, 7.0, 0.0),  # 64-row blocks, 2 weight tiles, chains of 512
    (64, 48, [20, 3, 0, 70], 90, 2, 4.0, 25.0),     # short K: a wave a tile
    (32, 32, [70, 33, 17, 1], 90, 1, 7.0, 0.0),     # the same, all row classes
    (160, 6176, [16, 9], 20, 1, 7.0, 0.0),          # a wave a tile by the number of tiles
]


@pytest.mark.parametrize("case", F32_CASES)
def test_fmt0_block_on_f32_matrix_cores(hip, orc, case):
    D, I, nr, S, act, a, b = case
    say("fmt0 block", case)
    rng = np.random.default_rng(D + I + len(nr))
    c = random_case(rng, 0, D, I, nr, S, act, a, b)
    hip.stats_reset()
    got = run_block(hip, c)
    st = hip.stats()
    exp = c.out.copy()
    assert orc.moe_block(*c.args(exp), act, a, b) == 1
    err = npref.rel_err(got, exp)
    say("  rel_err", err, "launches", st["launches_gate_up"], st["launches_down"])
    assert err < TOL_F32


@pytest.mark.parametrize("T,D,E,k,rscale,bias", [(1, 7168, 384, 8, 2.5, True),
                                                 (16, 2048, 64, 8, 1.0, False),
                                                 (300, 1024, 256, 8, 1.0, True),
                                                 (61, 2064, 384, 8, 2.5, True),
                                                 (100, 2048, 320, 64, 2.5, False),
                                                 (33, 2048, 512, 3, 1.0, True),
                                                 (5, 2048, 544, 4, 2.5, True),
                                                 (1, 48, 32, 31, 2.5, True)])
def test_router_matches_host_router(hip, orc, T, D, E, k, rscale, bias):
    say("router", T, D, E, k)
    rng = np.random.default_rng(T + D + E)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = (rng.standard_normal((E, D)) * (1.0 / np.sqrt(D))).astype(np.float32)
    bv = (rng.standard_normal(E) * 0.05).astype(np.float32) if bias else None
    f32 = dict(dtype=torch.float32, device="cuda")
    scores, choice = torch.empty((T, E), **f32), torch.empty((T, E), **f32)
    idx = torch.empty((T, k), dtype=torch.int32, device="cuda")
    wt = torch.empty((T, k), **f32)
    hip.router_dev(dev(x), dev(w), None if bv is None else dev(bv), T, D, E, k, rscale, scores,
                   choice, idx, wt)
    torch.cuda.synchronize()
    gi, gw = idx.cpu().numpy(), wt.cpu().numpy()
    ei, ew = orc.route(x, w, bv, k, rscale)
    # the host's choices in f64, for the gap between the k-th and (k+1)-th
    s64 = x.astype(np.float64) @ w.astype(np.float64).T
    ch = 1.0 / (1.0 + np.exp(-s64)) + (0.0 if bv is None else bv.astype(np.float64))
    srt = -np.sort(-ch, axis=1)
    gap = (srt[:, k - 1] - srt[:, k]) / np.maximum(np.abs(srt[:, k - 1]), 1e-30)
    clear = gap > 1e-5
    # as sets (two picks a few ulp apart inside the top k may swap places), weights matched
    # by expert id
    go, eo = np.argsort(gi, axis=1, kind="stable"), np.argsort(ei, axis=1, kind="stable")
    gi_s, ei_s = np.take_along_axis(gi, go, 1), np.take_along_axis(ei, eo, 1)
    gw_s, ew_s = np.take_along_axis(gw, go, 1), np.take_along_axis(ew, eo, 1)
    agree = np.all(gi_s == ei_s, axis=1)
    in_order = np.all(gi == ei, axis=1)
    say(f"  tokens {T}: clear {int(clear.sum())}, picks agree {int(agree.sum())}, same order "
        f"{int(in_order.sum())}")
    assert np.all(agree[clear])
    assert np.max(np.abs(gw_s[agree] - ew_s[agree]) /
                  np.maximum(np.abs(ew_s[agree]), 1e-30)) < 1e-5


@pytest.mark.parametrize("T,D,E,k", [(1, 7168, 384, 8), (61, 2048, 256, 6), (300, 2048, 64, 4)])
@pytest.mark.parametrize("shared", ["scores", "x"])
def test_router_workspace_shared(hip, T, D, E, k, shared):
    """choice in the memory of scores (no bias: both hold the mix) or of x, which is read
    before choice is written: the result of separate workspaces.  The split of K changes the
    sums' order only: a score by some 1e-6, and a pick where two choices are that close."""
    rng = np.random.default_rng(T + D + E)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = (rng.standard_normal((E, D)) / np.sqrt(D)).astype(np.float32)
    f32 = dict(dtype=torch.float32, device="cuda")
    wd, res = dev(w), []
    for own in (True, False):
        xd, scores = dev(x), torch.empty((T, E), **f32)
        choice = torch.empty((T, E), **f32) if own else scores if shared == "scores" else xd
        idx, wt = torch.empty((T, k), dtype=torch.int32, device="cuda"), torch.empty((T, k), **f32)
        hip.router_dev(xd, wd, None, T, D, E, k, 1.0, scores, choice, idx, wt)
        torch.cuda.synchronize()
        res.append((idx.cpu().numpy(), wt.cpu().numpy(), scores.cpu().numpy()))
    mix = 1.0 / (1.0 + np.exp(-(x.astype(np.float64) @ w.astype(np.float64).T)))
    srt = -np.sort(-mix, axis=1)
    clear = np.all((srt[:, :k] - srt[:, 1:k + 1]) / srt[:, :k] > 1e-5, axis=1)
    assert clear.any()
    for idx, wt, scores in res:
        assert np.max(np.abs(scores - mix) / mix) < 1e-5
        assert np.array_equal(idx[clear], np.argsort(-mix, axis=1)[clear, :k])
        exp = srt[:, :k] / srt[:, :k].sum(axis=1, keepdims=True)
        assert np.max(np.abs(wt - exp) / exp) < 1e-5


@pytest.mark.parametrize("fmt,O,K,n", [(0, 2048, 7168, 1), (0, 7168, 2048, 5), (0, 64, 48, 3),
                                       (4, 2048, 6144, 1), (4, 512, 1024, 40),
                                       (7, 7168, 2048, 3), (7, 256, 512, 70),
                                       (8, 2048, 7168, 1), (8, 7168, 2048, 4),
                                       (8, 7168, 7168, 1), (8, 96, 48, 37),
                                       (0, 32, 16, 1), (0, 480, 1040, 17), (0, 7200, 4112, 16),
                                       (8, 160, 4160, 33), (8, 7200, 4096, 2), (8, 32, 80, 65),
                                       (0, 4128, 80, 129), (0, 4128, 16, 300), (0, 4128, 1040, 300),
                                       (8, 4128, 144, 129), (8, 4128, 1040, 257),
                                       # a wave a tile: ragged workgroups, odd numbers of
                                       # blocks, either side of its lines
                                       (0, 160, 64, 16), (0, 12320, 304, 5), (0, 12256, 304, 5),
                                       (0, 32768, 496, 9), (0, 32800, 1008, 16), (0, 160, 64, 17),
                                       (0, 24608, 240, 32), (0, 32768, 512, 20), (0, 160, 32, 65),
                                       (0, 160, 16, 130), (0, 20512, 64, 40), (0, 49184, 80, 33),
                                       (8, 160, 64, 16), (8, 12320, 240, 7), (8, 32800, 496, 5),
                                       (8, 12288, 96, 17), (8, 32768, 240, 32), (8, 20512, 16, 40),
                                       (8, 28704, 32, 33), (8, 49184, 96, 64)])
def test_linear(hip, orc, fmt, O, K, n):
    """fmt 8 (QuantMat's int8 rows, MVLLM_DENSE_BITS=8) at K3's latent shapes, with codes
    and scales from the reference's quantizer rule (row amax / 127, clamp +-127) and an
    all-zero row (scale 0)."""
    say("linear", fmt, O, K, n)
    rng = np.random.default_rng(O + K + n + fmt)
    x = rng.standard_normal((n, K)).astype(np.float32)
    if fmt == 0:
        w = (rng.standard_normal((O, K)) * 0.05).astype(np.float32)
        sc = None
    elif fmt == 8:
        wf = (rng.standard_normal((O, K)) * 0.05).astype(np.float32)
        wf[1] = 0.0
        amax = np.abs(wf).max(axis=1)
        sc = (amax / np.float32(127.0)).astype(np.float32)
        inv = np.where(sc > 0, np.float32(1.0) / np.where(sc > 0, sc, 1), 0).astype(np.float32)
        w = np.clip(np.round(wf * inv[:, None]), -127, 127).astype(np.int8)
    else:
        e = expert_arrays(rng, fmt, K, O)   # gate: [O, K] codes and scales
        w, sc = e["gp"], e["gs"]
    y = torch.zeros((n, O), dtype=torch.float32, device="cuda")
    hip.linear_dev(fmt, dev(w), None if sc is None else dev(sc), O, K, dev(x), n, y)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    exp = orc.matmul(fmt, x, w, sc)
    err = npref.rel_err(got, exp)
    say("  rel_err", err)
    assert err < (TOL_F32 if fmt in (0, 8) else 1e-4)


def test_linear_refuses_odd_shapes(hip):
    """Shapes and formats the kernels do not take return 0 (the host runs them), with a
    message."""
    buf = torch.zeros(1 << 16, dtype=torch.float32, device="cuda")
    assert hip.lib().mvllm_hip_linear_dev(8, buf.data_ptr(), buf.data_ptr(), 100, 256,
                                          buf.data_ptr(), 1, buf.data_ptr(), None) == 0
    assert hip.lib().mvllm_hip_linear_dev(8, buf.data_ptr(), None, 256, 256,
                                          buf.data_ptr(), 1, buf.data_ptr(), None) == 0
    assert hip.lib().mvllm_hip_linear_dev(5, buf.data_ptr(), buf.data_ptr(), 256, 256,
                                          buf.data_ptr(), 1, buf.data_ptr(), None) == 0
    assert hip.lib().mvllm_hip_linear_dev(4, buf.data_ptr(), buf.data_ptr(), 100, 256,
                                          buf.data_ptr(), 1, buf.data_ptr(), None) == 0
    assert b"linear_dev" in hip.lib().mvllm_hip_last_error()


@pytest.mark.parametrize("rows,n,with_w", [(1, 7168, True), (9, 2048, True), (4, 333, False),
                                           (2, 4, True), (3, 2052, False), (2, 8192, True)])
def test_rmsnorm(hip, orc, rows, n, with_w):
    say("rmsnorm", rows, n)
    rng = np.random.default_rng(rows + n)
    x = (rng.standard_normal((rows, n)) * 3).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32) if with_w else None
    y = torch.zeros((rows, n), dtype=torch.float32, device="cuda")
    hip.rmsnorm_dev(dev(x), None if w is None else dev(w), y, rows, n, 1e-6)
    torch.cuda.synchronize()
    err = npref.rel_err(y.cpu().numpy(), orc.rmsnorm(x, w, 1e-6))
    say("  rel_err", err)
    assert err < 2e-6


@pytest.mark.parametrize("n,off", [(8196, 0), (16384, 0), (16388, 0), (2048, 1)])
def test_rmsnorm_against_64_bits(hip, n, off):
    """The last row in registers, the first in the loop, and rows that are not 16-byte
    aligned, against 64 bits (the host's sequential f32 sum is itself 2.5e-6 off at 16384).
    The register form's sum has at most 16 + 6 + 16 roundings of positive terms, the loop's
    ceil(n / 256) + 6 + 4, each 2^-24; the norm takes half of that, and four more roundings
    follow: below 2.9e-6."""
    rng = np.random.default_rng(n + off)
    x = (rng.standard_normal((2, n)) * 3).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    raw = torch.empty(2 * n + 1, device="cuda")
    xd = raw[off:off + 2 * n].view(2, n)
    xd.copy_(dev(x))
    y = torch.zeros((2, n), dtype=torch.float32, device="cuda")
    hip.rmsnorm_dev(xd, dev(w), y, 2, n, 1e-6)
    torch.cuda.synchronize()
    x64 = x.astype(np.float64)
    exp = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-6) * w
    assert npref.rel_err(y.cpu().numpy(), exp) < 2.9e-6


def test_k3_latent_chain(hip, orc):
    """K3's routed MoE around the block (src/model/kimi_k3.cpp:1973-2090) on the device:
    router on x -> top-k -> segments; z = lat_down(x) (int4); the batched block on z rows
    (MXFP4 experts, SiTU); acc -> rmsnorm(lat_n) -> lat_up (f32) -> uph.  The oracle runs
    the same chain from the device's routing (routing parity is the test above)."""
    say("k3 chain")
    rng = np.random.default_rng(2090)
    T, H, L, I, E, k = 12, 1024, 512, 256, 32, 4
    x = rng.standard_normal((T, H)).astype(np.float32)
    w_r = (rng.standard_normal((E, H)) / np.sqrt(H)).astype(np.float32)
    dn = expert_arrays(rng, 4, H, L)                      # lat_down: [L, H] int4-g64
    w_up = (rng.standard_normal((H, L)) * 0.05).astype(np.float32)   # lat_up: f32 [H, L]
    lat_n = rng.uniform(0.5, 1.5, L).astype(np.float32)
    experts = [expert_arrays(rng, 7, L, I) for _ in range(E)]
    f32 = dict(dtype=torch.float32, device="cuda")
    i32 = dict(dtype=torch.int32, device="cuda")
    # router -> segments
    scores, choice = torch.empty((T, E), **f32), torch.empty((T, E), **f32)
    idx, wt = torch.empty((T, k), **i32), torch.empty((T, k), **f32)
    hip.router_dev(dev(x), dev(w_r), None, T, H, E, k, 1.0, scores, choice, idx, wt)
    work, counts = torch.empty(2 * E + 1, **i32), torch.empty(2, **i32)
    eids, xoff, nr = (torch.empty(E, **i32) for _ in range(3))
    rows, rw = torch.empty(T * k, **i32), torch.empty(T * k, **f32)
    hip.moe_segments_dev(idx, wt, T, k, E, work, eids, xoff, nr, rows, rw, counts)
    # z = lat_down(x)
    z = torch.empty((T, L), **f32)
    hip.linear_dev(4, dev(dn["gp"]), dev(dn["gs"]), L, H, dev(x), T, z)
    torch.cuda.synchronize()
    nb, n_rows = (int(v) for v in counts.cpu())
    e_ids = eids.cpu().numpy()[:nb]
    xo, n_r = xoff.cpu().numpy()[:nb], nr.cpu().numpy()[:nb]
    rws, rwv = rows.cpu().numpy()[:n_rows], rw.cpu().numpy()[:n_rows]
    zg = z[torch.from_numpy(rws.astype(np.int64)).cuda()].contiguous()
    keep = []

    def L_(key):
        out = []
        for e in e_ids:
            t = dev(experts[int(e)][key])
            keep.append(t)
            out.append(t.data_ptr())
        return out
    acc = torch.zeros((T, L), **f32)
    hip.moe_block_dev(nb, L, I, 7, L_("gp"), L_("up"), L_("dp"), L_("gs"), L_("us"), L_("ds"),
                      zg, xo, n_r, rws, rwv, acc, T, 2, 4.0, 25.0)
    accn = torch.empty((T, L), **f32)
    hip.rmsnorm_dev(acc, dev(lat_n), accn, T, L, 1e-6)
    uph = torch.empty((T, H), **f32)
    hip.linear_dev(0, dev(w_up), None, H, L, accn, T, uph)
    torch.cuda.synchronize()
    got = uph.cpu().numpy()
    # the oracle chain, from the device's routing
    z_o = orc.matmul(4, x, dn["gp"], dn["gs"])
    ex = [experts[int(e)] for e in e_ids]
    acc_o = np.zeros((T, L), np.float32)
    assert orc.moe_block(nb, L, I, 7, [e["gp"] for e in ex], [e["up"] for e in ex],
                         [e["dp"] for e in ex], [e["gs"] for e in ex], [e["us"] for e in ex],
                         [e["ds"] for e in ex], np.ascontiguousarray(z_o[rws]), xo, n_r, rws,
                         rwv, acc_o, T, 2, 4.0, 25.0) == 1
    uph_o = orc.matmul(0, orc.rmsnorm(acc_o, lat_n, 1e-6), w_up)
    err = npref.rel_err(got, uph_o)
    say("  rel_err", err)
    assert err < 1e-4


def test_linear_int8_rows_aligned_to_four_bytes(hip, orc):
    """int8 rows whose base is only 4-byte aligned take 4 codes a load instead of 16."""
    rng = np.random.default_rng(88)
    O, K, n = 64, 256, 5
    x = rng.standard_normal((n, K)).astype(np.float32)
    w = rng.integers(-127, 128, (O, K)).astype(np.int8)
    sc = rng.uniform(0.001, 0.01, O).astype(np.float32)
    raw = torch.zeros(O * K + 16, dtype=torch.int8, device="cuda")
    raw[4:4 + O * K] = dev(w).reshape(-1)
    y = torch.zeros((n, O), dtype=torch.float32, device="cuda")
    hip.linear_dev(8, raw.data_ptr() + 4, dev(sc), O, K, dev(x), n, y)
    torch.cuda.synchronize()
    assert npref.rel_err(y.cpu().numpy(), orc.matmul(8, x, w, sc)) < TOL_F32


@pytest.mark.parametrize("fmt,O,K,n", [(4, 512, 7168, 1), (7, 256, 2304, 17), (4, 256, 2304, 100),
                                       (7, 512, 6144, 65), (4, 256, 2048, 16), (7, 256, 2048, 17),
                                       (4, 512, 1024, 32), (7, 256, 512, 64), (4, 256, 512, 65),
                                       (4, 512, 512, -5), (7, 2304, 2304, -33),
                                       # either side of the launches that stay whole
                                       (7, 32512, 2304, 17), (7, 32768, 2304, 17),
                                       (4, 40704, 2304, 3), (4, 40960, 2304, 3),
                                       (7, 40960, 4096, 2), (7, 41216, 4096, 2),
                                       # either side of the few-row launch by its workgroups
                                       (4, 8192, 256, 64), (4, 8192, 256, 65), (7, 4096, 256, 128),
                                       (7, 16384, 768, 32), (7, 16640, 768, 1), (4, 8448, 256, 48),
                                       (4, 8448, 1024, 8), (7, 8448, 1024, 9), (7, 8448, 512, 49)])
def test_linear_splits_against_64_bits(hip, fmt, O, K, n):
    """K split over workgroups (whole and ragged ranges of step pairs) and the few-row launch on
    either side of its line; n < 0: y overwrites x.  Two bf16 terms are 2^-17 of each product, the
    sums' roundings far below it: 1e-5."""
    rng = np.random.default_rng(O + K + abs(n) + fmt)
    m = abs(n)
    x = rng.standard_normal((m, K)).astype(np.float32)
    e = expert_arrays(rng, fmt, K, O)
    w = npref.dequant(fmt, e["gp"], e["gs"], K)
    xd = dev(x)
    y = xd if n < 0 else torch.zeros((m, O), dtype=torch.float32, device="cuda")
    for _ in range(2):
        xd.copy_(dev(x))
        hip.linear_dev(fmt, dev(e["gp"]), dev(e["gs"]), O, K, xd, m, y)
        torch.cuda.synchronize()
        assert npref.rel_err(y.cpu().numpy(), x.astype(np.float64) @ w.astype(np.float64).T) < 1e-5


@pytest.mark.parametrize("fmt", [4, 7])
def test_linears_wait_across_streams(hip, fmt):
    """An int4 / MXFP4 linear waits for the library's previous call on another stream, in
    every form it takes: planes (100 rows) -> few rows -> planes -> few rows, each on a stream
    of its own and reading the one before it, with a long product ahead of the first.  Equal
    bits to the same chain on one stream."""
    rng = np.random.default_rng(600 + fmt)
    shapes = [(512, 2048, 100), (2048, 512, 16), (512, 2048, 40), (256, 512, 8)]  # O, K, rows
    ws = [expert_arrays(rng, fmt, K, O) for O, K, _ in shapes]
    ws = [(dev(e["gp"]), dev(e["gs"])) for e in ws]
    x0 = dev(rng.standard_normal((100, 2048)).astype(np.float32))
    big = torch.randn(4096, 4096, device="cuda")

    def chain(streams):
        # a linear's input: the first K floats of each of its rows lie in the last output
        bufs = [x0] + [torch.zeros(100 * 2048, device="cuda") for _ in shapes]
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            p = big
            for _ in range(40):
                p = p @ big
        for i, (O, K, n) in enumerate(shapes):
            hip.linear_dev(fmt, *ws[i], O, K, bufs[i], n, bufs[i + 1], stream=streams[i])
        torch.cuda.synchronize()
        return [b.cpu().numpy() for b in bufs[1:]]

    s = [torch.cuda.Stream() for _ in shapes]
    exp = chain([s[0]] * len(shapes))
    got = chain(s)
    assert all(np.abs(e).max() > 0 for e in exp)
    for g, e in zip(got, exp):
        assert np.array_equal(g.view(np.uint32), e.view(np.uint32))


def same_nonfinite(got, exp):
    assert np.array_equal(np.isnan(got), np.isnan(exp))
    assert np.array_equal(np.isinf(got), np.isinf(exp))
    assert np.array_equal(np.sign(got[np.isinf(exp)]), np.sign(exp[np.isinf(exp)]))
    return np.isfinite(exp)


@pytest.mark.parametrize("fmt,O,K,n", [(0, 512, 2048, 5), (0, 2080, 1040, 200), (0, 96, 64, 20),
                                       (8, 512, 2048, 5), (8, 2080, 1040, 300), (8, 96, 48, 12)])
def test_linear_nonfinite_rows(hip, orc, fmt, O, K, n):
    """Inf and NaN in x (and in f32 weights, int8 row scales) through the split of K, the
    blocks through LDS (which pad K with zeros) and a wave a tile: they land where the
    reference's sums put them, in their own rows and columns."""
    rng = np.random.default_rng(O + K + n + fmt)
    x = rng.standard_normal((n, K)).astype(np.float32)
    x[1, K - 1], x[2, 0], x[n - 1, K // 2] = np.inf, np.nan, -np.inf
    if fmt == 0:
        w, sc = (rng.standard_normal((O, K)) * 0.05).astype(np.float32), None
        w[3, K - 2], w[O - 1, 5] = np.nan, np.inf
    else:
        w = rng.integers(-127, 128, (O, K)).astype(np.int8)
        w[5, K - 1] = 0  # 0 * inf
        sc = rng.uniform(0.001, 0.01, O).astype(np.float32)
        sc[7], sc[O - 1] = np.inf, np.nan
    y = torch.zeros((n, O), dtype=torch.float32, device="cuda")
    hip.linear_dev(fmt, dev(w), None if sc is None else dev(sc), O, K, dev(x), n, y)
    torch.cuda.synchronize()
    got, exp = y.cpu().numpy(), orc.matmul(fmt, x, w, sc)
    assert np.isnan(exp).any() and np.isinf(exp).any()
    fin = same_nonfinite(got, exp)
    assert npref.rel_err(got[fin], exp[fin]) < TOL_F32


@pytest.mark.parametrize("fmt", [4, 7])
@pytest.mark.parametrize("O,K,n", [(512, 512, 20), (256, 1024, 7), (512, 7168, 3), (512, 2304, 40),
                                   (256, 6144, 100)])
def test_linear_nonfinite_scales(hip, orc, fmt, O, K, n):
    """Non-finite int4 scales, ue8m0 bytes 0, 1, 254 and 255 and an infinite activation through
    the few-row launch and through K splits, whose ranges form such sums again by themselves."""
    rng = np.random.default_rng(O + K + n + fmt)
    x = rng.standard_normal((n, K)).astype(np.float32)
    x[n - 1, K - 3] = np.inf
    e = expert_arrays(rng, fmt, K, O)
    s = e["gs"]
    if fmt == 4:
        s[3, 0], s[O - 1, -1], s[40, s.shape[1] // 2] = np.inf, -np.inf, np.nan
    else:
        s[3, 0], s[O - 1, -1], s[40, s.shape[1] // 2], s[41, 1], s[42, 2] = 255, 255, 0, 1, 254
    y = torch.zeros((n, O), dtype=torch.float32, device="cuda")
    hip.linear_dev(fmt, dev(e["gp"]), dev(s), O, K, dev(x), n, y)
    torch.cuda.synchronize()
    got, exp = y.cpu().numpy(), orc.matmul(fmt, x, e["gp"], s)
    assert not np.isfinite(exp).all()
    fin = same_nonfinite(got, exp)
    rest = np.abs(exp) < 1e30  # byte 254: products of 2^127 stand apart from the rest
    assert npref.rel_err(got[fin & rest], exp[fin & rest]) < 1e-4


@pytest.mark.parametrize("T,D,E,k", [(3, 2048, 384, 8), (5, 1024, 64, 64), (40, 7168, 512, 4),
                                     (2, 64, 544, 6), (3, 64, 1024, 64)])
def test_router_nonfinite(hip, orc, T, D, E, k):
    """A bias of -inf masks experts (they are picked last, by index), +inf forces them; an
    infinite activation saturates the sigmoid; of a token of NaN activations the picks are
    distinct experts."""
    rng = np.random.default_rng(T + D + E)
    x = rng.standard_normal((T, D)).astype(np.float32)
    w = (rng.standard_normal((E, D)) / np.sqrt(D)).astype(np.float32)
    bias = (rng.standard_normal(E) * 0.05).astype(np.float32)
    bias[rng.permutation(E)[:E - min(k, E // 2)]] = -np.inf
    bias[np.nonzero(np.isfinite(bias))[0][0]] = np.inf
    x[0, 3], x[T - 1, 5] = np.inf, np.nan
    f32 = dict(dtype=torch.float32, device="cuda")
    scores, choice = torch.empty((T, E), **f32), torch.empty((T, E), **f32)
    idx, wt = torch.empty((T, k), dtype=torch.int32, device="cuda"), torch.empty((T, k), **f32)
    hip.router_dev(dev(x), dev(w), dev(bias), T, D, E, k, 2.5, scores, choice, idx, wt)
    torch.cuda.synchronize()
    gi, gw, mix = idx.cpu().numpy(), wt.cpu().numpy(), scores.cpu().numpy()
    ei, ew = orc.route(x[:T - 1], w, bias, k, 2.5)
    assert np.array_equal(np.sort(gi[:T - 1], axis=1), np.sort(ei, axis=1))
    go, eo = np.argsort(gi[:T - 1], axis=1), np.argsort(ei, axis=1)
    assert np.allclose(np.take_along_axis(gw[:T - 1], go, 1), np.take_along_axis(ew, eo, 1),
                       rtol=1e-5, atol=1e-7)
    assert np.isin(mix[0], (0.0, 1.0)).all() and np.isnan(mix[T - 1]).all()
    last = gi[T - 1]
    assert len(set(last)) == k and last.min() >= 0 and last.max() < E


@pytest.mark.parametrize("fmt,O,K,n", [(4, 512, 2048, 1), (7, 512, 2048, 16), (4, 256, 512, 64),
                                       (7, 256, 1024, 17), (7, 2048, 256, 33),
                                       # on the planes
                                       (4, 16640, 768, 1), (7, 8448, 1024, 16), (4, 8448, 2048, 16),
                                       (7, 7168, 256, 65), (4, 16640, 512, 40), (7, 10240, 1024, 32)])
def test_few_row_linear_holds_f32(hip, fmt, O, K, n):
    """Few rows of a short K enter as three exact terms, in one launch or, of many columns, on
    planes: against 64 bits on activations of all 24 bits the 2-norm error is that of at most 12
    roundings a wave's sum and 3 between waves (0.4 * 2^-24 each, the early ones less).  The
    planes hold the same: a group's products are summed smallest terms first, at most 8 groups
    follow one another in one of four sums, and 2 roundings join those (8.0e-8 measured).  Two
    terms are off by 2.5e-6, one chain of K by 1.2e-7 (int4) and 2.8e-7 (MXFP4)."""
    errs = []
    for seed in range(3):
        rng = np.random.default_rng(seed + O + K + n + fmt)
        x = rng.standard_normal((n, K)).astype(np.float32)
        e = expert_arrays(rng, fmt, K, O)
        y = torch.zeros((n, O), dtype=torch.float32, device="cuda")
        hip.linear_dev(fmt, dev(e["gp"]), dev(e["gs"]), O, K, dev(x), n, y)
        torch.cuda.synchronize()
        exp = x.astype(np.float64) @ npref.dequant(fmt, e["gp"], e["gs"], K).astype(np.float64).T
        errs.append(np.linalg.norm(y.cpu().numpy() - exp) / np.linalg.norm(exp))
    say("  errors", errs)
    assert np.mean(errs) < (1.2e-7 if O <= 2048 else 1e-7)


def test_linear_splits_workspace(hip):
    """The 32 MiB of the K splits are allocated by the first call that splits, not by one that
    does not need them; a capture before that call runs unsplit, replays give the same bits
    between eager work, and the split call agrees with 64 bits as well."""
    rng = np.random.default_rng(77)
    free = lambda: torch.cuda.mem_get_info()[0]  # noqa: E731
    mats = {}
    for O, K in ((512, 1024), (512, 7168), (256, 256)):
        e = expert_arrays(rng, 4, K, O)
        mats[O, K] = dev(e["gp"]), dev(e["gs"]), npref.dequant(4, e["gp"], e["gs"], K)
    xs = rng.standard_normal((3, 1, 7168)).astype(np.float32)
    few, x = dev(rng.standard_normal((32, 1024)).astype(np.float32)), dev(xs[0])
    out, y = torch.zeros((32, 512), device="cuda"), torch.zeros((1, 512), device="cuda")
    inplace = torch.ones((1, 256), device="cuda")
    w, s, w64 = mats[512, 7168]
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    hip.lib().mvllm_hip_shutdown()
    hip.init(0)
    before = free()
    hip.linear_dev(4, *mats[512, 1024][:2], 512, 1024, few, 32, out, stream=st)   # few rows
    hip.linear_dev(4, *mats[256, 256][:2], 256, 256, inplace, 1, inplace, stream=st)  # one K step
    torch.cuda.synchronize()
    assert before - free() < 16 << 20
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        hip.linear_dev(4, w, s, 512, 7168, x, 1, y, stream=st)
    seen = []
    for i in (0, 1, 2, 0):
        x.copy_(dev(xs[i]))
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        seen.append(y.cpu().numpy())
        assert npref.rel_err(seen[-1], xs[i].astype(np.float64) @ w64.astype(np.float64).T) < 1e-5
        hip.linear_dev(4, *mats[512, 1024][:2], 512, 1024, few, 32, out, stream=st)
    assert np.array_equal(seen[0], seen[3])
    before = free()
    hip.linear_dev(4, w, s, 512, 7168, x, 1, y, stream=st)
    torch.cuda.synchronize()
    assert before - free() >= 32 << 20
    assert npref.rel_err(y.cpu().numpy(), xs[0].astype(np.float64) @ w64.astype(np.float64).T) < 1e-5
