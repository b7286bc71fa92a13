"""GPU parity: the HIP library through its C ABI against the CPU oracle on the same seeded inputs.

Bars: ids and the dispatch permutation bit-exact; routing weights <= 1e-6 relative; layer outputs
<= 2e-3 max relative per token (tests/helpers.py).
"""
from __future__ import annotations

import os
import zlib

import numpy as np
import pytest

from oracle import oracle as O
from tests import helpers as H

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def F():
    import flashrt_amd
    flashrt_amd.lib()   # raises if the HIP library is not built
    return flashrt_amd


@pytest.fixture(scope="module")
def w0(F):
    return H.World(cfg=0)


def dev(a, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    return t.cuda() if dtype is None else t.to(dtype).cuda()


# ---------------------------------------------------------------- synthetic inputs

def test_generator_matches_oracle(F, w0):
    for e in (0, 7, 511):
        assert np.array_equal(w0.blob(e), O.gen_expert(0, 0, e, H.N, H.FF)), e
    sh = np.zeros(w0.eb, np.uint8)
    O.lib().orc_gen_expert(O.SEED, 0, 0, O.SHARED_TENSOR, H.N, H.FF, 0.02, sh)
    assert np.array_equal(w0.shared_h, sh)
    assert np.array_equal(w0.router_h.reshape(-1), O.gen_normal(0, 0, O.ROUTER_TENSOR, H.E * H.N, 0.02))
    assert np.array_equal(w0.gate_h, O.gen_normal(0, 0, O.GATE_TENSOR, H.N, 0.02))
    x = torch.empty(4096, dtype=torch.float32, device="cuda")
    F.gen.normal(x, 3, 0, O.X_TENSOR, 1.0, round_bf16=True)
    ref = O.gen_normal(3, 0, O.X_TENSOR, 4096)
    bits = ref.view(np.uint32).astype(np.uint64)
    rb = (((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32)).view(np.float32)
    assert np.array_equal(x.cpu().numpy(), rb)
    xc = torch.empty((3, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(xc, 1, 0, O.X_TENSOR, 3, H.N, 0.8)
    z0 = O.gen_normal(1, 0, O.X_TENSOR, H.N)
    a, b = np.sqrt(np.float32(0.8)), np.sqrt(np.float32(0.2))
    for t in range(3):
        zt = O.gen_normal(1, 0, O.X_TENSOR + 1 + t, H.N)
        assert np.array_equal(xc[t].cpu().numpy(), (a * z0 + b * zt).astype(np.float32))
    assert np.array_equal(F.gen.zipf_bias(2, 5, 512, 1.1), O.gen_zipf_bias(2, 5, 512, 1.1))


# ---------------------------------------------------------------- quantization and router

def test_quantize_q8_bit_exact(F):
    rng = np.random.default_rng(3)
    x = rng.standard_normal((5, 2048)).astype(np.float32)
    x[1, :32] = 0.0                  # an all-zero block: d = 0, codes 0
    x[2, 32:64] *= 1e4               # large values
    x[3, 64:96] = np.float32(-7.0)   # a constant block: codes -127
    x[4, 96:128] = np.arange(32, dtype=np.float32) * 0.5 - 8.0   # exact halves: roundf ties away from zero
    xq = torch.empty((5, 2048), dtype=torch.int8, device="cuda")
    xd = torch.empty((5, 64), dtype=torch.float32, device="cuda")
    F.quantize_q8(dev(x), 5, 2048, xq, xd)
    torch.cuda.synchronize()
    qs, d = O.quantize_q8(x)
    assert np.array_equal(xq.cpu().numpy().reshape(-1), qs)
    assert np.array_equal(xd.cpu().numpy().reshape(-1), d)


def _perm256(k):
    """Position of value k of a 256-wide stretch in the prefill operand rows: lane group g = k / 64
    holds its block's codes in the order the Q2_0 dwords unpack (code c of dword d at 2c bits)."""
    g, j = k >> 6, k & 63
    c = 4 * (j & 3) + (j >> 4)
    d = (j & 15) >> 2
    return 32 * (2 * d + ((c >> 2) & 1)) + 8 * g + 2 * (c & 3) + (c >> 3)


@pytest.mark.parametrize("rows,n,blk", [(5, 2048, 32), (3, 640, 32), (4, 2560, 64), (2, 128, 64)])
def test_quantize_pairs_exact(F, rows, n, blk):
    """The prefill GEMM's activation operand on its own: hi + lo equals the Q8_0 value q * d of the
    oracle exactly, hi is fp16(q * d) rounded to nearest even, value k of each stretch sits at
    perm256(k) (a permutation of the 256 positions), and the pad past n (rows of n rounded up to 512)
    is zero in both parts."""
    perm = np.array([_perm256(k) for k in range(256)])
    assert np.array_equal(np.sort(perm), np.arange(256))
    rng = np.random.default_rng(rows * n + blk)
    x = rng.standard_normal((rows, n)).astype(np.float32)
    x[0, :blk] = 0.0                      # a zero block
    x[-1, blk:2 * blk] *= 3e3             # large values
    np_ = (n + 511) // 512 * 512
    hi = torch.full((rows, np_), 0x7E00, dtype=torch.int16, device="cuda")   # NaN fill: every position written
    lo = torch.full((rows, np_), 0x7E00, dtype=torch.int16, device="cuda")
    F.quantize_pairs(dev(x), rows, n, blk, hi, lo)
    torch.cuda.synchronize()
    h = hi.cpu().numpy().view(np.float16).reshape(rows, np_ // 256, 256)
    l_ = lo.cpu().numpy().view(np.float16).reshape(rows, np_ // 256, 256)
    h, l_ = h[:, :, perm].reshape(rows, np_), l_[:, :, perm].reshape(rows, np_)   # back to value order
    qs, d = O.quantize_q8(x, blk)
    a = (qs.astype(np.float64) * np.repeat(d, 32).astype(np.float64)).reshape(rows, n)
    assert np.array_equal(h[:, :n].astype(np.float64) + l_[:, :n].astype(np.float64), a)
    assert np.array_equal(h[:, :n], a.astype(np.float32).astype(np.float16))
    assert not np.any(h[:, n:]) and not np.any(l_[:, n:])


@pytest.mark.parametrize("T,n,with_bias", [(1, 2048, False), (3, 2048, True), (17, 2048, True), (5, 2560, False)])
def test_router_logits_bit_exact(F, T, n, with_bias):
    E = 512
    rng = np.random.default_rng(T * 7 + n)
    x = rng.standard_normal((T, n)).astype(np.float32)
    W = (rng.standard_normal((E, n)) * 0.02).astype(np.float32)
    g = (rng.standard_normal(n) * 0.02).astype(np.float32)
    bias = (rng.standard_normal(E)).astype(np.float32) if with_bias else None
    lg = torch.empty((T, E), dtype=torch.float32, device="cuda")
    gt = torch.empty(T, dtype=torch.float32, device="cuda")
    F.router_logits(dev(x), T, dev(W), E, n, lg, bias=None if bias is None else dev(bias), gate_w=dev(g), gate=gt)
    torch.cuda.synchronize()
    ref = O.router_logits(x, W, bias)
    assert np.array_equal(lg.cpu().numpy(), ref)
    gref = np.array([O.dot_canon(g, x[t]) for t in range(T)], np.float32)
    assert np.array_equal(gt.cpu().numpy(), gref)


@pytest.mark.parametrize("n", [512, 1024, 4096])
@pytest.mark.parametrize("T", [1, 3, 4, 5, 6, 8, 16, 17])
def test_router_logits_small_calls(F, T, n):
    """Either side of the rule that gives a router row two waves (from 4 tokens and 3072 values on, within
    one token tile: 16 tokens, 5 at n = 4096): logits and gate bit for bit the oracle's, on an odd row count."""
    E = 33
    rng = np.random.default_rng(T * 11 + n)
    x = rng.standard_normal((T, n)).astype(np.float32)
    W = (rng.standard_normal((E, n)) * 0.02).astype(np.float32)
    g = (rng.standard_normal(n) * 0.02).astype(np.float32)
    lg = torch.full((T, E), float("nan"), dtype=torch.float32, device="cuda")
    gt = torch.full((T,), float("nan"), dtype=torch.float32, device="cuda")
    F.router_logits(dev(x), T, dev(W), E, n, lg, gate_w=dev(g), gate=gt)
    torch.cuda.synchronize()
    assert np.array_equal(lg.cpu().numpy(), O.router_logits(x, W, None))
    assert np.array_equal(gt.cpu().numpy(), np.array([O.dot_canon(g, x[t]) for t in range(T)], np.float32))


@pytest.mark.parametrize("T,n,with_bias", [(300, 2048, True), (2048, 2048, False), (70, 2560, True), (64, 1024, False),
                                            (100, 512, True), (65, 1536, False), (40, 3584, True)])
def test_router_logits_gemm_bit_exact(F, T, n, with_bias):
    """The prefill router GEMM (K split along the canonical tree; the chains on the matrix cores,
    whose f32 MFMA accumulates its four products as a chain of fmas in K order) equals the oracle's
    canonical order bit for bit, and the VALU kernel of the same GEMM equals it too."""
    E = 512
    rng = np.random.default_rng(T + n)
    x = rng.standard_normal((T, n)).astype(np.float32)
    W = (rng.standard_normal((E, n)) * 0.02).astype(np.float32)
    g = (rng.standard_normal(n) * 0.02).astype(np.float32)
    bias = (rng.standard_normal(E)).astype(np.float32) if with_bias else None
    ref = O.router_logits(x, W, bias)
    gref = np.array([O.dot_canon(g, x[t]) for t in range(T)], np.float32)
    for mfma in (1, 0):
        F.set_option("router_mfma", mfma)
        try:
            lg = torch.full((T, E), float("nan"), dtype=torch.float32, device="cuda")
            gt = torch.full((T,), float("nan"), dtype=torch.float32, device="cuda")
            F.router_logits_gemm(dev(x), T, dev(W), E, n, lg, bias=None if bias is None else dev(bias), gate_w=dev(g), gate=gt)
            torch.cuda.synchronize()
        finally:
            F.set_option("router_mfma", 1)
        assert np.array_equal(lg.cpu().numpy(), ref), mfma
        assert np.array_equal(gt.cpu().numpy(), gref), mfma


# ---------------------------------------------------------------- routing

def _route_gpu(F, lg, K, tail_from=1 << 30):
    T, E = lg.shape
    ids = torch.full((T, K), -1, dtype=torch.int32, device="cuda")
    w = torch.zeros((T, K), dtype=torch.float32, device="cuda")
    cnt = torch.zeros(E, dtype=torch.int32, device="cuda")
    tail = torch.zeros(E, dtype=torch.int32, device="cuda")
    F.moe_route_topk(None, dev(lg), T, E, K, ids, w, cnt, tail, tail_from)
    torch.cuda.synchronize()
    return ids.cpu().numpy(), w.cpu().numpy(), cnt.cpu().numpy(), tail.cpu().numpy()


def test_route_topk_reference_recipe(F):
    """tests/test_route_topk.cpp:22-69: T 16384, E 512, K 10, logits round(N(0,2)*4)/4 (many exact
    ties); ids == stable sort by logit, counts exact, weights vs a double softmax. The normals come
    from this build's generator (the reference draws std::mt19937 + libstdc++'s normal)."""
    T, E, K = 16384, 512, 10
    lg = (np.round(O.gen_normal(9, 0, 1, T * E, 2.0) * 4.0) / 4.0).astype(np.float32).reshape(T, E)
    ids, w, cnt, tail = _route_gpu(F, lg, K, tail_from=T - 100)
    oid, ow, ocnt = O.route_topk(lg, K)
    assert np.array_equal(ids, oid)
    assert np.array_equal(cnt.astype(np.uint32), ocnt)
    assert H.w_rel(w, ow) <= H.W_REL
    # the reference test's own definition: stable sort by logit, double softmax, < 1e-5 abs
    idx = np.argsort(-lg, axis=1, kind="stable")[:, :K]
    assert np.array_equal(ids, idx)
    mx = lg.max(axis=1, keepdims=True).astype(np.float64)
    p = np.exp(lg.astype(np.float64) - mx)
    p /= p.sum(axis=1, keepdims=True)
    ps = np.take_along_axis(p, idx, axis=1)
    assert np.abs(w - ps / ps.sum(axis=1, keepdims=True)).max() < 1e-5
    tref = np.bincount(oid[T - 100:].reshape(-1), minlength=E)
    assert np.array_equal(tail, tref)


@pytest.mark.parametrize("T,E,K", [(1, 512, 10), (3, 64, 1), (5, 1000, 32), (7, 1024, 8), (33, 96, 10)])
def test_route_topk_shapes(F, T, E, K):
    rng = np.random.default_rng(E + K)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    lg[0, :8] = 3.0   # exact ties at the top
    ids, w, cnt, _ = _route_gpu(F, lg, K)
    oid, ow, ocnt = O.route_topk(lg, K)
    assert np.array_equal(ids, oid)
    assert np.array_equal(cnt.astype(np.uint32), ocnt)
    assert H.w_rel(w, ow) <= H.W_REL


def test_route_topk_errors(F):
    lg = torch.zeros((2, 2048), dtype=torch.float32, device="cuda")
    ids = torch.zeros((2, 10), dtype=torch.int32, device="cuda")
    w = torch.zeros((2, 10), dtype=torch.float32, device="cuda")
    with pytest.raises(F.FrtError) as e:
        F.moe_route_topk(None, lg, 2, 2048, 10, ids, w)
    assert e.value.code == -1
    with pytest.raises(F.FrtError):
        F.moe_route_topk(None, lg, 2, 512, 33, ids, w)
    F.moe_route_topk(None, lg, 0, 512, 10, ids, w)   # T = 0: nothing to do


# ---------------------------------------------------------------- dispatch

@pytest.mark.parametrize("T,skew", [(1, 0.0), (3, 0.0), (2048, 1.2), (2457, 0.0), (8208, 3.0)])
def test_dispatch_bit_exact(F, T, skew):
    E, K = 512, 10
    rng = np.random.default_rng(T)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    if skew:
        lg += O.gen_zipf_bias(3, 0, E, skew)[None, :]
    ids, _, _ = O.route_topk(lg, K)
    b = torch.empty(E + 1, dtype=torch.int32, device="cuda")
    to = torch.empty(T * K, dtype=torch.int32, device="cuda")
    so = torch.empty(T * K, dtype=torch.int32, device="cuda")
    F.moe_dispatch(dev(ids), T, K, E, b, to, so)
    torch.cuda.synchronize()
    rb, rt, rs = O.dispatch(ids, E)
    assert np.array_equal(b.cpu().numpy(), rb)
    assert np.array_equal(so.cpu().numpy(), rs)
    assert np.array_equal(to.cpu().numpy(), rt)
    # a stable sort of (expert, slot), the definition in kernels/cuda/moe_q2.cu:83-168
    assert np.array_equal(rs, np.argsort(ids.reshape(-1), kind="stable"))


@pytest.mark.parametrize("T,E,K", [(1, 1, 1), (9, 3, 2), (37, 512, 10), (100, 1000, 32), (409, 1024, 10), (410, 512, 10),
                                   (4096, 7, 1), (4097, 7, 1)])
def test_dispatch_short_chunk(F, T, E, K):
    """Either side of the one-workgroup dispatch's limits (4096 slots, 1024 experts; batches of 64 slots per
    wave, empty waves): bounds, slots and tokens exactly those of the stable sort."""
    rng = np.random.default_rng(T + E)
    ids = np.stack([rng.permutation(E)[:K] for _ in range(T)]).astype(np.int32)
    b = torch.empty(E + 1, dtype=torch.int32, device="cuda")
    to = torch.empty(T * K, dtype=torch.int32, device="cuda")
    so = torch.empty(T * K, dtype=torch.int32, device="cuda")
    F.moe_dispatch(dev(ids), T, K, E, b, to, so)
    torch.cuda.synchronize()
    order = np.argsort(ids.reshape(-1), kind="stable")
    assert np.array_equal(b.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(ids.reshape(-1), minlength=E))]))
    assert np.array_equal(so.cpu().numpy(), order)
    assert np.array_equal(to.cpu().numpy(), order // K)


# ---------------------------------------------------------------- decode path (T <= 4)

def test_layer_decode_config0(F, w0):
    x = O.gen_normal(0, 0, O.X_TENSOR, H.N).reshape(1, H.N)
    out, ids, wts = w0.gpu_forward(x)
    ref, rid, rw, _ = w0.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL


@pytest.mark.parametrize("T", [1, 2, 8])
@pytest.mark.parametrize("E", [300, 128, 1000, 1024])
def test_layer_decode_other_expert_counts(F, E, T):
    """Decode routing with other expert counts. Each lane holds V consecutive logits (V = 8 for
    E <= 512, 16 above): E = 128 fills 16 lanes, 300 ends inside a lane (clamped loads, tail past
    E), 1000 and 1024 take the V = 16 selection. T = 1 runs the single-token selection, T = 2 and 8
    the window path's per-token selection (k_win_route) and its combine in the down kernel. Ids, weights and output against the oracle (the reference routes any E up to
    its kernel's bound, blocks.hpp:130-135)."""
    w = H.World(cfg=0, E=E)
    rng = np.random.default_rng(E + T)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    out, ids, wts = w.gpu_forward(x)
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL


def test_layer_reference_test_shape(F):
    """The reference tests' shape, d_model 2560 and expert ff 640 (tests/test_moe_q2.cpp:68-153),
    through the whole layer: decode at T = 1 and 3 and prefill at T = 128, every token's ids,
    weights and outputs against the oracle."""
    w = H.World(cfg=0, n=2560, ff=640)
    rng = np.random.default_rng(2560)
    for T in (1, 3, 128):
        x = rng.standard_normal((T, 2560)).astype(np.float32)
        out, ids, wts = w.gpu_forward(x)
        ref, rid, rw, _ = w.oracle_forward(x)
        assert np.array_equal(ids, rid), T
        assert H.w_rel(wts, rw) <= H.W_REL, T
        assert H.out_rel(out, ref) <= H.OUT_REL, T


@pytest.mark.parametrize("min_t", [2, 9])
def test_layer_decode_config1_window(F, min_t):
    """Config 1 (3 correlated tokens) through the window path (the default) and, with the window
    path switched off (window_min_t = 9), through the grouped decode kernels (four-wave routing in
    every gate/up workgroup, the combine lists in k_dec_down)."""
    w1 = H.World(cfg=1)
    xc = torch.empty((3, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(xc, 1, 0, O.X_TENSOR, 3, H.N, 0.8)
    x = xc.cpu().numpy()
    F.set_option("window_min_t", min_t)
    try:
        out, ids, wts = w1.gpu_forward(x)
    finally:
        F.set_option("window_min_t", 2)
    ref, rid, rw, _ = w1.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL
    # overlapping routes: the window reads fewer than 3 * 10 distinct experts
    assert len(set(ids.reshape(-1).tolist())) < 30
    # each token alone (the single-token path) selects the same experts and gives the same outputs
    # within the output bar (the window path forms the routing weights with the top-k kernel's
    # formula, so they can differ from the single-token path's in the last bits; the moe_hits
    # window itself equals its one-token calls bit for bit, test_moe_hits)
    for t in range(3):
        o1, i1, _ = w1.gpu_forward(x[t:t + 1])
        assert np.array_equal(i1[0], ids[t])
        assert H.out_rel(o1, out[t:t + 1]) <= H.OUT_REL


@pytest.mark.parametrize("T", [2, 3, 4])
def test_layer_window_persistent(F, T):
    """Windows of 2-4 tokens as one persistent launch (decodew.hip, the default where the shape fits)
    against the oracle and against the four-launch window path (option decode_window_persistent = 0):
    the same ids, outputs within the output bar of the oracle and equal to the four-launch path's bit
    for bit, the residual added exactly, the same bits on a second call, and the routing records
    (counts) of the window."""
    w1 = H.World(cfg=1)
    xc = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(xc, 1, 7, O.X_TENSOR, T, H.N, 0.8)
    x = xc.cpu().numpy()
    out, ids, wts = w1.gpu_forward(x)
    ref, rid, rw, _ = w1.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    err = H.out_rel(out, ref)
    print(f"persistent window T={T}: out rel err {err:.2e}, {len(set(ids.reshape(-1).tolist()))} distinct experts")
    assert err <= H.OUT_REL
    again = w1.gpu_forward(x)
    for a_, b_ in zip(again, (out, ids, wts)):
        assert np.array_equal(a_, b_)
    F.set_option("decode_window_persistent", 0)
    try:
        o4, i4, w4 = w1.gpu_forward(x)
    finally:
        F.set_option("decode_window_persistent", 1)
    assert np.array_equal(i4, ids)
    assert H.out_rel(o4, ref) <= H.OUT_REL
    # the same arithmetic in the same order as the four launches: the same bits
    assert np.array_equal(out, o4) and np.array_equal(wts, w4)
    r = O.gen_normal(1, 0, O.X_TENSOR + 9, T * H.N).reshape(T, H.N)
    out_r, _, _ = w1.gpu_forward(x, resid=r)
    assert np.array_equal(out_r, (r + out).astype(np.float32))
    counts = torch.zeros(H.E, dtype=torch.int32, device="cuda")
    xd = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    o = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    w1.layer_obj.forward(xd, o, T=T, counts=counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), np.bincount(ids.reshape(-1), minlength=H.E))


@pytest.mark.parametrize("path", ["T1", "T1_xcd", "T3", "T3_four_launch", "T6"])
def test_decode_h_in_cpu_order(F, path):
    """The decode paths sum each gate/up row's block terms in the CPU path's order (matvec_ref), so h
    takes the CPU's Q8 codes and the layer output differs from the oracle only by the order of the down
    and combine sums (~1e-7 relative). A pairwise tree moved h codes across Q8 boundaries on 2.6% of
    1000 single tokens (K = 4; 5.3% at K = 10), up to 2.5e-3 relative; in order, 1000 seeds gave at most
    1.9e-5. Here: 40 seeded windows per path, K = 4 (fewest experts, largest weight per flipped code),
    every token within 1e-4 of the oracle, ids bit-exact."""
    T = int(path.split("_")[0][1:])
    opts = {"T1_xcd": {"decode_xcd": 1}, "T3_four_launch": {"decode_window_persistent": 0}}.get(path, {})
    w = H.World(cfg=0, K=4)
    worst = 0.0
    try:
        for k, v in opts.items():
            F.set_option(k, v)
        for seed in range(40):
            x = np.random.default_rng(1000 + seed).standard_normal((T, w.n)).astype(np.float32)
            out, ids, wts = w.gpu_forward(x)
            ref, rid, rw, _ = w.oracle_forward(x)
            assert np.array_equal(ids, rid), seed
            worst = max(worst, H.out_rel(out, ref))
    finally:
        for k in opts:
            F.set_option(k, 1 if k == "decode_window_persistent" else 0)
    print(f"{path}: worst out rel err over 40 windows {worst:.2e}")
    assert worst <= 1e-4


@pytest.mark.parametrize("T", [5, 8])
def test_layer_verify_window(F, T):
    """Verify windows of 5 and 8 tokens (the reference's kMaxWindow = 8, moe_fast.cu:38; correlated
    tokens as in config 1) through the decode GEMV path (router with fused Q8_0, top-k, one moe_hits
    launch over every token's routed experts and the shared expert, combine): ids bit-exact, weights
    and outputs against the oracle; each token alone (the single-token path) gives the same ids and
    outputs within the output bar; a window with a residual adds it exactly."""
    w1 = H.World(cfg=1)
    xc = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(xc, 1, T, O.X_TENSOR, T, H.N, 0.8)
    x = xc.cpu().numpy()
    out, ids, wts = w1.gpu_forward(x)
    ref, rid, rw, _ = w1.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    err = H.out_rel(out, ref)
    print(f"verify window T={T}: out rel err {err:.2e}, {len(set(ids.reshape(-1).tolist()))} distinct experts")
    assert err <= H.OUT_REL
    for t in (0, T - 1):
        o1, i1, _ = w1.gpu_forward(x[t:t + 1])
        assert np.array_equal(i1[0], ids[t])
        assert H.out_rel(o1, out[t:t + 1]) <= H.OUT_REL
    r = O.gen_normal(1, 0, O.X_TENSOR + 9, T * H.N).reshape(T, H.N)
    out_r, _, _ = w1.gpu_forward(x, resid=r)
    assert np.array_equal(out_r, (r + out).astype(np.float32))


def test_layer_decode_resid(F, w0):
    x = O.gen_normal(0, 0, O.X_TENSOR + 5, 2 * H.N).reshape(2, H.N)
    r = O.gen_normal(0, 0, O.X_TENSOR + 6, 2 * H.N).reshape(2, H.N)
    out, _, _ = w0.gpu_forward(x)
    out_r, _, _ = w0.gpu_forward(x, resid=r)
    assert np.array_equal(out_r, (r + out).astype(np.float32))


ENVELOPE = [(1536, 768), (512, 2048), (4096, 4096)]


@pytest.mark.parametrize("n,ff", ENVELOPE)
def test_moe_hits_envelope(F, n, ff):
    """moe_hits at shapes of the reference's envelope outside the templated kernels (n % 512 == 0,
    ff % 64 == 0, ff <= 4096; arch/qwen4exp/moe_fast.cu:557): T = 1 and 3 tokens (a blob shared by
    two tokens, pad slots untouched), every written slot within 2e-3 of the oracle's expert_ffn;
    shapes the reference refuses are refused (FRT_ERR_SHAPE)."""
    E, K = 12, 4
    w = H.World(cfg=0, n=n, ff=ff, E=E, K=K)
    rng = np.random.default_rng(n + ff)
    for T in (1, 3):
        x = rng.standard_normal((T, n)).astype(np.float32)
        hit_n = np.array([K, K - 1, 2][:T], np.int32)
        experts = np.stack([rng.choice(E, size=K, replace=False) for _ in range(T)]).astype(np.int64)
        if T > 1:
            experts[1, 0] = experts[0, 0]
        ptr = torch.tensor((w.arena.data_ptr() + experts * w.stride).reshape(-1), dtype=torch.int64, device="cuda")
        yh = torch.full((T, K, n), float("nan"), dtype=torch.float32, device="cuda")
        scratch = torch.empty(F.moe_hits_scratch_bytes(K, ff, T), dtype=torch.uint8, device="cuda")
        F.moe_hits(ptr, dev(hit_n), K, dev(x), n, ff, scratch, yh, T=T)
        torch.cuda.synchronize()
        y = yh.cpu().numpy()
        for t in range(T):
            for k in range(K):
                if k >= hit_n[t]:
                    assert np.isnan(y[t, k]).all()
                    continue
                ref = O.expert_ffn(w.blob(int(experts[t, k])), n, ff, x[t])
                assert H.out_rel(y[t, k][None], ref) <= H.OUT_REL, (n, ff, T, t, k)
    x = torch.zeros((1, 1000), dtype=torch.float32, device="cuda")
    ptr = torch.tensor([w.arena.data_ptr()], dtype=torch.int64, device="cuda")
    one = torch.ones(1, dtype=torch.int32, device="cuda")
    yh = torch.empty((1, 1, 4096), dtype=torch.float32, device="cuda")
    scratch = torch.empty(1 << 24, dtype=torch.uint8, device="cuda")
    for bad_n, bad_ff in ((1000, ff), (n, 4160), (n, 96), (768, ff)):
        with pytest.raises(F.FrtError) as e:
            F.moe_hits(ptr, one, 1, x, bad_n, bad_ff, scratch, yh, T=1)
        assert e.value.code == -1, (bad_n, bad_ff)


@pytest.mark.parametrize("n,ff", ENVELOPE)
def test_layer_envelope_decode(F, n, ff):
    """Whole layers at those shapes for T = 1 and 3 (router, routing, the routed experts and the Q2_0
    shared expert through moe_hits, combine): ids bit-exact, weights 1e-6, outputs within 2e-3 of
    the oracle."""
    w = H.World(cfg=0, n=n, ff=ff, E=16, K=4)
    rng = np.random.default_rng(3 * n + ff)
    for T in (1, 3):
        x = rng.standard_normal((T, n)).astype(np.float32)
        out, ids, wts = w.gpu_forward(x)
        ref, rid, rw, _ = w.oracle_forward(x)
        assert np.array_equal(ids, rid), (n, ff, T)
        assert H.w_rel(wts, rw) <= H.W_REL
        assert H.out_rel(out, ref) <= H.OUT_REL, (n, ff, T)


@pytest.mark.parametrize("n,ff", ENVELOPE)
def test_moe_q2_run_envelope(F, n, ff):
    """moe_q2::run at those shapes, T = 200 (800 slots, tiles of up to 16 tokens): sampled slots within 2e-3 of
    the oracle's expert_ffn; bf16 yd with ff above 1024 and ff above 4096 are refused (FRT_ERR_SHAPE)."""
    T, K, E = 200, 4, 12
    w = H.World(cfg=0, n=n, ff=ff, E=E, K=K)
    rng = np.random.default_rng(7 * n + ff)
    x = rng.standard_normal((T, n)).astype(np.float32)
    ids = np.stack([rng.choice(E, size=K, replace=False) for _ in range(T)]).astype(np.int32)
    nb = F.moe_q2.workspace_bytes(T, K, n, ff, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T * K, n), float("nan"), dtype=torch.float32, device="cuda")
    F.moe_q2.run(w.arena.data_ptr(), w.stride, E, n, ff, dev(x), dev(ids), T, K, yd, ws, nb)
    torch.cuda.synchronize()
    y = yd.cpu().numpy().reshape(T, K, n)
    assert np.isfinite(y).all()
    for t in range(0, T, 23):
        for k in range(K):
            ref = O.expert_ffn(w.blob(int(ids[t, k])), n, ff, x[t])
            assert H.out_rel(y[t, k][None], ref) <= H.OUT_REL, (n, ff, t, k)
    if ff > 1024:
        yb = torch.empty((T * K, n), dtype=torch.bfloat16, device="cuda")
        with pytest.raises(F.FrtError) as e:
            F.moe_q2.run(w.arena.data_ptr(), w.stride, E, n, ff, dev(x), dev(ids), T, K, yb, ws, nb, None, False, True)
        assert e.value.code == -1
    with pytest.raises(F.FrtError) as e:
        F.moe_q2.workspace_bytes(T, K, n, 4224, E)
        F.moe_q2.run(w.arena.data_ptr(), w.stride, E, n, 4224, dev(x), dev(ids), T, K, yd, ws, nb)
    assert e.value.code in (-1, -2)


@pytest.mark.parametrize("n,ff", ENVELOPE)
def test_layer_envelope_prefill(F, n, ff):
    """Whole layers at those shapes for a 200-token chunk (router GEMM, routing, the grouped GEMMs
    with the shared expert as group E, combine): ids bit-exact, weights 1e-6, outputs 2e-3."""
    w = H.World(cfg=0, n=n, ff=ff, E=16, K=4)
    x = np.random.default_rng(5 * n + ff).standard_normal((200, n)).astype(np.float32)
    out, ids, wts = w.gpu_forward(x)
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid), (n, ff)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL, (n, ff)


def test_moe_hits(F, w0):
    """tests/test_moe_hits.cpp:42-166: per-slot expert outputs; pad entries (k >= hit_n) untouched."""
    T, K = 3, 16
    rng = np.random.default_rng(7)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    hit_n = np.array([9, 16, 1], np.int32)
    experts = rng.choice(512, size=(T, K), replace=True).astype(np.int64)
    experts[1, :4] = experts[0, :4]   # shared across tokens of the window
    base = w0.arena.data_ptr()
    ptr = torch.tensor((base + experts * w0.stride).reshape(-1), dtype=torch.int64, device="cuda")
    yh = torch.full((T, K, H.N), float("nan"), dtype=torch.float32, device="cuda")
    scratch = torch.empty(F.moe_hits_scratch_bytes(K, H.FF, T), dtype=torch.uint8, device="cuda")
    F.moe_hits(ptr, dev(hit_n), K, dev(x), H.N, H.FF, scratch, yh, T=T)
    torch.cuda.synchronize()
    y = yh.cpu().numpy()
    for t in range(T):
        for k in range(K):
            if k >= hit_n[t]:
                assert np.isnan(y[t, k]).all()
                continue
            ref = O.expert_ffn(w0.blob(int(experts[t, k])), H.N, H.FF, x[t])
            assert H.out_rel(y[t, k][None], ref) <= H.OUT_REL
    # window == one-token calls, exactly
    for t in range(T):
        y1 = torch.full((1, K, H.N), float("nan"), dtype=torch.float32, device="cuda")
        F.moe_hits(ptr[t * K:(t + 1) * K], dev(hit_n[t:t + 1]), K, dev(x[t:t + 1]), H.N, H.FF, scratch, y1, T=1)
        torch.cuda.synchronize()
        a = y1.cpu().numpy()[0, :hit_n[t]]
        assert np.array_equal(a, y[t, :hit_n[t]])


def test_moe_hits_repeated_blob(F, w0):
    """One blob hit more often in a window than one grouped entry holds (four token slots): twice
    by token 0 and once by each of tokens 1-3, plus a token listing another blob three times. Every
    slot against the oracle (the reference's k_moe_group keeps one slot per (expert, token),
    moe_fast.cu:195-232), pad slots untouched."""
    T, K = 4, 8
    rng = np.random.default_rng(21)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    hit_n = np.array([8, 6, 7, 8], np.int32)
    experts = rng.choice(512, size=(T, K), replace=True).astype(np.int64)
    experts[0, 1] = experts[0, 5] = experts[1, 0] = experts[2, 6] = experts[3, 3] = 77
    experts[3, 0] = experts[3, 4] = experts[3, 7] = 300
    base = w0.arena.data_ptr()
    ptr = torch.tensor((base + experts * w0.stride).reshape(-1), dtype=torch.int64, device="cuda")
    yh = torch.full((T, K, H.N), float("nan"), dtype=torch.float32, device="cuda")
    scratch = torch.empty(F.moe_hits_scratch_bytes(K, H.FF, T), dtype=torch.uint8, device="cuda")
    F.moe_hits(ptr, dev(hit_n), K, dev(x), H.N, H.FF, scratch, yh, T=T)
    torch.cuda.synchronize()
    y = yh.cpu().numpy()
    for t in range(T):
        assert np.isnan(y[t, hit_n[t]:]).all()
        for k in range(hit_n[t]):
            ref = O.expert_ffn(w0.blob(int(experts[t, k])), H.N, H.FF, x[t])
            assert H.out_rel(y[t, k][None], ref) <= H.OUT_REL, (t, k)
    assert np.array_equal(y[0, 1], y[0, 5])
    assert np.array_equal(y[3, 0], y[3, 4]) and np.array_equal(y[3, 0], y[3, 7])


@pytest.mark.parametrize("T,K", [(8, 10), (5, 32)])
def test_moe_hits_long_windows(F, w0, T, K):
    """Windows up to the reference's kMaxWindow (T = 8, moe_fast.cu:38) in one grouped launch (K = 10:
    three experts hit by all 8 tokens, so each opens a second entry after four tokens); with K = 32 a
    launch holds four tokens and the window runs in two. Every slot against the oracle, pad slots
    untouched, and each token equal to its one-token call bit for bit."""
    rng = np.random.default_rng(T * K)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    hit_n = rng.integers(1, K + 1, size=T).astype(np.int32)
    experts = rng.choice(512, size=(T, K), replace=True).astype(np.int64)
    experts[1:, :3] = experts[0, :3]   # shared across the window's chunks
    base = w0.arena.data_ptr()
    ptr = torch.tensor((base + experts * w0.stride).reshape(-1), dtype=torch.int64, device="cuda")
    yh = torch.full((T, K, H.N), float("nan"), dtype=torch.float32, device="cuda")
    scratch = torch.empty(F.moe_hits_scratch_bytes(K, H.FF, T), dtype=torch.uint8, device="cuda")
    F.moe_hits(ptr, dev(hit_n), K, dev(x), H.N, H.FF, scratch, yh, T=T)
    torch.cuda.synchronize()
    y = yh.cpu().numpy()
    for t in range(T):
        assert np.isnan(y[t, hit_n[t]:]).all()
        for k in range(hit_n[t]):
            ref = O.expert_ffn(w0.blob(int(experts[t, k])), H.N, H.FF, x[t])
            assert H.out_rel(y[t, k][None], ref) <= H.OUT_REL, (t, k)
        y1 = torch.full((1, K, H.N), float("nan"), dtype=torch.float32, device="cuda")
        F.moe_hits(ptr[t * K:(t + 1) * K], dev(hit_n[t:t + 1]), K, dev(x[t:t + 1]), H.N, H.FF, scratch, y1, T=1)
        torch.cuda.synchronize()
        assert np.array_equal(y1.cpu().numpy()[0, :hit_n[t]], y[t, :hit_n[t]]), t


def test_router_widen_gguf_types(F):
    """Router / gate tensors in the GGUF types a model ships (ggml F32, F16, BF16, Q8_0 blocks
    {fp16 d; int8 q[32]}) widen to fp32 exactly: against numpy's exact conversions; an unsupported
    type and a Q8_0 count off the block size fail loudly."""
    rng = np.random.default_rng(30)
    n = 512 * 64
    ref = (rng.standard_normal(n) * 0.02).astype(np.float32)
    out = torch.full((n,), float("nan"), dtype=torch.float32, device="cuda")
    h16 = ref.astype(np.float16)
    F.router_widen(torch.from_numpy(h16.view(np.uint8).copy()).cuda(), F.GGML_F16, n, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), h16.astype(np.float32))
    b16 = (ref.view(np.uint32) >> 16).astype(np.uint16)   # truncation: any bf16 bit pattern
    F.router_widen(torch.from_numpy(b16.view(np.uint8).copy()).cuda(), F.GGML_BF16, n, out)
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint32), b16.astype(np.uint32) << 16)
    nb = n // 32
    d = (np.abs(rng.standard_normal(nb)) * 1e-3).astype(np.float16)
    q = rng.integers(-127, 128, size=(nb, 32)).astype(np.int8)
    blocks = np.zeros((nb, 34), np.uint8)
    blocks[:, :2] = d.view(np.uint8).reshape(nb, 2)
    blocks[:, 2:] = q.view(np.uint8)
    F.router_widen(torch.from_numpy(blocks.reshape(-1)).cuda(), F.GGML_Q8_0, n, out)
    torch.cuda.synchronize()
    want = (d.astype(np.float32)[:, None] * q.astype(np.float32)).reshape(-1)
    assert np.array_equal(out.cpu().numpy(), want)
    src32 = torch.from_numpy(ref).cuda()
    F.router_widen(src32, F.GGML_F32, n, out)
    torch.cuda.synchronize()
    assert torch.equal(out, src32)
    with pytest.raises(F.FrtError):
        F.router_widen(src32, 2, n, out)          # Q4_0: not a router type here
    with pytest.raises(F.FrtError):
        F.router_widen(src32, F.GGML_Q8_0, 33, out)


# ---------------------------------------------------------------- prefill path

@pytest.mark.parametrize("yd_bf16", [False, True])
def test_moe_q2_run(F, w0, yd_bf16):
    """tests/test_moe_q2.cpp:97-153 shape: T = 96 tokens over 24 experts; per-slot outputs vs the
    oracle's expert_ffn (bf16 output: within bf16 rounding, 2^-8 relative)."""
    T, K, E = 96, 10, 24
    rng = np.random.default_rng(96)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    ids = np.stack([rng.choice(E, size=K, replace=False) for _ in range(T)]).astype(np.int32)
    nb = F.moe_q2.workspace_bytes(T, K, H.N, H.FF, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T * K, H.N), float("nan"), dtype=torch.bfloat16 if yd_bf16 else torch.float32, device="cuda")
    F.moe_q2.run(w0.arena.data_ptr(), w0.stride, E, H.N, H.FF, dev(x), dev(ids), T, K, yd, ws, nb, None, False, yd_bf16)
    torch.cuda.synchronize()
    y = yd.float().cpu().numpy().reshape(T, K, H.N)
    tol = 2 ** -8 if yd_bf16 else H.OUT_REL
    for t in range(0, T, 5):
        for k in range(K):
            ref = O.expert_ffn(w0.blob(int(ids[t, k])), H.N, H.FF, x[t])
            err = H.out_rel(y[t, k][None], ref)
            assert err <= tol, (t, k, err)
    with pytest.raises(F.FrtError) as e:
        F.moe_q2.run(w0.arena.data_ptr(), w0.stride, E, H.N, H.FF, dev(x), dev(ids), T, K, yd, ws, 4096)
    assert e.value.code == -2


@pytest.mark.parametrize("n,ff,T,K,E", [(2048, 512, 96, 10, 24), (640, 384, 40, 3, 5)])
def test_moe_q2_run_block64(F, n, ff, T, K, E):
    """moe_q2::run(block64 = true): x and h quantized in Q8 blocks of 64 (kernels/cuda/moe_q2.cu:58-81,
    AB = 64); every sampled slot against the oracle's expert_ffn with blk = 64. The block size changes
    the result (checked), so a kernel that ignored the flag would fail."""
    w = H.World(cfg=0, n=n, ff=ff, E=E, K=K)
    rng = np.random.default_rng(640 + n)
    x = rng.standard_normal((T, n)).astype(np.float32)
    ids = np.stack([rng.choice(E, size=K, replace=False) for _ in range(T)]).astype(np.int32)
    nb = F.moe_q2.workspace_bytes(T, K, n, ff, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T * K, n), float("nan"), dtype=torch.float32, device="cuda")
    F.moe_q2.run(w.arena.data_ptr(), w.stride, E, n, ff, dev(x), dev(ids), T, K, yd, ws, nb, None, True)
    torch.cuda.synchronize()
    y = yd.cpu().numpy().reshape(T, K, n)
    worst = 0.0
    for t in range(0, T, 3):
        for k in range(K):
            blob = w.blob(int(ids[t, k]))
            ref = O.expert_ffn(blob, n, ff, x[t], blk=64)
            err = H.out_rel(y[t, k][None], ref)
            worst = max(worst, err)
            assert err <= H.OUT_REL, (t, k, err)
    print(f"block64 n={n} ff={ff}: max out rel err {worst:.2e}")
    ref32 = O.expert_ffn(w.blob(int(ids[0, 0])), n, ff, x[0])
    assert H.out_rel(y[0, 0][None], ref32) > 0.0


@pytest.mark.parametrize("n,ff,T,K,E", [(1024, 1024, 40, 4, 6), (2048, 512, 8, 2, 8), (1024, 512, 200, 3, 4),
                                         (2560, 640, 90, 4, 6), (512, 128, 70, 2, 3), (1536, 384, 50, 3, 5),
                                         (640, 384, 60, 3, 5), (896, 256, 40, 2, 4), (128, 128, 30, 2, 3),
                                         (1152, 640, 20, 4, 6)])
def test_moe_q2_run_shapes(F, n, ff, T, K, E):
    """moe_q2::run at other shapes, in tiles of up to 16 tokens (at most 1536 slots), every slot against the
    oracle's expert_ffn: ff = 1024 (four weight stretches in the down product) with n = 1024 and about 27 rows
    per expert; groups of a row or two (T = 8, K = 2 over 8 experts) and of about 150 (T = 200, K = 3 over 4
    experts); ff not a multiple of 256 (the h rows padded to whole stretches: 640 = the reference tests'
    2560 / 640 shape, 128, 384) and n = 512 and 1536; n a multiple of 128 but not of 512
    (moe_q2.cu:516-517 accepts those: 640, 896, 128, 1152; the activations are padded with zeros to
    a multiple of 512 and the down GEMM's last row block is partial)."""
    w = H.World(cfg=0, n=n, ff=ff, E=E, K=K)
    rng = np.random.default_rng(n + ff + T)
    x = rng.standard_normal((T, n)).astype(np.float32)
    ids = np.stack([rng.choice(E, size=K, replace=False) for _ in range(T)]).astype(np.int32)
    nb = F.moe_q2.workspace_bytes(T, K, n, ff, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T * K, n), float("nan"), dtype=torch.float32, device="cuda")
    F.moe_q2.run(w.arena.data_ptr(), w.stride, E, n, ff, dev(x), dev(ids), T, K, yd, ws, nb)
    torch.cuda.synchronize()
    y = yd.cpu().numpy().reshape(T, K, n)
    for t in range(T):
        for k in range(K):
            ref = O.expert_ffn(w.blob(int(ids[t, k])), n, ff, x[t])
            err = H.out_rel(y[t, k][None], ref)
            assert err <= H.OUT_REL, (t, k, err)


@pytest.mark.parametrize("rep", [1, 3])
@pytest.mark.parametrize("n,ff", [(128, 128), (384, 256), (640, 384), (512, 640)])
def test_moe_q2_run_tile_edges(F, n, ff, rep):
    """Groups of every size class of the grouped GEMMs' tiles (16 tokens; 17-32 and 33-64 in the 32x32 shape;
    full tiles with a rest) in one call, each row against the oracle's expert: 716 slots, which all go in
    tiles of 16, and 2148."""
    sizes = [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 81, 128, 0, 2] * rep
    rng = np.random.default_rng(n + ff)
    ids = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    rng.shuffle(ids)
    T, E = ids.size, len(sizes)
    eb = F.expert_bytes(n, ff)
    arena = torch.empty(E * eb, dtype=torch.uint8, device="cuda")
    F.gen.experts(arena, eb, 7, 0, 0, E, n, ff)
    x = rng.standard_normal((T, n)).astype(np.float32)
    nb = F.moe_q2.workspace_bytes(T, 1, n, ff, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T, n), float("nan"), dtype=torch.float32, device="cuda")
    F.moe_q2.run(arena.data_ptr(), eb, E, n, ff, torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), T, 1, yd, ws, nb)
    torch.cuda.synchronize()
    y, ah = yd.cpu().numpy(), arena.cpu().numpy().reshape(E, eb)
    # the matrix cores' order of the gate / up sums moves an h code by one step on a few rows in a thousand.
    # One step is amax / 127 of its block; with a weight of at most 6.5 and an h of at most 6 times their root
    # mean squares, against a largest output of at least 3 root mean squares of ff terms, it moves the row by
    # at most 6.5 * 6 / (127 * 3 * sqrt(ff)) = 0.1 / sqrt(ff).
    err = np.array([H.out_rel(y[t][None], O.expert_ffn(ah[ids[t]], n, ff, x[t])) for t in range(T)])
    assert np.isfinite(err).all()
    assert err.max() <= max(H.OUT_REL, 0.1 / ff ** 0.5), (err.argmax(), ids[err.argmax()], err.max())
    assert (err > H.OUT_REL).mean() <= 0.005, (err > H.OUT_REL).sum()
    assert np.median(err) <= H.OUT_REL / 4


@pytest.mark.parametrize("n,ff,block64,bf16", [(640, 384, True, False), (512, 640, True, True), (1024, 256, False, True),
                                               (512, 1024, True, False), (1024, 1024, False, True), (512, 2048, False, False),
                                               (512, 4096, True, False)])
def test_moe_q2_run_large_tiles(F, n, ff, block64, bf16):
    """The 17-64-token tiles (chunks of more than 1536 slots: 2148 here) with Q8 blocks of 64, bf16 outputs and
    rows of 256 to 4096 in the down product: the rows at the edges of every tile and token column of groups of
    every size class, against the oracle's expert. The bounds are test_moe_q2_run_tile_edges', plus half a
    step of bf16."""
    sizes = [1, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 80, 81, 128, 0, 2] * 3
    rng = np.random.default_rng(n + ff)
    ids = np.repeat(np.arange(len(sizes)), sizes).astype(np.int32)
    rng.shuffle(ids)
    T, E = ids.size, len(sizes)
    assert T > 1536
    eb = F.expert_bytes(n, ff)
    arena = torch.empty(E * eb, dtype=torch.uint8, device="cuda")
    F.gen.experts(arena, eb, 7, 0, 0, E, n, ff)
    x = rng.standard_normal((T, n)).astype(np.float32)
    nb = F.moe_q2.workspace_bytes(T, 1, n, ff, E)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    yd = torch.full((T, n), float("nan"), dtype=torch.bfloat16 if bf16 else torch.float32, device="cuda")
    F.moe_q2.run(arena.data_ptr(), eb, E, n, ff, torch.from_numpy(x).cuda(), torch.from_numpy(ids).cuda(), T, 1, yd, ws, nb,
                 None, block64, bf16)
    torch.cuda.synchronize()
    y, ah = yd.float().cpu().numpy(), arena.cpu().numpy().reshape(E, eb)
    assert np.isfinite(y).all()
    rows = []
    for e in range(E):
        at = np.nonzero(ids == e)[0]   # (the group's rows in order)
        rows += [at[i] for i in sorted({0, 1, 15, 16, 31, 32, 47, 48, 63, 64, 79, 80, 127, len(at) - 1}) if 0 <= i < len(at)]
    step = 2.0 ** -9 if bf16 else 0.0
    err = np.array([H.out_rel(y[t][None], O.expert_ffn(ah[ids[t]], n, ff, x[t], blk=64 if block64 else 32)) for t in rows])
    print(f"large tiles n {n} ff {ff} block64 {block64} bf16 {bf16}: {len(rows)} rows, max {err.max():.2e}, "
          f"median {np.median(err):.2e}, above {(err > H.OUT_REL + step).sum()}")
    assert err.max() <= max(H.OUT_REL, 0.1 / ff ** 0.5) + step, (err.argmax(), err.max())
    assert (err > H.OUT_REL + step).mean() <= 0.01
    assert np.median(err) <= H.OUT_REL / 4 + step


@pytest.mark.parametrize("n,ff", [(512, 1024), (512, 2048), (1024, 4096)])
def test_layer_prefill_large_tiles(F, n, ff):
    """Whole layers of 400 tokens, K = 4 (2000 slots with the shared group: tiles of up to 64 tokens), at ff of 1024
    and above: ids bit-exact, weights 1e-6, outputs 2e-3."""
    w = H.World(cfg=0, n=n, ff=ff, E=16, K=4)
    x = np.random.default_rng(5 * n + ff).standard_normal((400, n)).astype(np.float32)
    out, ids, wts = w.gpu_forward(x)
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid), (n, ff)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL, (n, ff)


def test_moe_q2_run_shape_errors(F, w0):
    """The grouped GEMMs' shape limits (n and ff multiples of 128, ff up to 4096) fail loudly."""
    T, K = 4, 2
    x = torch.zeros((T, 2048), dtype=torch.float32, device="cuda")
    ids = torch.zeros((T, K), dtype=torch.int32, device="cuda")
    ids[:, 1] = 1
    yd = torch.empty((T * K, 2048), dtype=torch.float32, device="cuda")
    for n, ff in ((2048, 704), (1000, 512), (2048, 4224), (64, 512)):
        nb = F.moe_q2.workspace_bytes(T, K, n, ff, 8)
        ws = torch.empty(max(nb, 1 << 20), dtype=torch.uint8, device="cuda")
        with pytest.raises(F.FrtError) as e:
            F.moe_q2.run(w0.arena.data_ptr(), w0.stride, 8, n, ff, x, ids, T, K, yd, ws, ws.numel())
        assert e.value.code == -1


def test_layer_prefill_config3(F):
    """Config 3: 2048 bf16 tokens, Zipf(1.2) routing prior. Every token's ids are bit-exact; the
    outputs of 48 sampled tokens are checked against the oracle (a token's output depends only on
    that token)."""
    T = 2048
    bias = O.gen_zipf_bias(3, 0, H.E, H.ZIPF_S_PREFILL, H.PREFILL_ALPHA)
    w3 = H.World(cfg=3, bias=bias)
    xt = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xt, 3, 0, O.X_TENSOR, 1.0, round_bf16=True)
    x = xt.cpu().numpy()
    out, ids, wts = w3.gpu_forward(x)
    lg = O.router_logits(x, w3.router_h, bias)
    rid, rw, cnt = O.route_topk(lg, H.K)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert cnt.max() > 100 and (cnt == 0).sum() > 0   # ragged groups, some empty
    sel = np.random.default_rng(0).choice(T, size=48, replace=False)
    ref, sid, _, _ = w3.oracle_forward(x[sel])
    assert np.array_equal(sid, ids[sel])
    assert H.out_rel(out[sel], ref) <= H.OUT_REL
    assert np.isfinite(out).all()


def test_layer_prefill_config3_all_rows(F):
    """Config 3 (the bench's prefill layer and input), every one of the 2048 token rows against the
    oracle: ids bit-exact and each row within the output bar. The prefill path sums gate/up on the
    matrix cores and carries h and the per-slot outputs in fp16, so rows sit near 3e-4 (median) with a
    tail from h codes that the sum order moves: measured median 3.0e-4, 99th percentile 5.8e-4,
    worst 1.81e-3. Guards: median <= 5e-4, 99th percentile <= 1e-3, every row <= 2e-3."""
    T = 2048
    bias = O.gen_zipf_bias(3, 0, H.E, H.ZIPF_S_PREFILL, H.PREFILL_ALPHA)
    w3 = H.World(cfg=3, bias=bias)
    xt = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xt, 3, 0, O.X_TENSOR, 1.0, round_bf16=True)
    x = xt.cpu().numpy()
    out, ids, wts = w3.gpu_forward(x)
    ref, rid, rw, _ = w3.oracle_forward(x, threads=16)
    assert np.array_equal(ids, rid)
    g, r = out.astype(np.float64), ref.astype(np.float64)
    e = np.abs(g - r).max(axis=1) / np.abs(r).max(axis=1)
    print(f"prefill of 2048 tokens, all rows: median {np.median(e):.2e}, p99 {np.quantile(e, 0.99):.2e}, max {e.max():.2e}")
    assert np.median(e) <= 5e-4 and np.quantile(e, 0.99) <= 1e-3
    assert e.max() <= H.OUT_REL


def test_layer_prefill_repeatable(F):
    """The prefill kernels sum without atomics, so one input gives the same bits on every call: 8
    calls of the config 3 layer agree exactly on all 2048 tokens (a load that an LDS ring reads
    before it lands, or a missing barrier, shows up as differences between calls)."""
    T = 2048
    bias = O.gen_zipf_bias(3, 0, H.E, H.ZIPF_S_PREFILL, H.PREFILL_ALPHA)
    w3 = H.World(cfg=3, bias=bias)
    xt = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xt, 3, 0, O.X_TENSOR, 1.0, round_bf16=True)
    out = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    ws = w3.layer_obj.workspace(T)
    first = None
    for i in range(8):
        out.fill_(float("nan"))
        w3.layer_obj.forward(xt, out, T=T, ws=ws)
        cur = out.clone()
        if first is None:
            first = cur
            assert torch.isfinite(first).all()
        else:
            assert torch.equal(cur, first), i


def test_layer_prefill_graph_replays(F):
    """The prefill layer (router GEMM, top-k, dispatch, grouped GEMMs, combine) captured in a HIP
    graph replays to the eager result, bit for bit, on three replays with eager work and
    synchronizations between them (no fill node of the library's own in the graph)."""
    T = 2048
    bias = O.gen_zipf_bias(3, 0, H.E, H.ZIPF_S_PREFILL, H.PREFILL_ALPHA)
    w3 = H.World(cfg=3, bias=bias)
    xt = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xt, 3, 0, O.X_TENSOR, 1.0, round_bf16=True)
    ws = w3.layer_obj.workspace(T)
    ref = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    w3.layer_obj.forward(xt, ref, T=T, ws=ws)
    torch.cuda.synchronize()
    out = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        w3.layer_obj.forward(xt, out, T=T, ws=ws, stream=s)
    for i in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), i
        w3.layer_obj.forward(xt, ref, T=T, ws=ws)   # eager work between the replays
        torch.cuda.synchronize()


@pytest.mark.parametrize("T", [3, 8])
def test_layer_window_graph_replays(F, T):
    """A verify window (router, routing and grouping, moe_hits gate/up, the down kernel whose last
    workgroup per row group combines on a counter that the routing kernel zeroes) captured in a HIP
    graph replays to the eager result, bit for bit, on three replays with eager work of another
    window size and synchronizations between them; the eager result meets the oracle's bar."""
    w1 = H.World(cfg=1)
    xc = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(xc, 1, 40 + T, O.X_TENSOR, T, H.N, 0.8)
    x2 = torch.empty((2, H.N), dtype=torch.float32, device="cuda")
    F.gen.correlated(x2, 1, 50 + T, O.X_TENSOR, 2, H.N, 0.8)
    lo = w1.layer_obj
    ws = lo.workspace(T)
    ref = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    lo.forward(xc, ref, T=T, ws=ws)
    torch.cuda.synchronize()
    r, rid, _, _ = w1.oracle_forward(xc.cpu().numpy())
    assert H.out_rel(ref.cpu().numpy(), r) <= H.OUT_REL
    out = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    o2 = torch.empty((2, H.N), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        lo.forward(xc, out, T=T, ws=ws, stream=s)
    for i in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), i
        lo.forward(x2, o2, T=2, ws=ws)   # eager work between the replays, on the same workspace
        torch.cuda.synchronize()


def test_decode_stack_graph_replays(F):
    """Four config 2 decode layers (single token, RMS-normalised input, residual, the next layer's
    router warming) captured in a HIP graph, as the bench runs them: three replays, with eager work
    and synchronizations between them, each equal to the eager chain bit for bit (ids, weights and
    outputs)."""
    layers = []
    for layer in range(4):
        bias = O.gen_zipf_bias(2, layer, H.E, H.ZIPF_S_STACK)
        layers.append(H.World(cfg=2, layer=layer, bias=bias, norm_input=True))
    for l in range(4):
        layers[l].layer_obj.set_next_router(layers[(l + 1) % 4].router_w)
    x0 = torch.from_numpy(O.gen_normal(2, 0, O.X_TENSOR + 11, H.N).reshape(1, H.N)).cuda()
    ws = torch.empty(layers[0].layer_obj.workspace_bytes(1), dtype=torch.uint8, device="cuda")
    bufs = [torch.empty((1, H.N), dtype=torch.float32, device="cuda") for _ in range(4)]
    ids = torch.empty((4, H.K), dtype=torch.int32, device="cuda")
    wts = torch.empty((4, H.K), dtype=torch.float32, device="cuda")

    def chain(stream=None):
        cur = x0
        for l in range(4):
            layers[l].layer_obj.forward(cur, bufs[l], T=1, resid=cur, ids=ids[l], wts=wts[l], ws=ws, stream=stream)
            cur = bufs[l]

    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        chain(s)
    s.synchronize()
    ref = [b.clone() for b in bufs], ids.clone(), wts.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        chain(s)
    try:
        for i in range(3):
            for b in bufs:
                b.fill_(float("nan"))
            ids.fill_(-1)
            wts.fill_(0.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            for l in range(4):
                assert torch.equal(bufs[l], ref[0][l]), (i, l)
            assert torch.equal(ids, ref[1]), i
            assert torch.equal(wts, ref[2]), i
            with torch.cuda.stream(s):
                chain(s)   # eager work between the replays
            s.synchronize()
    finally:
        for l in range(4):
            layers[l].layer_obj.set_next_router(None)


def test_layer_mixed_config4(F):
    """Config 4: an 8192-token bf16 prefill chunk plus 16 uncorrelated fp32 decode tokens in one
    launch (T = 8208), with adversarial popularity: +2.8 on the logits of 16 seeded hot experts puts
    about 90% of the top-10 selections on them. All 8208 tokens' ids are bit-exact and the weights
    in tolerance; the outputs of 32 prefill and all 16 decode tokens are checked against the oracle."""
    import torch
    T_pf, T_dec = 8192, 16
    hot = np.random.default_rng(4).permutation(H.E)[:16]
    bias = np.zeros(H.E, np.float32)
    bias[hot] = 2.8
    w4 = H.World(cfg=4, bias=bias)
    xp = torch.empty((T_pf, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xp, 4, 0, O.X_TENSOR, 1.0, round_bf16=True)
    xd = torch.empty((T_dec, H.N), dtype=torch.float32, device="cuda")
    F.gen.normal(xd, 4, 0, O.X_TENSOR + 1, 1.0)
    x = np.concatenate([xp.cpu().numpy(), xd.cpu().numpy()])
    out, ids, wts = w4.gpu_forward(x)
    lg = O.router_logits(x, w4.router_h, bias)
    rid, rw, _ = O.route_topk(lg, H.K)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    frac = float(np.isin(ids, hot).mean())
    print(f"hot-expert share of the selections: {frac:.3f}")
    assert 0.85 <= frac <= 0.95
    sel = np.concatenate([np.random.default_rng(1).choice(T_pf, size=32, replace=False), np.arange(T_pf, T_pf + T_dec)])
    ref, sid, _, _ = w4.oracle_forward(x[sel])
    assert np.array_equal(sid, ids[sel])
    assert H.out_rel(out[sel], ref) <= H.OUT_REL
    assert np.isfinite(out).all()


def test_next_router_warming_keeps_results(F, w0):
    """A decode call that also loads the next layer's router rows into the caches
    (frt_moe_layer.next_router_w) returns exactly what it returns without."""
    x = np.random.default_rng(5).standard_normal((1, H.N)).astype(np.float32)
    out0, ids0, wts0 = w0.gpu_forward(x)
    w0.layer_obj.set_next_router(w0.router_w)
    try:
        out1, ids1, wts1 = w0.gpu_forward(x)
    finally:
        w0.layer_obj.set_next_router(None)
    assert np.array_equal(ids0, ids1)
    assert np.array_equal(wts0, wts1)
    assert np.array_equal(out0, out1)


def _edge_bias(case: str) -> np.ndarray:
    rng = np.random.default_rng(11)
    E = H.E
    pos = rng.permutation(E)
    if case == "all_equal":
        return np.zeros(E, np.float32)
    if case == "coarse":
        return (np.round(rng.standard_normal(E) * 2.0) / 2.0).astype(np.float32)
    b = (-1.0 - np.abs(rng.standard_normal(E))).astype(np.float32)
    if case == "tie10":          # 5 distinct leaders, then 12 equal values across the 10th place
        b[pos[:5]] = [10.0, 9.0, 8.0, 7.0, 6.0]
        b[pos[5:17]] = 5.0
    elif case in ("c64", "c65"):   # 3 leaders and 61 / 62 equal: 64 / 65 candidates
        b[pos[:3]] = [10.0, 9.0, 8.0]
        b[pos[3:3 + (61 if case == "c64" else 62)]] = 4.0
    elif case == "neg_inf":      # 6 finite logits; 4 of the selection are -inf (weight 0)
        b[:] = -np.inf
        b[pos[:6]] = [3.0, 1.0, 0.5, -2.0, -2.0, 7.0]
    elif case == "signed_zero":  # +0 and -0 leaders, equal as logits
        b[pos[:14]] = np.where(np.arange(14) % 2 == 0, 0.0, -0.0).astype(np.float32)
    return b


@pytest.mark.parametrize("case", ["tie10", "c64", "c65", "all_equal", "neg_inf", "signed_zero", "coarse"])
def test_decode_routing_edge_logits(F, case):
    """Decode routing on chosen logits: with the router matrix zero the logits are the bias
    exactly. Ties across the 10th place go to the lowest ids; 64 candidates stay on the one-wave
    selection of a single token, 65 and more (all equal) take the four-wave path; -inf logits get
    weight 0. T = 1 (one-wave path) and T = 2 (four-wave path) against the oracle."""
    w = H.World(cfg=0, bias=_edge_bias(case))
    w.router_w.zero_()
    w.router_h[:] = 0.0
    torch.cuda.synchronize()
    for T in (1, 2):
        x = O.gen_normal(0, 0, O.X_TENSOR + 9, T * H.N).reshape(T, H.N)
        out, ids, wts = w.gpu_forward(x)
        ref, rid, rw, _ = w.oracle_forward(x)
        assert np.array_equal(ids, rid), (case, T, ids, rid)
        nz = rw != 0
        assert np.array_equal(wts[~nz], rw[~nz]), (case, T)
        assert H.w_rel(wts[nz], rw[nz]) <= H.W_REL, (case, T)
        assert H.out_rel(out, ref) <= H.OUT_REL, (case, T)


SINGLE_TOKEN_ROUTES = [(1, 0), (8, 0), (1, 1)]   # options (route_waves, decode_xcd): the single token's routings


@pytest.mark.parametrize("E,K,finite", [(512, 10, 1), (512, 10, 9), (512, 32, 3), (1000, 32, 1), (40, 32, 5)])
@pytest.mark.parametrize("shared", ["q2", "dense"])
def test_routing_few_finite_logits(F, E, K, finite, shared):
    """Fewer finite logits than selections (-inf biases: masked experts), through every routing kernel: the rest of
    the selection are the lowest masked ids, each once (one lane of the selection holds only 8 or 16 of them),
    with weight 0: ids and weights the oracle's, outputs 2e-3 up to 8 tokens. The grouped products of 24 tokens sum
    h in another order, so that a code of h may move a step, and few experts carry the output: the bound of a
    single expert's rows there (test_moe_q2_run_tile_edges)."""
    b = np.full(E, -np.inf, np.float32)
    b[np.random.default_rng(E + K).permutation(E)[:finite]] = np.arange(finite) * 0.5
    kw = dict(cfg=0, n=1024, ff=256, E=E, K=K, bias=b)
    w = H.World(**kw) if shared == "q2" else _dense_world(H.GGML_Q8_0, 64, 3, **kw)
    w.router_w.zero_()
    w.router_h[:] = 0.0
    for T in (1, 2, 3, 4, 5, 8, 24):
        print(f"E {E} K {K} finite {finite} {shared} T {T}", flush=True)
        x = np.random.default_rng(T).standard_normal((T, w.n)).astype(np.float32)
        ref, rid, rw, _ = O.moe_layer(w.arena_h, w.stride, E, w.shared_h if shared == "q2" else w.dense, w.router_h, b,
                                      w.gate_h, w.n, w.ff, K, x, threads=8)
        nz = rw != 0
        for waves, xcd in SINGLE_TOKEN_ROUTES if T == 1 and shared == "q2" else SINGLE_TOKEN_ROUTES[:1]:
            try:
                F.set_option("route_waves", waves)
                F.set_option("decode_xcd", xcd)
                out, ids, wts = w.gpu_forward(x)
            finally:
                F.set_option("route_waves", 1)
                F.set_option("decode_xcd", 0)
            assert np.array_equal(ids, rid), (T, waves, xcd)
            assert np.array_equal(wts[~nz], rw[~nz]) and H.w_rel(wts[nz], rw[nz]) <= H.W_REL, (T, waves, xcd)
            assert H.out_rel(out, ref) <= (H.OUT_REL if T <= 8 else max(H.OUT_REL, 0.1 / w.ff ** 0.5)), (T, waves, xcd)
    ids = torch.full((4, K), -1, dtype=torch.int32, device="cuda")
    wts = torch.empty((4, K), dtype=torch.float32, device="cuda")
    F.moe_route_topk(None, dev(np.tile(b, (4, 1))), 4, E, K, ids, wts)
    torch.cuda.synchronize()
    assert np.array_equal(ids.cpu().numpy(), O.route_topk(np.tile(b, (4, 1)), K)[0])


@pytest.mark.parametrize("E,K", [(512, 10), (1000, 32), (40, 10)])
@pytest.mark.parametrize("bits", [0x7FC00000, 0xFFC00000, 0xFFFFFFFF])
@pytest.mark.parametrize("shared", ["q2", "dense"])
def test_routing_nan_logits(F, E, K, bits, shared):
    """NaN logits rank with -inf: a token of NaN selects K distinct experts in range and leaves the other tokens of
    its call as they are (the bounds of test_routing_few_finite_logits); experts whose logit alone is NaN (a NaN
    bias) are not selected."""
    some = np.random.default_rng(E).permutation(E)[:20]
    for bias_nan in (False, True):
        b = np.zeros(E, np.float32)
        if bias_nan:
            b.view(np.uint32)[some] = bits
        kw = dict(cfg=0, n=1024, ff=256, E=E, K=K, bias=b)
        w = H.World(**kw) if shared == "q2" else _dense_world(H.GGML_Q8_0, 64, 3, **kw)
        for T in (1, 2, 3, 4, 5, 8, 24):
            print(f"E {E} K {K} bits {bits:x} {shared} bias {bias_nan} T {T}", flush=True)
            x = np.random.default_rng(T).standard_normal((T, w.n)).astype(np.float32)
            if not bias_nan:
                x.view(np.uint32)[T // 2] = bits
            xd, out = dev(x), torch.empty((T, w.n), dtype=torch.float32, device="cuda")
            ids = torch.full((T, K), -1, dtype=torch.int32, device="cuda")
            cnt = torch.zeros(E, dtype=torch.int32, device="cuda")
            lg = O.router_logits(x, w.router_h, b)
            ref = np.argsort(-np.where(np.isnan(lg), -np.inf, lg), axis=1, kind="stable")[:, :K]
            for waves, xcd in SINGLE_TOKEN_ROUTES if T == 1 and shared == "q2" else SINGLE_TOKEN_ROUTES[:1]:
                ids.fill_(-1)
                cnt.zero_()
                try:
                    F.set_option("route_waves", waves)
                    F.set_option("decode_xcd", xcd)
                    w.layer_obj.forward(xd, out, T=T, ids=ids, counts=cnt)
                finally:
                    F.set_option("route_waves", 1)
                    F.set_option("decode_xcd", 0)
                assert np.array_equal(ids.cpu().numpy(), ref), (T, waves, xcd)
                assert np.array_equal(cnt.cpu().numpy(), np.bincount(ref.reshape(-1), minlength=E)), (T, waves, xcd)
            out = out.cpu().numpy()
            if not bias_nan and T > 1:
                ok = np.arange(T) != T // 2
                r = O.moe_layer(w.arena_h, w.stride, E, w.shared_h if shared == "q2" else w.dense, w.router_h, b,
                                w.gate_h, w.n, w.ff, K, x[ok], threads=8)[0]
                assert H.out_rel(out[ok], r) <= (H.OUT_REL if T <= 8 else max(H.OUT_REL, 0.1 / w.ff ** 0.5)), T


def test_layer_errors(F, w0):
    x = torch.zeros((1, H.N), dtype=torch.float32, device="cuda")
    out = torch.zeros((1, H.N), dtype=torch.float32, device="cuda")
    ws = w0.layer_obj.workspace(1)
    with pytest.raises(F.FrtError) as e:
        w0.layer_obj.forward(x, out, T=1, ws=ws[:16])
    assert e.value.code == -2


# ---------------------------------------------------------------- config 2: the stack's layers

@pytest.mark.parametrize("T", [1, 3, 64])
def test_stack_layers_teacher_forced(F, T):
    """Config 2 layers (Zipf(1.1) prior, RMS-normalised input, residual add), teacher-forced: the GPU
    and the oracle get the same layer input. Three layers, chained on the GPU's outputs."""
    x = O.gen_normal(2, 0, O.X_TENSOR, T * H.N).reshape(T, H.N) * np.float32(3.0)
    for layer in (0, 17, 47):
        bias = O.gen_zipf_bias(2, layer, H.E, H.ZIPF_S_STACK)
        w = H.World(cfg=2, layer=layer, bias=bias, norm_input=True)
        out, ids, wts = w.gpu_forward(x, resid=x)
        ref, rid, rw, _ = w.oracle_forward(x)
        assert np.array_equal(ids, rid), layer
        assert H.w_rel(wts, rw) <= H.W_REL
        # compare the MoE part (out - x) against the oracle's layer output
        assert H.out_rel(out - x, ref) <= H.OUT_REL, layer
        x = out


@pytest.mark.parametrize("T,n", [(3, 2048), (300, 2048), (1, 2560), (3, 1024), (300, 2560)])
def test_norm_input_routing(F, T, n):
    """The layer with the stack's RMS norm on its input (FRT_LAYER_NORM_INPUT): the single-token
    kernel (T = 1), a decode window (T = 3) and the prefill router GEMM (T = 300) route rmsnorm(x) as
    the oracle does, at chains of 32, 40 and 16 values (the canonical RMS sums each chain in four
    quarters): ids bit-exact, each selection's probability within 1e-6 relative of the oracle's
    softmax over its logits on rmsnorm(x), outputs within the layer bar."""
    bias = O.gen_zipf_bias(2, 5, H.E, H.ZIPF_S_STACK)
    w = H.World(cfg=2, layer=5, n=n, bias=bias, norm_input=True)
    x = (np.random.default_rng(T + n).standard_normal((T, n)) * 3).astype(np.float32)
    out = torch.empty((T, n), dtype=torch.float32, device="cuda")
    ids = torch.empty((T, H.K), dtype=torch.int32, device="cuda")
    wts = torch.empty((T, H.K), dtype=torch.float32, device="cuda")
    probs = torch.empty((T, H.K), dtype=torch.float32, device="cuda")
    w.layer_obj.forward(dev(x), out, T=T, ids=ids, wts=wts, probs=probs)
    torch.cuda.synchronize()
    ref, rid, rw, lg = w.oracle_forward(x)
    assert np.array_equal(ids.cpu().numpy(), rid)
    assert H.w_rel(wts.cpu().numpy(), rw) <= H.W_REL
    lg = lg.astype(np.float64)
    p = np.exp(lg - lg.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    want = np.take_along_axis(p, rid, axis=1)
    assert float((np.abs(probs.cpu().numpy() - want) / want).max()) <= 1e-6
    assert H.out_rel(out.cpu().numpy(), ref) <= H.OUT_REL
    # the default call (no probabilities asked for): the persistent kernels at T = 1 and 3
    o2, i2, _ = w.gpu_forward(x)
    assert np.array_equal(i2, rid)
    assert H.out_rel(o2, ref) <= H.OUT_REL


def test_cpp_mirror_gpu():
    """The C++ client of include/flashrt_moe.hpp on the GPU: moe_route_topk on the test_route_topk
    recipe against std::stable_sort and a double softmax, and an arena round trip."""
    import subprocess
    exe = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "cpp", "_build",
                       "test_shim")
    assert os.path.exists(exe), "build first: make -C flashrt_amd/csrc"
    r = subprocess.run([exe, "--gpu"], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "all passed" in r.stdout, r.stdout + r.stderr


# ---------------------------------------------------------------- the persistent single-token layer

def _fused_vs_three(F, w, x, resid=None, reps=3):
    """The single-token layer through the persistent launch of decode1.hip (several calls on one
    workspace, so the epochs advance) and through the three-kernel path: identical ids, weights and
    outputs, and no wait ran out of time."""
    ws = w.layer_obj.workspace(1)
    outs = []
    try:
        F.set_option("decode_xcd", 0)
        F.set_option("decode_fused", 0)
        ref = w.gpu_forward(x, resid=resid)
        F.set_option("decode_fused", 1)
        for _ in range(reps):
            outs.append(w.gpu_forward(x, resid=resid))
    finally:
        F.set_option("decode_fused", 1)
        F.set_option("decode_xcd", 0)   # (the default)
    assert not F.layer_sync_error(ws)
    for o in outs:
        for a, b in zip(o, ref):
            assert np.array_equal(a, b)
    return outs[0]


@pytest.mark.parametrize("case", ["cfg0", "stack", "E128", "E1000", "n2560", "n1024_ff1024", "K32", "n4096"])
def test_decode_fused_matches_three_kernel(F, case):
    """Persistent single-token layer == three-kernel path bit for bit, and within the bars of the
    oracle, over shapes: config 0; a config 2 layer (RMS norm, Zipf bias, residual); E = 128 and 1000
    (one and two wave-halves of logits per lane); the reference tests' 2560 / 640; n = 1024 with
    ff = 1024 (more h blocks than workgroups); K = 32 (33 entries, a second down batch); n = 4096
    (two 8-row output groups per workgroup)."""
    rng = np.random.default_rng(zlib.crc32(case.encode()) % 1000)
    kw = {}
    resid = None
    if case == "stack":
        kw = dict(cfg=2, layer=9, bias=O.gen_zipf_bias(2, 9, H.E, H.ZIPF_S_STACK), norm_input=True)
    elif case == "E128":
        kw = dict(cfg=0, E=128)
    elif case == "E1000":
        kw = dict(cfg=0, E=1000)
    elif case == "n2560":
        kw = dict(cfg=0, n=2560, ff=640)
    elif case == "n1024_ff1024":
        kw = dict(cfg=0, n=1024, ff=1024)
    elif case == "K32":
        kw = dict(cfg=0, K=32)
    elif case == "n4096":
        kw = dict(cfg=0, n=4096)
    else:
        kw = dict(cfg=0)
    w = H.World(**kw)
    x = (rng.standard_normal((1, w.n)) * (3.0 if case == "stack" else 1.0)).astype(np.float32)
    if case == "stack":
        resid = x
    out, ids, wts = _fused_vs_three(F, w, x, resid=resid)
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out - (x if resid is not None else 0), ref) <= H.OUT_REL


@pytest.mark.parametrize("T", [2, 3])
def test_layer_k32_short_windows(F, T):
    """K = 32 windows of 2 and 3 tokens: 33 slots per token exceed the window path's moe_hits launch
    (at most 32 slots), so the layer takes another path and must still match the oracle (ids
    bit-exact, weights 1e-6, outputs 2e-3), with the workspace the size query gives."""
    w = H.World(cfg=0, K=32)
    x = (np.random.default_rng(70 + T).standard_normal((T, H.N))).astype(np.float32)
    out, ids, wts = w.gpu_forward(x)
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out, ref) <= H.OUT_REL


def test_layer_workspace_size_independent_of_window_option(F):
    """The layer workspace size for T <= 8 does not change with "window_min_t": a workspace sized
    once serves calls after the option changes."""
    w = H.World(cfg=0)
    sizes = {}
    try:
        for mt in (2, 5, 9):
            F.set_option("window_min_t", mt)
            sizes[mt] = [w.layer_obj.workspace_bytes(T) for T in range(1, 9)]
    finally:
        F.set_option("window_min_t", 2)
    assert sizes[2] == sizes[5] == sizes[9]


@pytest.mark.parametrize("xcd", [0, 1])
def test_decode_fused_router_logits_bit_exact(F, xcd):
    """The persistent layer's router logits with the stack's RMS norm (read back from the
    workspace's tagged logit words) equal the oracle's canonical router on rmsnorm(x) bit for bit,
    the shared gate logit included (both persistent kernels)."""
    bias = O.gen_zipf_bias(2, 3, H.E, H.ZIPF_S_STACK)
    w = H.World(cfg=2, layer=3, bias=bias, norm_input=True)
    x = (np.random.default_rng(3).standard_normal((1, H.N)) * 4).astype(np.float32)
    ws = w.layer_obj.workspace(1)
    xd = dev(x)
    out = torch.empty((1, H.N), dtype=torch.float32, device="cuda")
    try:
        F.set_option("decode_xcd", xcd)
        w.layer_obj.forward(xd, out, T=1, ws=ws)
        torch.cuda.synchronize()
    finally:
        F.set_option("decode_xcd", 0)
    # the logit words follow the 4352-byte header, one every 4 words (32 bytes)
    words = ws[4352:4352 + 32 * (H.E + 1)].cpu().numpy().view(np.uint64)[::4]
    got = (words & np.uint64(0xFFFFFFFF)).astype(np.uint32).view(np.float32)
    u = O.rmsnorm(x)
    ref = O.router_logits(u, w.router_h, bias)[0]
    gate = O.router_logits(u, w.gate_h.reshape(1, H.N), None)[0, 0]
    assert np.array_equal(got[:H.E], ref)
    assert got[H.E] == gate


@pytest.mark.parametrize("xcd,T", [(0, 1), (1, 1), (0, 3)])
def test_decode_fused_timeout_path(F, w0, xcd, T):
    """With a zero wait bound the persistent layer cannot wait for the other workgroups: every call
    still completes (no hang), the next call reports it (FRT_ERR_SYNC, without a synchronisation),
    the error word reports it, and the next call with the normal bound returns the right answer
    again (both single-token persistent kernels, and the persistent window kernel at T = 3)."""
    F.set_option("decode_xcd", xcd)
    try:
        _timeout_path(F, w0, T)
    finally:
        F.set_option("decode_xcd", 0)


def _timeout_path(F, w0, T=1):
    x = O.gen_normal(0, 0, O.X_TENSOR, T * H.N).reshape(T, H.N)
    ws = w0.layer_obj.workspace(T)
    good = w0.gpu_forward(x)
    assert not F.layer_sync_error(ws)
    try:
        F.set_option("sync_ticks", 0)
        w0.gpu_forward(x)   # completes (a 256-workgroup join cannot finish within zero ticks)
    finally:
        F.set_option("sync_ticks", 20000000)
    # the next call reports the time-out without a synchronisation and launches nothing
    with pytest.raises(F.FrtError) as e:
        w0.gpu_forward(x)
    assert e.value.code == -6, e.value
    assert "ran out of time" in str(e.value)
    # the workspace's error word still tells (and is cleared by the check)
    assert F.layer_sync_error(ws)
    again = w0.gpu_forward(x)
    assert not F.layer_sync_error(ws)
    for a, b in zip(again, good):
        assert np.array_equal(a, b)
    # a time-out reported by layer_sync_error is not reported again by the next call
    try:
        F.set_option("sync_ticks", 0)
        w0.gpu_forward(x)
    finally:
        F.set_option("sync_ticks", 20000000)
    assert F.layer_sync_error(ws)
    again = w0.gpu_forward(x)
    for a, b in zip(again, good):
        assert np.array_equal(a, b)


# ---------------------------------------------------------------- the shared expert in a dense GGUF type

def _dense_world(gtype, ffs, seed, **kw):
    w = H.World(**kw)
    rng = np.random.default_rng(seed)
    raw = [H.dense_tensor(gtype, r, c, rng) for r, c in ((ffs, w.n), (ffs, w.n), (w.n, ffs))]
    dv = [torch.from_numpy(a).cuda() for a in raw]
    w.layer_obj.set_shared_dense(gtype, *dv, ffs)
    w.dense = (gtype, *raw, ffs)
    w._dense_keep = dv
    return w


@pytest.mark.parametrize("gtype", [H.GGML_Q8_0, H.GGML_F16, H.GGML_BF16, H.GGML_F32])
@pytest.mark.parametrize("T", [1, 3, 8, 200])
def test_layer_dense_shared_expert(F, gtype, T):
    """The layer with the shared expert in the model's own GGUF type (frt_moe_layer.shared_dense;
    the reference runs ffn_*_shexp through linear(), moe_ref.cu:117-123): ids bit-exact, weights
    1e-6 and outputs within 2e-3 of the oracle's layer with orc_shexp_ffn, for a single token, a
    3- and an 8-token window (moe_hits) and a 200-token chunk (moe_q2::run), shared ff 768 (not the
    experts' 512)."""
    w = _dense_world(gtype, 768, 30 + gtype, cfg=0)
    x = np.random.default_rng(T + gtype).standard_normal((T, H.N)).astype(np.float32)
    out, ids, wts = w.gpu_forward(x)
    ref, rid, rw, _ = O.moe_layer(w.arena_h, w.stride, w.E, w.dense, w.router_h, w.bias_h, w.gate_h, w.n, w.ff, w.K,
                                  x, threads=8)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    err = H.out_rel(out, ref)
    print(f"type {gtype} T {T}: out rel err {err:.2e}")
    assert err <= H.OUT_REL


def _shared_only(F, gtype, T, n, ffs, seed, ff=128, E=16, K=2, weights=None):
    """A layer whose routed experts have zero scales, so that it gives sigmoid(gate) * shared: its output,
    and the same in float64 on the weights' exact values (Q8_0: activations and h rounded to codes).
    weights: a function that changes the float64 gate / up / down matrices' raw bytes in place."""
    rng = np.random.default_rng(seed)
    eb = F.expert_bytes(n, ff)
    stride = (eb + 4095) // 4096 * 4096
    arena = torch.zeros(E * stride, dtype=torch.uint8, device="cuda")
    router = torch.from_numpy((rng.standard_normal((E, n)) * 0.02).astype(np.float32)).cuda()
    gate = (rng.standard_normal(n) * 0.02).astype(np.float32)
    raw = [H.dense_tensor(gtype, r, c, rng) for r, c in ((ffs, n), (ffs, n), (n, ffs))]
    if weights is not None:
        weights(raw)
    dv = [torch.from_numpy(a).cuda() for a in raw]
    gate_d = torch.from_numpy(gate).cuda()
    ml = F.MoeLayer(arena.data_ptr(), stride, E, 0, router, gate_d, n, ff, K)
    ml.set_shared_dense(gtype, *dv, ffs)
    x = rng.standard_normal((T, n)).astype(np.float32)
    out = torch.full((T, n), float("nan"), dtype=torch.float32, device="cuda")
    ml.forward(torch.from_numpy(x).cuda(), out, T=T)
    torch.cuda.synchronize()
    g, u, d = (H.dense_values(gtype, a, r, c) for a, (r, c) in zip(raw, ((ffs, n), (ffs, n), (n, ffs))))
    xx = x.astype(np.float64)
    if gtype == H.GGML_Q8_0:
        q, s = O.quantize_q8(x)
        xx = (q.reshape(T, n // 32, 32) * s.reshape(T, n // 32, 1).astype(np.float64)).reshape(T, n)
    with np.errstate(all="ignore"):
        gg = xx @ g.T
        h = gg / (1 + np.exp(-gg)) * (xx @ u.T)
        if gtype == H.GGML_Q8_0:
            q, s = O.quantize_q8(h.astype(np.float32))
            h = (q.reshape(T, ffs // 32, 32) * s.reshape(T, ffs // 32, 1).astype(np.float64)).reshape(T, ffs)
        ref = (h @ d.T) / (1 + np.exp(-(x.astype(np.float64) @ gate)))[:, None]
    return out.cpu().numpy(), ref


@pytest.mark.parametrize("gtype", [H.GGML_F16, H.GGML_F32])
@pytest.mark.parametrize("T,n,ffs", [(9, 512, 64), (16, 512, 4096), (20, 512, 4096), (21, 512, 4096), (20, 512, 64), (21, 512, 64),
                                     (8, 4096, 2048), (9, 4096, 2048)])
def test_shared_expert_short_calls(F, gtype, T, n, ffs):
    """F16 and F32 shared experts on either side of the rule that sends a short call to the row kernel (up to
    20 tokens, fewer than 72 M products), against float64: a root mean square error of at most 2^-20 of the
    outputs', four times what fp32 sums of these lengths show (2.5e-7)."""
    out, ref = _shared_only(F, gtype, T, n, ffs, 31 * T + ffs)
    err = np.sqrt(((out - ref) ** 2).mean() / (ref ** 2).mean())
    print(f"short type {gtype} T {T} n {n} ffs {ffs}: rms {err:.2e}")
    assert err <= 2.0 ** -20


@pytest.mark.parametrize("gtype", [H.GGML_F16, H.GGML_BF16, H.GGML_F32])
@pytest.mark.parametrize("case", ["gate", "up", "down", "overflow"])
def test_shared_expert_nonfinite(F, gtype, case):
    """An infinite weight of the shared expert, or weights whose h overflows fp32: the outputs of a call on the
    matrix cores are infinite, NaN and finite where the same tokens' are in a short call (fma chains): an
    infinity's products with the zero parts of the other operand do not turn it into a NaN."""
    def plant(raw):
        view = {H.GGML_F16: np.float16, H.GGML_BF16: np.uint16, H.GGML_F32: np.float32}[gtype]
        inf = np.uint16(0x7F80) if gtype == H.GGML_BF16 else np.inf
        if case == "overflow":
            if gtype == H.GGML_F16:   # (fp16 weights cannot: an infinite down weight of another row instead)
                raw[2].view(view).reshape(512, 128)[300, 7] = inf
                return
            big = np.uint16(0x6951) if gtype == H.GGML_BF16 else np.float32(1.6e25)   # (bf16: 1.58e25)
            raw[0].view(view).reshape(128, 512)[9, 4] = big
            raw[1].view(view).reshape(128, 512)[9, 4] = big
        else:
            m = ("gate", "up", "down").index(case)
            raw[m].view(view).reshape(512 if m == 2 else 128, -1)[100, 11] = inf
    long, _ = _shared_only(F, gtype, 24, 512, 128, 5, weights=plant)
    short, _ = _shared_only(F, gtype, 8, 512, 128, 5, weights=plant)
    long = long[:8]
    assert np.isinf(short).any()
    assert np.array_equal(np.isnan(long), np.isnan(short))
    assert np.array_equal(np.isinf(long), np.isinf(short))
    assert np.array_equal(np.sign(long[np.isinf(long)]), np.sign(short[np.isinf(short)]))
    ok = np.isfinite(short)
    assert np.abs(long[ok] - short[ok]).max(initial=0.0) <= 1e-5 * np.abs(short[ok]).max(initial=1.0)


@pytest.mark.parametrize("n,ff", [(512, 128), (1024, 256)])
@pytest.mark.parametrize("ffs", [64, 320, 2112, 4096])
@pytest.mark.parametrize("T", [1, 4, 5, 8])
def test_shared_expert_q8_windows(F, T, ffs, n, ff):
    """A Q8_0 shared expert of a window, whose down product quantizes h for itself: h of two blocks up to
    4096 values (part of one staging batch up to several, whole ones and a rest), through the slot path
    (512 / 128) and the window kernels (1024 / 256), against float64. A code of h may move by one step of
    its block (1/127 of the block's largest value, one of ffs terms): 2e-3."""
    out, ref = _shared_only(F, H.GGML_Q8_0, T, n, ffs, 7 * T + ffs, ff=ff)
    err = H.out_rel(out, ref)
    print(f"T {T} n {n} ffs {ffs}: {err:.2e}")
    assert err <= 2e-3


@pytest.mark.parametrize("gtype", [H.GGML_Q8_0, H.GGML_F16, H.GGML_BF16, H.GGML_F32])
@pytest.mark.parametrize("T,n,ffs", [(9, 512, 64), (16, 512, 64), (17, 1024, 192), (32, 512, 64), (33, 512, 128), (700, 2560, 640),
                                     (1025, 2560, 640), (1055, 2560, 640)])
def test_shared_expert_many_tokens(F, gtype, T, n, ffs):
    """The dense shared expert of more than 8 tokens: edges of the 16- and 32-token and 32-row tiles of the matrix
    cores (32 tokens from 512 workgroups on: the down product at 700 tokens, both at 1025, whose last workgroups
    have a token column wholly past the end, and at 1055), one to twenty K-steps per wave, against float64 on the
    weights' exact values. The dense types' products are exact and summed in fp32: a root mean square error of at most
    2^-20, four times what such sums show (2.5e-7); a plane or a cross product left out shows 4e-6 and more. Q8_0
    rounds h to codes, so a code may move by one step of its block (1/127 of the block's largest value, one of ffs
    terms): 2e-3."""
    out, ref = _shared_only(F, gtype, T, n, ffs, T + gtype)
    err, rms = H.out_rel(out, ref), np.sqrt(((out - ref) ** 2).mean() / (ref ** 2).mean())
    print(f"type {gtype} T {T} n {n} ffs {ffs}: {err:.2e} rms {rms:.2e}")
    assert err <= (2e-3 if gtype == H.GGML_Q8_0 else 4 * (n + ffs) * 2.0 ** -24)
    assert gtype == H.GGML_Q8_0 or rms <= 2.0 ** -20


@pytest.mark.parametrize("gtype", [H.GGML_Q8_0, H.GGML_BF16])
@pytest.mark.parametrize("n,ff,E,K,T,win", [(2048, 512, 1000, 10, 3, True), (2048, 512, 1024, 16, 7, True), (2560, 640, 64, 10, 8, True),
                                            (1024, 1024, 128, 31, 4, True), (1024, 256, 31, 31, 1, True),
                                            (2048, 512, 10, 10, 8, True), (2048, 512, 64, 16, 8, False), (1024, 256, 64, 31, 5, False),
                                            (4096, 256, 64, 32, 1, False)])
def test_layer_dense_window_shapes(F, gtype, n, ff, E, K, T, win):
    """Windows of a layer with a dense shared expert, RMS norm and residual on either side of the rule that sends
    them to the window kernels (K + 1 <= 32 slots a token, at most 128 in all): more than 512 experts, wide K,
    ff = 640, experts that all tokens share (two entries each); the path by the kernels that run, ids bit-exact,
    weights 1e-6, outputs 2e-3."""
    w = _dense_world(gtype, 192, 40 + gtype, cfg=0, n=n, ff=ff, E=E, K=K, norm_input=True)
    x = (np.random.default_rng(T + n + K).standard_normal((T, n)) * 2).astype(np.float32)
    out, ids, wts = w.gpu_forward(x, resid=x)
    ref, rid, rw, _ = O.moe_layer(w.arena_h, w.stride, w.E, w.dense, w.router_h, w.bias_h, w.gate_h, w.n, w.ff, w.K,
                                  x, threads=8, norm_input=True)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    assert H.out_rel(out - x, ref) <= H.OUT_REL
    xd, o = dev(x), torch.empty((T, n), dtype=torch.float32, device="cuda")
    assert ("win_route" in _kernels(F, lambda: w.layer_obj.forward(xd, o, T=T, resid=xd))) == win


def test_layer_dense_shared_expert_stack_norm(F):
    """Config 2 layers (RMS norm, Zipf bias, residual) with a Q8_0 shared expert of ff 512, chained
    by a two-layer stack call (layer by layer: the persistent kernels take only the Q2_0 blob), each
    layer checked teacher-forced against the oracle, and the stack call equal to the layer calls."""
    ws_ = []
    for layer in (0, 1):
        bias = O.gen_zipf_bias(2, layer, H.E, H.ZIPF_S_STACK)
        ws_.append(_dense_world(H.GGML_Q8_0, 512, 60 + layer, cfg=2, layer=layer, bias=bias, norm_input=True))
    x = O.gen_normal(2, 0, O.X_TENSOR, H.N).reshape(1, H.N) * np.float32(3.0)
    cur = x
    for w in ws_:
        out, ids, wts = w.gpu_forward(cur, resid=cur)
        ref, rid, rw, _ = O.moe_layer(w.arena_h, w.stride, w.E, w.dense, w.router_h, w.bias_h, w.gate_h, w.n, w.ff,
                                      w.K, cur, threads=8, norm_input=True)
        assert np.array_equal(ids, rid)
        assert H.w_rel(wts, rw) <= H.W_REL
        assert H.out_rel(out - cur, ref) <= H.OUT_REL
        cur = out
    st = F.MoeStack([w.layer_obj for w in ws_])
    o = torch.empty((1, H.N), dtype=torch.float32, device="cuda")
    st.forward(dev(x), o)
    torch.cuda.synchronize()
    assert np.array_equal(o.cpu().numpy(), cur)


def _kernels(F, fn):
    """The library kernels fn() launches (names of its per-kernel timing)."""
    import ctypes as C
    L = F.lib()
    L.frt_timing_begin()
    fn()
    names = C.create_string_buffer(64 * 32)
    ms = (C.c_double * 32)()
    cnt = (C.c_int * 32)()
    n = L.frt_timing_end(names, 32, ms, cnt, 32)
    return {names.raw[i * 32:(i + 1) * 32].split(b"\0")[0].decode() for i in range(n)}


@pytest.mark.parametrize("case", ["cfg0", "stack", "E128", "E1000", "n1024_ff1024", "n4096_ff256", "K32", "K4",
                                  "K7", "n3072"])
def test_decode_xcd_layer_matches_oracle(F, case):
    """The single-token layer through decode2.hip (joins split by XCD): ids bit-exact, weights 1e-6,
    outputs within 2e-3 of the oracle, over shapes: config 0; a config 2 layer (RMS norm, Zipf
    bias, residual); E = 128 and 1000; n = 1024 / ff = 1024 (4 blocks per XCD); n = 4096 / ff = 256
    (one 32-row block per XCD, 128 down rows per workgroup); K = 32 (4 owned entries per XCD and one
    split), K = 4 (no owned entry: every entry split over the XCDs), K = 7 (one owned entry per XCD, none
    split); n = 3072. Repeated calls
    on one workspace give the same bits, and no wait runs out of time."""
    rng = np.random.default_rng(zlib.crc32(case.encode()) % 1000 + 5)
    kw = dict(cfg=0)
    resid = None
    if case == "stack":
        kw = dict(cfg=2, layer=11, bias=O.gen_zipf_bias(2, 11, H.E, H.ZIPF_S_STACK), norm_input=True)
    elif case == "E128":
        kw = dict(cfg=0, E=128)
    elif case == "E1000":
        kw = dict(cfg=0, E=1000)
    elif case == "n1024_ff1024":
        kw = dict(cfg=0, n=1024, ff=1024)
    elif case == "n4096_ff256":
        kw = dict(cfg=0, n=4096, ff=256)
    elif case == "K32":
        kw = dict(cfg=0, K=32)
    elif case == "K4":
        kw = dict(cfg=0, K=4)
    elif case == "K7":
        kw = dict(cfg=0, K=7)
    elif case == "n3072":
        kw = dict(cfg=0, n=3072)
    w = H.World(**kw)
    x = (rng.standard_normal((1, w.n)) * (3.0 if case == "stack" else 1.0)).astype(np.float32)
    if case == "stack":
        resid = x
    ws = w.layer_obj.workspace(1)
    try:
        F.set_option("decode_xcd", 1)
        got = [w.gpu_forward(x, resid=resid) for _ in range(3)]
        assert not F.layer_sync_error(ws)
        xd = dev(x)
        o = torch.empty((1, w.n), dtype=torch.float32, device="cuda")
        assert "dec2_layer" in _kernels(F, lambda: w.layer_obj.forward(xd, o, T=1, ws=ws)), case
    finally:
        F.set_option("decode_xcd", 0)
    for g in got[1:]:
        for a, b in zip(g, got[0]):
            assert np.array_equal(a, b)
    out, ids, wts = got[0]
    ref, rid, rw, _ = w.oracle_forward(x)
    assert np.array_equal(ids, rid)
    assert H.w_rel(wts, rw) <= H.W_REL
    err = H.out_rel(out - (x if resid is not None else 0), ref)
    print(f"{case}: out rel err {err:.2e}")
    assert err <= H.OUT_REL


@pytest.mark.parametrize("xcd", [0, 1])
@pytest.mark.parametrize("E", [512, 128, 300])
def test_decode_route_waves_equal(F, xcd, E):
    """The persistent kernels' single-token routing by all 8 waves (option route_waves = 8) gives the
    one-wave routing's ids, weights and outputs bit for bit, also with coarse (tied) logits."""
    w = H.World(cfg=0, E=E)
    rng = np.random.default_rng(E + xcd)
    xs = [(rng.standard_normal((1, H.N))).astype(np.float32), np.round(rng.standard_normal((1, H.N)) * 2) / 2]
    try:
        F.set_option("decode_xcd", xcd)
        for x in xs:
            x = x.astype(np.float32)
            F.set_option("route_waves", 1)
            a = w.gpu_forward(x)
            F.set_option("route_waves", 8)
            b = w.gpu_forward(x)
            for p, q in zip(a, b):
                assert np.array_equal(p, q)
            ref, rid, rw, _ = w.oracle_forward(x)
            assert np.array_equal(b[1], rid)
    finally:
        F.set_option("route_waves", 1)
        F.set_option("decode_xcd", 0)


def _stack_worlds(nl, x_seed=21):
    layers = []
    for layer in range(nl):
        bias = O.gen_zipf_bias(2, layer, H.E, H.ZIPF_S_STACK)
        layers.append(H.World(cfg=2, layer=layer, bias=bias, norm_input=True))
    x0 = torch.from_numpy(O.gen_normal(2, 0, O.X_TENSOR + x_seed, H.N).reshape(1, H.N)).cuda()
    return layers, x0


def _layer_chain(layers, x0):
    cur = x0
    outs, ids, wts = [], torch.empty((len(layers), H.K), dtype=torch.int32, device="cuda"), \
        torch.empty((len(layers), H.K), dtype=torch.float32, device="cuda")
    for l, w in enumerate(layers):
        nxt = torch.empty((1, H.N), dtype=torch.float32, device="cuda")
        w.layer_obj.forward(cur, nxt, T=1, resid=cur, ids=ids[l], wts=wts[l])
        outs.append(nxt)
        cur = nxt
    torch.cuda.synchronize()
    return outs, ids, wts


@pytest.mark.parametrize("nl", [1, 6])
@pytest.mark.parametrize("xcd", [0, 1])
def test_decode_stack_call_matches_layer_calls(F, nl, xcd):
    """frt_moe_stack_forward (config 2 layers: RMS norm, Zipf bias, residual chain) as one
    persistent launch equals the chain of single-layer calls bit for bit (ids, weights, output);
    decode1.hip's kernel equals the three-kernel layer-by-layer path too, and decode2.hip's (xcd = 1)
    is within the layer bar of it; three graph replays of the stack call equal it."""
    F.set_option("decode_xcd", xcd)
    try:
        _stack_vs_layers(F, nl, xcd)
    finally:
        F.set_option("decode_xcd", 0)


def _stack_vs_layers(F, nl, xcd):
    layers, x0 = _stack_worlds(nl)
    st = F.MoeStack([w.layer_obj for w in layers])
    outs, ids_ref, wts_ref = _layer_chain(layers, x0)
    out = torch.empty((1, H.N), dtype=torch.float32, device="cuda")
    ids = torch.full((nl, H.K), -1, dtype=torch.int32, device="cuda")
    wts = torch.zeros((nl, H.K), dtype=torch.float32, device="cuda")
    ws = st.workspace()
    st.forward(x0, out, ids=ids, wts=wts, ws=ws)
    torch.cuda.synchronize()
    assert not F.layer_sync_error(ws)
    assert torch.equal(ids, ids_ref)
    assert torch.equal(wts, wts_ref)
    assert torch.equal(out, outs[-1])
    kn = _kernels(F, lambda: st.forward(x0, out, ws=ws))
    assert (kn & {"dec2_stack", "dec2_layer"}) if xcd else (kn & {"dec1_stack", "dec1_layer"}), kn
    # decode1.hip's stack kernel equals the three-kernel path layer by layer bit for bit; decode2.hip's
    # result is within the layer bar of it (same ids)
    try:
        F.set_option("decode_xcd", 0)
        out1 = torch.empty_like(out)
        ids1 = torch.full((nl, H.K), -1, dtype=torch.int32, device="cuda")
        st.forward(x0, out1, ids=ids1, ws=ws)
        F.set_option("decode_fused", 0)
        out3 = torch.empty_like(out)
        st.forward(x0, out3, ws=ws)
        torch.cuda.synchronize()
    finally:
        F.set_option("decode_fused", 1)
        F.set_option("decode_xcd", xcd)
    assert torch.equal(out3, out1)
    assert torch.equal(ids1, ids_ref)
    if xcd:
        assert H.out_rel((out1 - x0).cpu().numpy(), (out - x0).cpu().numpy()) <= H.OUT_REL
    else:
        assert torch.equal(out1, out)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        st.forward(x0, out, ids=ids, wts=wts, ws=ws, stream=s)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        st.forward(x0, out, ids=ids, wts=wts, ws=ws, stream=s)
    for i in range(3):
        out.fill_(float("nan"))
        ids.fill_(-1)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[-1]), i
        assert torch.equal(ids, ids_ref), i
        with torch.cuda.stream(s):
            st.forward(x0, out, ws=ws, stream=s)   # eager work between the replays
        s.synchronize()
    assert not F.layer_sync_error(ws)


# ---------------------------------------------------------------- loader, routing records

def test_load_experts_into_arena_and_layer(F, tmp_path):
    """frt_load_experts: ggml-layout Q2_0 slabs of a 2-layer, 12-expert model (d_model 1024, ff 256)
    written to a file at GGUF-like 4 KiB-aligned offsets, read into the HBM arena: every blob equals
    the host repack of its bytes, and a layer over the loaded arena matches the oracle (ids bit-exact,
    outputs within 2e-3). The reference model (FLASHRT_TEST_MODEL) is not in this image."""
    rng = np.random.default_rng(9)
    L_, E_, n, ff, K_ = 2, 12, 1024, 256, 4
    shapes = ((ff, n), (ff, n), (n, ff))
    path = str(tmp_path / "experts.gguf")
    slabs, data, off = [], [], 4096
    with open(path, "wb") as f:
        f.write(b"\0" * 4096)
        for l in range(L_):
            for r, c in shapes:
                nb = r * (c // 64) * E_
                blocks = np.zeros((nb, 18), np.uint8)
                blocks[:, 2:] = rng.integers(0, 256, (nb, 16), dtype=np.uint8)
                blocks[:, :2] = (rng.uniform(0.005, 0.02, nb).astype(np.float16)).view(np.uint8).reshape(nb, 2)
                raw = blocks.reshape(-1)
                slabs.append((0, off))
                data.append(raw)
                f.write(raw.tobytes())
                off += raw.size
                pad = (-off) % 4096
                f.write(b"\0" * pad)
                off += pad
    eb = F.expert_bytes(n, ff)
    arena = F.arena_alloc(L_, E_, eb)
    try:
        secs, nread = F.load_experts([path], slabs, n, ff, arena, threads=3)
        assert nread >= sum(d.size for d in data)
        for l in range(L_):
            for e in range(E_):
                parts = [data[3 * l + k][e * r * (c // 64) * 18:(e + 1) * r * (c // 64) * 18]
                         for k, (r, c) in enumerate(shapes)]
                want = F.q2_repack_expert(*parts, n, ff)
                got = torch.empty(eb, dtype=torch.uint8, device="cuda")
                import ctypes as C
                hip = C.CDLL("libamdhip64.so")
                assert hip.hipMemcpy(C.c_void_p(got.data_ptr()), C.c_void_p(arena.blob(l, e)), C.c_size_t(eb), 3) == 0
                assert np.array_equal(got.cpu().numpy(), want), (l, e)
        # a layer over the loaded experts (layer 1; the shared expert is layer 0's expert 11)
        arena_h = np.zeros(E_ * arena.stride, np.uint8)
        for e in range(E_):
            parts = [data[3 + k][e * r * (c // 64) * 18:(e + 1) * r * (c // 64) * 18] for k, (r, c) in enumerate(shapes)]
            arena_h[e * arena.stride:e * arena.stride + eb] = F.q2_repack_expert(*parts, n, ff)
        sh_parts = [data[k][11 * r * (c // 64) * 18:12 * r * (c // 64) * 18] for k, (r, c) in enumerate(shapes)]
        shared_h = F.q2_repack_expert(*sh_parts, n, ff)
        router = (rng.standard_normal((E_, n)) * 0.02).astype(np.float32)
        gate = (rng.standard_normal(n) * 0.02).astype(np.float32)
        rd, gd = dev(router), dev(gate)
        ml = F.MoeLayer(arena.blob(1, 0), arena.stride, E_, arena.blob(0, 11), rd, gd, n, ff, K_)
        for T in (1, 3, 40):
            x = rng.standard_normal((T, n)).astype(np.float32)
            out = torch.empty((T, n), dtype=torch.float32, device="cuda")
            ids = torch.empty((T, K_), dtype=torch.int32, device="cuda")
            wts = torch.empty((T, K_), dtype=torch.float32, device="cuda")
            ml.forward(dev(x), out, T=T, ids=ids, wts=wts)
            torch.cuda.synchronize()
            ref, rid, rw, _ = O.moe_layer(arena_h, arena.stride, E_, shared_h, router, None, gate, n, ff, K_, x)
            assert np.array_equal(ids.cpu().numpy(), rid), T
            assert H.w_rel(wts.cpu().numpy(), rw) <= H.W_REL, T
            assert H.out_rel(out.cpu().numpy(), ref) <= H.OUT_REL, T
    finally:
        F.arena_free(arena)


@pytest.mark.parametrize("T", [1, 3, 300])
def test_layer_routing_records(F, w0, T):
    """frt_moe_layer_forward_ex: probs (before renormalisation) and tail_counts, as moe_block's
    MoeTrace and moe_route_topk's tail_counts (blocks.hpp:130-135, :280-283), against the oracle's
    softmax: probs within 1e-6 relative, their renormalisation the weights, tail counts exact."""
    rng = np.random.default_rng(T)
    x = rng.standard_normal((T, H.N)).astype(np.float32)
    out = torch.empty((T, H.N), dtype=torch.float32, device="cuda")
    ids = torch.empty((T, H.K), dtype=torch.int32, device="cuda")
    wts = torch.empty((T, H.K), dtype=torch.float32, device="cuda")
    probs = torch.empty((T, H.K), dtype=torch.float32, device="cuda")
    counts = torch.zeros(H.E, dtype=torch.int32, device="cuda")
    tail = torch.zeros(H.E, dtype=torch.int32, device="cuda")
    tail_from = T // 2
    w0.layer_obj.forward(dev(x), out, T=T, ids=ids, wts=wts, counts=counts, tail_counts=tail, tail_from=tail_from,
                         probs=probs)
    torch.cuda.synchronize()
    lg = O.router_logits(x, w0.router_h, None).astype(np.float64)
    p = np.exp(lg - lg.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    i = ids.cpu().numpy()
    want = np.take_along_axis(p, i, axis=1)
    got = probs.cpu().numpy()
    assert float((np.abs(got - want) / want).max()) <= 1e-6
    assert H.w_rel(wts.cpu().numpy(), (want / want.sum(axis=1, keepdims=True)).astype(np.float32)) <= 1e-5
    tc = np.bincount(i[tail_from:].reshape(-1), minlength=H.E)
    assert np.array_equal(tail.cpu().numpy(), tc)
    assert np.array_equal(counts.cpu().numpy(), np.bincount(i.reshape(-1), minlength=H.E))
