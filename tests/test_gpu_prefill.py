"""GPU tests of prompt prefill (multi-token GEMMs on matrix cores, token-
batched attention) through the C ABI.

Each prefill GEMM row is compared with the oracle's serial GEMV of that row
(<= 1e-5 relative, normwise: the products are exact in fp32 -- fp32 W on the
fp32 MFMA, bf16 W against x split into three bf16 parts -- so only the fp32
summation order differs).  Token-batched attention must equal the decode
attention of each token bit for bit (same splits, same units).  At model
level, prefilling a prompt must give the stepped prompt's logits and KV
cache within tolerance and the same greedy tokens, including the C1 golden
fixture.
"""
import ctypes
import json
import os

import numpy as np
import pytest

import oracle
from ammon_amd import LlamaModel, _abi
from ammon_amd._abi import BF16, F32, AmmonError, call

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
RTOL = 1e-5
# bf16 KV: the two sides' fp32 K/V differ only by summation order, which can
# flip a bf16 rounding by one ulp (at most 2^-7 of the element): stored rows
# within 2^-7 normwise, logits within 1e-3 normwise
KV_STORE_TOL = 2.0**-7
BF16_KV_TOL = 1e-3


def rel_err(got, want):
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    return float(np.max(np.abs(got - want)) / max(np.max(np.abs(want)), 1e-30))


def up(rt, a):
    return rt.upload(np.ascontiguousarray(a))


def npdt(dtype):
    return np.uint16 if dtype == BF16 else np.float32


def head_major(pm, kv_heads, seq, head):
    return np.ascontiguousarray(pm.reshape(seq, kv_heads, head).transpose(1, 0, 2))


def pos_major(hm, kv_heads, seq, head):
    return np.ascontiguousarray(hm.reshape(kv_heads, seq, head).transpose(1, 0, 2))


# ---- GEMM -----------------------------------------------------------------------------------
# (d, n, tokens): tails in every dimension -- rows past a 64-row tile, n past
# a 256-wide chunk (288 = 256 + 32), tokens past 16- and 32-token tiles.  The
# library splits the reduction over a workgroup's waves (16-row tiles) when
# 64-row tiles would not fill the device; the last two shapes take 64-row
# tiles (16- and 32-token variants).  From 64 tokens bf16 weights take 64-token
# tiles with 2 or 4 16-row tiles per wave: tails in rows (520, 1000), in the
# 64-wide reduction chunks (4104, 520) and in tokens (130 = 2 * 64 + 2).
GEMM_SHAPES = [(4096, 4096, 16), (1024, 4096, 33), (288, 288, 8), (768, 288, 40),
               (288, 768, 7), (100, 264, 5), (5, 8, 3), (64, 256, 1), (130, 4104, 64),
               (32768, 64, 16), (4096, 264, 256), (1000, 520, 130), (520, 4104, 64),
               (8192, 1024, 100)]


@pytest.mark.parametrize("d,n,tokens", GEMM_SHAPES)
@pytest.mark.parametrize("w_dtype", [BF16, F32])
def test_prefill_gemm_matches_oracle_gemv(rt, d, n, tokens, w_dtype):
    wh = oracle.storage(oracle.normal(d * n, 201, std=0.02), w_dtype).reshape(d, n)
    xh = oracle.normal(tokens * n, 202).reshape(tokens, n) * 2
    w, x, y = up(rt, wh), up(rt, xh), rt.alloc(tokens * d * 4)
    call("ammon_prefill_gemm", rt.handle, None, w, w_dtype, d, n, x, tokens, y, None)
    got = y.download((tokens, d))
    want = np.stack([oracle.gemv(wh, w_dtype, xh[t]) for t in range(tokens)])
    assert rel_err(got, want) <= RTOL
    # residual epilogue in place (x += W h, per row)
    rh = oracle.normal(tokens * d, 203).reshape(tokens, d)
    r = up(rt, rh)
    call("ammon_prefill_gemm", rt.handle, None, w, w_dtype, d, n, x, tokens, r, r)
    assert rel_err(r.download((tokens, d)), rh + want) <= RTOL


@pytest.mark.parametrize("d,n,tokens", [(1024, 8192, 64), (520, 4104, 100), (256, 2048, 40)])
def test_prefill_gemm_split_reduction(rt, d, n, tokens):
    """With a workspace, few-row projections split the reduction into ranges
    summed in order by a second launch: oracle parity, the residual form in
    place, repeatable to the bit, and equal within rounding to the unsplit
    GEMM."""
    wh = oracle.storage(oracle.normal(d * n, 205, std=0.02), BF16).reshape(d, n)
    xh = oracle.normal(tokens * n, 206).reshape(tokens, n)
    w, x = up(rt, wh), up(rt, xh)
    nbytes = _abi.lib.ammon_prefill_gemm_workspace_bytes(d, tokens)
    assert nbytes == 8 * tokens * d * 4
    ws = rt.alloc(nbytes)
    want = np.stack([oracle.gemv(wh, BF16, xh[t]) for t in range(tokens)])
    y1, y2, y0 = rt.alloc(tokens * d * 4), rt.alloc(tokens * d * 4), rt.alloc(tokens * d * 4)
    for y in (y1, y2):
        call("ammon_prefill_gemm_ws", rt.handle, None, w, BF16, d, n, x, tokens, y, None, ws, nbytes)
    call("ammon_prefill_gemm", rt.handle, None, w, BF16, d, n, x, tokens, y0, None)
    g1, g2, g0 = (b.download((tokens, d)) for b in (y1, y2, y0))
    np.testing.assert_array_equal(g1.view(np.uint32), g2.view(np.uint32))
    assert rel_err(g1, want) <= RTOL and rel_err(g1, g0) <= RTOL
    rh = oracle.normal(tokens * d, 207).reshape(tokens, d)
    r = up(rt, rh)
    call("ammon_prefill_gemm_ws", rt.handle, None, w, BF16, d, n, x, tokens, r, r, ws, nbytes)
    assert rel_err(r.download((tokens, d)), rh + want) <= RTOL
    with pytest.raises(AmmonError, match="workspace overlaps"):
        call("ammon_prefill_gemm_ws", rt.handle, None, w, BF16, d, n, x, tokens, y1, None, y1,
             nbytes)


# Row tails of one to four rows per lane, first and last tokens of a tile, and y
# at a 4-byte boundary (a lane's four rows go out as one store): every element
# right, the ones before and behind y untouched.
@pytest.mark.parametrize("d,n,tokens,w_dtype", [
    (1001, 264, 65, BF16), (1002, 264, 64, BF16), (1003, 264, 130, BF16), (1004, 264, 127, BF16),
    (515, 4104, 33, BF16), (517, 72, 17, BF16), (37, 64, 16, F32), (39, 64, 31, F32),
    (40, 64, 33, F32),
    (32770, 136, 16, BF16), (24577, 648, 1, BF16),  # 16-token tiles of many rows
])
def test_prefill_gemm_row_tails(rt, d, n, tokens, w_dtype):
    wh = oracle.storage(oracle.normal(d * n, 208, std=0.02), w_dtype).reshape(d, n)
    xh = oracle.normal(tokens * n, 209).reshape(tokens, n)
    want = np.stack([oracle.gemv(wh, w_dtype, xh[t]) for t in range(tokens)])
    w, x = up(rt, wh), up(rt, xh)
    for residual in (False, True):
        host = np.full(tokens * d + 8, 7.0, np.float32)
        if residual:
            host[1:1 + tokens * d] = oracle.normal(tokens * d, 210)
        y = up(rt, host)
        at = ctypes.c_void_p(y.ptr + 4)
        call("ammon_prefill_gemm", rt.handle, None, w, w_dtype, d, n, x, tokens, at,
             at if residual else None)
        got = y.download(tokens * d + 8)
        base = host[1:1 + tokens * d].reshape(tokens, d) if residual else 0
        assert rel_err(got[1:1 + tokens * d].reshape(tokens, d), base + want) <= RTOL
        assert got[0] == 7.0 and (got[1 + tokens * d:] == 7.0).all()


# 16-token tiles (enough row blocks for the device): first and last tokens, row
# blocks and 128-wide chunks of k that end early; 17 tokens take the next tile.
@pytest.mark.parametrize("dim,hidden,tokens", [(200, 12300, 1), (136, 12288, 16), (640, 12289, 9),
                                               (264, 12300, 17)])
def test_prefill_gate_up_short(rt, dim, hidden, tokens):
    w1 = oracle.storage(oracle.normal(hidden * dim, 211, std=0.05), BF16).reshape(hidden, dim)
    w3 = oracle.storage(oracle.normal(hidden * dim, 212, std=0.05), BF16).reshape(hidden, dim)
    xh = oracle.normal(tokens * dim, 213).reshape(tokens, dim)
    hb = rt.alloc(tokens * hidden * 4)
    call("ammon_prefill_gate_up_swiglu", rt.handle, None, up(rt, xh), tokens, up(rt, w1), up(rt, w3),
         BF16, dim, hidden, hb)
    got = hb.download((tokens, hidden))
    for t in range(tokens):
        gate, lift = (oracle.gemv(w, BF16, xh[t]).astype(np.float64) for w in (w1, w3))
        assert rel_err(got[t], gate / (1 + np.exp(-gate)) * lift) <= RTOL


def test_prefill_gemm_random_shapes(rt):
    """Seeded random shapes through every tile family and the split
    reduction (rows, reduction length and tokens off every tile multiple),
    bf16 weights, with and without a workspace, against the oracle."""
    rng = np.random.default_rng(12)
    for case in range(16):
        d = int(rng.integers(1, 700))
        n = 8 * int(rng.integers(1, 700))
        tokens = int(rng.choice([1, 3, 16, 17, 31, 33, 63, 64, 65, 100, 130]))
        wh = oracle.storage(oracle.normal(d * n, 300 + case, std=0.05), BF16).reshape(d, n)
        xh = oracle.normal(tokens * n, 400 + case).reshape(tokens, n)
        rh = oracle.normal(tokens * d, 500 + case).reshape(tokens, d)
        want = np.stack([oracle.gemv(wh, BF16, xh[t]) for t in range(tokens)])
        w, x = up(rt, wh), up(rt, xh)
        nbytes = _abi.lib.ammon_prefill_gemm_workspace_bytes(d, tokens)
        ws = rt.alloc(nbytes)
        for use_ws in (False, True):
            r = up(rt, rh)
            if use_ws:
                call("ammon_prefill_gemm_ws", rt.handle, None, w, BF16, d, n, x, tokens, r, r, ws,
                     nbytes)
            else:
                call("ammon_prefill_gemm", rt.handle, None, w, BF16, d, n, x, tokens, r, r)
            # the projection part (y - residual: exact but for y's rounding)
            got = r.download((tokens, d)).astype(np.float64) - rh
            assert rel_err(got, want) <= 2 * RTOL, (d, n, tokens, use_ws)


def test_prefill_gemm_identity_is_exact(rt):
    # the reference's identity GEMV (tests/kernels.rs:83-97) per row: exact
    for w_dtype in (F32, BF16):
        n = 64
        wh = oracle.storage(np.eye(n, dtype=np.float32), w_dtype)
        xh = oracle.normal(3 * n, 204).reshape(3, n)
        w, x, y = up(rt, wh), up(rt, xh), rt.alloc(3 * n * 4)
        call("ammon_prefill_gemm", rt.handle, None, w, w_dtype, n, n, x, 3, y, None)
        np.testing.assert_array_equal(y.download((3, n)), xh)


def test_prefill_gemm_validation(rt):
    w = up(rt, np.zeros((8, 12), np.float32))
    x = up(rt, np.zeros((2, 12), np.float32))
    y = rt.alloc(2 * 8 * 4)
    with pytest.raises(AmmonError, match="multiple of 8"):
        call("ammon_prefill_gemm", rt.handle, None, w, F32, 8, 12, x, 2, y, None)
    x8 = up(rt, np.zeros((2, 8), np.float32))
    with pytest.raises(AmmonError, match="y overlaps x"):
        call("ammon_prefill_gemm", rt.handle, None, w, F32, 8, 8, x8, 2, x8, None)
    with pytest.raises(AmmonError, match="empty shape"):
        call("ammon_prefill_gemm", rt.handle, None, w, F32, 8, 8, x8, 0, y, None)


@pytest.mark.parametrize("dim,hidden,tokens,w_dtype",
                         [(288, 768, 8, F32), (4096, 14336, 16, BF16), (64, 200, 35, BF16),
                          (64, 16400, 16, BF16), (64, 4100, 100, F32), (256, 1000, 130, BF16),
                          (512, 8192, 64, BF16)])
def test_prefill_gate_up_swiglu(rt, dim, hidden, tokens, w_dtype):
    w1 = oracle.storage(oracle.normal(hidden * dim, 211, std=0.02), w_dtype).reshape(hidden, dim)
    w3 = oracle.storage(oracle.normal(hidden * dim, 212, std=0.02), w_dtype).reshape(hidden, dim)
    xh = oracle.normal(tokens * dim, 213).reshape(tokens, dim)
    d1, d3, x, hb = up(rt, w1), up(rt, w3), up(rt, xh), rt.alloc(tokens * hidden * 4)
    call("ammon_prefill_gate_up_swiglu", rt.handle, None, x, tokens, d1, d3, w_dtype, dim,
         hidden, hb)
    want = np.stack([oracle.swiglu(oracle.gemv(w1, w_dtype, xh[t]), oracle.gemv(w3, w_dtype, xh[t]))
                     for t in range(tokens)])
    assert rel_err(hb.download((tokens, hidden)), want) <= RTOL


@pytest.mark.parametrize("shape", ["c1", "c4", "c4_long"])
@pytest.mark.parametrize("kv_dtype", [F32, BF16])
@pytest.mark.parametrize("use_ws", [False, True])
def test_prefill_qkv_rope_store(rt, shape, kv_dtype, use_ws):
    """use_ws: the workspace entry, whose c4 shape (6144 rows, 40 tokens)
    splits the reduction and rotates / stores in the summing launch."""
    if shape == "c1":
        dim, q_heads, kv_heads, head, seq, w_dtype, theta, p0, T = 288, 6, 6, 48, 64, F32, 1e4, 0, 9
    elif shape == "c4":
        dim, q_heads, kv_heads, head, seq, w_dtype, theta, p0, T = 4096, 32, 8, 128, 96, BF16, 5e5, 30, 40
    else:  # enough token tiles for 64-row tiles; a narrow model keeps the oracle quick
        dim, q_heads, kv_heads, head, seq, w_dtype, theta, p0, T = 512, 32, 8, 128, 256, BF16, 5e5, 5, 200
    qd, kd = q_heads * head, kv_heads * head
    wq = oracle.storage(oracle.normal(qd * dim, 221, std=0.02), w_dtype).reshape(qd, dim)
    wk = oracle.storage(oracle.normal(kd * dim, 222, std=0.02), w_dtype).reshape(kd, dim)
    wv = oracle.storage(oracle.normal(kd * dim, 223, std=0.02), w_dtype).reshape(kd, dim)
    xh = oracle.normal(T * dim, 224).reshape(T, dim)
    table_h = oracle.rope_table(theta, head, seq)
    kc_pm = np.zeros((seq, kv_heads, head), npdt(kv_dtype))
    vc_pm = np.zeros_like(kc_pm)
    want_q = np.zeros((T, qd), np.float32)
    for t in range(T):
        q = oracle.gemv(wq, w_dtype, xh[t])
        oracle.rope_store(q, oracle.gemv(wk, w_dtype, xh[t]), kc_pm, kv_dtype, head, p0 + t, table_h)
        oracle.cache_store(oracle.gemv(wv, w_dtype, xh[t]), vc_pm, kv_dtype, p0 + t)
        want_q[t] = q
    kc = up(rt, np.zeros((kv_heads, seq, head), npdt(kv_dtype)))
    vc = up(rt, np.zeros((kv_heads, seq, head), npdt(kv_dtype)))
    x, q, table = up(rt, xh), rt.alloc(T * qd * 4), up(rt, table_h)
    step = rt.step(0, p0)
    if use_ws:
        nbytes = _abi.lib.ammon_prefill_gemm_workspace_bytes(qd + 2 * kd, T)
        call("ammon_prefill_qkv_rope_store_ws", rt.handle, None, x, T, up(rt, wq), up(rt, wk),
             up(rt, wv), w_dtype, dim, q_heads, kv_heads, head, q, kc, vc, kv_dtype, seq, step,
             table, rt.alloc(nbytes), nbytes)
    else:
        call("ammon_prefill_qkv_rope_store", rt.handle, None, x, T, up(rt, wq), up(rt, wk),
             up(rt, wv), w_dtype, dim, q_heads, kv_heads, head, q, kc, vc, kv_dtype, seq, step,
             table)
    assert rel_err(q.download((T, qd)), want_q) <= RTOL
    got_k = pos_major(kc.download((kv_heads, seq, head), npdt(kv_dtype)), kv_heads, seq, head)
    got_v = pos_major(vc.download((kv_heads, seq, head), npdt(kv_dtype)), kv_heads, seq, head)
    tol = RTOL if kv_dtype == F32 else KV_STORE_TOL
    for got, want in ((got_k, kc_pm), (got_v, vc_pm)):
        assert rel_err(oracle.widen(got, kv_dtype), oracle.widen(want, kv_dtype)) <= tol
        # rows outside [p0, p0 + T) untouched
        np.testing.assert_array_equal(got[:p0], 0)
        np.testing.assert_array_equal(got[p0 + T:], 0)


def test_prefill_qkv_positions_past_cache_poison_q(rt):
    # tokens whose position reaches seq: q rows are NaN, no cache write
    dim, q_heads, kv_heads, head, seq, T = 64, 2, 1, 32, 20, 8
    qd, kd = q_heads * head, kv_heads * head
    wq = oracle.storage(oracle.normal(qd * dim, 231, std=0.1), BF16).reshape(qd, dim)
    wk = oracle.storage(oracle.normal(kd * dim, 232, std=0.1), BF16).reshape(kd, dim)
    wv = oracle.storage(oracle.normal(kd * dim, 233, std=0.1), BF16).reshape(kd, dim)
    kc = up(rt, np.zeros((kv_heads, seq + 4, head), np.float32))  # guard rows past seq
    vc = up(rt, np.zeros((kv_heads, seq + 4, head), np.float32))
    x, q = up(rt, oracle.normal(T * dim, 234).reshape(T, dim)), rt.alloc(T * qd * 4)
    table = up(rt, oracle.rope_table(5e5, head, seq))
    step = rt.step(0, seq - 3)
    call("ammon_prefill_qkv_rope_store", rt.handle, None, x, T, up(rt, wq), up(rt, wk), up(rt, wv),
         BF16, dim, q_heads, kv_heads, head, q, kc, vc, F32, seq, step, table)
    got_q = q.download((T, qd))
    assert np.isfinite(got_q[:3]).all() and np.isnan(got_q[3:]).all()
    for c in (kc, vc):
        rows = c.download((kv_heads, seq + 4, head))[0]
        assert np.count_nonzero(rows[seq - 3:seq].any(axis=1)) == 3
        np.testing.assert_array_equal(rows[seq:], 0)


# ---- rmsnorm rows ---------------------------------------------------------------------------
# Rows held in registers, at the edges of 1, 2, 4 and 8 quads per lane, the loops
# beyond, and weights at 2-, 4- and 8-byte boundaries; in place too.
@pytest.mark.parametrize("dim", [4, 1020, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 1030])
@pytest.mark.parametrize("w_dtype,shift", [(F32, 0), (F32, 1), (BF16, 0), (BF16, 1), (BF16, 4)])
def test_rmsnorm_row_widths(rt, dim, w_dtype, shift):
    rows = 3
    xh = oracle.normal(rows * dim, 221).reshape(rows, dim)
    wh = oracle.storage(oracle.normal(dim + shift, 222) + np.float32(1), w_dtype)
    x, w, o = up(rt, xh), up(rt, wh), rt.alloc(rows * dim * 4)
    at = ctypes.c_void_p(w.ptr + shift * wh.itemsize)
    call("ammon_rmsnorm", rt.handle, None, x, at, w_dtype, o, rows, dim, 1e-5)
    got = o.download((rows, dim))
    want = oracle.rmsnorm(xh, wh[shift:], w_dtype)
    assert rel_err(got, want) <= RTOL
    call("ammon_rmsnorm", rt.handle, None, x, at, w_dtype, x, rows, dim, 1e-5)
    np.testing.assert_array_equal(x.download((rows, dim)), got)


# The same row gives the same bits however its weights are aligned: weights one
# bf16 off an 8-byte boundary take the loop over the row, aligned ones the forms
# that hold it in registers.
@pytest.mark.parametrize("dim", [4, 1020, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196])
def test_rmsnorm_does_not_depend_on_alignment(rt, dim):
    rows = 64
    x, o = up(rt, oracle.normal(rows * dim, 223)), rt.alloc(rows * dim * 4)
    w = oracle.storage(oracle.normal(dim, 224) + np.float32(1), BF16)
    got = []
    for shift in (0, 1):
        at = up(rt, np.concatenate([np.zeros(shift, w.dtype), w]))
        call("ammon_rmsnorm", rt.handle, None, x, ctypes.c_void_p(at.ptr + 2 * shift), BF16, o, rows,
             dim, 1e-5)
        got.append(o.download((rows, dim)))
    np.testing.assert_array_equal(got[0], got[1])


# ---- attention ------------------------------------------------------------------------------
@pytest.mark.parametrize("q_heads,kv_heads,head,seq,p0,T,split,kv_dtype", [
    (32, 8, 128, 512, 0, 40, 16, BF16),
    (32, 8, 128, 512, 300, 17, 64, BF16),
    (6, 6, 48, 256, 0, 9, 16, F32),
    (4, 2, 64, 80, 10, 70, 8, F32),
    (8, 1, 128, 300, 250, 50, 32, F32),
    (4, 2, 64, 1200, 1100, 5, 8, F32),    # 138..139 live splits: several per split lane
    (2, 1, 32, 4200, 4100, 3, 8, BF16),   # 513+: the decode merge's second pass
])
def test_attention_prefill_equals_decode_per_token(rt, q_heads, kv_heads, head, seq, p0, T, split,
                                                  kv_dtype):
    dt = npdt(kv_dtype)
    kc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 241), kv_dtype).reshape(
        seq, kv_heads, head)
    vc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 242), kv_dtype).reshape(
        seq, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 243).reshape(T, q_heads, head)
    kc, vc = up(rt, head_major(kc_pm, kv_heads, seq, head)), up(rt, head_major(vc_pm, kv_heads, seq, head))
    q, out = up(rt, qh), rt.alloc(T * q_heads * head * 4)
    ctx = p0 + T
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    part = up(rt, np.full(nbytes // 4, np.nan, np.float32))
    step = rt.step(0, p0)
    call("ammon_attention_prefill", rt.handle, None, q, T, q_heads, kc, vc, kv_dtype, kv_heads,
         head, seq, step, ctx, split, part, nbytes, out)
    got = out.download((T, q_heads, head))
    # the decode attention of each token at its position: identical units
    dpart_n = _abi.lib.ammon_attention_scratch_bytes(q_heads, head, seq, split)
    dpart, dout = rt.alloc(dpart_n), rt.alloc(q_heads * head * 4)
    for t in range(T):
        qt = up(rt, qh[t])
        rt.deposit(step, 0, p0 + t)
        call("ammon_attention_decode", rt.handle, None, qt, q_heads, kc, vc, kv_dtype, kv_heads,
             head, seq, step, split, dpart, dpart_n, dout)
        np.testing.assert_array_equal(got[t], dout.download((q_heads, head)))
    # and the oracle's split attention (split 8) within tolerance
    for t in (0, T // 2, T - 1):
        want = oracle.attention(qh[t], kc_pm, vc_pm, kv_dtype, p0 + t)
        assert rel_err(got[t], want) <= RTOL


# The matrix-core tiles (128 query rows x 64 or 32 positions), which long prompts
# take: heads of one to four 32-dim blocks, whole and ragged; groups that do not
# divide a tile; last tiles and chunks of a few rows; one split (the scratch stays
# untouched) and several (start far into the cache).  A token's V that is not
# finite must reach the tokens from it on and no earlier one, and a position past
# ctx gives NaN.
TILE_SHAPES = [  # q_heads, kv_heads, head, kv_dtype, start, tokens, split_len
    (32, 8, 128, BF16, 0, 333, 1024), (32, 8, 128, BF16, 1100, 130, 64),
    (16, 16, 128, F32, 0, 900, 1024), (16, 2, 120, BF16, 700, 200, 128),
    (14, 2, 96, F32, 600, 300, 64), (15, 5, 72, BF16, 0, 500, 512),
    (32, 8, 64, F32, 1, 511, 1024), (24, 24, 40, BF16, 3, 650, 1024),
    (32, 32, 24, BF16, 0, 700, 1024), (64, 8, 128, F32, 1000, 65, 256),
]


@pytest.mark.parametrize("q_heads,kv_heads,head,kv_dtype,p0,T,split", TILE_SHAPES)
def test_attention_prefill_tiles(rt, q_heads, kv_heads, head, kv_dtype, p0, T, split):
    ctx, late = p0 + T - 2, T // 2  # the last two tokens lie past ctx
    seq = ctx + 3
    kc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 261), kv_dtype).reshape(
        seq, kv_heads, head)
    vc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 262), kv_dtype).reshape(
        seq, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 263).reshape(T, q_heads, head)
    kc, q = up(rt, head_major(kc_pm, kv_heads, seq, head)), up(rt, qh)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    step = rt.step(0, p0)
    bad_pm = vc_pm.copy()
    inf = np.inf if kv_dtype == F32 else np.uint16(0x7f80)
    nan = np.nan if kv_dtype == F32 else np.uint16(0x7fc0)
    bad_pm[p0 + late, :, 3], bad_pm[p0 + late, :, head - 1] = inf, nan
    for v_pm, first_bad in ((vc_pm, T - 2), (bad_pm, late)):
        vc, out = up(rt, head_major(v_pm, kv_heads, seq, head)), rt.alloc(T * q_heads * head * 4)
        part = up(rt, np.full(nbytes // 4, 7.0, np.float32))
        call("ammon_attention_prefill", rt.handle, None, q, T, q_heads, kc, vc, kv_dtype, kv_heads,
             head, seq, step, ctx, split, part, nbytes, out)
        got = out.download((T, q_heads, head))
        if split >= ctx:  # one split: a tile writes the result itself
            np.testing.assert_array_equal(part.download(nbytes // 4), 7.0)
        for t in (0, 1, 31, 32, late - 1, late, T - 3):
            if t < first_bad:
                want = oracle.attention(qh[t], kc_pm, vc_pm, kv_dtype, p0 + t)
                assert rel_err(got[t], want) <= RTOL, t
        assert np.isfinite(got[:first_bad]).all()
        assert np.isnan(got[first_bad:T - 2, :, head - 1]).all()
        assert (got[first_bad:T - 2, :, 3] == np.inf).all()
        assert np.isnan(got[T - 2:]).all()


# Every token and head of the tiles against 64 bits; and tiles they are: q at a
# 4-byte boundary takes the units, whose results are other bits.
@pytest.mark.parametrize("q_heads,kv_heads,head,kv_dtype,p0,T,split", TILE_SHAPES + [
    (32, 8, 128, BF16, 0, 700, 1024), (24, 8, 128, BF16, 0, 333, 1024), (32, 8, 16, F32, 0, 1600, 1024),
    (32, 32, 32, F32, 0, 700, 1024), (32, 8, 32, F32, 400, 300, 256), (16, 16, 128, BF16, 5, 450, 1024),
    (24, 6, 48, F32, 0, 1000, 1024), (16, 16, 16, BF16, 0, 900, 1024),
])
def test_attention_prefill_every_token(rt, q_heads, kv_heads, head, kv_dtype, p0, T, split):
    ctx = p0 + T
    kv = oracle.storage(oracle.normal(2 * ctx * kv_heads * head, 274), kv_dtype).reshape(
        2, ctx, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 275)
    kc, vc = (up(rt, head_major(a, kv_heads, ctx, head)) for a in kv)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    out, part, got = rt.alloc(T * q_heads * head * 4), rt.alloc(nbytes), []
    for shift in (0, 1):
        q = up(rt, np.concatenate([np.zeros(shift, np.float32), qh]))
        call("ammon_attention_prefill", rt.handle, None, ctypes.c_void_p(q.ptr + 4 * shift), T, q_heads,
             kc, vc, kv_dtype, kv_heads, head, ctx, rt.step(0, p0), ctx, split, part, nbytes, out)
        got.append(out.download((T, q_heads, head)))
    assert (got[0] != got[1]).any()
    k, v = (oracle.widen(a, kv_dtype).astype(np.float64) for a in kv)
    qh, want = qh.astype(np.float64).reshape(T, q_heads, head), np.empty((T, q_heads, head))
    late = np.arange(ctx)[None] > p0 + np.arange(T)[:, None]
    for h in range(q_heads):
        g = h // (q_heads // kv_heads)
        s = np.where(late, -np.inf, qh[:, h] @ k[:, g].T / np.sqrt(head))
        w = np.exp(s - s.max(-1, keepdims=True))
        want[:, h] = (w @ v[:, g]) / w.sum(-1, keepdims=True)
    for t in range(T):
        assert rel_err(got[0][t], want[t]) <= RTOL, t
        assert rel_err(got[1][t], want[t]) <= RTOL, t


# Odd heads: the merge writes every dim once, nothing into the next head and nothing
# behind the last one; positions past ctx too.
@pytest.mark.parametrize("head", [1, 5, 63])
def test_attention_prefill_odd_heads(rt, head):
    q_heads, kv_heads, T, p0, split = 4, 2, 9, 30, 16
    seq, ctx = p0 + T, p0 + T - 1
    kv = oracle.normal(2 * seq * kv_heads * head, 272).reshape(2, seq, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 273).reshape(T, q_heads, head)
    kc, vc = (up(rt, head_major(a, kv_heads, seq, head)) for a in kv)
    out = up(rt, np.full(T * q_heads * head + 4, 7.0, np.float32))
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    call("ammon_attention_prefill", rt.handle, None, up(rt, qh), T, q_heads, kc, vc, F32, kv_heads, head,
         seq, rt.step(0, p0), ctx, split, rt.alloc(nbytes), nbytes, out)
    got = out.download(T * q_heads * head + 4)
    assert (got[T * q_heads * head:] == 7.0).all()
    got = got[:T * q_heads * head].reshape(T, q_heads, head)
    for t in range(T - 1):
        assert rel_err(got[t], oracle.attention(qh[t], kv[0], kv[1], F32, p0 + t)) <= RTOL, t
    assert np.isnan(got[T - 1]).all()


# Splits fill the workgroups that are resident at once: two per CU (the bf16 tile
# of 4:1 heads of 128), one (3:1, whose q is kept whole).  As many tiles as CUs are
# split in two in the first case and write their results themselves in the second,
# leaving the scratch as it was.
@pytest.mark.parametrize("q_heads,kv_heads,splits", [(32, 8, 2), (24, 8, 1)])
def test_attention_prefill_splits_follow_residency(rt, q_heads, kv_heads, splits):
    head, split = 128, 256
    tiles = rt.info.compute_units // kv_heads
    T = tiles * 128 // (q_heads // kv_heads)
    kv = oracle.storage(oracle.normal(2 * T * kv_heads * head, 270), BF16).reshape(2, T, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 271).reshape(T, q_heads, head)
    kc, vc = (up(rt, head_major(a, kv_heads, T, head)) for a in kv)
    out = rt.alloc(T * q_heads * head * 4)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, T, split)
    part = up(rt, np.full(nbytes // 4, 7.0, np.float32))
    call("ammon_attention_prefill", rt.handle, None, up(rt, qh), T, q_heads, kc, vc, BF16, kv_heads,
         head, T, rt.step(0, 0), T, split, part, nbytes, out)
    got, rest = out.download((T, q_heads, head)), part.download(nbytes // 4)
    used = T * q_heads * splits * (head + 2) if splits > 1 else 0
    np.testing.assert_array_equal(rest[used:], 7.0)
    assert splits == 1 or (rest[:used] != 7.0).any()
    for t in (0, 1, 127, 128, T // 2, T - 1):
        assert rel_err(got[t], oracle.attention(qh[t], kv[0], kv[1], BF16, t)) <= RTOL, t


# K and V that are not finite give what they give the oracle, whichever tile, chunk
# or split they fall into: an infinite V its infinity in its column (two of both
# signs NaN), an infinite K a NaN row or a weight of 0, and neither reaches an
# earlier token or another column.  Column 9 holds 1e36 and the first 64 scores
# are 0: its sums fit with weights of at most 1, not with weights against 0.
@pytest.mark.parametrize("q_heads,kv_heads,head,kv_dtype,p0,T,split", [
    (32, 8, 128, BF16, 0, 333, 1024), (32, 8, 128, BF16, 1100, 130, 64),
    (24, 8, 128, BF16, 0, 333, 1024), (14, 2, 96, BF16, 300, 300, 64), (15, 5, 64, BF16, 0, 500, 512),
    (32, 32, 24, BF16, 0, 700, 1024), (16, 16, 128, F32, 0, 900, 1024), (14, 2, 96, F32, 600, 300, 64),
    (32, 8, 64, F32, 1, 511, 1024), (32, 32, 32, F32, 0, 700, 1024),
])
def test_attention_prefill_not_finite(rt, q_heads, kv_heads, head, kv_dtype, p0, T, split):
    seq = ctx = p0 + T
    k, v = (oracle.normal(seq * kv_heads * head, s).reshape(seq, kv_heads, head) for s in (267, 268))
    qh = oracle.normal(T * q_heads * head, 269).reshape(T, q_heads, head)
    k[:64] = 0
    v[:, :, 9] = 1e36
    v[17, :, 3] = v[40, :, 5] = np.inf
    v[90, :, 5] = -np.inf
    v[100, :, 7] = np.nan
    v[p0 + T // 2, :, 1] = -np.inf
    k[p0 + T // 2 + 2, 0, 4] = np.inf
    kp, vp = (oracle.storage(a.ravel(), kv_dtype).reshape(seq, kv_heads, head) for a in (k, v))
    kc, vc = (up(rt, head_major(a, kv_heads, seq, head)) for a in (kp, vp))
    out = rt.alloc(T * q_heads * head * 4)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    call("ammon_attention_prefill", rt.handle, None, up(rt, qh), T, q_heads, kc, vc, kv_dtype,
         kv_heads, head, seq, rt.step(0, p0), ctx, split, rt.alloc(nbytes), nbytes, out)
    got = out.download((T, q_heads, head))
    late = T // 2
    edges = {0, 1, 16, 17, 39, 40, 41, 63, 64, 90, 101, late - 1, late, late + 1, late + 2, late + 3, T - 1}
    for t in sorted(edges | set(range(0, T, 13))):
        want = oracle.attention_serial(qh[t], kp, vp, kv_dtype, p0 + t)
        np.testing.assert_array_equal(np.isnan(got[t]), np.isnan(want), err_msg=str(t))
        same = np.isinf(want)
        np.testing.assert_array_equal(got[t][same], want[same], err_msg=str(t))
        for cols in (np.arange(head) != 9, np.arange(head) == 9):
            use = np.isfinite(want) & cols
            if use.any():
                assert rel_err(got[t][use], want[use]) <= RTOL, t


# Long contexts: the tiles' sums (up to 2048 positions each) are no further off
# than the units', which run the same tokens one by one.  q = 0 makes every weight
# exactly 1: only the value sums are left to round.  Over 24 tokens x 8 heads x 128
# outputs the two root mean squares are known within 1 / sqrt(2 x 24576), 0.5%.
@pytest.mark.parametrize("ctx", [16384, 32768])
@pytest.mark.parametrize("q_heads,kv_heads,kv_dtype", [(8, 1, BF16), (8, 1, F32), (6, 1, BF16)])
@pytest.mark.parametrize("q_scale", [0.0, 1.0])
def test_attention_prefill_long_context_error(rt, q_heads, kv_heads, kv_dtype, ctx, q_scale):
    head, T, split = 128, 8192, 1024
    p0 = ctx - T
    k = oracle.storage(oracle.normal(ctx * head, 264), kv_dtype).reshape(ctx, head)
    v = oracle.storage(oracle.normal(ctx * head, 265), kv_dtype).reshape(ctx, head)
    qh = (oracle.normal(T * q_heads * head, 266) * np.float32(q_scale)).reshape(T, q_heads, head)
    kc, vc, q, out = up(rt, k), up(rt, v), up(rt, qh), rt.alloc(T * q_heads * head * 4)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    part = rt.alloc(nbytes)

    def attention(at, tokens, first):
        call("ammon_attention_prefill", rt.handle, None, at, tokens, q_heads, kc, vc, kv_dtype,
             kv_heads, head, ctx, rt.step(0, first), first + tokens, split, part, nbytes, out)
        return out.download((T, q_heads, head))

    kw, vw = (oracle.widen(a, kv_dtype).astype(np.float64) for a in (k, v))
    tiles = attention(q, T, p0)
    off = {"tiles": 0.0, "units": 0.0}
    for t in range(T // 24 - 1, T, T // 24):
        n = p0 + t + 1
        s = qh[t].astype(np.float64) @ kw[:n].T / np.sqrt(head)
        w = np.exp(s - s.max(-1, keepdims=True))
        want = (w @ vw[:n]) / w.sum(-1, keepdims=True)
        unit = attention(ctypes.c_void_p(q.ptr + t * q_heads * head * 4), 1, p0 + t)[0]
        off["tiles"] += np.square(tiles[t] - want).sum() / np.square(want).mean()
        off["units"] += np.square(unit - want).sum() / np.square(want).mean()
    print({n: (x / (24 * q_heads * head)) ** 0.5 for n, x in off.items()})
    assert off["tiles"] <= off["units"] * 1.01 ** 2


@pytest.mark.parametrize("kv_dtype", [F32, BF16])
def test_attention_prefill_positions_past_ctx_are_poisoned(rt, kv_dtype):
    # The grid and the scratch cover ctx positions; the host cannot see
    # step->position, so a token at position >= ctx (but < seq) must get NaN
    # and write no partial instead of silently dropping the keys past ctx.
    q_heads, kv_heads, head, seq, split, T, ctx, p0 = 4, 2, 64, 64, 8, 6, 20, 17
    kc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 251), kv_dtype).reshape(
        seq, kv_heads, head)
    vc_pm = oracle.storage(oracle.normal(seq * kv_heads * head, 252), kv_dtype).reshape(
        seq, kv_heads, head)
    qh = oracle.normal(T * q_heads * head, 253).reshape(T, q_heads, head)
    kc, vc = up(rt, head_major(kc_pm, kv_heads, seq, head)), up(rt, head_major(vc_pm, kv_heads, seq, head))
    q, out = up(rt, qh), rt.alloc(T * q_heads * head * 4)
    nbytes = _abi.lib.ammon_attention_prefill_scratch_bytes(T, q_heads, head, ctx, split)
    part_h = np.full(nbytes // 4, 7.0, np.float32)  # a sentinel no write leaves
    part = up(rt, part_h)
    step = rt.step(0, p0)
    call("ammon_attention_prefill", rt.handle, None, q, T, q_heads, kc, vc, kv_dtype, kv_heads,
         head, seq, step, ctx, split, part, nbytes, out)
    got = out.download((T, q_heads, head))
    live = ctx - p0  # tokens at positions p0 .. ctx - 1
    for t in range(live):
        want = oracle.attention(qh[t], kc_pm, vc_pm, kv_dtype, p0 + t)
        assert rel_err(got[t], want) <= RTOL, t
    assert np.isnan(got[live:]).all()
    splits = _abi.lib.ammon_attention_splits(ctx, split)
    per_token = q_heads * splits * (head + 2)
    after = part.download(nbytes // 4)
    np.testing.assert_array_equal(after[live * per_token:], 7.0)


def test_attention_prefill_validation(rt):
    q = up(rt, np.zeros((2, 2, 64), np.float32))
    kc = up(rt, np.zeros((1, 16, 64), np.float32))
    step = rt.step(0, 0)
    out = rt.alloc(2 * 2 * 64 * 4)
    part = rt.alloc(1 << 16)
    with pytest.raises(AmmonError, match="ctx"):
        call("ammon_attention_prefill", rt.handle, None, q, 2, 2, kc, kc, F32, 1, 64, 16, step, 17,
             8, part, 1 << 16, out)
    with pytest.raises(AmmonError, match="partial scratch"):
        call("ammon_attention_prefill", rt.handle, None, q, 2, 2, kc, kc, F32, 1, 64, 16, step, 16,
             8, part, 16, out)


# ---- model ----------------------------------------------------------------------------------
@pytest.mark.parametrize("heads,kv_dtype,w_dtype", [((32, 8), BF16, BF16), ((4, 4), F32, F32),
                                                    ((8, 2), F32, BF16)])
def test_model_prefill_matches_stepping(rt, heads, kv_dtype, w_dtype):
    n_heads, n_kv = heads
    cfg = oracle.LlamaConfig(dim=128 * n_heads if n_heads > 4 else 256, n_layers=2,
                             n_heads=n_heads, n_kv_heads=n_kv, hidden=1544, vocab=5003,
                             max_seq=300, theta=500000.0, w_dtype=w_dtype, kv_dtype=kv_dtype)
    stepped = LlamaModel.synthetic(rt, cfg, seed=41, std=0.05)
    filled = LlamaModel(rt, cfg, stepped.weights)
    # 100 tokens: the 64-token GEMM tiles for bf16 weights
    prompt = [int(t) for t in np.arange(100) * 131 % 5003]
    for pos, tok in enumerate(prompt):
        want = stepped.step(tok, pos)
    got = filled.prefill(prompt)
    # fp32 KV: only summation order differs; bf16 KV: a last-bit difference
    # in an fp32 K/V value can flip its bf16 rounding by one ulp
    tol = 1e-4 if kv_dtype == F32 else BF16_KV_TOL
    kv_tol = 1e-4 if kv_dtype == F32 else KV_STORE_TOL
    assert rel_err(got, want) <= tol
    for l in range(cfg.n_layers):
        for g, w in zip(filled.kv_layer(l), stepped.kv_layer(l)):
            g, w = oracle.widen(g, kv_dtype), oracle.widen(w, kv_dtype)  # bf16 storage bits
            assert rel_err(g[: len(prompt)], w[: len(prompt)]) <= kv_tol
            np.testing.assert_array_equal(g[len(prompt):], 0)
    # decoding on from the prefilled cache gives the stepped model's tokens
    nxt = oracle.sample_argmax(want)
    np.testing.assert_array_equal(filled.decode(nxt, len(prompt), 12, read_tokens=True),
                                  stepped.decode(nxt, len(prompt), 12, read_tokens=True))
    # the prefill entry also works mid-sequence (a second chunk of positions)
    more = [3, 17, 400, 5002, 1]
    p0 = len(prompt) + 12
    for i, tok in enumerate(more):
        want2 = stepped.step(tok, p0 + i)
    assert rel_err(filled.prefill(more, p0), want2) <= tol
    filled.close()
    stepped.close()


def test_generate_prefill_matches_device_loop(rt):
    cfg = oracle.LlamaConfig(dim=512, n_layers=2, n_heads=4, n_kv_heads=2, hidden=1024,
                             vocab=3001, max_seq=128, theta=500000.0, w_dtype=BF16,
                             kv_dtype=F32)
    m = LlamaModel.synthetic(rt, cfg, seed=43, std=0.05)
    prompt = [5, 900, 2999, 17, 4, 4, 1200, 31, 77, 2048, 6]
    toks_d, logits_d, _ = m.generate_tokens_device(prompt, 60)
    toks_p, logits_p, tps = m.generate_tokens_prefill(prompt, 60)
    np.testing.assert_array_equal(toks_p, toks_d)
    assert rel_err(logits_p, logits_d) <= 1e-4
    assert tps > 0
    # stop token and a limit inside the prompt behave as the stepped loop
    stop = int(toks_d[len(prompt) + 3])
    np.testing.assert_array_equal(m.generate_tokens_prefill(prompt, 60, stop_on=stop)[0],
                                  m.generate_tokens_device(prompt, 60, stop_on=stop)[0])
    np.testing.assert_array_equal(m.generate_tokens_prefill(prompt, 6)[0],
                                  m.generate_tokens_device(prompt, 6)[0])
    m.close()


def test_c1_prefill_greedy_matches_fixture(rt):
    f = np.load(os.path.join(HERE, "golden", "c1_greedy.npz"))
    cfg = oracle.LlamaConfig(**json.loads(str(f["config"])))
    weights = oracle.random_weights(cfg, seed=int(f["weight_seed"]), std=0.02)
    m = LlamaModel.from_host(rt, cfg, weights)
    toks, logits, _ = m.generate_tokens_prefill(f["prompt"], int(f["max_new_tokens"]))
    np.testing.assert_array_equal(toks, f["tokens"])
    assert rel_err(logits, f["logits"]) <= 1e-4
    m.close()


def test_model_prefill_validation(rt):
    cfg = oracle.LlamaConfig(dim=256, n_layers=1, n_heads=2, n_kv_heads=1, hidden=512, vocab=300,
                             max_seq=32, theta=500000.0, w_dtype=BF16, kv_dtype=BF16)
    m = LlamaModel.synthetic(rt, cfg, seed=44, std=0.05)
    with pytest.raises(AmmonError, match="outside the vocab"):
        m.prefill([1, 300])
    with pytest.raises(AmmonError, match="exceeds max_seq"):
        m.prefill(list(range(20)), 20)
    m.close()
