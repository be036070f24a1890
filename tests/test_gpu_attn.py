"""GPU parity of decode attention over the FP8 KV cache and of the KV write
(mxfp4_attn_decode, mxfp4_kv_write), the reference's attn_decode / kv_write
(src/ext/mxfp4_decode.cu:352-490).

Oracle: oracle/attn.py, pinned in tests/test_oracle_attn.py.  The KV bytes
are compared bit-exactly; attention output against the float64 oracle on the
same cache bytes with the per-op tolerance (cos >= 0.99999, norm-wise
max-rel <= 1e-4), the raw scores written to `sc` with max-rel <= 1e-5.
"""
import ctypes

import numpy as np
import pytest
import torch

from moe_fused_inference_amd import _lib
from oracle import attn
from oracle import mxfp4 as fmt
from tests.gpu_helpers import DEV, assert_close, log, np_

pytestmark = pytest.mark.gpu


def _bf16(a):
    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16()


def _mixed_values(rng, shape):
    """bf16 values over the codec's regimes: sub-2^-6, normal, ties, >= 248."""
    x = rng.standard_normal(shape).astype(np.float32)
    scale = rng.choice(np.array([1e-3, 0.02, 0.5, 3.0, 60.0, 400.0], np.float32), size=shape)
    x *= scale
    flat = x.reshape(-1)
    ties = np.array([1.0625, -1.1875, 0.03125 * 1.0625, 17.0, 240.0, 248.0, -250.0, 2.0 ** -7, 0.0, -0.0],
                    np.float32)
    flat[:ties.size] = ties
    return _bf16(x)


@pytest.mark.parametrize("M,Hkv,base,max_pos", [(1, 4, 5, 64), (9, 4, 30, 64), (4, 8, 62, 64), (3, 2, -1, 16)])
def test_kv_write_bit_exact(dext, M, Hkv, base, max_pos):
    rng = np.random.default_rng(M * 100 + Hkv + max_pos)
    D = 128
    k, v = _mixed_values(rng, (M, Hkv, D)), _mixed_values(rng, (M, Hkv, D))
    init_k = rng.integers(0, 256, size=(max_pos, Hkv, D), dtype=np.uint8)
    init_v = rng.integers(0, 256, size=(max_pos, Hkv, D), dtype=np.uint8)
    kvk, kvv = torch.from_numpy(init_k.copy()).to(DEV), torch.from_numpy(init_v.copy()).to(DEV)
    dpos = torch.tensor([base], dtype=torch.int32, device=DEV)
    dext.kv_write(k.to(DEV), v.to(DEV), kvk, kvv, dpos, M)
    torch.cuda.synchronize()
    wk, wv = attn.kv_write_ref(k.float().numpy(), v.float().numpy(), init_k.copy(), init_v.copy(), base)
    assert np.array_equal(np_(kvk), wk) and np.array_equal(np_(kvv), wv)
    written = max(0, min(M, max_pos - base)) if base >= 0 else 0
    log(f"  kv_write M={M} Hkv={Hkv} base={base}: {written} rows written, bit-exact")


def _cache(rng, max_pos, Hkv, D, scale=0.5):
    return attn.e4m3_ref_encode(rng.standard_normal((max_pos, Hkv, D)).astype(np.float32) * scale)


@pytest.mark.parametrize("M,Hq,Hkv,max_pos,base", [(1, 32, 4, 4096, 4095), (1, 32, 4, 4096, 0),
                                                  (9, 32, 4, 4096, 2000), (2, 8, 8, 256, 100),
                                                  (3, 16, 1, 300, 250), (1, 4, 2, 128, 70),
                                                  # more than 64 chunks: the two-pass merge
                                                  (2, 32, 4, 8192, 6000), (1, 8, 2, 8192, 8191)])
def test_attn_decode_vs_oracle(dext, M, Hq, Hkv, max_pos, base):
    rng = np.random.default_rng(Hq * 7 + max_pos + base)
    D = 128
    kvk_np, kvv_np = _cache(rng, max_pos, Hkv, D), _cache(rng, max_pos, Hkv, D)
    q = _bf16(rng.standard_normal((M, Hq, D)))
    sc = torch.full((M, Hq, max_pos), float("nan"), dtype=torch.float32, device=DEV)
    o = dext.attn_decode(q.to(DEV), torch.from_numpy(kvk_np).to(DEV), torch.from_numpy(kvv_np).to(DEV),
                         torch.tensor([base], dtype=torch.int32, device=DEV), sc, M)
    torch.cuda.synchronize()
    ref, scores = attn.attn_decode_ref(q.float().numpy(), kvk_np, kvv_np, base)
    assert_close(np_(o), ref, what=f"attn_decode M={M} Hq={Hq} Hkv={Hkv} S={base + 1}..")
    for m in range(M):
        S = base + m + 1
        got = np_(sc[m, :, :S]).astype(np.float64)
        err = np.abs(got - scores[m]).max() / np.abs(scores[m]).max()
        assert err <= 1e-5, (m, err)


def test_attn_decode_rows_past_the_cache_are_skipped(dext):
    """Token rows whose position falls outside [0, max_pos) write nothing
    (src/ext/mxfp4_decode.cu:378,410)."""
    rng = np.random.default_rng(5)
    M, Hq, Hkv, D, max_pos = 3, 8, 2, 128, 64
    kvk = torch.from_numpy(_cache(rng, max_pos, Hkv, D)).to(DEV)
    kvv = torch.from_numpy(_cache(rng, max_pos, Hkv, D)).to(DEV)
    q = _bf16(rng.standard_normal((M, Hq, D))).to(DEV)
    o = torch.full((M, Hq, D), float("nan"), dtype=torch.float32, device=DEV)
    sc = torch.zeros((M, Hq, max_pos), dtype=torch.float32, device=DEV)
    dpos = torch.tensor([max_pos - 1], dtype=torch.int32, device=DEV)
    lib = _lib.load()
    wsb = lib.mxfp4_attn_decode_workspace_size(M, Hq, max_pos)
    ws = torch.zeros(wsb, dtype=torch.uint8, device=DEV)
    _lib.check(lib.mxfp4_attn_decode(q.data_ptr(), kvk.data_ptr(), kvv.data_ptr(), dpos.data_ptr(), sc.data_ptr(),
                                     o.data_ptr(), M, Hq, Hkv, D, max_pos, ws.data_ptr(), wsb,
                                     torch.cuda.current_stream().cuda_stream), "attn_decode")
    torch.cuda.synchronize()
    assert not torch.isnan(o[0]).any() and torch.isnan(o[1:]).all()
    ref, _ = attn.attn_decode_ref(q.float().cpu().numpy(), np_(kvk), np_(kvv), max_pos - 1)
    assert_close(np_(o[0]), ref[0], what="last cache row")


def test_attn_decode_in_graph_follows_dpos(dext):
    """attn_decode + kv_write captured once; dpos updated between replays
    (how runtime/model_runner_v3.py:98-126 drives them)."""
    rng = np.random.default_rng(6)
    M, Hq, Hkv, D, max_pos = 1, 32, 4, 128, 512
    kvk_np, kvv_np = _cache(rng, max_pos, Hkv, D), _cache(rng, max_pos, Hkv, D)
    kvk, kvv = torch.from_numpy(kvk_np.copy()).to(DEV), torch.from_numpy(kvv_np.copy()).to(DEV)
    q = _bf16(rng.standard_normal((M, Hq, D))).to(DEV)
    k = _bf16(rng.standard_normal((M, Hkv, D))).to(DEV)
    v = _bf16(rng.standard_normal((M, Hkv, D))).to(DEV)
    dpos = torch.tensor([10], dtype=torch.int32, device=DEV)
    sc = torch.empty((M, Hq, max_pos), dtype=torch.float32, device=DEV)
    out = torch.empty((M, Hq, D), dtype=torch.float32, device=DEV)

    def step():
        dext.kv_write(k, v, kvk, kvv, dpos, M)
        out.copy_(dext.attn_decode(q, kvk, kvv, dpos, sc, M))

    step()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        step()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            step()
    torch.cuda.synchronize()
    ck, cv = kvk_np.copy(), kvv_np.copy()
    attn.kv_write_ref(k.float().cpu().numpy(), v.float().cpu().numpy(), ck, cv, 10)
    for pos in (50, 300, 511):
        dpos.fill_(pos)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        attn.kv_write_ref(k.float().cpu().numpy(), v.float().cpu().numpy(), ck, cv, pos)
        assert np.array_equal(np_(kvk), ck) and np.array_equal(np_(kvv), cv)
        ref, _ = attn.attn_decode_ref(q.float().cpu().numpy(), ck, cv, pos)
        assert_close(np_(out), ref, what=f"graph replay at dpos={pos}")


@pytest.mark.parametrize("M,Hq,Hkv,max_pos,base", [(1, 32, 4, 4096, 4095), (4, 32, 4, 1000, 700), (3, 16, 1, 200, 0),
                                                   (2, 8, 8, 128, 63)])
def test_attn_decode_mx_quantized_output(M, Hq, Hkv, max_pos, base):
    """The attention output written as MXFP4 rows of bf16(o) equals
    mxfp4_quantize_rows (bf16 mode) of the fp32 output bit for bit, o itself
    equals the plain entry point's bit for bit, on three calls in a row
    that share one workspace."""
    lib = _lib.load()
    rng = np.random.default_rng(M * 1000 + base)
    D = 128
    kvk = torch.from_numpy(_cache(rng, max_pos, Hkv, D)).to(DEV)
    kvv = torch.from_numpy(_cache(rng, max_pos, Hkv, D)).to(DEV)
    dpos = torch.tensor([base], dtype=torch.int32, device=DEV)
    sc = torch.zeros((M, Hq, max_pos), dtype=torch.float32, device=DEV)
    wsb = lib.mxfp4_attn_decode_workspace_size(M, Hq, max_pos)
    ws = torch.zeros(wsb, dtype=torch.uint8, device=DEV)
    st = torch.cuda.current_stream().cuda_stream
    for call in range(3):
        q = _bf16(rng.standard_normal((M, Hq, D)) * (1 + call)).to(DEV)
        o1 = torch.zeros((M, Hq, D), dtype=torch.float32, device=DEV)
        o2 = torch.zeros((M, Hq, D), dtype=torch.float32, device=DEV)
        oq = torch.zeros((M, Hq * D // 2), dtype=torch.uint8, device=DEV)
        os_ = torch.zeros((M, Hq * D // 32), dtype=torch.uint8, device=DEV)
        _lib.check(lib.mxfp4_attn_decode(q.data_ptr(), kvk.data_ptr(), kvv.data_ptr(), dpos.data_ptr(), sc.data_ptr(),
                                         o1.data_ptr(), M, Hq, Hkv, D, max_pos, ws.data_ptr(), wsb, st), "attn_decode")
        _lib.check(lib.mxfp4_attn_decode_mx(q.data_ptr(), kvk.data_ptr(), kvv.data_ptr(), dpos.data_ptr(),
                                            sc.data_ptr(), o2.data_ptr(), oq.data_ptr(), os_.data_ptr(), M, Hq, Hkv, D,
                                            max_pos, ws.data_ptr(), wsb, st), "attn_decode_mx")
        torch.cuda.synchronize()
        live = [m for m in range(M) if base + m < max_pos]
        assert torch.equal(o1[live], o2[live]), f"call {call}"
        rq, rs = fmt.quantize_rows(fmt.bf16_round(np_(o2).reshape(M, Hq * D)))
        assert np.array_equal(np_(oq)[live], rq[live]) and np.array_equal(np_(os_)[live], rs[live]), f"call {call}"
        ref, _ = attn.attn_decode_ref(q.float().cpu().numpy(), np_(kvk), np_(kvv), base)
        assert_close(np_(o2)[live], ref[live], what=f"attn_decode_mx call {call}")


# several tokens over a cache of more than 4096 positions: one, two and three row tiles and more than one row group,
# a split's edges (32- and 128-position multiples and their neighbours), a context far shorter than the cache, score rows
# that are not 16-byte aligned (max_pos % 4 != 0), positions outside the cache
@pytest.mark.parametrize("M,Hq,Hkv,max_pos,base", [(2, 4, 4, 4100, 4098), (2, 32, 4, 4097, 31), (3, 32, 4, 8192, 127),
                                                   (5, 32, 4, 5001, 4996), (6, 8, 8, 4224, 4223), (9, 32, 4, 6000, 5000),
                                                   (13, 16, 1, 4160, 1000), (16, 32, 2, 4352, 32), (2, 16, 16, 4104, -1),
                                                   (300, 2, 2, 4500, 4300)])
def test_attn_decode_split_vs_oracle(dext, M, Hq, Hkv, max_pos, base):
    """The context-split path: output and raw scores against the oracle; sc
    untouched past a token's position; a V cache that starts at any dword
    gives the same bits."""
    rng = np.random.default_rng(M * 11 + max_pos + base)
    kvk_np, kvv_np = _cache(rng, max_pos, Hkv, 128), _cache(rng, max_pos, Hkv, 128)
    kvk_np[5::701] = _cache(rng, max_pos, Hkv, 128, 150.0)[5::701]      # exponent field 15 among them
    kvv_np[3::97] = _cache(rng, max_pos, Hkv, 128, 300.0)[3::97]
    q = _bf16(rng.standard_normal((M, Hq, 128)))
    sc = torch.full((M, Hq, max_pos), float("nan"), dtype=torch.float32, device=DEV)
    kvk, kvv = torch.from_numpy(kvk_np).to(DEV), torch.from_numpy(kvv_np).to(DEV)
    dpos = torch.tensor([base], dtype=torch.int32, device=DEV)
    o = dext.attn_decode(q.to(DEV), kvk, kvv, dpos, sc, M)
    moved = torch.empty(kvv.numel() + 16, dtype=torch.uint8, device=DEV)[4:4 + kvv.numel()].view(kvv.shape)
    moved.copy_(kvv)
    o4 = dext.attn_decode(q.to(DEV), kvk, moved, dpos, torch.empty_like(sc), M)
    torch.cuda.synchronize()
    ref, scores = attn.attn_decode_ref(q.float().numpy(), kvk_np, kvv_np, base)
    live = [m for m in range(M) if 0 <= base + m < max_pos]
    # 21 bits of each probability, fp32 sums: ten times what 32 bits leave
    assert_close(np_(o)[live], ref[live], what=f"attn split M={M} Hq={Hq} Hkv={Hkv} base={base}", rel_max=1e-5)
    assert torch.equal(o[live], o4[live])
    for m in live[:20]:
        S = base + m + 1
        err = np.abs(np_(sc[m, :, :S]).astype(np.float64) - scores[m]).max() / np.abs(scores[m]).max()
        assert err <= 1e-5, (m, err)
    assert torch.isnan(sc[live[0], :, base + live[0] + 1:]).all()


# fewer splits than 128-position pieces of the cache, so a split's share follows the context (attn_split.hip's
# units_per_split): 128, 64, 42 and 32 splits (each merge kernel), one, two and three row tiles; a cache that is full, one
# that is nearly empty (the share at its floor), tokens on both sides of a split's edge, the first of a new round of shares;
# q of standard deviation 1, and 4, whose softmax spreads over more than 2^20
@pytest.mark.parametrize("M,Hq,Hkv,max_pos,base,qs", [
    (4, 32, 4, 23040, 23036, 1), (4, 32, 4, 23040, 700, 1), (4, 32, 4, 23040, 19966, 4), (4, 32, 4, 23040, 16380, 1),
    (9, 32, 4, 16640, 16631, 1), (9, 32, 4, 16640, 250, 4), (9, 32, 4, 16640, 12283, 4), (16, 32, 4, 8448, 8432, 1),
    (16, 32, 4, 8448, 5368, 1), (16, 32, 8, 8448, 8000, 4), (2, 8, 8, 16640, 16500, 1), (2, 8, 8, 16640, 8191, 4)])
def test_attn_decode_split_shares_vs_oracle(dext, M, Hq, Hkv, max_pos, base, qs):
    """As test_attn_decode_split_vs_oracle where splits are shares of the context."""
    rng = np.random.default_rng(M * 13 + max_pos + base)
    kvk_np, kvv_np = _cache(rng, max_pos, Hkv, 128), _cache(rng, max_pos, Hkv, 128)
    kvv_np[3::97] = _cache(rng, max_pos, Hkv, 128, 300.0)[3::97]
    q = _bf16(rng.standard_normal((M, Hq, 128)) * qs)
    sc = torch.full((M, Hq, max_pos), float("nan"), dtype=torch.float32, device=DEV)
    o = dext.attn_decode(q.to(DEV), torch.from_numpy(kvk_np).to(DEV), torch.from_numpy(kvv_np).to(DEV),
                         torch.tensor([base], dtype=torch.int32, device=DEV), sc, M)
    torch.cuda.synchronize()
    ref, scores = attn.attn_decode_ref(q.float().numpy(), kvk_np, kvv_np, base)
    assert_close(np_(o), ref, what=f"attn shares M={M} Hq={Hq} Hkv={Hkv} base={base} q*{qs}", rel_max=1e-5)
    for m in range(M):
        S = base + m + 1
        err = np.abs(np_(sc[m, :, :S]).astype(np.float64) - scores[m]).max() / np.abs(scores[m]).max()
        assert err <= 1e-5, (m, err)
        assert torch.isnan(sc[m, :, S:]).all()


# one score of q * sqrt(128) / 16 of a context's n = base + 1 .. positions, 0 for the others; the values' codes at that
# position and at the others.  The weight of a small score against the large one is rounded in its exponent (below 2^5, so
# by 2^-20) where the scores' scale is applied, where a wave takes its reference and where records are merged: 3 * 2^-20 *
# ln 2 = 2e-6, which the result follows where the small terms make it up, and by a fortieth of that in the first case
@pytest.mark.parametrize("M,Hkv,max_pos,base,a,first,rest,tol", [
    (16, 2, 65536, 65515, 1.546875, 0x38, 0x58, 1e-6),     # e^17.5 against 65520 ones, values 1 and 16
    (16, 2, 65536, 65515, 1.546875, 0x01, 0x78, 3e-6),     # values 2^-6 and 448
    (16, 2, 65536, 65515, 1.890625, 0x01, 0x78, 3e-6),     # e^21.4
    (9, 4, 23040, 22992, 1.234375, 0x01, 0x78, 3e-6),      # e^14
    (9, 4, 23040, 22992, 1.890625, 0x00, 0x38, 3e-6),      # the large one's value is 0
    (2, 4, 8192, 37, 1.546875, 0x01, 0x78, 3e-6),          # all in two units of one wave each
    (5, 8, 4200, 4100, 6.0, 0x00, 0x38, 1.2e-5)])          # e^67.9: exponents up to 2^7, rounded by 2^-18
def test_attn_decode_split_one_large_score(dext, M, Hkv, max_pos, base, a, first, rest, tol):
    """A position that takes most of the weight leaves the sum of the many small
    ones, whose probabilities keep their bits at any size."""
    Hq = 32
    kvk = torch.zeros((max_pos, Hkv * 128), dtype=torch.uint8, device=DEV)
    kvv = torch.full_like(kvk, rest)
    kvk[0], kvv[0] = 0x38, first                                         # 1
    q = torch.full((M, Hq, 128), a, dtype=torch.bfloat16, device=DEV)
    o = dext.attn_decode(q, kvk.view(max_pos, Hkv, 128), kvv.view(max_pos, Hkv, 128),
                         torch.tensor([base], dtype=torch.int32, device=DEV),
                         torch.empty((M, Hq, max_pos), dtype=torch.float32, device=DEV), M)
    torch.cuda.synchronize()
    vf, vr = (float(attn.e4m3_ref_decode(np.uint8(c))) for c in (first, rest))
    w = np.exp(-a * 128 / np.sqrt(128.0))
    n = base + np.arange(M, dtype=np.float64)
    ref = ((vf + vr * w * n) / (1 + w * n))[:, None, None]
    err = np.abs(np_(o) / ref - 1).max()
    log(f"  one large score, M={M} base={base} a={a}: {err:.2e}")
    assert err <= tol


@pytest.mark.parametrize("M,Hq,Hkv,scale", [(2, 8, 2, 28), (9, 32, 4, 28), (3, 32, 4, 60)])
def test_attn_decode_split_scores_past_fp32_resolution(dext, M, Hq, Hkv, scale):
    """Scores so large that their exponents are whole numbers of bits apart: the
    largest takes all, as in the oracle."""
    rng = np.random.default_rng(77)
    max_pos, base = 4352, 4300
    kvk_np, kvv_np = _cache(rng, max_pos, Hkv, 128), _cache(rng, max_pos, Hkv, 128)
    q = _bf16(rng.standard_normal((M, Hq, 128)) * 2.0 ** scale)
    o = dext.attn_decode(q.to(DEV), torch.from_numpy(kvk_np).to(DEV), torch.from_numpy(kvv_np).to(DEV),
                         torch.tensor([base], dtype=torch.int32, device=DEV),
                         torch.empty((M, Hq, max_pos), dtype=torch.float32, device=DEV), M)
    torch.cuda.synchronize()
    ref, _ = attn.attn_decode_ref(q.float().numpy(), kvk_np, kvv_np, base)
    assert_close(np_(o), ref, what=f"attn split, scores of 2^{scale}, M={M}", rel_max=1e-5)


def test_attn_decode_split_rows_without_numbers(dext):
    """Query rows with infinities and NaN have NaN where a token alone has it,
    and the rows that share their tiles keep their results."""
    rng = np.random.default_rng(3)
    M, Hq, Hkv, max_pos, base = 3, 32, 4, 4352, 4300
    kvk, kvv = (torch.from_numpy(_cache(rng, max_pos, Hkv, 128)).to(DEV) for _ in range(2))
    good = _bf16(rng.standard_normal((M, Hq, 128))).to(DEV)
    bad = good.clone()
    bad[0, 0], bad[0, 5, 3], bad[1, 9, 7], bad[2, 31, 0] = float("nan"), float("inf"), -float("inf"), float("nan")
    hit = torch.zeros((M, Hq), dtype=torch.bool, device=DEV)
    hit[0, 0] = hit[0, 5] = hit[1, 9] = hit[2, 31] = True

    def attend(q, first, n):
        sc = torch.empty((n, Hq, max_pos), dtype=torch.float32, device=DEV)
        return dext.attn_decode(q[first:first + n].contiguous(), kvk, kvv,
                                torch.tensor([base + first], dtype=torch.int32, device=DEV), sc, n)

    clean, o = attend(good, 0, M), attend(bad, 0, M)
    alone = torch.cat([attend(bad, m, 1) for m in range(M)])
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(o), torch.isnan(alone)) and torch.isnan(o[hit]).all()
    # (a tile with an infinite reference rounds the products in the exponents of its other rows too: below 2^5 here, 2^-20)
    assert_close(np_(o[~hit]), np_(clean[~hit]), what="rows beside", rel_max=1e-5)


@pytest.mark.parametrize("Hq,Hkv,max_pos,base", [(32, 4, 4096, 4000), (8, 8, 4096, 63), (32, 4, 4352, 4200)])
def test_attn_decode_token_alone_and_in_company(dext, Hq, Hkv, max_pos, base):
    """A token's result up to max_pos 4096 has the same bits in any company;
    past it, one token and several take different sums of the same terms: the
    chunk pass's 16 bits of a probability (2e-6 in the sums) apart."""
    rng = np.random.default_rng(max_pos + base)
    M = 9
    kvk, kvv = (torch.from_numpy(_cache(rng, max_pos, Hkv, 128)).to(DEV) for _ in range(2))
    q = _bf16(rng.standard_normal((M, Hq, 128))).to(DEV)

    def attend(first, n):
        sc = torch.empty((n, Hq, max_pos), dtype=torch.float32, device=DEV)
        return dext.attn_decode(q[first:first + n].contiguous(), kvk, kvv,
                                torch.tensor([base + first], dtype=torch.int32, device=DEV), sc, n)

    whole = attend(0, M)
    for first, n in ((0, 1), (4, 1), (8, 1), (0, 4), (3, 5)):
        part = attend(first, n)
        torch.cuda.synchronize()
        if max_pos <= 4096:
            assert torch.equal(part, whole[first:first + n]), (first, n)
        else:
            assert_close(np_(part), np_(whole[first:first + n]), what=f"tokens {first}..{first + n - 1}", rel_max=1e-5)


@pytest.mark.parametrize("codec", [0, 1])
def test_attn_decode_fused_split_matches_two_ops(codec):
    """Past 4096 positions mxfp4_attn_decode_fused with several tokens still
    equals qk_norm_rope_kv followed by attn_decode_mx bit for bit."""
    from tests.test_gpu_decode_step import test_attn_decode_fused_matches_two_ops as check
    check(5, 32, 4, 6001, 5998, codec)


@pytest.mark.parametrize("M,Hq,Hkv,max_pos,base", [(1, 32, 4, 300, 290), (5, 8, 8, 200, 190)])
def test_attn_decode_chunks_every_byte(dext, M, Hq, Hkv, max_pos, base):
    """The chunk pass over caches that hold every codec byte, exponent fields 0
    and 15 among them."""
    rng = np.random.default_rng(M + Hq)
    kvk_np = rng.integers(0, 256, size=(max_pos, Hkv, 128), dtype=np.uint8)
    kvv_np = rng.integers(0, 256, size=(max_pos, Hkv, 128), dtype=np.uint8)
    q = _bf16(rng.standard_normal((M, Hq, 128)) * 1e-3)      # scores of order one
    sc = torch.empty((M, Hq, max_pos), dtype=torch.float32, device=DEV)
    o = dext.attn_decode(q.to(DEV), torch.from_numpy(kvk_np).to(DEV), torch.from_numpy(kvv_np).to(DEV),
                         torch.tensor([base], dtype=torch.int32, device=DEV), sc, M)
    torch.cuda.synchronize()
    ref, _ = attn.attn_decode_ref(q.float().numpy(), kvk_np, kvv_np, base)
    assert_close(np_(o), ref, what=f"every cache byte, M={M}")
