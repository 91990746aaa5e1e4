"""End-to-end decoder on the GPU: the dense kernels (RMSNorm, rotary + KV cache,
attention, GEMV) against CPU restatements of the Hugging Face modules the reference runs,
and the whole engine (prefill + greedy decode, graph-replayed and eager, all-resident and
offload) against the CPU reference decoder, teacher-forced on the engine's tokens."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from decoder_ref import RefDecoder, rel_l2, rmsnorm, rope, top2_gap
from helpers import bits

pytestmark = pytest.mark.gpu


def _bf16(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to(torch.bfloat16)


def _ulps(a: torch.Tensor, b: torch.Tensor) -> np.ndarray:
    x = bits(a).astype(np.int32)
    y = bits(b).astype(np.int32)
    # bf16 bit patterns -> ordered integers (sign-magnitude to two's complement)
    x = np.where(x & 0x8000, -(x & 0x7FFF), x)
    y = np.where(y & 0x8000, -(y & 0x7FFF), y)
    return np.abs(x - y)


@pytest.mark.parametrize("T,H,with_res", [(1, 4096, True), (40, 4096, True), (3, 512, False)])
def test_add_rmsnorm(cuda_device, T, H, with_res):
    from moeinfra_amd import _lib

    x, r, w = _bf16((T, H), 1), _bf16((T, H), 2), _bf16((H,), 3, 0.5)
    dev = lambda t: t.to(cuda_device)
    out = torch.empty((T, H), dtype=torch.bfloat16, device=cuda_device)
    r_out = torch.empty_like(out)
    xd, rd, wd = dev(x), dev(r), dev(w)
    _lib.check(_lib.lib().moe_add_rmsnorm_bf16(xd.data_ptr(), rd.data_ptr() if with_res else 0,
                                               wd.data_ptr(), 1e-5, T, H,
                                               r_out.data_ptr() if with_res else 0, out.data_ptr(),
                                               torch.cuda.current_stream().cuda_stream), "norm")
    torch.cuda.synchronize()
    resid = x + r if with_res else x
    if with_res:
        np.testing.assert_array_equal(bits(r_out), bits(resid))        # one bf16 add: exact
    want = rmsnorm(resid, w, 1e-5)
    u = _ulps(out.cpu(), want)
    assert u.max() <= 1 and (u > 0).mean() < 0.02                     # fp32 sum order only


def test_rope_and_cache_write(cuda_device):
    from moeinfra_amd import _lib
    from moeinfra_amd.engine.decoder import MixtralShape, rope_inv_freq

    s = MixtralShape()
    T, p0, max_seq = 5, 37, 128
    qkv = _bf16((T, s.qkv_rows), 4)
    inv = rope_inv_freq(s)
    kc = torch.zeros((s.n_kv_heads, max_seq, s.head_dim), dtype=torch.bfloat16, device=cuda_device)
    vc = torch.zeros_like(kc)
    q = torch.empty((T, s.n_heads * s.head_dim), dtype=torch.bfloat16, device=cuda_device)
    pos = torch.tensor([p0], dtype=torch.int32, device=cuda_device)
    qd, invd = qkv.to(cuda_device), inv.to(cuda_device)
    _lib.check(_lib.lib().moe_rope_kv_bf16(qd.data_ptr(), T, s.n_heads, s.n_kv_heads, s.head_dim,
                                           invd.data_ptr(), pos.data_ptr(), max_seq, q.data_ptr(),
                                           kc.data_ptr(), vc.data_ptr(),
                                           torch.cuda.current_stream().cuda_stream), "rope")
    torch.cuda.synchronize()
    nq, nkv, hd = s.n_heads, s.n_kv_heads, s.head_dim
    positions = torch.arange(p0, p0 + T)
    want_q = rope(qkv[:, :nq * hd].reshape(T, nq, hd), positions, inv).reshape(T, -1)
    want_k = rope(qkv[:, nq * hd:(nq + nkv) * hd].reshape(T, nkv, hd), positions, inv)
    want_v = qkv[:, (nq + nkv) * hd:].reshape(T, nkv, hd)
    kc, vc = kc.cpu(), vc.cpu()
    assert _ulps(q.cpu(), want_q).max() <= 1                              # cos/sin libm last bit
    assert _ulps(kc[:, p0:p0 + T].transpose(0, 1).contiguous(), want_k).max() <= 1
    np.testing.assert_array_equal(bits(vc[:, p0:p0 + T].transpose(0, 1).contiguous()), bits(want_v))
    assert not kc[:, :p0].any() and not kc[:, p0 + T:].any()              # other rows untouched


@pytest.mark.parametrize("T,p0,max_seq,hd", [(1, 0, 256, 128), (1, 71, 256, 128), (40, 0, 256, 128),
                                             (7, 20, 256, 128), (1, 3000, 4096, 128),
                                             (16, 2040, 4096, 128),
                                             # a score sums over hd / 8 lanes: 4, 8 and 32 lanes
                                             (1, 71, 256, 32), (3, 200, 512, 64), (2, 129, 256, 256)])
def test_attention(cuda_device, T, p0, max_seq, hd):
    from moeinfra_amd import _lib

    nq, nkv = 32, 8
    S = p0 + T
    q = _bf16((T, nq, hd), 5)
    k = _bf16((nkv, S, hd), 6)
    v = _bf16((nkv, S, hd), 7)
    kc = torch.zeros((nkv, max_seq, hd), dtype=torch.bfloat16)
    vc = torch.zeros_like(kc)
    kc[:, :S], vc[:, :S] = k, v
    out = torch.empty((T, nq * hd), dtype=torch.bfloat16, device=cuda_device)
    pos = torch.tensor([p0], dtype=torch.int32, device=cuda_device)
    qd, kd, vd = q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device)
    _lib.check(_lib.lib().moe_attention_bf16(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), T, nq, nkv,
                                             hd, pos.data_ptr(), max_seq, hd ** -0.5, out.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream), "attention")
    torch.cuda.synchronize()
    # Reference: eager attention in fp32 with the bf16 roundings of the bf16 module.
    K = k.float().repeat_interleave(nq // nkv, dim=0)
    V = v.float().repeat_interleave(nq // nkv, dim=0)
    sc = torch.matmul(q.float().transpose(0, 1), K.transpose(1, 2)).to(torch.bfloat16)
    sc = (sc.float() * (hd ** -0.5)).to(torch.bfloat16).float()
    mask = torch.full((T, S), float("-inf"))
    for t in range(T):
        mask[t, :p0 + t + 1] = 0.0
    p = torch.softmax(sc + mask, dim=-1).to(torch.bfloat16).float()
    want = torch.matmul(p, V).transpose(0, 1).reshape(T, nq * hd)
    assert rel_l2(out.cpu(), want) < 4e-3


def _attend(q, kc, vc, p0, ws, scaling=None):
    """moe_attention_ws_bf16 (moe_attention_bf16 with ws None) of q [T, nq, hd] on the GPU."""
    from moeinfra_amd import _lib

    (T, nq, hd), (nkv, max_seq, _) = q.shape, kc.shape
    out = torch.empty((T, nq * hd), dtype=torch.bfloat16, device=q.device)
    pos = torch.tensor([p0], dtype=torch.int32, device=q.device)
    args = (q.data_ptr(), kc.data_ptr(), vc.data_ptr(), T, nq, nkv, hd, pos.data_ptr(), max_seq,
            hd ** -0.5 if scaling is None else scaling, out.data_ptr())
    st = torch.cuda.current_stream().cuda_stream
    if ws is None:
        _lib.check(_lib.lib().moe_attention_bf16(*args, st), "attention")
    else:
        _lib.check(_lib.lib().moe_attention_ws_bf16(*args, ws.data_ptr(), ws.numel(), st), "attention")
    return out


def _attend_ref(q, k, v, p0, scaling=None):
    """Eager attention in fp32 with the bf16 roundings of the bf16 module, one query at a time
    over the keys that it sees."""
    T, nq, hd = q.shape
    grp = nq // k.shape[0]
    out = torch.empty((T, nq, hd))
    for t in range(T):
        K = k[:, :p0 + t + 1].float().repeat_interleave(grp, dim=0)
        V = v[:, :p0 + t + 1].float().repeat_interleave(grp, dim=0)
        sc = torch.einsum("hd,hkd->hk", q[t].float(), K).to(torch.bfloat16)
        sc = (sc.float() * (hd ** -0.5 if scaling is None else scaling)).to(torch.bfloat16).float()
        p = torch.softmax(sc, dim=-1).to(torch.bfloat16).float()
        out[t] = torch.einsum("hk,hkd->hd", p, V)
    return out.reshape(T, -1)


# Above 8 tokens the matrix form: row tiles of 128 (token, head of the group) rows, key tiles
# of 64 keys, taken in pairs (a lone pair by one wave group); up to 384 keys its row instances
# where the units, 1 or 2 heads of a token, are 512 or fewer.  Up to 8 tokens a row's keys are
# shared between workgroups above 384 of them.
@pytest.mark.parametrize("T,p0,max_seq,nq,nkv,hd", [
    (17, 0, 64, 4, 4, 128), (18, 46, 64, 8, 2, 64), (2, 0, 64, 4, 4, 128), (9, 50, 64, 8, 2, 64), (8, 380, 400, 8, 2, 64), (33, 95, 128, 32, 8, 128), (32, 128, 256, 4, 1, 128),
    (129, 0, 256, 2, 2, 64), (65, 127, 200, 6, 2, 128), (17, 700, 1024, 8, 8, 64),
    (5, 2500, 4096, 32, 8, 128), (40, 1000, 2048, 7, 1, 128),
    (1, 383, 4096, 32, 8, 128), (1, 384, 4096, 32, 8, 128), (1, 640, 1000, 6, 3, 64),
    (1, 8191, 8192, 8, 8, 256), (1, 2900, 4096, 8, 8, 128),
    (129, 0, 256, 16, 2, 64), (65, 127, 200, 24, 4, 128), (66, 64, 130, 16, 16, 128),
    (100, 0, 128, 16, 4, 128), (60, 0, 64, 32, 8, 64), (60, 68, 128, 32, 8, 128),
    (16, 368, 400, 32, 8, 128), (16, 369, 400, 32, 8, 128), (9, 5, 64, 7, 7, 64),
    (30, 300, 400, 32, 4, 128), (17, 3, 64, 34, 17, 64),
    (3, 700, 1024, 6, 1, 128), (8, 300, 1024, 21, 7, 64), (2, 900, 1024, 5, 5, 256)])
def test_attention_forms(cuda_device, T, p0, max_seq, nq, nkv, hd):
    """Matrix form and shared keys: against the module's arithmetic, with cache rows past the
    last key NaN; the workspace's counters return to zero, a second call repeats the bits."""
    from moeinfra_amd import _lib

    S = p0 + T
    q, k, v = _bf16((T, nq, hd), 5), _bf16((nkv, S, hd), 6), _bf16((nkv, S, hd), 7)
    kc = torch.full((nkv, max_seq, hd), float("nan"), dtype=torch.bfloat16)
    vc = kc.clone()
    kc[:, :S], vc[:, :S] = k, v
    qd, kd, vd = q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device)
    n = _lib.lib().moe_attention_workspace_bytes(T, nq, nkv, hd, max_seq)
    ws = torch.zeros((max(n, 16),), dtype=torch.uint8, device=cuda_device)
    want = _attend_ref(q, k, v, p0)
    got = _attend(qd, kd, vd, p0, ws)
    # As test_attention: bf16 rounding of the probabilities and of the output, 2^-9 each.
    assert rel_l2(got.cpu(), want) < 4e-3
    assert rel_l2(_attend(qd, kd, vd, p0, None).cpu(), want) < 4e-3
    assert not ws[:4096].any()
    assert torch.equal(_attend(qd, kd, vd, p0, ws), got)


@pytest.mark.parametrize("T,p0,hd,nq", [(40, 70, 128, 8), (130, 0, 64, 8), (20, 1500, 128, 8), (6, 1500, 128, 8),
                                        (60, 40, 128, 32), (50, 0, 64, 32), (40, 100, 128, 32)])
def test_attention_nonfinite_values(cuda_device, T, p0, hd, nq):
    """An infinity or NaN in a V row reaches the queries that see the row and no others."""
    from moeinfra_amd import _lib

    nkv, max_seq, S = 2, 2048, p0 + T
    q, k, v = _bf16((T, nq, hd), 15), _bf16((nkv, S, hd), 16), _bf16((nkv, S, hd), 17)
    clean = v.clone()
    bad = p0 + T // 2
    v[0, bad, 3], v[1, bad + 1, hd - 1] = float("inf"), float("nan")
    kc = torch.zeros((nkv, max_seq, hd), dtype=torch.bfloat16)
    vc = kc.clone()
    kc[:, :S], vc[:, :S] = k, v
    qd, kd, vd = q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device)
    n = _lib.lib().moe_attention_workspace_bytes(T, nq, nkv, hd, max_seq)
    ws = torch.zeros((max(n, 16),), dtype=torch.uint8, device=cuda_device)
    want = _attend_ref(q, k, clean, p0).reshape(T, nq, hd)
    for w in (None, ws):
        got = _attend(qd, kd, vd, p0, w).cpu().float().reshape(T, nq, hd)
        t = torch.arange(T) + p0
        hit = torch.zeros((T, nq, hd), dtype=torch.bool)
        hit[t >= bad, :nq // 2, 3] = True
        hit[t >= bad + 1, nq // 2:, hd - 1] = True
        assert not torch.isfinite(got[hit]).any() and torch.isfinite(got[~hit]).all()
        assert rel_l2(got.masked_fill(hit, 0.0), want.masked_fill(hit, 0.0)) < 4e-3


@pytest.mark.parametrize("T", [1, 8, 40])
@pytest.mark.parametrize("lost", ["one pass", "one NaN", "all"])
def test_attention_scores_of_minus_infinity(cuda_device, T, lost):
    """Keys whose scores overflow to -inf have probability zero, also where they are all that a
    workgroup sharing the row's keys has (128 keys a pass at head dim 128); a NaN among them,
    or no finite score at all, gives NaN as in the module's softmax."""
    from moeinfra_amd import _lib

    nq, nkv, hd, p0, max_seq = 8, 2, 128, 1000, 2048
    S = p0 + T
    q, k, v = _bf16((T, nq, hd), 25).abs() + 0.125, _bf16((nkv, S, hd), 26), _bf16((nkv, S, hd), 27)
    if lost == "all":
        k[:] = -3e38
    else:
        k[:, 128:256] = -3e38
    if lost == "one NaN":
        k[1, 200, 5] = float("nan")
    kc = torch.zeros((nkv, max_seq, hd), dtype=torch.bfloat16)
    vc = kc.clone()
    kc[:, :S], vc[:, :S] = k, v
    n = _lib.lib().moe_attention_workspace_bytes(T, nq, nkv, hd, max_seq)
    ws = torch.zeros((n,), dtype=torch.uint8, device=cuda_device)
    want = _attend_ref(q, k, v, p0).reshape(T, nq, hd)
    nan = torch.zeros((T, nq, hd), dtype=torch.bool)
    if lost != "one pass":
        nan[:, 0 if lost == "all" else nq // 2:] = True
    assert torch.equal(torch.isnan(want), nan)
    for w in (None, ws):
        got = _attend(q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device), p0, w)
        got = got.cpu().float().reshape(T, nq, hd)
        assert torch.equal(torch.isnan(got), nan)
        if lost != "all":
            # As test_attention: bf16 rounding of the probabilities and of the output.
            assert rel_l2(got.masked_fill(nan, 0.0), want.masked_fill(nan, 0.0)) < 4e-3


@pytest.mark.parametrize("T,hd", [(20, 128), (140, 64), (6, 128)])
@pytest.mark.parametrize("scores", ["high", "low", "both"])
@pytest.mark.parametrize("bad_value", [False, True])
def test_attention_scores_near_the_largest(cuda_device, T, hd, scores, bad_value):
    """Finite scores up to 3.3e38 in magnitude (times log2 e beyond fp32): differences are
    taken before anything is scaled.  ``bad_value``: the last V row holds an infinity, which
    takes the matrix form through its row-by-row branch and reaches the last query alone."""
    from moeinfra_amd import _lib

    nq, nkv, p0, max_seq = 4, 2, 500, 1024
    S = p0 + T
    q = torch.zeros((T, nq, hd), dtype=torch.bfloat16)
    q[:, :, 0] = 1.0
    k, v = _bf16((nkv, S, hd), 36), _bf16((nkv, S, hd), 37)
    hot = torch.rand((nkv, S), generator=torch.Generator().manual_seed(8)) < 0.1
    hot[:, 0] = True
    top, rest = {"high": (3.3e38, 2.5e38), "low": (-2.5e38, -3.3e38), "both": (3.3e38, -3.3e38)}[scores]
    k[:, :, 0] = torch.where(hot, top, rest).to(torch.bfloat16)
    clean = v.clone()
    if bad_value:
        v[:, S - 1, 3] = float("inf")
    kc = torch.zeros((nkv, max_seq, hd), dtype=torch.bfloat16)
    vc = kc.clone()
    kc[:, :S], vc[:, :S] = k, v
    n = _lib.lib().moe_attention_workspace_bytes(T, nq, nkv, hd, max_seq)
    ws = torch.zeros((max(n, 16),), dtype=torch.uint8, device=cuda_device)
    want = _attend_ref(q, k, clean, p0, 1.0).reshape(T, nq, hd)
    hit = torch.zeros((T, nq, hd), dtype=torch.bool)
    hit[T - 1, :, 3] = bad_value
    for w in (None, ws):
        got = _attend(q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device), p0, w, 1.0)
        got = got.cpu().float().reshape(T, nq, hd)
        assert torch.isfinite(got[~hit]).all() and not torch.isfinite(got[hit]).any()
        # As test_attention: bf16 rounding of the probabilities and of the output.
        assert rel_l2(got.masked_fill(hit, 0.0), want.masked_fill(hit, 0.0)) < 4e-3


@pytest.mark.parametrize("hd", [64, 128])
def test_attention_splits_join_in_order(cuda_device, hd):
    """The partial outputs of a row's key splits add up in split order, whichever workgroup
    finishes last.  With q = 0 every key has weight one; the first two splits (256 keys each)
    sum to +-2^28 and cancel, the others to 8 each, which a sum that starts with one of them
    (fp32: a unit of 32 at 2^28) loses."""
    from moeinfra_amd import _lib

    T, n, max_seq = 40, 8, 8192
    p0 = max_seq - T
    q = torch.zeros((T, n, hd), dtype=torch.bfloat16, device=cuda_device)
    k = _bf16((n, max_seq, hd), 46).to(cuda_device)
    v = torch.full((n, max_seq, hd), 2.0 ** -5, dtype=torch.bfloat16, device=cuda_device)
    v[:, :256], v[:, 256:512] = 2.0 ** 20, -(2.0 ** 20)
    ws = torch.zeros((_lib.lib().moe_attention_workspace_bytes(T, n, n, hd, max_seq),),
                     dtype=torch.uint8, device=cuda_device)
    keys = torch.arange(p0 + 1, max_seq + 1, device=cuda_device, dtype=torch.float32)
    want = ((keys - 512) / 32 / keys)[:, None].expand(T, n * hd)
    for _ in range(3):
        got = _attend(q, k, v, p0, ws)
        # one bf16 rounding (a lost split is 3.4 % off)
        assert torch.allclose(got.float(), want, rtol=2.0 ** -8, atol=0.0)


@pytest.mark.parametrize("T,p0,nq,nkv,hd", [(9, 0, 32, 8, 128), (16, 368, 32, 8, 128), (13, 40, 7, 7, 64),
                                            (17, 0, 32, 8, 128), (32, 352, 32, 8, 128), (17, 100, 34, 17, 64)])
def test_attention_short_context_by_rows(cuda_device, T, p0, nq, nkv, hd):
    """A few dozen tokens with up to 384 keys run row by row: each token's outputs have the bits
    of a call of that token alone (pairs of key tiles on the matrix cores took these prompts
    twice as long and round the probabilities before the division)."""
    from moeinfra_amd import _lib

    max_seq, S = 400, p0 + T
    q, k, v = _bf16((T, nq, hd), 55), _bf16((nkv, S, hd), 56), _bf16((nkv, S, hd), 57)
    kc = torch.full((nkv, max_seq, hd), float("nan"), dtype=torch.bfloat16)
    vc = kc.clone()
    kc[:, :S], vc[:, :S] = k, v
    qd, kd, vd = q.to(cuda_device), kc.to(cuda_device), vc.to(cuda_device)
    n = _lib.lib().moe_attention_workspace_bytes(T, nq, nkv, hd, max_seq)
    ws = torch.zeros((max(n, 16),), dtype=torch.uint8, device=cuda_device)
    want = torch.cat([_attend(qd[t:t + 1], kd, vd, p0 + t, None) for t in range(T)])
    for w in (None, ws):
        np.testing.assert_array_equal(bits(_attend(qd, kd, vd, p0, w)), bits(want))


@pytest.mark.parametrize("T,p0,nq,nkv,hd", [(9, 1000, 32, 8, 128), (16, 500, 8, 8, 64), (60, 700, 8, 1, 128)])
def test_attention_without_workspace(cuda_device, T, p0, nq, nkv, hd):
    """Without a workspace to share keys through, rows that the device holds all at once run one
    workgroup each, at any context length: the bits of one-token calls."""
    max_seq, S = 1100, p0 + T
    q, k, v = _bf16((T, nq, hd), 65), _bf16((nkv, max_seq, hd), 66), _bf16((nkv, max_seq, hd), 67)
    qd, kd, vd = q.to(cuda_device), k.to(cuda_device), v.to(cuda_device)
    want = torch.cat([_attend(qd[t:t + 1], kd, vd, p0 + t, None) for t in range(T)])
    np.testing.assert_array_equal(bits(_attend(qd, kd, vd, p0, None)), bits(want))
    assert rel_l2(want.cpu(), _attend_ref(q, k[:, :S], v[:, :S], p0)) < 4e-3


@pytest.mark.parametrize("T,N,K", [(1, 6144, 4096), (1, 4096, 4096), (1, 1000, 512), (4, 515, 1024)])
def test_gemv(cuda_device, T, N, K):
    from moeinfra_amd import _lib

    W = _bf16((N, K), 8, 0.02)
    x = _bf16((T, K), 9)
    y = torch.empty((T, N), dtype=torch.bfloat16, device=cuda_device)
    Wd, xd = W.to(cuda_device), x.to(cuda_device)
    _lib.check(_lib.lib().moe_gemv_bf16(Wd.data_ptr(), xd.data_ptr(), T, N, K, y.data_ptr(),
                                        torch.cuda.current_stream().cuda_stream), "gemv")
    torch.cuda.synchronize()
    want = (x.float() @ W.float().t()).to(torch.bfloat16)
    u = _ulps(y.cpu(), want)
    assert u.max() <= 1 and (u > 0).mean() < 0.05


# --------------------------------------------------------------------------- fused step
def _stream():
    return torch.cuda.current_stream().cuda_stream


def _unfused_norm(lib, x, res, w, eps=1e-5):
    out = torch.empty_like(x)
    r_out = torch.empty_like(x)
    _lib_check(lib.moe_add_rmsnorm_bf16(x.data_ptr(), 0 if res is None else res.data_ptr(),
                                        w.data_ptr(), eps, x.shape[0], x.shape[1], r_out.data_ptr(),
                                        out.data_ptr(), _stream()), "norm")
    return r_out, out


def _unfused_gemv(lib, W, x):
    y = torch.empty((x.shape[0], W.shape[0]), dtype=torch.bfloat16, device=x.device)
    _lib_check(lib.moe_gemv_bf16(W.data_ptr(), x.data_ptr(), x.shape[0], W.shape[0], W.shape[1],
                                 y.data_ptr(), _stream()), "gemv")
    return y


def _lib_check(rc, what):
    from moeinfra_amd import _lib

    _lib.check(rc, what)


@pytest.mark.parametrize("H,nq,nkv,hd,pos,row,with_res", [
    (4096, 32, 8, 128, 41, 7, True),     # Mixtral layer > 0
    (4096, 32, 8, 128, 0, 3, False),     # Mixtral layer 0: embedding row, no residual
    (512, 8, 2, 64, 13, -5, False),      # row ids outside the table clamp (to 0)
    (1024, 4, 4, 128, 63, 99, True),     # ... and to the last row
])
def test_qkv_rope_fused_matches_unfused(cuda_device, H, nq, nkv, hd, pos, row, with_res):
    """norm + q/k/v projection + rotary + cache write in one launch == the three kernels."""
    from moeinfra_amd import _lib
    from moeinfra_amd.engine.decoder import MixtralShape, rope_inv_freq

    lib = _lib.lib()
    rows, max_seq = 20, 64
    dev = cuda_device
    table = _bf16((rows, H), 11).to(dev)
    res = _bf16((1, H), 12).to(dev) if with_res else None
    nw = _bf16((H,), 13, 0.5).to(dev)
    W = _bf16(((nq + 2 * nkv) * hd, H), 14, 0.02).to(dev)
    inv = rope_inv_freq(MixtralShape(head_dim=hd)).to(dev)
    p0 = torch.tensor([pos], dtype=torch.int32, device=dev)
    rid = torch.tensor([row], dtype=torch.int64, device=dev)
    caches = [torch.zeros((nkv, max_seq, hd), dtype=torch.bfloat16, device=dev) for _ in range(4)]
    q_f = torch.empty((1, nq * hd), dtype=torch.bfloat16, device=dev)
    h_f = torch.empty((1, H), dtype=torch.bfloat16, device=dev)
    _lib.check(lib.moe_qkv_rope_bf16(W.data_ptr(), table.data_ptr(), rid.data_ptr(), rows,
                                     None if res is None else res.data_ptr(), nw.data_ptr(), 1e-5, H,
                                     nq, nkv, hd, inv.data_ptr(), p0.data_ptr(), max_seq,
                                     h_f.data_ptr(), q_f.data_ptr(), caches[0].data_ptr(),
                                     caches[1].data_ptr(), _stream()), "qkv_rope")
    x = table[min(max(row, 0), rows - 1)][None].contiguous()
    h_u, xn = _unfused_norm(lib, x, res, nw)
    qkv = _unfused_gemv(lib, W, xn)
    q_u = torch.empty_like(q_f)
    _lib.check(lib.moe_rope_kv_bf16(qkv.data_ptr(), 1, nq, nkv, hd, inv.data_ptr(), p0.data_ptr(),
                                    max_seq, q_u.data_ptr(), caches[2].data_ptr(),
                                    caches[3].data_ptr(), _stream()), "rope")
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bits(h_f), bits(h_u))
    np.testing.assert_array_equal(bits(q_f), bits(q_u))
    np.testing.assert_array_equal(bits(caches[0]), bits(caches[2]))   # k rows, others zero
    np.testing.assert_array_equal(bits(caches[1]), bits(caches[3]))   # v rows
    assert caches[0][:, pos].abs().sum() > 0 and not caches[0][:, :pos].any()


def test_head_argmax(cuda_device):
    """final norm + lm_head + argmax + step bookkeeping: logits equal the unfused kernels,
    the token is torch.argmax of them, ties go to the lower index, and gen[ctr] is written
    only inside gen_cap while ctr and pos always advance."""
    from moeinfra_amd import _lib

    lib = _lib.lib()
    dev = cuda_device
    V, H = 32000, 4096
    x = _bf16((1, H), 32).to(dev)
    res = _bf16((1, H), 33).to(dev)
    nw = torch.ones((H,), dtype=torch.bfloat16, device=dev)
    _, xn0 = _unfused_norm(lib, x, res, nw)
    W = _bf16((V, H), 31, 0.02).to(dev)
    # rows 777 and 20000 equal and aligned with the normalised input: a tie at the maximum
    W[777] = (xn0[0].float().sign() * 0.05).to(torch.bfloat16)
    W[20000] = W[777]
    logits = torch.empty((1, V), dtype=torch.bfloat16, device=dev)
    cu = torch.cuda.get_device_properties(dev).multi_processor_count
    cand = torch.empty((8 * 4 * cu,), dtype=torch.uint8, device=dev)
    tok = torch.full((1,), -1, dtype=torch.int64, device=dev)
    gen = torch.full((3,), -1, dtype=torch.int64, device=dev)
    gctr = torch.tensor([1], dtype=torch.int64, device=dev)
    pos = torch.tensor([9], dtype=torch.int32, device=dev)
    for cand_bytes in (cand.numel(), 8 * 3):  # full grid, then only three workgroups
        _lib.check(lib.moe_head_argmax_bf16(W.data_ptr(), x.data_ptr(), res.data_ptr(), nw.data_ptr(),
                                            1e-5, V, H, logits.data_ptr(), cand.data_ptr(),
                                            cand_bytes, tok.data_ptr(),
                                            gen.data_ptr(), gen.numel(), gctr.data_ptr(),
                                            pos.data_ptr(), _stream()), "head")
        torch.cuda.synchronize()
        _, xn = _unfused_norm(lib, x, res, nw)
        want = _unfused_gemv(lib, W, xn)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits(logits), bits(want))
        lg = want.float().cpu()[0]
        assert float(lg[777]) == float(lg[20000]) == float(lg.max())
        assert int(tok.item()) == int(torch.argmax(lg)) == 777
    assert gen.tolist() == [-1, 777, 777] and int(gctr.item()) == 3 and int(pos.item()) == 11
    # gen_ctr at the capacity: nothing written, the counter still advances
    _lib.check(lib.moe_head_argmax_bf16(W.data_ptr(), x.data_ptr(), res.data_ptr(), nw.data_ptr(),
                                        1e-5, V, H, logits.data_ptr(), cand.data_ptr(), cand.numel(),
                                        tok.data_ptr(), gen.data_ptr(), gen.numel(),
                                        gctr.data_ptr(), None, _stream()), "head")
    torch.cuda.synchronize()
    assert gen.tolist() == [-1, 777, 777] and int(gctr.item()) == 4 and int(pos.item()) == 11


@pytest.mark.parametrize("form", ["full", "small", "wide"])
def test_layer_norm_fused_matches_unfused(cuda_device, form):
    """The single-token MoE layer with the post-attention residual add + norm in its gate/up
    kernel == moe_add_rmsnorm_bf16 then moe_layer_forward_nf4, bit for bit (output,
    residual, routing weights and ids), on two calls in a row.  Hidden 4096 and 512 take the
    one-chunk-per-thread norm, 6144 the form with up to four chunks per thread."""
    from moeinfra_amd import _lib
    from moeinfra_amd.engine.decoder import MixtralShape, synthesize

    lib = _lib.lib()
    dev = cuda_device
    shape = {"full": MixtralShape(layers=1),
             "small": MixtralShape(hidden=512, ffn=1024, layers=1, n_heads=8, n_kv_heads=2,
                                   head_dim=64, vocab=64),
             "wide": MixtralShape(hidden=6144, ffn=1536, layers=1, n_heads=48, n_kv_heads=8,
                                  head_dim=128, vocab=64)}[form]
    w = synthesize(shape, seed=41, device=dev)
    lw = w.layers[0]
    H, F, E, k = shape.hidden, shape.ffn, shape.experts, shape.top_k
    nw = _bf16((H,), 42, 0.5).to(dev)
    ws_n = torch.empty((lib.moe_layer_norm_workspace_bytes(k, E, H, F),), dtype=torch.uint8, device=dev)
    ws_u = torch.empty((lib.moe_layer_workspace_bytes(1, k, E, H, F),), dtype=torch.uint8, device=dev)
    for seed in (43, 44):
        y = _bf16((1, H), seed).to(dev)
        h = _bf16((1, H), seed + 10).to(dev)
        outs = {}
        for fused in (True, False):
            r = torch.empty((1, H), dtype=torch.bfloat16, device=dev)
            out = torch.empty((1, H), dtype=torch.bfloat16, device=dev)
            wt = torch.empty((1, k), dtype=torch.float32, device=dev)
            idx = torch.empty((1, k), dtype=torch.int64, device=dev)
            if fused:
                _lib.check(lib.moe_layer_forward_nf4_norm(
                    lw.table, E, lw.gate.data_ptr(), y.data_ptr(), h.data_ptr(), nw.data_ptr(), 1e-5,
                    H, F, k, r.data_ptr(), out.data_ptr(), wt.data_ptr(), idx.data_ptr(),
                    ws_n.data_ptr(), ws_n.numel(), _stream()), "fused")
            else:
                x2 = torch.empty_like(y)
                _lib.check(lib.moe_add_rmsnorm_bf16(y.data_ptr(), h.data_ptr(), nw.data_ptr(), 1e-5, 1,
                                                    H, r.data_ptr(), x2.data_ptr(), _stream()), "norm")
                _lib.check(lib.moe_layer_forward_nf4(
                    lw.table, E, lw.gate.data_ptr(), None, x2.data_ptr(), 1, H, F, k, out.data_ptr(),
                    None, wt.data_ptr(), idx.data_ptr(), ws_u.data_ptr(), ws_u.numel(), _stream()),
                    "layer")
            torch.cuda.synchronize()
            outs[fused] = (bits(r), bits(out), wt.cpu().numpy(), idx.cpu().numpy())
        for a, b in zip(outs[True], outs[False]):
            np.testing.assert_array_equal(a, b)
        assert np.abs(outs[True][1].astype(np.int32)).sum() > 0


def test_decode_step_matches_forward(cuda_device):
    """The fused decode step == forward() + argmax, bit for bit, over several positions."""
    from moeinfra_amd.engine.decoder import NativeDecoder

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (7,), generator=torch.Generator().manual_seed(8))
    a = NativeDecoder(w, 32, cuda_device)
    b = NativeDecoder(w, 32, cuda_device)
    assert a.fused_step_supported()
    la = a.forward(prompt.to(cuda_device))
    lb = b.forward(prompt.to(cuda_device))
    tok = la.argmax(dim=-1)
    tok_b = tok.clone()
    for _ in range(5):
        lf = a.decode_step(tok)                       # writes the next token into tok
        lu = b.forward(tok_b)
        np.testing.assert_array_equal(bits(lf), bits(lu))
        tok_b = lu.argmax(dim=-1)
        assert int(tok.item()) == int(tok_b.item())
    assert int(a.pos.item()) == int(b.pos.item()) == 12
    np.testing.assert_array_equal(bits(a.k_cache), bits(b.k_cache))
    np.testing.assert_array_equal(bits(a.v_cache), bits(b.v_cache))


# --------------------------------------------------------------------------- engine
def _small_shape():
    from moeinfra_amd.engine.decoder import MixtralShape

    return MixtralShape(hidden=512, ffn=1024, layers=2, n_heads=8, n_kv_heads=2, head_dim=64,
                        vocab=640, experts=8, top_k=2)


_E2E = {}


def _small_engine_weights(device):
    if "w" not in _E2E:
        from moeinfra_amd.engine.decoder import synthesize

        _E2E["w"] = synthesize(_small_shape(), seed=5, device=device)
    return _E2E["w"]


def _check_against_reference(res, weights, prompt, tol=2e-2):
    ref = RefDecoder(weights)
    want = ref.forward(prompt[0].tolist())
    toks = res.token_ids
    logits_seen = [want]
    for t in toks[:-1]:
        logits_seen.append(ref.forward([t]))
    for step, (tok, lg) in enumerate(zip(toks, logits_seen)):
        if int(lg.argmax()) != tok:
            assert top2_gap(lg) < 0.05 * float(lg.abs().max()), (step, tok, int(lg.argmax()))
    assert rel_l2(res.logits.float().cpu().reshape(-1), logits_seen[-1].reshape(-1)) < tol


@pytest.mark.parametrize("use_graph", [True, False])
def test_engine_matches_reference(cuda_device, use_graph):
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 12), generator=torch.Generator().manual_seed(3))
    eng = InferenceEngine(w, max_seq=64, device=cuda_device, use_graph=use_graph)
    res = eng.generate(ForwardRequest(prompt, max_new_tokens=8))
    assert len(res.token_ids) == 8 and res.tps > 0 and res.ttft_ms > 0
    _check_against_reference(res, w, prompt)
    _E2E.setdefault("tokens", {})[use_graph] = (res.token_ids, bits(res.logits))


def test_engine_graph_replays_match_eager(cuda_device):
    """Graph replays give bit-identical tokens and logits to eager steps, also when the
    engine generates twice (a second prefill resets the position and cache)."""
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 9), generator=torch.Generator().manual_seed(4))
    outs = []
    for use_graph in (False, True):
        eng = InferenceEngine(w, max_seq=64, device=cuda_device, use_graph=use_graph)
        for _ in range(2):
            res = eng.generate(ForwardRequest(prompt, max_new_tokens=10))
            outs.append((res.token_ids, bits(res.logits)))
    for toks, lg in outs[1:]:
        assert toks == outs[0][0]
        np.testing.assert_array_equal(lg, outs[0][1])


@pytest.mark.parametrize("policy,slots,per_layer,evict", [
    ("NONE", 4, None, "lru"), ("NEXT_LAYER", 4, None, "lru"), ("NEXT_ROUTER", 4, None, "lru"),
    ("NONE", 3, 1, "lru"), ("NEXT_ROUTER", 6, 3, "lru"),
    ("NEXT_ROUTER", 4, None, "lfu"), ("NONE", 4, 2, "lfu"),
    ("NEXT_ROUTER", 4, None, "arc"), ("NONE", 4, 2, "arc")])
def test_engine_offload_matches_reference(cuda_device, policy, slots, per_layer, evict):
    """Offload mode: the NF4 store pinned on the host, a few GPU expert slots (fewer than a
    40-token prefill routes to per layer), the prefetch policies, the per-layer GPU tier
    that keeps transferred experts across tokens, and the LRU / LFU / ARC GPU tiers."""
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest, PrefetchPolicy
    from moeinfra_amd.transfer import scheduler as sched_mod

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 6), generator=torch.Generator().manual_seed(6))
    eng = InferenceEngine(w, max_seq=64, device=cuda_device, offload=True, gpu_expert_slots=slots,
                          prefetch=PrefetchPolicy[policy], gpu_slots_per_layer=per_layer,
                          cache_policy=evict, prefetch_prefix_bytes=None)  # whole copies
    assert eng.cache_manager.policy.value == evict
    n_prof = len(sched_mod.EXECUTE_NEXT_PROFILE)
    res = eng.generate(ForwardRequest(prompt, max_new_tokens=5))
    _check_against_reference(res, w, prompt)
    assert eng.pinned_store.pinned_bytes > 0
    assert all(p.get("source", "image") == "image"                 # never staged
               for p in sched_mod.EXECUTE_NEXT_PROFILE[n_prof:])
    used = eng.cache_manager.stats().gpu_slots_used
    if per_layer is not None:                # transferred experts are kept, per layer
        assert 0 < used <= per_layer * w.shape.layers
        assert all(sum(1 for k in eng.cache_manager._gpu_cache if k[0] == l) <= per_layer
                   for l in range(w.shape.layers))
    elif policy == "NONE":                   # the reference's contract: demoted after use
        assert used == 0


@pytest.mark.parametrize("prefix,slots,per_layer", [
    (4096, 4, None), ("half", 4, None), ("whole", 4, None), ("half", 6, 3)])
def test_engine_offload_prefix_prefetch_matches_reference(cuda_device, prefix, slots, per_layer):
    """NEXT_ROUTER with bounded prefixes: the first bytes of each guessed expert's image go
    ahead into a spare slot; the layer's transfer copies the rest into the same slot (a
    prefix of a few KB, half the image, the whole image), or the unused prefix is dropped."""
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest, PrefetchPolicy

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 6), generator=torch.Generator().manual_seed(7))
    probe = InferenceEngine(w, max_seq=64, device=cuda_device, offload=True, gpu_expert_slots=slots)
    image = probe.cache_manager.peek_cpu(0, 0).image_layout.nbytes
    del probe
    nbytes = {"half": image // 2 + 3, "whole": image}.get(prefix, prefix)
    eng = InferenceEngine(w, max_seq=64, device=cuda_device, offload=True, gpu_expert_slots=slots,
                          prefetch=PrefetchPolicy.NEXT_ROUTER, gpu_slots_per_layer=per_layer,
                          prefetch_prefix_bytes=nbytes)
    res = eng.generate(ForwardRequest(prompt, max_new_tokens=6))
    _check_against_reference(res, w, prompt)
    c = eng.prefetch_engine.counts
    assert c["prefixes"] > 0 and c["started"] == 0       # prefixes only, no whole copies
    assert c["prefixes_used"] > 0
    assert c["prefixes_used"] + c["prefixes_dropped"] <= c["prefixes"]
    assert eng.transfer_scheduler.copies["prefix"] == c["prefixes"]


def test_engine_full_mixtral_layer_matches_reference(cuda_device):
    """One decoder layer at the full Mixtral-8x7B shape (hidden 4096, 32/8 heads of 128,
    8 NF4 experts of 14336, vocab 32000): prefill of 6 tokens and 4 graph-replayed decode
    tokens against the CPU oracle decoder, teacher-forced on the engine's tokens."""
    from moeinfra_amd.engine.decoder import MixtralShape, synthesize
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest

    w = synthesize(MixtralShape(layers=1), seed=12, device=cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 6), generator=torch.Generator().manual_seed(13))
    eng = InferenceEngine(w, max_seq=32, device=cuda_device)
    res = eng.generate(ForwardRequest(prompt, max_new_tokens=5))
    assert len(res.token_ids) == 5
    _check_against_reference(res, w, prompt)


def test_engine_fills_max_seq_and_lookahead_offload(cuda_device):
    """A prompt plus generated tokens that fill the KV cache exactly, graph-replayed; and the
    offload engine with look-ahead prefetch, both against the oracle decoder."""
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest, PrefetchPolicy

    w = _small_engine_weights(cuda_device)
    prompt = torch.randint(0, w.shape.vocab, (1, 10), generator=torch.Generator().manual_seed(21))
    eng = InferenceEngine(w, max_seq=16, device=cuda_device)
    res = eng.generate(ForwardRequest(prompt, max_new_tokens=7))      # positions 0 .. 15
    assert len(res.token_ids) == 7
    _check_against_reference(res, w, prompt)
    eng = InferenceEngine(w, max_seq=32, device=cuda_device, offload=True, gpu_expert_slots=3,
                          prefetch=PrefetchPolicy.LOOKAHEAD, prefetch_depth=2)
    res = eng.generate(ForwardRequest(prompt[:, :5], max_new_tokens=4))
    _check_against_reference(res, w, prompt[:, :5])


def test_engine_rejects_bad_requests(cuda_device):
    from moeinfra_amd.engine.engine import InferenceEngine
    from moeinfra_amd.engine.types import ForwardRequest

    w = _small_engine_weights(cuda_device)
    eng = InferenceEngine(w, max_seq=16, device=cuda_device)
    with pytest.raises(ValueError):
        eng.generate(ForwardRequest(torch.zeros((12,), dtype=torch.long)))
    with pytest.raises(ValueError):
        eng.generate(ForwardRequest(torch.zeros((1, 20), dtype=torch.long)))
    with pytest.raises(ValueError):
        eng.generate(ForwardRequest(torch.zeros((1, 4), dtype=torch.long), max_new_tokens=-1))


def test_long_context_step_replays(cuda_device):
    """Decode steps that cross the length from which workgroups share a row's keys (384): a
    captured step, replayed with the program's own eager prefill between the replays, gives
    the bits of eager steps, and forward() of one token those of decode_step()."""
    from moeinfra_amd.engine.decoder import MixtralShape, NativeDecoder, synthesize

    shape = MixtralShape(hidden=512, ffn=512, layers=2, n_heads=8, n_kv_heads=2, head_dim=64, vocab=640)
    w = synthesize(shape, seed=11, device=cuda_device)
    ids = torch.randint(0, shape.vocab, (381,), generator=torch.Generator().manual_seed(4)).to(cuda_device)
    a, b, c, other = (NativeDecoder(w, 640, cuda_device) for _ in range(4))
    for d in (a, b, c):
        d.forward(ids)
    np.testing.assert_array_equal(bits(a.k_cache), bits(b.k_cache))
    toks = {d: ids[:1].clone() for d in (a, b, c)}
    a_pos, side = b.pos.clone(), torch.cuda.Stream(cuda_device)
    kv = b.k_cache.clone(), b.v_cache.clone()
    side.wait_stream(torch.cuda.current_stream(cuda_device))
    with torch.cuda.stream(side):
        b.decode_step(toks[b])
    torch.cuda.current_stream(cuda_device).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lg = b.decode_step(toks[b])
    b.pos.copy_(a_pos), b.k_cache.copy_(kv[0]), b.v_cache.copy_(kv[1]), toks[b].copy_(ids[:1])
    for step in range(7):                       # positions 381 .. 387
        want = a.decode_step(toks[a]).clone()
        graph.replay()
        other.reset()
        other.forward(ids[:40 + step])          # eager work of another decoder
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits(lg), bits(want))
        got = c.forward(toks[c])
        np.testing.assert_array_equal(bits(got), bits(want))
        toks[c].copy_(toks[a])
        assert torch.equal(toks[a], toks[b])
    assert not b._attn_ws[:4096].any()
