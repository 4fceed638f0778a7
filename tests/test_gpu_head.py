"""GPU parity of the vocabulary-chunked LM head (dk_head_chunk / dk_head_finalize between the
fp16-weight GEMMs) with the oracle: loss, entropy, argmax hit and lse per row, and d(hidden), on a
ragged last chunk, rows without a target, and a batch with no targets at all."""

import numpy as np
import pytest

from tests.helpers import assert_close, host, log

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    return t


def _case(n, v, d, seed, frac_no_target):
    rng = np.random.default_rng(seed)
    y = rng.standard_normal((n, d)).astype(np.float16)
    emb = (rng.standard_normal((v, d)) * 0.05).astype(np.float16)
    tgt = rng.integers(0, v, n).astype(np.int32)
    tgt[rng.random(n) < frac_no_target] = -1
    return y, emb, tgt


# chunk widths from 1024 to 65,536 columns (the full-vocabulary test below: 32,768 and a last
# chunk of 20,864), with a ragged last chunk in each case but the second
@pytest.mark.parametrize("n,v,chunk,frac,gscale", [(300, 9984, 4096, 0.2, 4.0),
                                                   (64, 4096, 1024, 1.0, 1.0),
                                                   (64, 20480, 16384, 0.5, 1.0),
                                                   (48, 70016, 65536, 0.8, 2.0)])
def test_streamed_head(torch, n, v, chunk, frac, gscale):
    from decentrik_prime_amd import k_head
    from oracle import head
    d = 1536
    log(f"LM head N={n} V={v} chunk={chunk}")
    y, emb, tgt = _case(n, v, d, 11 + n, frac)
    perm = np.concatenate([np.nonzero(tgt >= 0)[0], np.nonzero(tgt < 0)[0]]).astype(np.int32)
    tgt_sorted = tgt[perm]
    n_lab = int((tgt >= 0).sum())
    temb = torch.from_numpy(emb).cuda()
    src = k_head.ResidentEmbedding(temb, chunk)
    tps = torch.from_numpy(tgt_sorted).cuda()
    et = temb.index_select(0, tps[:n_lab].long()).contiguous()
    loss, stats, dy = k_head.streamed_head(torch.from_numpy(y).cuda(), src, tps,
                                           torch.from_numpy(perm).cuda(), n_lab, et, gscale)
    torch.cuda.synchronize()
    ref_stats, ref_dy = head.head(y, emb, tgt, gscale)
    got = np.empty_like(ref_stats)
    got[perm] = host(stats)                       # sorted order -> token order
    assert_close(got[:, 0], ref_stats[:, 0], 2e-3, 2e-3, "loss")
    assert_close(got[:, 1], ref_stats[:, 1], 2e-3, 2e-3, "entropy")
    assert_close(got[:, 3], ref_stats[:, 3], 1e-3, 2e-3, "lse")
    # argmax hits agree wherever the top two logits are not within a GEMM rounding of each other
    x = np.sort(head.logits16(y, emb).astype(np.float64), 1)
    clear = (x[:, -1] - x[:, -2]) > 2e-2
    assert np.array_equal(got[clear, 2], ref_stats[clear, 2]), "argmax hits"
    assert abs(float(loss) - ref_stats[:, 0].sum()) <= 2e-3 * max(1.0, abs(ref_stats[:, 0].sum()))
    s = float(np.abs(ref_dy).max()) or 1.0
    assert_close(host(dy).astype(np.float64) / s, ref_dy / s, 1e-2, 2e-2, "d(hidden)")
    assert not np.any(host(dy)[tgt < 0]), "rows without a target get a zero gradient"


def test_streamed_head_full_vocabulary(torch):
    """Qwen2.5's 151,936-token vocabulary at the default chunk (four full chunks of 32,768 and a
    partial last chunk of 20,864), a few dozen rows: targets in the last partial chunk and on
    chunk boundaries, and argmax ties planted across chunk boundaries and inside the last chunk
    (two identical embedding rows that are a row's clear maximum: the first index is the argmax,
    so the hit is 1 only when the target is the first of the pair)."""
    from decentrik_prime_amd import k_head
    from oracle import head
    n, v, d = 48, 151936, 1536
    chunk = k_head.CHUNK
    log(f"LM head N={n} V={v} chunk={chunk}")
    y, emb, tgt = _case(n, v, d, 123, 0.1)
    rng = np.random.default_rng(124)
    last0 = (v // chunk) * chunk                       # first column of the partial last chunk
    tgt[8:32] = rng.integers(last0, v, 24)             # targets in the last partial chunk
    tgt[32:36] = [chunk - 1, chunk, 2 * chunk - 1, last0]   # targets on chunk boundaries
    # (row, first column of an identical pair or None for a single planted maximum, target)
    planted = [(0, chunk - 1, chunk - 1), (1, 2 * chunk - 1, 2 * chunk), (2, v - 2, v - 1),
               (3, None, last0), (4, 3 * chunk - 1, 3 * chunk - 1), (5, 3 * chunk + 7, 3 * chunk + 8)]
    cols = [c for _, c, t in planted for c in ((t,) if c is None else (c, c + 1))]
    assert len(set(cols)) == len(cols), "planted columns overlap"
    for row, c, t in planted:
        e = (y[row].astype(np.float32) * 0.01).astype(np.float16)
        if c is None:
            emb[t] = e
        else:
            emb[c] = emb[c + 1] = e
        tgt[row] = t
    perm = np.concatenate([np.nonzero(tgt >= 0)[0], np.nonzero(tgt < 0)[0]]).astype(np.int32)
    tgt_sorted = tgt[perm]
    n_lab = int((tgt >= 0).sum())
    temb = torch.from_numpy(emb).cuda()
    src = k_head.ResidentEmbedding(temb)
    assert src.chunk == chunk and src.n_chunks == 5
    tps = torch.from_numpy(tgt_sorted).cuda()
    et = temb.index_select(0, tps[:n_lab].long()).contiguous()
    loss, stats, dy = k_head.streamed_head(torch.from_numpy(y).cuda(), src, tps,
                                           torch.from_numpy(perm).cuda(), n_lab, et, 2.0)
    torch.cuda.synchronize()
    ref_stats, ref_dy = head.head(y, emb, tgt, 2.0)
    got = np.empty_like(ref_stats)
    got[perm] = host(stats)
    assert_close(got[:, 0], ref_stats[:, 0], 2e-3, 2e-3, "loss")
    assert_close(got[:, 1], ref_stats[:, 1], 2e-3, 2e-3, "entropy")
    assert_close(got[:, 3], ref_stats[:, 3], 1e-3, 2e-3, "lse")
    for row, c, t in planted:
        want = 1.0 if (c is None or t == c) else 0.0
        assert got[row, 2] == want == ref_stats[row, 2], f"row {row}: argmax hit at target {t}"
    x = np.sort(head.logits16(y, emb).astype(np.float64), 1)
    clear = (x[:, -1] - x[:, -2]) > 2e-2
    assert np.array_equal(got[clear, 2], ref_stats[clear, 2]), "argmax hits"
    assert abs(float(loss) - ref_stats[:, 0].sum()) <= 2e-3 * max(1.0, abs(ref_stats[:, 0].sum()))
    s = float(np.abs(ref_dy).max()) or 1.0
    assert_close(host(dy).astype(np.float64) / s, ref_dy / s, 1e-2, 2e-2, "d(hidden)")
    assert not np.any(host(dy)[tgt < 0]), "rows without a target get a zero gradient"


@pytest.mark.parametrize("vc", [8, 2040, 2048, 8184, 8192, 8200, 10248])
def test_chunk_rows(torch, vc):
    """The row kernel alone at the edges of its strides (256 threads x 8 columns x 4 pieces), with
    ties, infinite logits, rows of -inf and a NaN.  The sums' bound: vc / 512 + 24 roundings (a
    thread's two chains, then the lanes' and waves' sums), 2 ulp per exponential, and z's own
    rounding, |z| 2^-24 of e^z with |z| under 26 where it counts; P is a rounding to fp16 of values
    within that of the exact ones."""
    from decentrik_prime_amd import _lib
    lib = _lib.lib()
    rng = np.random.default_rng(vc)
    n, n_lab, d, v0, scale = 12, 9, 64, 40, 64.0
    x = (rng.standard_normal((n, vc)) * 3).astype(np.float16)
    top = x.max(1)
    x[1, [vc // 2, vc - 1]] = top[1] + np.float16(1)            # a tie: the first counts
    x[2, : vc // 2] = -np.inf
    x[3] = -np.inf
    x[3, vc - 3] = -5.0
    x[4] = np.float16(-60000.0)                                 # far from the maximum: e^z is 0
    x[4, 5] = 60000.0
    x[5] = np.float16(2.0)                                      # all equal
    x[11, 3] = np.nan
    tgt = rng.integers(v0, v0 + vc, n).astype(np.int32)
    tgt[6], tgt[7] = v0 - 1, v0 + vc                            # outside the chunk
    tgt[9:] = -1
    lg, st = torch.from_numpy(x).cuda(), torch.zeros(n, 8, device="cuda")
    st[:, 0] = float("-inf")
    acc = torch.ones(n, d, device="cuda")
    t = torch.from_numpy(tgt).cuda()
    log(f"head rows, {vc} columns")
    rc = lib.dk_head_chunk(_lib.ptr(lg), _lib.ptr(t), _lib.ptr(st), _lib.ptr(acc), n, n_lab, vc, v0,
                           scale, d, _lib.stream_handle(lg.device))
    _lib.check(rc, "dk_head_chunk")
    p, got = host(lg), host(st).astype(np.float64)
    assert np.isnan(got[11, 1])
    x64 = x[:11].astype(np.float64)
    m = x64.max(1)
    z = x64 - m[:, None]
    ev = np.exp(z)
    bound = (vc / 512 + 24 + 4 + 26) * 2.0 ** -24
    assert np.array_equal(got[:11, 0], m) and np.array_equal(got[:11, 3], x64.argmax(1) + v0)
    assert np.all(np.abs(got[:11, 1] - ev.sum(1)) <= bound * ev.sum(1)), "s"
    ok = [r for r in range(11) if r not in (2, 3)]              # 0 x -inf there, as in the definition
    tt = (ev[ok] * z[ok]).sum(1)
    assert np.all(np.abs(got[ok, 2] - tt) <= bound * np.abs(tt) + 2.0 ** -120), "t"
    assert np.isnan(got[2, 2]) and np.isnan(got[3, 2])
    inside = (tgt[:11] >= v0) & (tgt[:11] < v0 + vc)
    rows = np.nonzero(inside)[0]
    assert np.array_equal(got[rows, 4], x64[rows, tgt[rows] - v0])
    want = ev[:n_lab] * scale
    for r in range(n_lab):
        if inside[r]:
            want[r, tgt[r] - v0] = 0.0
    assert np.all(np.abs(p[:n_lab] - want) <= (2.0 ** -11 + 2.0 ** -18) * want + 2.0 ** -25), "P"
    assert np.array_equal(p[n_lab:], x[n_lab:], equal_nan=True), "rows without a target stay"


def test_chunk_rows_small_probabilities(torch):
    """Probabilities below the normal range count: with a scale of 2^126 they come out in P.  e^z is
    a multiple of 2^-149, half of which is the bound's last term; the first is P's own rounding and
    2 ulp of e^z, the second half the smallest subnormal of fp16."""
    from decentrik_prime_amd import _lib
    lib = _lib.lib()
    vc, scale = 4096, 2.0 ** 126
    log("head rows, probabilities below the normal range")
    x = np.zeros((1, vc), dtype=np.float16)
    x[0, 1:] = -np.linspace(87.5, 102.0, vc - 1).astype(np.float16)
    lg, st = torch.from_numpy(x).cuda(), torch.zeros(1, 8, device="cuda")
    st[:, 0] = float("-inf")
    acc, t = torch.zeros(1, 64, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(lib.dk_head_chunk(_lib.ptr(lg), _lib.ptr(t), _lib.ptr(st), _lib.ptr(acc), 1, 1, vc, 0,
                                 scale, 64, _lib.stream_handle(lg.device)), "dk_head_chunk")
    want = np.exp(x[0, 1:].astype(np.float64)) * scale
    err = np.abs(host(lg)[0, 1:].astype(np.float64) - want)
    bound = (2.0 ** -11 + 2.0 ** -22) * want + 2.0 ** -25 + 2.0 ** -149 * scale
    assert np.all(err <= bound), float((err / want).max())
