"""GPU tests at the edges of the kernels' tiles and of their dispatch rules, against the
CPU oracle.  Tolerances as in test_gpu_branches.py (fp32 outputs 1e-5, gradients 1e-4; bf16
2e-2, the oracle fed the bf16-rounded inputs)."""
import math

import numpy as np
import oracle
import pytest
import torch

from nsa import NSAAttention, NSAConfig, NSAKVCache, _ops
from nsa.kernels import _CompressTokens, score_and_select
from test_gpu_branches import _check, _make

pytestmark = pytest.mark.gpu


def _lists(seed, B, G, T, n, nb):
    """n slots a row in any order: random blocks (later ones and repeats among them), -1."""
    g = torch.Generator().manual_seed(seed)
    idx = torch.randint(0, nb, (B, G, T, n), generator=g)
    idx[torch.rand(B, G, T, n, generator=g) < 0.2] = -1
    return idx


# a wave's block bitmaps: 31 / 32 / 33 / 65 blocks (word edges), one to seventeen timesteps a
# wave (1, 2, 3, 4, 15, 20 heads a group), blocks of one, two and three 16-key groups
@pytest.mark.parametrize("hpg,T,lp,n", [(1, 512, 16, 5), (2, 496, 16, 16), (3, 528, 16, 7), (4, 1040, 16, 16),
                                        (15, 130, 48, 3), (20, 131, 32, 64)])
@pytest.mark.parametrize("dtype,dk,dv", [(torch.float32, 64, 64), (torch.bfloat16, 64, 64),
                                         (torch.float32, 192, 128), (torch.bfloat16, 128, 128)])
def test_selection_bitmap_edges(dev, hpg, T, lp, n, dtype, dk, dv):
    B, G = 1, 2
    q, kp, v, do = _make(hpg, B, G * hpg, G, T, T, dk, dv, dtype, dev)
    idx = _lists(hpg + T, B, G, T, n, (T + lp - 1) // lp).to(dev)
    _check(_ops.SELECTION, q, kp, v, do, 1 / math.sqrt(dk), dtype, indices=idx, lprime=lp)


# scoring with few rows (one MFMA tile per wave) and few timesteps (heads across waves): rows
# about 16 / 64 (the tile and the rule's edge; past 16 rows 2048 / 2112 and 8192 / 8704 waves: the
# other edges), 1 / 3 / 20 heads a group, block counts at the
# 256-block pieces and 64-block tiles, both remaps (l/d = 2, l'/d = 4 and another), dk with a
# remainder piece; indices and scores bit for bit
@pytest.mark.parametrize("B,G,hpg,T,N,dk,l,lp", [(1, 2, 16, 1, 255, 64, 32, 64), (2, 2, 3, 5, 257, 40, 32, 64),
                                                 (1, 1, 16, 4, 64, 192, 32, 64), (1, 1, 13, 5, 65, 96, 32, 64),
                                                 (1, 2, 20, 3, 1030, 64, 32, 64), (3, 1, 4, 17, 600, 128, 64, 32),
                                                 (1, 2, 1, 64, 70, 64, 32, 64), (1, 1, 2, 1024, 100, 32, 32, 64),
                                                 (1, 1, 2, 1025, 100, 32, 32, 64), (1, 1, 64, 1, 4096, 32, 32, 64),
                                                 (2, 4, 4, 8, 2048, 32, 32, 64), (2, 4, 4, 8, 2049, 32, 32, 64),
                                                 (8, 4, 4, 16, 1024, 32, 32, 64), (8, 4, 4, 16, 1025, 32, 32, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_score_few_rows(dev, B, G, hpg, T, N, dk, l, lp, dtype):
    g = torch.Generator().manual_seed(N + T)
    q = torch.randn(B, G * hpg, T, dk, generator=g).to(dtype)
    k = torch.randn(B, G, dk, N, generator=g).to(dtype)
    be = torch.arange(N, dtype=torch.int32) * 16 + l - 1
    q0 = max(0, 16 * N - 3 * T)  # the last rows see every block, the first ones do not
    cfg = NSAConfig(head_dim_qk=dk, n_heads=G * hpg, n_kv_groups=G, l=l, l_prime=lp, n=9)
    got = score_and_select(q.to(dev), k.to(dev), be.to(dev), 0.2, cfg, return_scores=True, q_offset=q0)
    want = oracle.score_topn(q.float().numpy(), k.float().numpy(), be.numpy(), np.float32(0.2), l=l, d=16, lprime=lp,
                             n=9, positions=np.arange(q0, q0 + T, dtype=np.int32), want_scores=True)
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a.cpu().numpy(), b)


# a query row with a NaN: its group's sums are NaN at every block, and what is left to take is the
# first entry past the last block (here 100 of 100), never an index that no block can have; the
# rows beside it are untouched.  A wave per timestep and a timestep's heads across waves
@pytest.mark.parametrize("T", [4, 1500])
@pytest.mark.parametrize("fixed", [False, True])
def test_score_nan_row(dev, T, fixed):
    cfg = NSAConfig(head_dim_qk=64, n_heads=4, n_kv_groups=1, n=9, include_fixed_in_selection=fixed)
    N, q0 = 400, 16 * 379 + 31  # l' = 4 d: 100 blocks, the own one of row 0 is 95
    g = torch.Generator().manual_seed(0)
    q = torch.randn(1, 4, T, 64, generator=g).to(dev)
    k = torch.randn(1, 1, 64, N, generator=g).to(dev)
    be = torch.arange(N, dtype=torch.int32, device=dev) * 16 + 31
    clean = score_and_select(q, k, be, 0.2, cfg, q_offset=q0)
    q[:, 1, 0] = float("nan")
    got = score_and_select(q, k, be, 0.2, cfg, q_offset=q0)
    assert got[0, 0, 0].tolist() == ([0, 94, 95] + 6 * [100] if fixed else 9 * [100])
    assert torch.equal(got[:, :, 1:], clean[:, :, 1:])


# the decode step's split over 256-key workgroups and 64-key waves: positions at their edges and
# at block edges, no compressed token / one / 256 / 257, 1 / 4 / 16 / 17 / 40 heads a group (head
# tiles), every compiled width, windows of one key and past the sequence, empty slots, caches of
# either layout
@pytest.mark.parametrize("B,G,hpg,t,n_cmp,dk,dv,lp,n,w,act", [
    (1, 1, 16, 0, 0, 64, 64, 64, 1, 512, 1), (2, 2, 4, 255, 15, 32, 32, 16, 5, 1, 2),
    (1, 2, 1, 256, 1, 128, 128, 48, 16, 256, 0), (1, 2, 17, 4159, 257, 64, 64, 64, 16, 257, 1),
    (3, 1, 40, 4160, 256, 192, 128, 64, 4, 9000, 2), (1, 1, 16, 319, 18, 128, 128, 32, 64, 65, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_attention_edges(dev, B, G, hpg, t, n_cmp, dk, dv, lp, n, w, act, dtype):
    H, T = G * hpg, t + 7  # the cache is longer than the sequence
    g = torch.Generator().manual_seed(t + dk)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dtype)

    q, gates = rnd(B, H, 1, dk), rnd(B, 1, H, 3).permute(0, 2, 1, 3)
    nc = max(n_cmp, 1) + 3
    kv = [rnd(B, G, nc, dk), rnd(B, nc, G, dv).transpose(1, 2), rnd(B, G, T, dk), rnd(B, G, T, dv),
          rnd(B, T, G, dk).transpose(1, 2), rnd(B, G, T, dv)]
    nb = t // lp + 1
    idx = torch.stack([torch.randperm(max(nb + 2, n), generator=g)[:n] for _ in range(B * G)]).view(B, G, 1, n)
    idx[torch.rand(B, G, 1, n, generator=g) < 0.2] = -1
    idx[0, 0] = -1  # a row without any block takes its own
    # what lies past the sequence never reaches a result
    for x, e in ((kv[0], n_cmp), (kv[1], n_cmp), *((x, t + 1) for x in kv[2:])):
        x[:, :, e:] = float("nan")
    dkv = [x.to(dev) for x in kv]
    assert _ops.decode_direct(q.to(dev), dkv, n, lp)
    out = _ops.decode_attn(q.to(dev), dkv, n_cmp, idx.to(dev), gates.to(dev), act, t, dk ** -0.5, lp, w)
    pos = dict(positions=np.array([t], np.int32))
    a = [x.double().numpy() for x in kv]
    be = np.arange(n_cmp, dtype=np.int32) * 0
    cut = [x[:, :, :t + 1] for x in a[2:]]
    qd = q.double().numpy()
    sel = idx.numpy().copy()
    sel[(sel < 0).all(-1)] = t // lp
    o = [oracle.attn_fwd(oracle.COMPRESSION, qd, a[0][:, :, :n_cmp], a[1][:, :, :n_cmp], dk ** -0.5, block_ends=be,
                         **pos)[0] if n_cmp else np.zeros((B, H, 1, dv)),
         oracle.attn_fwd(oracle.SELECTION, qd, cut[0], cut[1], dk ** -0.5, indices=sel, lprime=lp, **pos)[0],
         oracle.attn_fwd(oracle.SLIDING, qd, cut[2], cut[3], dk ** -0.5, window=w, **pos)[0]]
    z = gates.double()
    z = (z, torch.sigmoid(z), torch.softmax(z, -1))[act].numpy()
    want = sum(z[..., i:i + 1] * o[i] for i in range(3))
    err = np.linalg.norm(out.double().cpu().numpy() - want) / np.linalg.norm(want)
    assert err < (2e-2 if dtype == torch.bfloat16 else 1e-5), err


# a NaN or an infinite score within the visible keys of each branch in turn reaches the output of
# every head that sees it, and no other (with an infinite key: the heads whose query makes it
# +inf, as exp(inf - inf); the others give that key the weight 0)
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("br", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_attention_keeps_nan(dev, br, bad, dtype):
    B, G, hpg, t, n_cmp, d, lp, n, w = 2, 2, 4, 300, 17, 64, 16, 5, 100
    g = torch.Generator().manual_seed(br)

    def rnd(*s):
        return torch.randn(*s, generator=g).to(dtype).to(dev)

    q, gates = rnd(B, G * hpg, 1, d), rnd(B, G * hpg, 1, 3)
    kv = [rnd(B, G, n_cmp if i < 2 else t + 1, d) for i in range(6)]
    idx = torch.tensor([0, 3, 7, 12, 18]).expand(B, G, 1, n).contiguous().to(dev)
    args = (n_cmp, idx, gates, 1, t, 0.1, lp, w)
    clean = _ops.decode_attn(q, kv, *args)
    kv[2 * br][1, 0, (5, 7 * lp + 3, t - 50)[br], 11] = bad
    out = _ops.decode_attn(q, kv, *args)
    hit = torch.zeros(B, G, hpg, dtype=torch.bool, device=dev)
    hit[1, 0] = True if math.isnan(bad) else q[1, :hpg, 0, 11] > 0
    hit = hit.view(B, G * hpg, 1)
    assert hit.any() and torch.equal(out.isnan(), hit.unsqueeze(-1).expand_as(out))
    assert torch.equal(out[:, hpg:], clean[:, hpg:]) and torch.equal(out[0], clean[0])


# repeated blocks count once, as in the forward kernels (whose cleaned lists are the same set): the
# same bits as with -1 in the repeats' place
@pytest.mark.parametrize("n", [2, 16, 64])
def test_decode_attention_repeated_blocks(dev, n):
    t, lp, d, w = 1500, 32, 64, 40
    g = torch.Generator().manual_seed(n)
    q, gates = torch.randn(2, 8, 1, d, generator=g).to(dev), torch.randn(2, 8, 1, 3, generator=g).to(dev)
    kv = [torch.randn(2, 2, 20 if i < 2 else t + 1, d, generator=g).to(dev) for i in range(6)]
    idx = torch.randint(0, max(n // 2, 1), (2, 2, 1, n), generator=g)
    idx[0, 0, 0] = 5
    once = idx.clone()
    for row in once.view(-1, n):
        for j in range(n - 1, 0, -1):
            if row[j] in row[:j]:
                row[j] = -1
    a, b = (_ops.decode_attn(q, kv, 17, x.to(dev), gates, 1, t, 0.1, lp, w) for x in (idx, once))
    assert torch.equal(a, b)


# few-row linear layers: rows at the 16-row tiles, widths at the 16-feature tiles, inputs at the
# 32- (16-) feature chunks, the eight waves' turns and a last chunk of one piece; several jobs,
# grouped outputs, bias, relu.  fp32 sums: 1e-6 norm-relative; bf16 rounding of the result 2^-9
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("K", [8, 40, 256, 2568])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_few(dev, rows, K, dtype):
    g = torch.Generator().manual_seed(rows + K)
    x = torch.randn(rows, K + 8, generator=g).to(dtype).to(dev)[:, :K]  # padded rows
    jobs, want = [], []
    for i, (n, group) in enumerate([(1, 1), (17, 17), (96, 32), (15, 40), (208, 208)]):
        w = (torch.randn(n, K, generator=g) / K ** 0.5).to(dtype).to(dev)
        b = torch.randn(n, generator=g).to(dtype).to(dev) if i % 2 else None
        ng, gs = -(-n // group), group + 3
        o = torch.full((rows, ng, gs), 7.0, dtype=dtype, device=dev)
        y = x.double() @ w.double().t() + (b.double() if b is not None else 0)
        y = y.relu() if i % 3 == 1 else y
        r = o.double()
        for j in range(ng):
            r[:, j, :min(group, n - j * group)] = y[:, j * group:(j + 1) * group]
        jobs.append((w, b, o, o.stride(0), o.stride(1), group, int(i % 3 == 1)))
        want.append(r)
    _ops.linear_few(x, jobs)
    for (_, _, o, *_), r in zip(jobs, want):
        assert ((o.double() - r).norm() / r.norm()).item() < (2 ** -9 if dtype == torch.bfloat16 else 1e-6)
        assert torch.equal(o[..., -3:].double(), r[..., -3:])  # nothing past a group


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decode_projections_direct_and_through_modules(dev, dtype):
    """Biased layers, several sequences: the token's projections in one launch against the
    modules' own (taken when a layer carries a hook), on outputs and every cache."""
    cfg = NSAConfig(d_model=96, head_dim_qk=64, head_dim_v=64, n_heads=8, n_kv_groups=2, l_prime=32, n=4, w=40,
                    use_bias=True)
    torch.manual_seed(3)
    m = NSAAttention(cfg).to(dev, dtype).eval()
    x = torch.randn(3, 90, 96, device=dev).to(dtype)
    calls, res = [], []
    for hooked in (False, True):
        h = m.k_select.register_forward_hook(lambda *_: calls.append(1)) if hooked else None
        cache = NSAKVCache(cfg, 3, 90, dev, dtype)
        m.prefill(x[:, :70], cache)
        calls.clear()
        out = torch.cat([m.decode(x[:, t:t + 1], cache)[0] for t in range(70, 90)], 1)
        res.append((out, cache.k_cmp_in, cache.v_cmp_in, cache.k_sel, cache.v_sel, cache.k_win, cache.v_win))
        assert len(calls) == (20 if hooked else 0) and cache.length == 90
        if h:
            h.remove()
    for a, b in zip(*res):
        assert ((a.double() - b.double()).norm() / b.double().norm()).item() < (1e-2 if dtype == torch.bfloat16 else 1e-5)
    with pytest.raises(ValueError):
        m.decode(x[:, :1], cache)  # the cache is full


# the compression dK/dV work list: one to five key tiles of which the last ones are padding or
# partly so, spans cut into segments down to 32 rows and into more than the list's cap of equal
# cuts, 1 / 4 / 16 / 40 heads a group (row chunks of one timestep and of many), rows that see
# nothing, no row that sees anything
@pytest.mark.parametrize("B,G,hpg,T,l,d,dtype,dk,dv", [
    (1, 1, 16, 300, 32, 16, torch.bfloat16, 64, 64), (2, 2, 16, 2100, 8, 8, torch.bfloat16, 128, 128),
    (1, 2, 4, 1290, 4, 2, torch.bfloat16, 64, 64), (1, 1, 1, 700, 2, 1, torch.float32, 32, 32),
    (1, 1, 40, 257, 32, 16, torch.bfloat16, 192, 128), (3, 1, 3, 20, 32, 16, torch.float32, 64, 64),
    (1, 1, 8, 1060, 32, 4, torch.float32, 64, 64)])
def test_compression_work_list(dev, B, G, hpg, T, l, d, dtype, dk, dv):
    n_act = max((T - l) // d + 1, 0)
    n_pad = 1
    while n_pad < n_act:
        n_pad *= 2
    be = torch.full((n_pad,), 999999, dtype=torch.int32)
    be[:n_act] = torch.arange(n_act, dtype=torch.int32) * d + l - 1
    q, kp, v, do = _make(T, B, G * hpg, G, T, n_pad, dk, dv, dtype, dev)
    _check(_ops.COMPRESSION, q, kp, v, do, 1 / math.sqrt(dk), dtype, block_ends=be.to(dev))


# dK/dV items of less than 128 entries (small launches) keep their partials in fp32: 128 rows of 16
# heads whose dO, multiples of 1/128 that one key (selection: one block of 16, of weight 1/16 each)
# takes whole, cancel but for one entry.  All sums are exact in fp32; a sum of 32 rows is not in bf16
@pytest.mark.parametrize("branch", [_ops.SLIDING, _ops.COMPRESSION, _ops.SELECTION])
def test_small_launch_partials_are_fp32(dev, branch):
    T, hpg, d = 128, 16, 64
    g = torch.Generator().manual_seed(branch)
    half = torch.randint(-128, 129, (T * hpg // 2, d), generator=g).double() / 128
    do = torch.cat([half, -half[torch.randperm(len(half), generator=g)]])
    do[7] = 0
    want = do.sum(0)
    do = do.view(T, hpg, d).permute(1, 0, 2).unsqueeze(0).to(torch.bfloat16).to(dev)
    n = {_ops.SLIDING: T, _ops.COMPRESSION: 1, _ops.SELECTION: 16}[branch]
    k = torch.zeros(1, 1, n, d, device=dev, dtype=torch.bfloat16)
    q = torch.zeros(1, hpg, T, d, device=dev, dtype=torch.bfloat16)
    if branch == _ops.SLIDING:  # scores 32 for key 0, -32 for the others
        q[..., 0], k[..., 0] = 16, -16
        k[:, :, 0, 0] = 16
    v = torch.zeros(1, 1, n, d, device=dev, dtype=torch.bfloat16)
    kw = {_ops.SLIDING: dict(window=T), _ops.COMPRESSION: dict(block_ends=torch.zeros(1, dtype=torch.int32, device=dev)),
          _ops.SELECTION: dict(indices=torch.zeros(1, 1, T, 1, dtype=torch.int64, device=dev), lprime=16, causal=False)}
    out, L, M = _ops.attn_fwd(branch, q, k, v, 0.125, **kw[branch])
    _, _, dv = _ops.attn_bwd(branch, q, k, v, out, do, L, M, 0.125, **kw[branch])
    want = (want / 16 if branch == _ops.SELECTION else want).to(torch.bfloat16).double()
    assert want.abs().max() > 0 and torch.equal(dv[0, 0, 0].double().cpu(), want)


# sliding-window dK/dV: a wave whose 16 keys no row of a chunk sees skips it.  Windows below, at
# and past a wave's keys and a row chunk, shorter and longer than the sequence; chunks of less
# than a timestep to 32 of them; with and without stored dS; one item per key tile (256 tiles).
# (Window 2 is the smallest: at 1 the probability is 1 and the exact dQ and dK are zero, so a
# relative error has no meaning.)
@pytest.mark.parametrize("B,G,hpg,T,w,dtype,dk,dv", [
    (1, 1, 16, 700, 2, torch.bfloat16, 64, 64), (1, 2, 16, 403, 17, torch.bfloat16, 192, 128),
    (2, 1, 16, 257, 600, torch.bfloat16, 128, 128), (1, 1, 1, 1500, 128, torch.bfloat16, 64, 64),
    (1, 2, 40, 150, 33, torch.bfloat16, 128, 128), (2, 128, 1, 100, 16, torch.bfloat16, 32, 32),
    (1, 1, 4, 391, 48, torch.float32, 64, 64), (1, 1, 3, 200, 2, torch.float32, 32, 32)])
def test_sliding_chunks_out_of_sight(dev, B, G, hpg, T, w, dtype, dk, dv):
    q, k, v, do = _make(T + w, B, G * hpg, G, T, T, dk, dv, dtype, dev)
    _check(_ops.SLIDING, q, k, v, do, 1 / math.sqrt(dk), dtype, window=w)


# compress_tokens as one call each way: one block / a power of two of them / padding, tokens past
# the last block, one and several batches and groups in either storage order, every width of the
# weight-gradient tiles, row counts about its 64- (32-) row steps, overlapping and disjoint blocks.
# Against the same formula in float64: fp32 1e-5 (rounding of the sums).  bf16: 1e-2 for outputs;
# gradients 6e-2, because a pre-activation within its bf16 rounding (2^-9 of |y| ~ 1) of zero has
# its unit's gradient switched: about 2^-9 of the units, sqrt(2^-9) = 4.4e-2 of the norm
@pytest.mark.parametrize("B,G,T,dk,dv,l,d,major", [
    (1, 1, 8, 64, 8, 8, 8, False), (1, 2, 32, 64, 64, 32, 16, True), (2, 3, 177, 128, 40, 32, 16, True),
    (2, 2, 95, 192, 128, 32, 32, False), (1, 4, 1056, 192, 128, 32, 16, True), (3, 1, 130, 64, 128, 64, 16, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_compress_tokens_edges(dev, B, G, T, dk, dv, l, d, major, dtype, monkeypatch):
    cfg = NSAConfig(d_model=64, head_dim_qk=dk, head_dim_v=dv, n_heads=G, n_kv_groups=G, l=l, d=d, l_prime=64 if 64 % d == 0
                    else d)
    torch.manual_seed(T)
    m = NSAAttention(cfg).to(dev, dtype)

    def rnd(w):
        x = torch.randn(B, T, G, w, device=dev).to(dtype)
        return (x.transpose(1, 2) if major else x.transpose(1, 2).contiguous()).detach().requires_grad_()

    k, v = rnd(dk), rnd(dv)
    kc, vc, be, n = m.compress_tokens(k, v)
    npad = kc.shape[-1]
    assert n == (T - l) // d + 1 and npad >= n and (npad & (npad - 1)) == 0
    assert not kc[..., n:].any() and not vc[:, :, n:].any()
    gk, gv = torch.randn_like(kc), torch.randn_like(vc)
    gk[..., n:], gv[:, :, n:] = float("nan"), float("nan")  # the padding's gradients are dropped
    names = ("compress_mlp.0.weight", "compress_mlp.0.bias", "compress_mlp.2.weight", "compress_mlp.2.bias",
             "pos_embed.weight")
    ps = [m.get_parameter(x) for x in names]
    got = torch.autograd.grad([kc, vc], [k, v, *ps], [gk, gv])
    W1, b1, W2, b2, E = P = [p.detach().double().requires_grad_() for p in ps]
    kd, vd = (x.detach().double().requires_grad_() for x in (k, v))
    y = (kd @ W1[:, :dk].t()).unfold(2, l, d).transpose(-1, -2) + (E @ W1[:, dk:].t() + b1)
    rk, rv = torch.relu(y).mean(-2) @ W2.t() + b2, vd.unfold(2, l, d).mean(-1)
    want = torch.autograd.grad([rk, rv], [kd, vd, *P], [gk[..., :n].transpose(-1, -2).double(), gv[:, :, :n].double()])

    def err(a, b):
        return ((a.double() - b).norm() / b.norm()).item()

    bf = dtype == torch.bfloat16
    assert max(err(kc[..., :n].transpose(-1, -2), rk), err(vc[:, :, :n], rv)) < (1e-2 if bf else 1e-5)
    errs = {x: err(a, b) for x, a, b in zip(("k", "v") + names, got, want)}
    assert max(errs.values()) < (6e-2 if bf else 1e-5), errs
    # the output layer as a GEMM of the caller's (many rows): the same pooled rows, the same zeros
    monkeypatch.setattr(_CompressTokens, "OWN_OUT", 0)
    gc, gvc, _, _ = m.compress_tokens(k, v)
    assert torch.equal(gvc, vc) and not gc[..., n:].any() and err(gc[..., :n].transpose(-1, -2), rk) < (1e-2 if bf else 1e-5)
    for a, b in zip(torch.autograd.grad([gc, gvc], [k, v, *ps], [gk, gv]), got):
        assert torch.equal(a, b)
    # and, in fp32, the token half of the first layer's weight gradient
    monkeypatch.setattr(_CompressTokens, "OWN_WGRAD32", 0)
    gc, gvc, _, _ = m.compress_tokens(k, v)
    for x, a, b, w in zip(("k", "v") + names, torch.autograd.grad([gc, gvc], [k, v, *ps], [gk, gv]), got, want):
        assert torch.equal(a, b) if bf or x != names[0] else err(a, w) < 1e-5, x
    monkeypatch.undo()
    # frozen layers: the other gradients are the same
    for p in ps[2:]:
        p.requires_grad_(False)
    kc, vc, _, _ = m.compress_tokens(k, v)
    part = torch.autograd.grad([kc, vc], [k, v, *ps[:2]], [gk, gv])
    for a, b in zip(part, got):
        assert torch.equal(a, b)


def test_compress_tokens_broadcast_bias(dev):
    """A bias of one element broadcasts, as in F.linear (the one-call form reads whole biases)."""
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=2, n_kv_groups=2)
    torch.manual_seed(0)
    m = NSAAttention(cfg).to(dev)
    k, v = (torch.randn(1, 2, 100, 64, device=dev) for _ in range(2))
    res = []
    for one in (True, False):
        for lay in (m.compress_mlp[0], m.compress_mlp[2]):
            b = torch.full((1,), 0.3, device=dev)
            lay.bias = torch.nn.Parameter(b if one else b.expand(lay.out_features).clone())
        assert _CompressTokens.usable(k, v, m.compress_mlp[0].weight, m.compress_mlp[0].bias, m.compress_mlp[2].weight,
                                      m.compress_mlp[2].bias, m.pos_embed.weight, cfg.l) is not one
        kc = m.compress_tokens(k, v)[0]
        kc.square().sum().backward()
        res.append((kc.double(), *(lay.bias.grad.double().sum() for lay in (m.compress_mlp[0], m.compress_mlp[2]))))
    for a, b in zip(*res):
        assert ((a - b).norm() / b.norm()).item() < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_compress_tokens_backward_under_autocast(dev, dtype):
    """A backward that runs inside an autocast region (the forward outside) takes its products in
    the tensors' own type: autocast's float16 ones would be read as another type by the call."""
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=2, n_kv_groups=2)
    torch.manual_seed(0)
    m = NSAAttention(cfg).to(dev, dtype)
    k, v = (torch.randn(2, 2, 177, 64, device=dev, dtype=dtype, requires_grad=True) for _ in range(2))
    ps = [k, v, *m.compress_mlp.parameters(), m.pos_embed.weight]
    gs, res = None, []
    for on in (False, True):
        kc, vc, _, _ = m.compress_tokens(k, v)
        gs = gs or [torch.randn_like(kc), torch.randn_like(vc)]
        with torch.autocast("cuda", dtype=torch.float16, enabled=on):
            res.append(torch.autograd.grad([kc, vc], ps, gs))
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_compress_tokens_saved_tensor_hooks(dev):
    """Saved tensors that a hook hands back with other strides (each element twice as far apart)
    or off their 16-byte alignment give the same gradients."""
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=2, n_kv_groups=2)
    torch.manual_seed(0)
    m = NSAAttention(cfg).to(dev, torch.bfloat16)
    k, v = (torch.randn(2, 2, 177, 64, device=dev, dtype=torch.bfloat16, requires_grad=True) for _ in range(2))
    ps = [k, v, *m.compress_mlp.parameters(), m.pos_embed.weight]

    def strided(x):
        return torch.stack([x, torch.zeros_like(x)], -1)[..., 0]

    def shifted(x):
        y = x.new_empty(x.numel() + 1)[1:].view(x.shape)
        return y.copy_(x)

    gs, res = None, []
    for unpack in (lambda x: x, strided, shifted):
        with torch.autograd.graph.saved_tensors_hooks(lambda x: x.detach(), unpack):
            kc, vc, _, _ = m.compress_tokens(k, v)
        gs = gs or [torch.randn_like(kc), torch.randn_like(vc)]
        res.append(torch.autograd.grad([kc, vc], ps, gs))
    for other in res[1:]:
        for a, b in zip(other, res[0]):
            assert torch.equal(a, b)


# the 32-column selection forward: one timestep a wave (32 to 96 heads a group, from 2048 waves on,
# from 4096 where all of more than 512 keys' blocks fit the slots: the rule's edges from both
# sides; a partly filled last workgroup; five rows: a lone key has an exact dQ of zero, so no relative error), several that
# share most blocks (from 65536 rows and at most
# four blocks a slot on: the rule's edges from both sides), timesteps that straddle waves, blocks
# of half a tile and of one and a half; the forward's workgroup orders for whole and partial rounds
# of XCDs (the stored-dS dQ's: test_selection_dq_workgroup_order)
@pytest.mark.parametrize("B,G,hpg,T,lp,n,dtype,dk,dv", [
    (1, 2, 32, 77, 64, 4, torch.bfloat16, 128, 128), (1, 1, 64, 5, 16, 1, torch.bfloat16, 64, 64),
    (1, 1, 64, 130, 48, 7, torch.bfloat16, 192, 128), (4, 4, 4, 1024, 32, 8, torch.bfloat16, 32, 32),
    (4, 4, 4, 1025, 32, 8, torch.bfloat16, 32, 32), (4, 4, 4, 1023, 16, 16, torch.bfloat16, 32, 32),
    (8, 4, 3, 700, 64, 5, torch.bfloat16, 64, 64), (1, 1, 64, 1023, 16, 3, torch.bfloat16, 64, 64),
    (1, 1, 64, 1025, 16, 3, torch.bfloat16, 64, 64), (1, 1, 64, 1030, 48, 5, torch.bfloat16, 192, 128),
    (1, 2, 32, 1029, 32, 33, torch.bfloat16, 64, 64), (2, 2, 32, 1025, 32, 33, torch.bfloat16, 64, 64),
    (1, 1, 96, 1400, 16, 1, torch.bfloat16, 32, 32), (4, 1, 32, 512, 64, 8, torch.bfloat16, 32, 32),
    (4, 1, 32, 513, 64, 9, torch.bfloat16, 32, 32)])
def test_selection_forward_32_columns(dev, B, G, hpg, T, lp, n, dtype, dk, dv):
    q, kp, v, do = _make(hpg + T, B, G * hpg, G, T, T, dk, dv, dtype, dev)
    idx = _lists(T, B, G, T, n, (T + lp - 1) // lp).to(dev)
    _check(_ops.SELECTION, q, kp, v, do, 1 / math.sqrt(dk), dtype, indices=idx, lprime=lp)


# the dQ kernel of the stored dS (16 and 32 heads a group, blocks of 64 keys) has ceil(waves / 4)
# workgroups: a multiple of neither 8 nor the batch-groups when T % 4 is 1, 2 or 3, with 8 and 16
# batch-groups, which the XCDs share out whole, and 6, which they do not.  Added to a given dQ the
# result is the overwritten one plus it: both rounded to bf16 once, 2^-8 of the sum
@pytest.mark.parametrize("B,G,hpg,T", [(2, 4, 16, 301), (8, 1, 16, 202), (4, 4, 16, 129), (1, 8, 32, 67),
                                       (4, 2, 16, 5), (3, 2, 16, 131), (2, 8, 16, 100)])
def test_selection_dq_workgroup_order(dev, B, G, hpg, T):
    lp, n, dk, dt = 64, 4, 64, torch.bfloat16
    q, kp, v, do = _make(hpg + T, B, G * hpg, G, T, T, dk, dk, dt, dev)
    idx = _lists(T, B, G, T, n, (T + lp - 1) // lp).to(dev)
    out, (dq, _, _) = _check(_ops.SELECTION, q, kp, v, do, 1 / math.sqrt(dk), dt, indices=idx, lprime=lp)
    k = kp.transpose(-1, -2)
    _, L, M = _ops.attn_fwd(_ops.SELECTION, q, k, v, 1 / math.sqrt(dk), indices=idx, lprime=lp)
    base = torch.randn_like(q)
    acc, _, _ = _ops.attn_bwd(_ops.SELECTION, q, k, v, out, do, L, M, 1 / math.sqrt(dk), indices=idx, lprime=lp,
                              dq=base.clone(), dq_accumulate=True)
    want = base.double() + dq.double()
    assert ((acc.double() - want).abs() <= 2 ** -8 * (want.abs() + dq.double().abs()) + 1e-6).all()


@pytest.mark.parametrize("what", ["gate_mlp", "gate_mlp.1", "k_select", "prefill", "_project_kv"])
def test_decode_runs_what_was_replaced(dev, what):
    """A forward replaced on a module's instance, or a method on the layer's, runs in a decode step
    (which otherwise passes the modules by), with the step's own result."""
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=8, n_kv_groups=2, l_prime=32, n=4, w=40)
    torch.manual_seed(0)
    m = NSAAttention(cfg).to(dev, torch.bfloat16).eval()
    x = torch.randn(2, 37, 64, device=dev).to(torch.bfloat16)
    calls, res = [], []
    for replaced in (False, True):
        c = NSAKVCache(cfg, 2, 40, dev, torch.bfloat16)
        m.prefill(x[:, :35], c)
        if replaced:
            owner, name = (m, what) if hasattr(type(m), what) else (m.get_submodule(what), "forward")
            real = getattr(owner, name)
            setattr(owner, name, lambda *a: (calls.append(1), real(*a))[1])
        res.append(torch.cat([m.decode(x[:, t:t + 1], c)[0] for t in (35, 36)], 1).double())
    assert len(calls) == 2 and (res[0] - res[1]).norm() < 1e-2 * res[0].norm()


def test_decode_output_in_the_layers_type(dev):
    """Projections that cast an fp32 token to bf16 before a plain bf16 output projection: the output
    is of that projection's type, as F.linear's is."""
    class Cast(torch.nn.Linear):
        def forward(self, x):
            return super().forward(x.to(self.weight.dtype))

    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=8, n_kv_groups=2, l_prime=32, n=4, w=40)
    torch.manual_seed(0)
    m = NSAAttention(cfg).to(dev, torch.bfloat16).eval()
    x = torch.randn(2, 37, 64, device=dev).to(torch.bfloat16)
    res = []
    for dt in (torch.bfloat16, torch.float32):
        cache = NSAKVCache(cfg, 2, 40, dev, torch.bfloat16)
        if dt == torch.float32:
            for name in ("q_proj", "k_compress", "v_compress", "k_select", "v_select", "k_sliding", "v_sliding"):
                getattr(m, name).__class__ = Cast
            m.gate_mlp[0].__class__ = Cast
        m.prefill(x[:, :35].to(dt), cache)
        res.append(torch.cat([m.decode(x[:, t:t + 1].to(dt), cache)[0] for t in (35, 36)], 1))
    assert res[1].dtype == torch.bfloat16
    assert (res[0].double() - res[1].double()).norm() < 1e-2 * res[0].double().norm()


@pytest.mark.parametrize("rows,own", [(32, True), (33, False)])
def test_decode_output_projection_rule(dev, rows, own, monkeypatch):
    """The output projection of a decode step is F.linear's from the size on at which it is the
    faster one (the rule's line moved to 32 rows of a small layer), with and without a bias, in
    the whole step and in its parts alike."""
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=8, n_kv_groups=2, l_prime=32, n=4, w=48,
                    use_bias=rows == 33)
    monkeypatch.setitem(_ops.LINEAR_ONE_WORK, torch.bfloat16, 32 * 64 * 512)
    torch.manual_seed(rows)
    m = NSAAttention(cfg).to(dev, torch.bfloat16).eval()
    x = torch.randn(rows, 45, 64, device=dev).to(torch.bfloat16)
    real, calls, res = torch.nn.functional.linear, [], []
    for parts in (False, True):
        cache = NSAKVCache(cfg, rows, 45, dev, torch.bfloat16)
        m.prefill(x[:, :40], cache)
        monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: (calls.append(a[1].shape), real(*a))[1])
        res.append(torch.cat([m.decode(x[:, t:t + 1], cache, output_attentions=parts)[0] for t in range(40, 45)], 1))
        monkeypatch.setattr(torch.nn.functional, "linear", real)
    assert calls == ([] if own else 10 * [(64, 512)]) and torch.equal(*res)


# the whole decode step in one call against its parts (taken when the attention details are
# asked for): the same kernels, so the same bits, with blocks completing on the way, before the
# first block, with every gate mode, with and without fixed blocks, after a prompt and from empty
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T0,n,gate,fixed,bias", [(1, 0, 4, "sigmoid", True, False), (3, 61, 5, "softmax", False, True),
                                                    (17, 300, 8, "sigmoid", True, True)])
def test_decode_step_matches_its_parts(dev, dtype, B, T0, n, gate, fixed, bias):
    cfg = NSAConfig(d_model=64, head_dim_qk=64, head_dim_v=64, n_heads=8, n_kv_groups=2, l_prime=32, n=n, w=48,
                    gate_mode=gate, include_fixed_in_selection=fixed, use_bias=bias)
    torch.manual_seed(B)
    m = NSAAttention(cfg).to(dev, dtype).eval()
    T = T0 + 40
    x = torch.randn(B, T, 64, device=dev).to(dtype)
    res = []
    for parts in (False, True):
        cache = NSAKVCache(cfg, B, T, dev, dtype)
        if T0:
            m.prefill(x[:, :T0], cache)
        if not parts:
            assert m._decode_step(x[:, T0:T0 + 1], cache) is not None and cache.length == T0 + 1
            cache.length, cache.n_act = T0, max((T0 - 32) // 16 + 1, 0)
        outs = [m.decode(x[:, t:t + 1], cache, output_attentions=parts)[0] for t in range(T0, T)]
        assert cache.length == T and cache.n_act == (T - 32) // 16 + 1
        res.append((torch.cat(outs, 1), cache.k_cmp_in, cache.v_cmp_in, cache.k_sel, cache.v_sel, cache.k_win,
                    cache.v_win, cache.K_cmp, cache.V_cmp, cache.block_ends))
    for i, (a, b) in enumerate(zip(*res)):
        if i or B <= 16:  # above 16 rows the parts' output projection is torch's
            assert torch.equal(a, b), i
        else:
            assert ((a.double() - b.double()).norm() / b.double().norm()).item() < (2 ** -8 if dtype == torch.bfloat16 else 1e-6)
