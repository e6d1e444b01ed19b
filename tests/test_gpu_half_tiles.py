"""The attention kernels' half-tile (32-key) steps at the edges of their ring
schedule, against the float64 oracle: prefixes of one to nine tiles (prologue
only, then the first slots reused; in split plans here up to three tiles a
chunk), last tiles that end in their first or second half (the tail's other
half is empty or masked), windows that start inside a page (every tile then takes
the per-row loads), trees of one to four key tiles, bf16 and fp8 prefixes, head
sizes 64 and 128, split plans (one body for both levels up to three key tiles of
the tree) and fused ones.  The second test has chunks of up to ten tiles in
split plans: the steady loop, whose loads go out between the MFMAs (from 5 full
tiles at head size 128 and 7 at 64), and the steps after it.

Tolerances as stated in test_gpu_parity.py (check_close)."""
import numpy as np
import pytest
import torch

import d2sd
from test_gpu_parity import bf16_randn, check_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _tree(n, rng):
    parent = [-1] + [int(rng.integers(0, i)) for i in range(1, n)]
    m = np.zeros((n, n), dtype=bool)
    for i, p in enumerate(parent):
        if p >= 0:
            m[i] = m[p]
        m[i, i] = True
    return m


@pytest.mark.parametrize("d,fp8", [(128, False), (64, False), (128, True)])
@pytest.mark.parametrize("nodes", [1, 33, 65, 129, 200])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("paged", [True, False])
def test_half_tile_edges(d, fp8, nodes, splits, paged):
    rng = np.random.default_rng(d + nodes)
    gen = torch.Generator().manual_seed(nodes)
    hq, hkv, P = 8, 2, 16
    mask = _tree(nodes, rng)
    q, ks, vs = bf16_randn(gen, nodes, hq, d), bf16_randn(gen, nodes, hkv, d), bf16_randn(gen, nodes, hkv, d)
    for L, window in [(1, -1), (31, -1), (32, -1), (33, -1), (64, -1), (97, -1), (128, -1), (161, -1), (224, -1),
                      (257, -1), (320, -1), (333, -1), (512, -1), (300, 170), (530, 321)]:
        kp, vp = bf16_randn(gen, L, hkv, d), bf16_randn(gen, L, hkv, d)
        if fp8:
            kp, vp = kp.to(torch.float8_e4m3fn), vp.to(torch.float8_e4m3fn)
        sees = np.ones((nodes, L), dtype=bool)
        if window >= 0:
            sees[:, :max(0, L - window)] = False
        full = torch.from_numpy(np.concatenate([sees, mask], 1))
        o_ref, lse_ref = _oracle(q, torch.cat([kp.float(), ks.float()]), torch.cat([vp.float(), vs.float()]), full)
        kw = dict(kv_layout="NHD")
        if paged:
            n = -(-L // P)
            table = torch.randperm(n + 1, generator=gen)[:n]
            pool = torch.zeros(2, (n + 1) * P, hkv, d)
            rows = (table[:, None] * P + torch.arange(P)).reshape(-1)[:L]
            pool[0, rows], pool[1, rows] = kp.float(), vp.float()
            kd, vd = (x.reshape(n + 1, P, hkv, d).to(kp.dtype).to(DEV) for x in pool)
            kw.update(page_size=P, page_indptr=[0, n], page_table=table.to(torch.int32).to(DEV))
        else:
            kd, vd = kp.to(DEV), vp.to(DEV)
        if fp8:
            one = torch.ones(hkv, device=DEV)
            kw.update(kv_dtype=torch.float8_e4m3fn, k_scale=one, v_scale=one)
        attn = d2sd.CascadeVerifyAttention(DEV).plan([0, nodes], [L], hq, hkv, d, tree_masks=[mask], max_splits=splits,
                                                     window_left=window, **kw)
        o, lse = attn.run(q.to(DEV), ks.to(DEV), vs.to(DEV), kd, vd)
        torch.cuda.synchronize()
        check_close(o, o_ref, lse, lse_ref, f"L {L} window {window}")


@pytest.mark.parametrize("d,waves", [(128, 4), (128, 2), (128, 8), (64, 4), (64, 2), (64, 8)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("P", [16, 64, 0])
@pytest.mark.parametrize("L", [2 * 320, 2 * 448 + 17, 2 * 512 + 40, 2 * 640 + 63])
def test_split_chunks_past_the_ring(d, waves, fp8, P, L):
    nodes, hq, hkv = 70, 8, 2
    gen = torch.Generator().manual_seed(L + d)
    mask = _tree(nodes, np.random.default_rng(L))
    q, ks, vs = bf16_randn(gen, nodes, hq, d), bf16_randn(gen, nodes, hkv, d), bf16_randn(gen, nodes, hkv, d)
    kp, vp = bf16_randn(gen, L, hkv, d), bf16_randn(gen, L, hkv, d)
    kw = dict(kv_layout="NHD")
    if fp8:
        kp, vp = kp.to(torch.float8_e4m3fn), vp.to(torch.float8_e4m3fn)
        one = torch.ones(hkv, device=DEV)
        kw.update(kv_dtype=torch.float8_e4m3fn, k_scale=one, v_scale=one)
    kd, vd = kp.to(DEV), vp.to(DEV)
    if P:
        n = -(-L // P)
        table = torch.randperm(n + 1, generator=gen)[:n]
        pool = torch.zeros(2, (n + 1) * P, hkv, d)
        rows = (table[:, None] * P + torch.arange(P)).reshape(-1)[:L]
        pool[0, rows], pool[1, rows] = kp.float(), vp.float()
        kd, vd = (x.reshape(n + 1, P, hkv, d).to(kp.dtype).to(DEV) for x in pool)
        kw.update(page_size=P, page_indptr=[0, n], page_table=table.to(torch.int32).to(DEV))
    attn = d2sd.CascadeVerifyAttention(DEV).plan([0, nodes], [L], hq, hkv, d, tree_masks=[mask], max_splits=2,
                                                 waves_per_block=waves, **kw)
    assert not attn.info.fused and attn.info.max_splits_used == 2, "two chunks of 5 to 11 tiles"
    full = torch.from_numpy(np.concatenate([np.ones((nodes, L), dtype=bool), mask], 1))
    o_ref, lse_ref = _oracle(q, torch.cat([kp.float(), ks.float()]), torch.cat([vp.float(), vs.float()]), full)
    o, lse = attn.run(q.to(DEV), ks.to(DEV), vs.to(DEV), kd, vd)
    torch.cuda.synchronize()
    check_close(o, o_ref, lse, lse_ref, f"L {L}")


def _oracle(q, k, v, mask):
    """Masked softmax attention in float64: O [n, hq, d] and natural-log LSE."""
    g = q.shape[1] // k.shape[1]
    qd, kd, vd = q.double(), k.double().repeat_interleave(g, 1), v.double().repeat_interleave(g, 1)
    s = torch.matmul(qd.transpose(0, 1), kd.permute(1, 2, 0).contiguous()) * q.shape[2] ** -0.5
    s = s.masked_fill(~mask[None], float("-inf"))
    lse = torch.logsumexp(s, -1)
    o = torch.matmul(torch.exp(s - lse[..., None]), vd.transpose(0, 1).contiguous())
    return o.transpose(0, 1), lse.transpose(0, 1)
