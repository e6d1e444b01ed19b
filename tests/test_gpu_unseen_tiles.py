"""Suffix tiles that none of a wave's rows sees take no part in its result: values
of +inf there (0 * inf would be NaN in the PV product) leave the rows that do not
see them finite and equal to the float64 oracle.  Causal suffixes (the tiles
past a row block's diagonal) and trees whose blocks see tiles in the middle and
at the end only, over every kind of plan.  Tolerances as stated in
test_gpu_parity.py (check_close)."""
import numpy as np
import pytest
import torch

import d2sd
from test_gpu_half_tiles import _oracle
from test_gpu_parity import bf16_randn, check_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mask(kind, n):
    if kind == "causal":
        return np.tril(np.ones((n, n), dtype=bool))
    if kind == "blocks":  # 32-node blocks that see themselves
        return np.kron(np.eye(-(-n // 32), dtype=bool), np.ones((32, 32), dtype=bool))[:n, :n]
    m = np.zeros((n, n), dtype=bool)  # a chain per 64 nodes below node 0; the odd chains see the one before
    for i in range(n):
        m[i, (i // 64) * 64:i + 1] = True
        m[i, 0] = True
        if (i // 64) % 2:
            m[i, (i // 64 - 1) * 64:(i // 64) * 64] = True
    return m


@pytest.mark.parametrize("d,waves", [(128, 4), (128, 2), (128, 8), (64, 4), (64, 2), (64, 8)])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("kind", ["causal", "blocks", "chains"])
@pytest.mark.parametrize("n,L,splits", [(200, 0, 0), (256, 300, 3), (256, 130, 1), (330, 700, 0)])
def test_unseen_tiles_are_left_out(d, waves, fp8, kind, n, L, splits):
    gen = torch.Generator().manual_seed(n + d)
    hq, hkv = 8, 2
    mask = _mask(kind, n)
    q, ks, vs = bf16_randn(gen, n, hq, d), bf16_randn(gen, n, hkv, d), bf16_randn(gen, n, hkv, d)
    kp, vp = bf16_randn(gen, max(L, 1), hkv, d), bf16_randn(gen, max(L, 1), hkv, d)
    kw = {}
    if fp8:
        kp, vp = kp.to(torch.float8_e4m3fn), vp.to(torch.float8_e4m3fn)
        one = torch.ones(hkv, device=DEV)
        kw = dict(kv_dtype=torch.float8_e4m3fn, k_scale=one, v_scale=one)
    full = torch.from_numpy(np.concatenate([np.ones((n, L), dtype=bool), mask], 1))
    o_ref, lse_ref = _oracle(q, torch.cat([kp.float()[:L], ks.float()]), torch.cat([vp.float()[:L], vs.float()]), full)
    # tiles made infinite: one in the middle, and the last one
    for t in (1, (n - 1) // 64):
        vi = vs.clone()
        vi[64 * t:64 * t + 64] = float("inf")
        # rows of wave row blocks (at most 64 rows = 16 nodes) none of whose rows sees the tile
        blind = ~mask[:, 64 * t:64 * t + 64].any(1)
        clean = np.array([blind[i // 16 * 16:i // 16 * 16 + 16].all() for i in range(n)])
        assert clean.sum() >= 64
        if kind == "causal":
            kw2 = dict(mask_mode="causal")
        else:
            kw2 = dict(tree_masks=[mask])
        attn = d2sd.CascadeVerifyAttention(DEV).plan([0, n], [L], hq, hkv, d, kv_layout="NHD", max_splits=splits,
                                                     waves_per_block=waves, **kw, **kw2)
        o, lse = attn.run(q.to(DEV), ks.to(DEV), vi.to(DEV), kp.to(DEV), vp.to(DEV))
        torch.cuda.synchronize()
        check_close(o[clean], o_ref[clean], lse[clean], lse_ref[clean], f"tile {t}")
        # with finite values everywhere, every row
        o, lse = attn.run(q.to(DEV), ks.to(DEV), vs.to(DEV), kp.to(DEV), vp.to(DEV))
        torch.cuda.synchronize()
        check_close(o, o_ref, lse, lse_ref, f"tile {t}, finite")


@pytest.mark.parametrize("d,waves", [(128, 4), (128, 2), (64, 4)])
@pytest.mark.parametrize("n", [192, 193, 257])
@pytest.mark.parametrize("P", [0, 16])
@pytest.mark.parametrize("dynamic", [False, True])
def test_trees_at_the_kernels_boundary(d, waves, n, P, dynamic):
    """Split plans take kernels with two bodies from 4 mask words per row on (193
    nodes): both sides of that line, contiguous and paged, also with the prefix
    length read at run time, eager and replayed from a graph."""
    gen = torch.Generator().manual_seed(n + d)
    hq, hkv, L, cap = 8, 2, 461, 600
    mask = _mask("chains", n)
    q, ks, vs = bf16_randn(gen, n, hq, d), bf16_randn(gen, n, hkv, d), bf16_randn(gen, n, hkv, d)
    kp, vp = bf16_randn(gen, cap, hkv, d), bf16_randn(gen, cap, hkv, d)
    kw = {}
    kd, vd = kp.to(DEV), vp.to(DEV)
    if P:
        pages = -(-cap // P)
        table = torch.randperm(pages, generator=gen)
        pool = torch.zeros(2, pages * P, hkv, d, dtype=torch.bfloat16)
        rows = (table[:, None] * P + torch.arange(P)).reshape(-1)[:cap]
        pool[0, rows], pool[1, rows] = kp, vp
        kd, vd = (x.reshape(pages, P, hkv, d).to(DEV) for x in pool)
        kw = dict(page_size=P, page_indptr=[0, pages if dynamic else -(-L // P)],
                  page_table=(table if dynamic else table[:-(-L // P)]).to(torch.int32).to(DEV))
    attn = d2sd.CascadeVerifyAttention(DEV).plan([0, n], [cap if dynamic else L], hq, hkv, d, tree_masks=[mask],
                                                 kv_layout="NHD", max_splits=3, waves_per_block=waves,
                                                 dynamic_prefix=dynamic, **kw)
    assert not attn.info.fused
    if dynamic:
        attn.set_prefix_len([L])
    full = torch.from_numpy(np.concatenate([np.ones((n, L), dtype=bool), mask], 1))
    o_ref, lse_ref = _oracle(q, torch.cat([kp[:L], ks]).float(), torch.cat([vp[:L], vs]).float(), full)
    args = [x.to(DEV) for x in (q, ks, vs)] + [kd, vd]
    out, lse = torch.zeros(n, hq, d, dtype=torch.bfloat16, device=DEV), torch.zeros(n, hq, device=DEV)
    attn.run(*args, out=out, lse=lse)
    torch.cuda.synchronize()
    check_close(out, o_ref, lse, lse_ref, "eager")
    eager = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        attn.run(*args, out=out, lse=lse)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
