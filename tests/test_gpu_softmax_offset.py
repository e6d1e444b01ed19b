"""The exponents' offset is a maximum over whole 64-key tiles: a row whose
largest score lies in the upper 32 keys of the tile in which its running max
grows has exp2(0) = 1 for that key, which bf16 holds exactly.

One key (position 40 of tile t) carries more than 92% of each row; key 0 of the
tile is 3.6 to 7.8 log2 units below it (less than the kernel's slack of 8, so
that an offset taken from the lower 32 keys would stay), everything else far
below.  bf16 rounds to half a unit in the last place, 2^-8 / m of a value of
mantissa m: rms 2^-8 / sqrt(3) * sqrt(E[1 / m^2]) = 2^-8 / sqrt(6) = 1.6e-3 over
uniform mantissas.  A probability P of that key other than 1 puts this error on
the whole row.  The roundings of the output and of a partial state are
independent per element: on the row's scale (the projection on the float64
result) they leave 1.6e-3 sqrt(sum v^4) / sum v^2, 1.6e-3 sqrt(3 / D) for normal
values: 3.5e-4 for D = 64, 4.9e-4 with a partial state.  Rows' scale errors have
to stay under 9e-4 rms, between the two."""
import pytest
import torch

import d2sd
from test_gpu_parity import bf16_randn

pytestmark = pytest.mark.gpu
DEV = "cuda"
LOW = -384.0  # with a query's component in [1, 2): at least 49 log2 units below 0


def _keys(n, t, hkv, d):
    """Scores LOW r, but 0 for key 64 t and 30 r for key 64 t + 40 (D = 128; 21 r for 64)."""
    k = torch.zeros(n, hkv, d)
    k[:, :, 0] = LOW
    if t is not None:
        k[64 * t, :, 0] = 0.0
        k[64 * t + 40, :, 0] = 30.0 if d == 128 else 21.0
    return k.to(torch.bfloat16)


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("nodes,splits", [(40, 1), (40, 0), (80, 1)])
@pytest.mark.parametrize("where", ["prefix 0", "prefix 1", "prefix 3", "prefix 7", "suffix 0", "suffix 1"])
def test_offset_is_a_tile_maximum(d, fp8, nodes, splits, where):
    level, t = where.split()
    t = int(t)
    gen = torch.Generator().manual_seed(nodes + d)
    hq, hkv, L = 8, 2, 512
    if level == "suffix":
        nodes = 64 * t + 64
    q = bf16_randn(gen, nodes, hq, d)
    q[:, :, 0] = (1.0 + torch.rand(nodes, hq, generator=gen) * 0.99).to(torch.bfloat16)
    kp, ks = _keys(L, t if level == "prefix" else None, hkv, d), _keys(nodes, t if level == "suffix" else None, hkv, d)
    vp, vs = bf16_randn(gen, L, hkv, d), bf16_randn(gen, nodes, hkv, d)
    kw = {}
    if fp8:
        kp, vp = kp.to(torch.float8_e4m3fn), vp.to(torch.float8_e4m3fn)
        one = torch.ones(hkv, device=DEV)
        kw = dict(kv_dtype=torch.float8_e4m3fn, k_scale=one, v_scale=one)
    attn = d2sd.CascadeVerifyAttention(DEV).plan([0, nodes], [L], hq, hkv, d, mask_mode="none", kv_layout="NHD",
                                                 max_splits=splits, **kw)
    o, _ = attn.run(q.to(DEV), ks.to(DEV), vs.to(DEV), kp.to(DEV), vp.to(DEV))
    k, v = torch.cat([kp.double(), ks.double()]), torch.cat([vp.double(), vs.double()])
    g = hq // hkv
    s = torch.matmul(q.double().transpose(0, 1), k.repeat_interleave(g, 1).permute(1, 2, 0).contiguous()) * d ** -0.5
    ref = torch.matmul(torch.softmax(s, -1), v.repeat_interleave(g, 1).transpose(0, 1).contiguous()).transpose(0, 1)
    scale = (o.cpu().double() * ref).sum(-1) / (ref * ref).sum(-1) - 1
    rms = scale.square().mean().sqrt().item()
    assert rms < 9e-4, f"scale error {rms:.2e} (rms over rows)"
