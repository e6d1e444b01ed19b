"""QK RMSNorm + RoPE where one operand's rows are off 16-byte boundaries (its base or
one of its strides), which takes the kernel of one wave per head: against the
oracle, with the tolerances of test_gpu_qk_rope.py.  Each operand is misaligned
alone; the aligned call on the same values has to agree as closely."""
import pytest
import torch

from oracle import cascade_oracle as orc
import d2sd
from test_gpu_qk_rope import _close, _rope_scale, _rope_table

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _place(x, how, pad=3):
    """x on the device: "base" one element off a 16-byte boundary, "token" / "head"
    with `pad` elements between its tokens / heads."""
    if how == "base":
        buf = torch.zeros(x.numel() + 1, dtype=x.dtype, device=DEV)
        out = buf[1:].view(x.shape)
    elif how == "token":
        n = x[0].numel()
        buf = torch.zeros(x.shape[0], n + pad, dtype=x.dtype, device=DEV)
        out = buf[:, :n].unflatten(1, x.shape[1:]) if x.dim() > 2 else buf[:, :n]
    elif how == "head":
        buf = torch.zeros(*x.shape[:-1], x.shape[-1] + pad, dtype=x.dtype, device=DEV)
        out = buf[..., :x.shape[-1]]
    else:
        return x.to(DEV)
    out.copy_(x)
    return out


@pytest.mark.parametrize("d,half", [(64, True), (128, False), (256, False)])
@pytest.mark.parametrize("operand,how", [("q", "base"), ("q", "token"), ("q", "head"), ("k", "base"), ("k", "token"),
                                         ("k", "head"), ("q_norm", "base"), ("k_norm", "base"), ("cos", "base"),
                                         ("cos", "token")])
def test_unaligned_rows(d, half, operand, how):
    g = torch.Generator().manual_seed(d)
    T, hq, hkv = 37, 6, 2
    q = (torch.randn(T, hq, d, generator=g) * 2).to(torch.bfloat16)
    k = (torch.randn(T, hkv, d, generator=g) * 2).to(torch.bfloat16)
    wq = (torch.rand(d, generator=g) + 0.5).to(torch.bfloat16)
    wk = (torch.rand(d, generator=g) + 0.5).to(torch.bfloat16)
    cos, sin = _rope_table(T, d, half, g)
    at = lambda name: how if operand == name else None
    qd, kd = _place(q, at("q")), _place(k, at("k"))
    # (cos and sin share one stride; "base" moves cos alone, then sin alone)
    tables = [(_place(cos, at("cos")), _place(sin, at("cos") if how == "token" else None))]
    if operand == "cos" and how == "base":
        tables.append((cos.to(DEV), _place(sin, "base")))
    ref_q, ref_k = (orc.qk_norm_rope_ref(x, w, cos, sin, 1e-6) for x, w in ((q, wq), (k, wk)))
    scale_q, scale_k = (_rope_scale(orc.qk_norm_rope_ref(x, w, None, None, 1e-6)) for x, w in ((q, wq), (k, wk)))
    for c, s in tables:
        qd.copy_(q)
        kd.copy_(k)
        d2sd.qk_norm_rope(qd, kd, _place(wq, at("q_norm")), _place(wk, at("k_norm")), c, s, 1e-6)
        torch.cuda.synchronize()
        _close(qd, ref_q, scale_q, 4, "q")
        _close(kd, ref_k, scale_k, 4, "k")
        # what lies between the rows is untouched
        for x in (qd, kd):
            if x._base is not None:
                inside = torch.zeros_like(x._base, dtype=torch.bool)
                torch.as_strided(inside, x.shape, x.stride(), x.storage_offset()).fill_(True)
                assert (x._base[~inside] == 0).all()
