"""GPU: the bf16 row gather's sums on the matrix cores (gather.hip
gather_slots_mx) at its edges: slot counts around a step (4 slots a lane group) and
a block of 64, one to 512 slots, head dimensions that fill 4, 8, 16 (with unused
lanes) and 16 lanes and the first one that takes the plain form (16), with and
without key sums, both layouts, invalid slots, repeated indices, empty rows.  Against
float64 sums over the same lists (outputs: half a bf16 step of the largest
magnitude, 2^-8 leaves one bit) and, before the rounding, against the plain form, which
fp32 copies of the same rows take: its outputs rounded to bf16 may differ by one
step where the order of the sums decides.  A row of inf that a query row selects
gives it what the plain form gives; one that it does not select stays out."""

import pytest
import torch

from sgsa_amd.retrieval import gather_masked

pytestmark = pytest.mark.gpu


def _lists(B, H, Tq, Tk, k, off, gen, dev):
    pos = torch.arange(Tq) + off
    idx = (torch.rand(B, H, Tq, k, generator=gen) * (pos[:, None] + 1)).long().clamp(max=Tk - 1)   # repeats in it
    sc = 3 * torch.randn(B, H, Tq, k, generator=gen)
    cnt = torch.minimum(pos + 1, torch.full_like(pos, k)).expand(B, H, Tq).clone()
    cnt[:, :, 5] = 0
    return idx.int().to(dev), sc.to(dev), cnt.int().to(dev)


def _top2(sc, cnt, valid):
    n = torch.arange(sc.shape[-1], device=sc.device) < cnt[..., None]
    if valid is not None:
        n = n & (valid != 0)
    s = torch.where(n, sc, torch.full_like(sc, torch.finfo(torch.float32).min))
    return torch.nn.functional.pad(s, (0, 1), value=torch.finfo(torch.float32).min).topk(2).values.contiguous(), n


@pytest.mark.parametrize("H,D,Tq,Tk,k,keys,masked", [
    (2, 128, 130, 130, 100, True, False), (3, 128, 77, 100, 65, False, True), (1, 128, 700, 700, 512, True, True),
    (2, 64, 130, 131, 64, True, True), (2, 96, 90, 90, 63, False, False), (4, 32, 70, 300, 257, True, False),
    (2, 128, 20, 20, 1, False, False), (2, 128, 20, 20, 3, True, False), (1, 16, 40, 40, 20, True, False)])
def test_mx_gather(dev, H, D, Tq, Tk, k, keys, masked):
    gen = torch.Generator().manual_seed(Tq + k)
    B, off = 2, Tk - Tq
    rnd = lambda *s: torch.randn(*s, generator=gen).to(dev).bfloat16()
    hm = 0 if keys else 1
    V = rnd(B, Tk, H, D) if keys else rnd(B, H, Tk, D)
    K = rnd(B, Tk, H, D) if keys else None
    idx, sc, cnt = _lists(B, H, Tq, Tk, k, off, gen, dev)
    valid = (torch.rand(idx.shape, generator=gen).to(dev) < 0.8).to(torch.uint8) if masked else None
    top2, n = _top2(sc, cnt, valid)
    run = lambda K, V: gather_masked(K, V, idx, sc, valid, top2, cnt, q_offset=off, kv_layout=hm, return_weights=True)
    r, plain = run(K, V), run(None if K is None else K.float(), V.float())
    w = torch.where(n, sc.double() - top2[..., :1].double(), torch.full_like(sc, -float("inf")).double()).exp()
    w = w / w.sum(-1, keepdim=True).clamp_min(1e-300)
    assert (r["weights"].double() - w).abs().max() <= 1e-6
    assert torch.equal(r["weights"], plain["weights"])
    full = torch.zeros(B, H, Tq, Tk, dtype=torch.float64, device=dev).scatter_add_(3, idx.long(), w)
    for X, name in ((K, "k_hat"), (V, "v_hat")):
        if X is None:
            continue
        xh = X.transpose(1, 2) if hm == 0 else X
        ref = torch.matmul(full, xh.double().contiguous()).transpose(1, 2)
        got = r[name].double()
        assert torch.isfinite(got).all()
        assert (got - ref).abs().max() <= 2.0 ** -8 * ref.abs().max()
        assert ((got - plain[name].bfloat16().double()).abs() <= 2.0 ** -7 * ref.abs() + 1e-6).all()


def test_mx_gather_nonfinite_rows(dev):
    B, H, T, k, D = 1, 4, 300, 40, 128
    gen = torch.Generator().manual_seed(3)
    V = torch.randn(B, T, H, D, generator=gen).to(dev).bfloat16()
    idx, sc, cnt = _lists(B, H, T, T, k, 0, gen, dev)
    V[:, 7, 3, 11], V[:, 200, 2, 5] = float("inf"), float("nan")
    top2, n = _top2(sc, cnt, None)
    out = gather_masked(V, V, idx, sc, None, top2, cnt)["v_hat"]
    plain = gather_masked(V.float(), V.float(), idx, sc, None, top2, cnt)["v_hat"]
    hit = ((idx[0, 3] == 7) & n[0, 3]).any(-1)
    assert hit.any() and (out[0, hit, 3, 11] == float("inf")).all()
    assert torch.equal(out.isnan(), plain.isnan()) and torch.equal(out.isinf(), plain.isinf())
    assert out.isnan().any() and torch.isfinite(out[:, :, :2]).all()
