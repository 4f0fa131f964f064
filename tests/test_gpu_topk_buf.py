"""GPU: the score-buffer form of the row lists (topk_buf.hip) at the edges of its
tiles, registers and LDS lists: key counts around 64, 256 and the 2048-, 4096- and
8192-key register forms, more slots than the sorted list holds (512), bins that
overflow it (mass ties), infinite scores, and dimensions and alignments that take
the staged score kernel.  Indices and scores must equal the lowest-index top-k of
the exact scores score_dump returns, bit for bit, sorted and unsorted."""

import pytest
import torch

from oracle import sgsa_oracle as O

pytestmark = pytest.mark.gpu

import sgsa_amd  # noqa: E402

CASES = [  # dtype, B, Tq, Tk, H, D, top_k, kind
    ("bf16", 1, 1, 1, 1, 128, 4, "random"), ("bf16", 1, 63, 63, 2, 128, 8, "random"),
    ("bf16", 2, 65, 257, 3, 128, 100, "random"), ("bf16", 1, 256, 256, 2, 96, 64, "random"),
    ("bf16", 1, 96, 2049, 2, 128, 512, "random"), ("bf16", 1, 130, 2048, 2, 128, 513, "random"),
    ("bf16", 1, 70, 4096, 2, 128, 65, "random"), ("bf16", 1, 70, 8192, 2, 64, 700, "random"),
    ("bf16", 1, 70, 5000, 2, 40, 33, "random"), ("bf16", 1, 64, 700, 2, 35, 128, "shift"),
    ("fp32", 1, 65, 640, 2, 64, 129, "random"), ("fp32", 1, 64, 1025, 2, 128, 300, "random"),
    ("fp32", 1, 64, 300, 2, 5, 64, "shift"), ("bf16", 1, 70, 2000, 2, 128, 600, "tied"),
    ("bf16", 1, 70, 2000, 2, 128, 100, "equal"), ("fp32", 1, 70, 900, 1, 64, 700, "equal"),
    ("bf16", 1, 70, 600, 2, 128, 90, "infinite"), ("fp32", 1, 70, 600, 2, 64, 550, "infinite"),
]


def _inputs(dt, B, Tq, Tk, H, D, kind, dev):
    g = torch.Generator().manual_seed(17)
    q, k = torch.randn(B, Tq, H, D, generator=g), torch.randn(B, Tk, H, D, generator=g)
    if kind == "tied":   # few distinct keys: thousands of equal scores
        k = k[:, :3].repeat(1, Tk // 3 + 1, 1, 1)[:, :Tk]
    if kind == "equal":
        k = k[:, :1].expand(B, Tk, H, D)
    if kind == "infinite":   # every 37th key overflows the product to +inf or -inf, by the query's sign
        k = k.clone()
        k[:, ::37] = 0.0
        k[:, ::37, :, 0] = 3e38
        q[..., 0] = torch.sign(q[..., 0]) * 1e3
    out = []
    for x in (q, k):
        buf = torch.empty(x.numel() + 1, dtype=dt, device=dev)
        s = 1 if kind == "shift" else 0
        buf[s:s + x.numel()] = x.reshape(-1).to(dt)
        out.append(buf[s:s + x.numel()].view(x.shape))
    return out


@pytest.mark.parametrize("dt,B,Tq,Tk,H,D,top_k,kind", CASES)
def test_score_buffer_select(dev, dt, B, Tq, Tk, H, D, top_k, kind):
    q, k = _inputs(torch.bfloat16 if dt == "bf16" else torch.float32, B, Tq, Tk, H, D, kind, dev)
    print(f"score buffer {dt} {B} {Tq} {Tk} {H} {D} {top_k} {kind}", flush=True)
    for causal in (True, False):
        off = max(0, Tk - Tq) if causal else 0
        dump = sgsa_amd.score_dump(q, k, 0, Tq, causal=causal, q_offset=off).cpu()
        for srt in (True, False):
            idx, sc, top2, cnt = (t.cpu() for t in sgsa_amd.score_topk(q, k, top_k, causal=causal, q_offset=off,
                                                                       sorted=srt, fast=False))
            kk = idx.shape[-1]
            nv = torch.arange(Tq) + off + 1 if causal else torch.full((Tq,), Tk)
            want_n = nv.clamp(max=min(kk, Tk))
            assert torch.equal(cnt, want_n.to(torch.int32).expand(B, H, Tq))
            for b in range(B):
                for h in range(H):
                    for r in range(0, Tq, 7):
                        n = int(want_n[r])
                        row = dump[b, h, r, :int(nv[r])]
                        vals, want = (t[0] for t in O.topk_lowest_index(row[None], n))
                        got, gs = idx[b, h, r, :n].long(), sc[b, h, r, :n]
                        if not srt:
                            got, order = got.sort()
                            gs = gs[order]
                            want, order = want.sort()
                            vals = vals[order]
                        assert torch.equal(got, want), (b, h, r)
                        assert torch.equal(gs, vals)
                        assert (idx[b, h, r, n:] == 0).all()
                        assert top2[b, h, r, 0] == row.max()
