"""GPU: the score-buffer form of the row lists (topk_buf.hip) at the edges of its
tiles, registers and LDS lists: key counts around 64, 256 and the 2048-, 4096- and
8192-key register forms, more slots than the sorted list holds (512), bins that
overflow it (mass ties), infinite scores, and dimensions and alignments that take
the staged score kernel.  Indices and scores must equal the lowest-index top-k of
the exact scores score_dump returns, bit for bit, sorted and unsorted.  The first
list runs on whichever form the dispatch takes (its calls of few rows and many keys
take the row kernel); FORMS names the form, which shows in an unsorted row's runs.
NaN scores sort by their bits as the order key has them, a positive NaN above +inf."""

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
    if kind == "nan":   # keys whose scores are NaN
        k = k.clone()
        k[:, 3::41, :, D // 2] = float("nan")
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


def _buffer_form(B, Tq, Tk, H, D, k, srt, causal, off):
    """topk_buf.hip topk_buf_fits: whether a call takes this form or the row kernel."""
    sorts = srt and k <= 512
    if Tk > ((4096 if sorts else 2048) if D == 128 else 8192):
        return False

    def keys(n):
        rows = torch.arange(n)
        return int((rows + off + 1).clamp(0, Tk).sum()) if causal else n * Tk

    if D == 128 and not sorts:
        kept = Tq if k >= Tk else min(Tq, max(0, k - off)) if causal else 0
        longest = min(Tk, Tq + off) if causal else Tk
        if 0 < keys(kept) >= 512 * (Tq - kept) and B * H * keys(Tq) >= (84 if kept < Tq else 42) * 256 * longest:
            return False
    pitch = (Tk + 255) // 256 * 256 + 64
    room = B * H * Tq * 512 * 8 // (64 * pitch * 4)
    return room * ((pitch + 1023) // 1024 + 1) >= B * H * ((Tq + 63) // 64)


def _keys(x):   # the order-preserving key of an fp32 score, -0 as +0
    b = torch.where(x == 0, torch.zeros_like(x), x).contiguous().view(torch.int32).long() & 0xffffffff
    return torch.where(b >= 2 ** 31, 2 ** 32 - 1 - b, b + 2 ** 31)


def _check_form(dev, dt, B, Tq, Tk, H, D, top_k, kind, causal, srt, form):
    """Every row against a stable sort of score_dump's keys, on the form that the rule names: the buffer form leaves
    an unsorted row as one ascending run, the row kernel the keys of the cut's bin after the others."""
    q, k = _inputs(torch.bfloat16 if dt == "bf16" else torch.float32, B, Tq, Tk, H, D, kind, dev)
    off = max(0, Tk - Tq) if causal else 0
    kk = min(top_k, Tk)
    assert _buffer_form(B, Tq, Tk, H, D, kk, srt, causal, off) == form
    dump = sgsa_amd.score_dump(q, k, 0, Tq, causal=causal, q_offset=off)
    got = sgsa_amd.score_topk(q, k, top_k, causal=causal, q_offset=off, sorted=srt, fast=False, return_split=not srt)
    idx, sc, top2, cnt = got[:4]
    if not srt and kind == "random":
        assert torch.equal(got[4], cnt) == form
    nv = (torch.arange(Tq, device=dev) + off + 1).clamp(max=Tk) if causal else torch.full((Tq,), Tk, device=dev)
    n = nv.clamp(max=kk)
    assert torch.equal(cnt, n.int().expand(B, H, Tq))
    valid = torch.arange(Tk, device=dev) < nv[:, None]
    for h in range(H):   # by head: the sorts take 24 bytes a score
        d = dump[:, h]
        order = torch.sort(torch.where(valid, _keys(d), torch.full((), -1, device=dev)), dim=-1, descending=True, stable=True)[1][..., :kk]
        used = torch.arange(kk, device=dev) < n[:, None]
        gi, gs = idx[:, h].long(), sc[:, h]
        if not srt:
            big = torch.where(used, gi, torch.full((), Tk, device=dev)).sort(dim=-1)
            gi, gs = big[0], gs.gather(-1, big[1])
            order = torch.where(used, order, torch.full((), Tk, device=dev)).sort(dim=-1)[0]
        want = d.gather(-1, order.clamp(max=Tk - 1))
        u = used.expand(B, Tq, kk)
        assert torch.equal(gi[u], order[u]), h
        assert torch.equal(_keys(gs[u]), _keys(want[u])), h
        assert (idx[:, h][~u] == 0).all()
        best = torch.where(valid & ~d.isnan(), d, torch.full((), torch.finfo(torch.float32).min, device=dev)).amax(-1)
        assert torch.equal(top2[:, h, :, 0], best)


@pytest.mark.parametrize("dt", ["bf16", "fp32"])
@pytest.mark.parametrize("H,T,top_k,causal,form", [(128, 640, 520, True, False), (64, 640, 520, True, True),
                                                   (128, 640, 520, False, True), (96, 600, 300, True, True)])
def test_mostly_kept_rows_take_the_row_kernel(dev, dt, H, T, top_k, causal, form):
    print(f"score buffer form {dt} {H} {T} {top_k} {causal}", flush=True)
    _check_form(dev, dt, 1, T, T, H, 128, top_k, "random", causal, False, form)


FORMS = [  # dtype, B, Tq, Tk, H, D, top_k, kind, the buffer form when sorted and when not
    # the registers of a row: 1, 2, 4, 8, 16 and 32 vectors of 256 keys
    ("bf16", 1, 100, 192, 2, 128, 1, "random", True, True), ("bf16", 1, 128, 257, 2, 128, 64, "random", True, True),
    ("fp32", 2, 129, 600, 3, 64, 65, "random", True, True), ("bf16", 1, 200, 1100, 2, 128, 128, "random", True, True),
    ("bf16", 1, 300, 2300, 2, 64, 129, "random", True, True), ("fp32", 1, 320, 4097, 2, 96, 257, "random", True, True),
    ("bf16", 1, 640, 5000, 2, 40, 33, "random", True, True), ("fp32", 1, 640, 5000, 2, 64, 512, "random", True, True),
    ("bf16", 1, 320, 8192, 2, 64, 700, "random", True, True),
    # D = 128: the key limits of the sorted and unsorted calls, and lists that are too long to sort here
    ("bf16", 1, 320, 4096, 2, 128, 65, "random", True, False), ("fp32", 1, 320, 4000, 2, 128, 512, "random", True, False),
    ("bf16", 1, 320, 4097, 2, 128, 65, "random", False, False), ("bf16", 1, 300, 2049, 2, 128, 256, "random", True, False),
    ("bf16", 1, 300, 2048, 2, 128, 513, "random", True, True), ("fp32", 1, 300, 2048, 2, 128, 600, "random", True, True),
    # too few rows for a slab of the buffer
    ("bf16", 1, 256, 8192, 2, 64, 33, "random", False, False), ("bf16", 1, 70, 4096, 2, 128, 65, "random", False, False),
    # and the row kernel's sort of 256 and 512 slots in registers, and of more in LDS
    ("bf16", 1, 70, 4500, 2, 128, 256, "random", False, False), ("fp32", 1, 70, 4500, 2, 128, 512, "random", False, False),
    ("bf16", 1, 70, 4500, 2, 128, 513, "random", False, False),
    # scores that no histogram separates, and those that are no numbers
    ("bf16", 1, 640, 5000, 2, 64, 300, "tied", True, True), ("fp32", 1, 640, 5000, 2, 64, 600, "equal", True, True),
    ("bf16", 1, 320, 4096, 2, 128, 500, "equal", True, False), ("fp32", 1, 320, 3000, 2, 64, 400, "infinite", True, True),
    ("bf16", 1, 320, 4096, 2, 128, 300, "infinite", True, False), ("bf16", 1, 130, 700, 2, 128, 90, "nan", True, True),
    ("bf16", 1, 130, 700, 2, 128, 600, "nan", True, True), ("fp32", 1, 320, 4100, 2, 64, 64, "nan", True, True),
    ("fp32", 1, 130, 300, 2, 40, 3, "nan", True, True),
]


@pytest.mark.parametrize("dt,B,Tq,Tk,H,D,top_k,kind,srt,uns", FORMS)
def test_select_forms(dev, dt, B, Tq, Tk, H, D, top_k, kind, srt, uns):
    print(f"score buffer forms {dt} {B} {Tq} {Tk} {H} {D} {top_k} {kind}", flush=True)
    for causal in (True, False):
        for s, form in ((True, srt), (False, uns)):
            _check_form(dev, dt, B, Tq, Tk, H, D, top_k, kind, causal, s, form)
