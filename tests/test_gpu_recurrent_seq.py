"""GPU: the recurrence over several tokens (recurrent_seq_kernel) at the edges of its
chunks of 8 tokens, of both row-group forms (D <= 64 and above) and of the element-wise
loads, on few and many heads.  Every sum is taken in the one-token kernel's order, so the
outputs and the state must equal as many one-token calls bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from sgsa_amd.recurrent import recurrent_sgsa_fwd  # noqa: E402


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,H,D,sparse,shift", [(1, 4, 1, 128, True, 0), (2, 7, 3, 64, True, 0), (1, 8, 2, 65, True, 0),
                                                  (3, 9, 2, 128, False, 0), (1, 17, 2, 20, False, 0),
                                                  (1, 5, 3, 35, True, 1), (1, 23, 1, 128, True, 2),
                                                  (16, 6, 16, 128, True, 0), (16, 10, 16, 64, True, 0)])
def test_tokens_equal_single_steps(dev, dt, B, T, H, D, sparse, shift):
    g = torch.Generator().manual_seed(41)
    r = lambda *s: torch.randn(*s, generator=g)

    def put(t):   # rows `shift` elements into their storage
        buf = torch.empty(t.numel() + shift, dtype=dt, device=dev)
        buf[shift:] = t.reshape(-1).to(dt)
        return buf[shift:].view(t.shape)

    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    x = [put(unit(r(B, T, H, D))), put(unit(r(B, T, H, D))), put(r(B, T, H, D)), torch.sigmoid(r(B, T, H)).to(dev),
         torch.sigmoid(r(B, T, H) + 3.0).to(dev)]
    x += [put(unit(r(B, T, H, D))), put(r(B, T, H, D)), (0.25 * torch.sigmoid(r(B, T, H))).to(dev)] if sparse \
        else [None] * 3
    st = (0.1 * r(B, H, D, D)).to(dev)
    print(f"recurrent seq {dt} B={B} T={T} H={H} D={D} sparse={sparse} shift={shift}", flush=True)
    o, end = recurrent_sgsa_fwd(*x, initial_state=st, output_final_state=True)
    for t in range(T):
        one, st = recurrent_sgsa_fwd(*(None if a is None else a[:, t:t + 1] for a in x), initial_state=st,
                                     output_final_state=True)
        assert torch.equal(o[:, t:t + 1], one), t
    assert torch.equal(end, st)


@pytest.mark.parametrize("T,D,sparse", [(4, 128, True), (9, 128, False), (13, 64, True), (15, 65, True), (16, 128, True)])
def test_infinite_last_write(dev, T, D, sparse):
    """An infinite value written by the last token stays where it was written: the final state is that of
    one-token calls, infinite entries and finite neighbours, whatever T leaves of the last chunk of 8."""
    g = torch.Generator().manual_seed(43)
    r = lambda *s: torch.randn(*s, generator=g)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    B, H = 2, 3
    x = [unit(r(B, T, H, D)), unit(r(B, T, H, D)), r(B, T, H, D), torch.sigmoid(r(B, T, H)), torch.sigmoid(r(B, T, H) + 3.0)]
    x += [unit(r(B, T, H, D)), r(B, T, H, D), 0.25 * torch.sigmoid(r(B, T, H))] if sparse else [None] * 3
    x[2][0, -1, 1, 5] = float("inf")
    x[1][0, -1, 1, 3] = 0.0   # inf * 0 in one row of that column
    x = [None if t is None else t.to(dev) for t in x]
    st = (0.1 * r(B, H, D, D)).to(dev)
    print(f"recurrent seq infinite T={T} D={D} sparse={sparse}", flush=True)
    o, end = recurrent_sgsa_fwd(*x, initial_state=st, output_final_state=True)
    for t in range(T):
        one, st = recurrent_sgsa_fwd(*(None if a is None else a[:, t:t + 1] for a in x), initial_state=st,
                                     output_final_state=True)
        assert torch.equal(o[:, t:t + 1].isnan(), one.isnan()) and torch.equal(o[:, t:t + 1].nan_to_num(), one.nan_to_num()), t
    assert end[0, 1, :, 5].isinf().sum() == D - 1
    assert torch.equal(end.isnan(), st.isnan()) and torch.equal(end.nan_to_num(), st.nan_to_num())
