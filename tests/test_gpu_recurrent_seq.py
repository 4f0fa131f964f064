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
