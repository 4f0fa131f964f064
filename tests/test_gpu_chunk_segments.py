"""GPU: the bf16 chunk forward where the number of segments of its state pass
changes (chunk_bf16.hip seg_count): 8 chunks, the last length that runs as one
segment, and 9, the first in several; a ragged last segment; more segments than
the chunks fill (one head of 130 chunks: 26 of 32, the last ones empty); more
heads than CUs.  Output and final state against the recurrent oracle in float64;
2^-8 of the largest magnitude for both: the output's own rounding is half of that,
and the rounding of the kernels' bf16 operands adds 7e-4 (emulated on the CPU)."""

import pytest
import torch

from oracle import sgsa_oracle as O

pytestmark = pytest.mark.gpu

import sgsa_amd  # noqa: E402


@pytest.mark.parametrize("B,T,H,D", [(1, 512, 2, 128), (1, 513, 2, 128), (2, 513, 2, 64), (1, 2117, 3, 128),
                                     (1, 8300, 1, 128), (1, 8300, 1, 64), (2, 600, 130, 64)])
def test_segments(dev, B, T, H, D):
    g = torch.Generator().manual_seed(T + D)
    r = lambda *s: torch.randn(*s, generator=g)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    q, k, sk = (unit(r(B, T, H, D)).bfloat16() for _ in range(3))
    v, sv = r(B, T, H, D).bfloat16(), r(B, T, H, D).bfloat16()
    beta, gamma, alpha = torch.sigmoid(r(B, T, H)), torch.sigmoid(r(B, T, H) + 4), 0.25 * torch.sigmoid(r(B, T, H))
    h0 = 0.1 * r(B, H, D, D)
    d = lambda *ts: [t.to(dev) for t in ts]
    out, st = sgsa_amd.chunk_sgsa(*d(q, k, v, beta, gamma), initial_state=h0.to(dev), output_final_state=True,
                                  **dict(zip(("sparse_k", "sparse_v", "alpha"), d(sk, sv, alpha))))
    f = lambda *ts: [t.double() for t in ts]
    ro, rs = O.naive_recurrent_sgsa(*f(q, k, v, beta, gamma, sk, sv, alpha, h0), True)
    for got, ref in ((out, ro), (st, rs)):
        err = (got.double().cpu() - ref).abs().max() / ref.abs().max()
        assert err <= 2.0 ** -8, err
