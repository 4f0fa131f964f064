"""GPU: the fp32 chunk kernels (chunk.hip's forward, chunk_bwd.hip's backward for
both input types) at the edges of their tiles: head dimensions on either side of
the 64- and 128-wide forms, chunks of one token and one token past a chunk, with
and without the sparse write, and rows whose start is not 16-byte aligned (the
element-wise loads).  Outputs, final states and every input's gradient against
the torch form of the same function in float64 (sgsa_amd.backward); the bound is
of the largest magnitude: 2e-5 for fp32 (sums of up to 128 terms per product,
about six products deep: 6 x sqrt(128) x 2^-24 = 4e-6), 1e-2 for bf16 outputs."""

import pytest
import torch

pytestmark = pytest.mark.gpu

import sgsa_amd  # noqa: E402
from sgsa_amd.backward import chunk_sgsa_torch, recompute_grads  # noqa: E402

NAMES = ["q", "k", "v", "beta", "gamma", "sparse_k", "sparse_v", "alpha", "initial_state"]


def _inputs(B, T, H, D, dt, sparse, shift, dev):
    g = torch.Generator().manual_seed(31)
    r = lambda *s: torch.randn(*s, generator=g)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)

    def put(t):   # rows `shift` elements into their storage
        buf = torch.empty(t.numel() + shift, dtype=dt, device=dev)
        buf[shift:] = t.reshape(-1).to(dt)
        return buf[shift:].view(t.shape)

    x = [put(r(B, T, H, D)), put(unit(r(B, T, H, D))), put(r(B, T, H, D)), torch.sigmoid(r(B, T, H)).to(dev),
         torch.sigmoid(r(B, T, H) + 3.0).to(dev)]
    x += [put(unit(r(B, T, H, D))), put(r(B, T, H, D)), (0.25 * torch.sigmoid(r(B, T, H))).to(dev)] if sparse \
        else [None] * 3
    return x + [(0.1 * r(B, H, D, D)).to(dev)], r(B, T, H, D).to(dev, dt), r(B, H, D, D).to(dev)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,D,sparse,shift", [(1, 64, True, 0), (64, 63, True, 0), (65, 64, True, 1), (129, 65, True, 0),
                                              (130, 128, True, 3), (200, 128, True, 0), (63, 128, False, 0),
                                              (129, 64, False, 0), (66, 128, False, 2), (191, 20, False, 0)])
def test_chunk_f32_edges(dev, dt, T, D, sparse, shift):
    x, do, dht = _inputs(2, T, 3, D, dt, sparse, shift, dev)
    print(f"chunk f32 {dt} T={T} D={D} sparse={sparse} shift={shift}", flush=True)
    x64 = [None if t is None else t.double() for t in x]
    o, st = sgsa_amd.chunk_sgsa(*x, output_final_state=True)
    wo, wst = chunk_sgsa_torch(*x64)
    needs = [t is not None for t in x]
    got = sgsa_amd.chunk_sgsa_bwd(x, needs, do, dht)
    want = recompute_grads(x64, needs, do.double(), dht.double())
    torch.cuda.synchronize()
    tol = 2e-5 if dt == torch.float32 else 1e-2
    for name, a, b in [("o", o, wo), ("state", st, wst)] + [("d" + n, a, b) for n, a, b in zip(NAMES, got, want)]:
        if b is None:
            assert a is None, name
            continue
        a, b = a.double(), b.double()
        assert torch.isfinite(a).all(), f"{name}: non-finite"
        err = ((a - b).abs().max() / b.abs().max().clamp_min(1e-12)).item()
        assert err <= tol, f"{name}: {err:.3e}"


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,D,sparse", [(1000, 128, True), (1000, 64, True), (700, 128, False), (700, 50, False)])
def test_gradients_repeat(dev, dt, T, D, sparse):
    """Fixed inputs give the same gradients bit for bit, the gates' (sums over a chunk's waves) among them."""
    x, do, dht = _inputs(2, T, 6, D, dt, sparse, 0, dev)
    print(f"gradients repeat {dt} T={T} D={D} sparse={sparse}", flush=True)
    needs = [t is not None for t in x]
    first = sgsa_amd.chunk_sgsa_bwd(x, needs, do, dht)
    for _ in range(12):
        again = sgsa_amd.chunk_sgsa_bwd(x, needs, do, dht)
        for name, a, b in zip(NAMES, first, again):
            assert a is None or torch.equal(a, b), name
