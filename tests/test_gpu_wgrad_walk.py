"""Walk of the persistent small-K weight gradient (GPU): tile counts per expert
that do not divide a team's workgroups, fewer experts than teams (with few and
with many tiles), experts without rows.

Tolerance: fp32 sums of K products (K 2^-23 of the sum of their magnitudes for
the two sides) and one bf16 rounding (2^-8 relative, twice half an ulp)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,n1,n2", [
    (1, 256, 256), (3, 512, 768),        # fewer experts than teams, few tiles
    (1, 4096, 4096), (8, 2048, 2048),    # one team from one tile per workgroup on
    (5, 4096, 2048), (15, 1536, 2048),   # the same with several tiles per workgroup
    (16, 256, 256), (17, 768, 768),      # 1 and 9 tiles per expert over 16-workgroup teams
    (40, 2048, 768),                     # 24 tiles: one and a half rounds per expert
])
def test_persistent_walk(E, n1, n2, monkeypatch):
    from mega_moe.ops import _kernels as K

    monkeypatch.setenv("MM_WGRAD_KERNEL", "wide")
    g = torch.Generator(device="cuda").manual_seed(E + n1)
    counts = [(0, 1, 33, 70)[e % 4] if E > 1 else 40 for e in range(E)]
    offs = torch.zeros(E + 1, dtype=torch.int32)
    offs[1:] = torch.tensor(counts, dtype=torch.int32).cumsum(0)
    R = int(offs[-1])
    p = torch.randn(R, n1, generator=g, device="cuda").bfloat16()
    q = torch.randn(R, n2, generator=g, device="cuda").bfloat16()
    c = K.grouped_wgrad(p, None, q, None, offs.cuda(), n1, n2, max_rows=R)
    torch.cuda.synchronize()
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        pe, qe = p[r0:r1].float(), q[r0:r1].float()
        ref, mag = pe.t() @ qe, pe.abs().t() @ qe.abs()
        err = (c[e].float() - ref).abs()
        assert bool((err <= 2.0 ** -8 * ref.abs() + max(1, r1 - r0) * 2.0 ** -23 * mag).all()), (e, counts[e])


@pytest.mark.parametrize("E,hot,rows", [
    (16, 0, 700), (40, 39, 700), (67, 64, 1500),  # one expert's rows load its team: the grid is one team
    (40, 7, 40),                                  # too little to matter: teams
])
def test_uneven_rows(E, hot, rows, monkeypatch):
    from mega_moe.ops import _kernels as K

    monkeypatch.setenv("MM_WGRAD_KERNEL", "wide")
    n1, n2 = 2048, 1536  # 48 tiles an expert: three rounds of a 16-workgroup team
    g = torch.Generator(device="cuda").manual_seed(E + rows)
    counts = [rows if e == hot else (0, 1, 5, 33)[e % 4] for e in range(E)]
    offs = torch.zeros(E + 1, dtype=torch.int32)
    offs[1:] = torch.tensor(counts, dtype=torch.int32).cumsum(0)
    R = int(offs[-1])
    p = torch.randn(R, n1, generator=g, device="cuda").bfloat16()
    q = torch.randn(R, n2, generator=g, device="cuda").bfloat16()
    c = K.grouped_wgrad(p, None, q, None, offs.cuda(), n1, n2, max_rows=R)
    torch.cuda.synchronize()
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        pe, qe = p[r0:r1].float(), q[r0:r1].float()
        ref, mag = pe.t() @ qe, pe.abs().t() @ qe.abs()
        err = (c[e].float() - ref).abs()
        assert bool((err <= 2.0 ** -8 * ref.abs() + max(1, r1 - r0) * 2.0 ** -23 * mag).all()), (e, counts[e])
