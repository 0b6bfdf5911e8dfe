"""Row GEMMs of 256-row tiles where N is no multiple of 256 (GPU): 128 columns,
ragged last tiles, both weight layouts, K loops shorter and longer than the
stage ring, and the gated epilogue; from 160 rows per expert on.

Tolerance: fp32 sums of K products (error at most K 2^-24 of the sum of their
magnitudes, doubled for the two sides) and one bf16 rounding (2^-8 relative,
doubled half an ulp)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

COUNTS = [256, 1, 0, 257, 511, 512, 63, 64, 65, 300]  # 203 rows on average


def _close(c, ref, mag, k):
    return bool(((c.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + k * 2.0 ** -23 * mag).all())


@pytest.mark.parametrize("n", [128, 384])
@pytest.mark.parametrize("k", [64, 128, 192, 320])
@pytest.mark.parametrize("n_contig", [True, False])
@pytest.mark.parametrize("gather", [True, False])
def test_row_gemm(n, k, n_contig, gather):
    from mega_moe.ops import _kernels as K

    g = torch.Generator(device="cuda").manual_seed(n + k)
    E, R = len(COUNTS), sum(COUNTS)
    offs = torch.tensor([0] + COUNTS, dtype=torch.int32).cumsum(0).int()
    a = torch.randn(R, k, generator=g, device="cuda").bfloat16()
    rows = torch.randperm(R, generator=g, device="cuda").int() if gather else None
    b = torch.randn((E, k, n) if n_contig else (E, n, k), generator=g, device="cuda").bfloat16()
    bl = b if n_contig else b.transpose(1, 2)
    c = K.grouped_gemm(a, rows, b, bl.stride(0), bl.stride(2), bl.stride(1), offs.cuda(), R, n, k)
    torch.cuda.synchronize()
    src = a[rows.long()] if gather else a
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        ae, be = src[r0:r1].float(), bl[e].float()
        assert _close(c[r0:r1], ae @ be, ae.abs() @ be.abs(), k), (e, COUNTS[e])


@pytest.mark.parametrize("inter", [64, 192])
@pytest.mark.parametrize("fmt", ["bf16", "fp16"])
def test_gated(inter, fmt):
    from mega_moe.ops import _kernels as K

    hidden, E, R = 192, len(COUNTS), sum(COUNTS)
    g = torch.Generator(device="cuda").manual_seed(inter)
    offs = torch.tensor([0] + COUNTS, dtype=torch.int32).cumsum(0).int()
    x = torch.randn(R, hidden, generator=g, device="cuda").bfloat16()
    w1 = (0.1 * torch.randn(E, hidden, 2 * inter, generator=g, device="cuda")).bfloat16()
    wp = torch.rand(R, generator=g, device="cuda")
    act, fc1, _ = K.fc1_swiglu(x, None, w1, offs.cuda(), wp, R, "swiglu", 1.0, None, 7.0, save_fc1=True, fc1_dtype=fmt)
    torch.cuda.synchronize()
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        xe, we = x[r0:r1].float(), w1[e].float()
        assert _close(fc1[r0:r1], xe @ we, xe.abs() @ we.abs(), hidden), (e, COUNTS[e])
    gate, up = fc1.float()[:, :inter], fc1.float()[:, inter:]
    ref = torch.nn.functional.silu(gate) * up * wp[:, None]
    # fp32 arithmetic on the rounded gate and up, one bf16 rounding; an fp16 save
    # holds values below 2^-14 up to 2^-25 off (|silu'| <= 1.1)
    tol = 2.0 ** -7 * ref.abs() + 1e-30
    if fmt == "fp16":
        tol = tol + 2.0 ** -25 * (1.1 * up.abs() + gate.abs()) * wp[:, None]
    assert bool(((act.float() - ref).abs() <= tol).all())
