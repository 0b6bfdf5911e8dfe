"""Weight-streaming row GEMMs (GPU): every slab count (32 rows, at most 5), ragged ends,
each tile width (128, 256 and 512 columns) and weight layout, K loops shorter
and longer than the stage ring, the three tile orders, and the gated epilogue.

Tolerance: fp32 sums of K products (error at most K 2^-24 of the sum of their
magnitudes, doubled for the two sides) and one bf16 rounding (2^-8 relative,
doubled half an ulp)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 0]


def _offsets(E):
    counts = [ROWS[e % len(ROWS)] for e in range(E)]
    offs = torch.zeros(E + 1, dtype=torch.int32)
    offs[1:] = torch.tensor(counts, dtype=torch.int32).cumsum(0)
    return offs, counts


def _check(c, a, b, rows):
    ref, mag = a.float() @ b.float(), a.float().abs() @ b.float().abs()
    err = (c.float() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + b.shape[0] * 2.0 ** -23 * mag).all()), rows


# N per width for 100 experts: 128 -> 128 columns, 512 -> 256, 1024 -> 512
# (N-contiguous weights); few experts (one round of 128 columns) -> 128, flat order
@pytest.mark.parametrize("E,n", [(100, 128), (100, 384), (100, 512), (100, 1024), (13, 256), (13, 512)])
@pytest.mark.parametrize("k", [64, 192, 640])
@pytest.mark.parametrize("n_contig", [True, False])
def test_stream_gemm(E, n, k, n_contig):
    from mega_moe.ops import _kernels as K

    g = torch.Generator(device="cuda").manual_seed(E + n + k)
    offs, counts = _offsets(E)
    R = int(offs[-1])
    a = torch.randn(R + 5, k, generator=g, device="cuda").bfloat16()
    rows = torch.randperm(R + 5, generator=g, device="cuda")[:R].int()
    b = torch.randn((E, k, n) if n_contig else (E, n, k), generator=g, device="cuda").bfloat16()
    bl = b if n_contig else b.transpose(1, 2)  # [E, k, n]
    # max_rows below 148 per expert selects these tiles
    c = K.grouped_gemm(a, rows, b, bl.stride(0), bl.stride(2), bl.stride(1), offs.cuda(), R, n, k)
    torch.cuda.synchronize()
    for e in range(min(E, 2 * len(ROWS) + 1)):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        if r1 > r0:
            _check(c[r0:r1], a[rows[r0:r1].long()], bl[e], (e, counts[e]))


@pytest.mark.parametrize("E,inter", [(100, 64), (100, 192), (100, 256), (100, 512), (13, 128)])
@pytest.mark.parametrize("fmt", ["bf16", "fp16"])
def test_stream_gated(E, inter, fmt):
    from mega_moe.ops import _kernels as K

    hidden = 256
    g = torch.Generator(device="cuda").manual_seed(E + inter)
    offs, counts = _offsets(E)
    R = int(offs[-1])
    x = torch.randn(R, hidden, generator=g, device="cuda").bfloat16()
    w1 = (0.1 * torch.randn(E, hidden, 2 * inter, generator=g, device="cuda")).bfloat16()
    wp = torch.rand(R, generator=g, device="cuda")
    act, fc1, _ = K.fc1_swiglu(x, None, w1, offs.cuda(), wp, R, "swiglu", 1.0, None, 7.0, save_fc1=True,
                               fc1_dtype=fmt)
    torch.cuda.synchronize()
    for e in range(len(ROWS)):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        if r1 > r0:
            _check(fc1[r0:r1], x[r0:r1], w1[e], (e, counts[e]))
    gate, up = fc1.float()[:, :inter], fc1.float()[:, inter:]
    ref = torch.nn.functional.silu(gate) * up * wp[:, None]
    # from the same rounded gate and up: fp32 arithmetic, one bf16 rounding. An
    # fp16 save holds values below 2^-14 in steps of 2^-24, i.e. up to 2^-25 off
    # the value the activation was computed from: |silu'| <= 1.1 bounds its share.
    tol = 2.0 ** -7 * ref.abs() + 1e-30
    if fmt == "fp16":
        tol = tol + 2.0 ** -25 * (1.1 * up.abs() + gate.abs()) * wp[:, None]
    assert bool(((act.float() - ref).abs() <= tol).all())
