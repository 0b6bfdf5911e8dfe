"""Weight-streaming row GEMMs (GPU): every slab count (32 rows, at most 5), ragged ends,
each tile width (128, 256 and 512 columns) and weight layout, K loops shorter
and longer than the stage ring, the three tile orders, and the gated epilogue
with each save format.

Tolerance: fp32 sums of K products (error at most K 2^-24 of the sum of their
magnitudes, doubled for the two sides) and one bf16 rounding (2^-8 relative,
doubled half an ulp)."""

import ctypes

import pytest
import torch

from oracle import moe_oracle as O

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


def _tile(R, E, n, k, n_contig, saves=False):
    from mega_moe import _lib

    rows, cols = ctypes.c_int32(), ctypes.c_int32()
    _lib.call("mm_row_tile", R, E, n, k, n_contig, saves, ctypes.byref(rows), ctypes.byref(cols))
    return rows.value, cols.value


# 100 experts: the M tiles in XCD order (not a multiple of 8 of them), MM_XCD_MOD=0 in
# contiguous shares; 13: in flat order. (E, n, columns with N- / K-contiguous weights)
@pytest.mark.parametrize("E,n,wide,narrow", [(100, 128, 128, 128), (100, 384, 128, 128), (100, 512, 256, 256),
                                             (100, 1024, 512, 256), (13, 256, 128, 128), (13, 512, 128, 128)])
@pytest.mark.parametrize("k", [64, 192, 640])
@pytest.mark.parametrize("n_contig", [True, False])
@pytest.mark.parametrize("xcd_mod", ["1", "0"])
def test_stream_gemm(E, n, wide, narrow, k, n_contig, xcd_mod, monkeypatch):
    from mega_moe.ops import _kernels as K

    monkeypatch.setenv("MM_XCD_MOD", xcd_mod)
    g = torch.Generator(device="cuda").manual_seed(E + n + k)
    offs, counts = _offsets(E)
    R = int(offs[-1])
    a = torch.randn(R + 5, k, generator=g, device="cuda").bfloat16()
    rows = torch.randperm(R + 5, generator=g, device="cuda")[:R].int()
    b = torch.randn((E, k, n) if n_contig else (E, n, k), generator=g, device="cuda").bfloat16()
    bl = b if n_contig else b.transpose(1, 2)  # [E, k, n]
    assert _tile(R, E, n, k, n_contig) == (160, wide if n_contig else narrow)
    assert E < 64 or sum(-(-c // 160) for c in counts) % 8
    c = K.grouped_gemm(a, rows, b, bl.stride(0), bl.stride(2), bl.stride(1), offs.cuda(), R, n, k)
    torch.cuda.synchronize()
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        if r1 > r0:
            _check(c[r0:r1], a[rows[r0:r1].long()], bl[e], (e, counts[e]))


@pytest.mark.parametrize("E,inter,cols", [(100, 64, 128), (100, 192, 128), (100, 256, 256), (100, 512, 512),
                                          (13, 128, 256)])
@pytest.mark.parametrize("fmt", ["bf16", "fp16"])
def test_stream_gated(E, inter, cols, fmt):
    from mega_moe.ops import _kernels as K

    hidden = 256
    g = torch.Generator(device="cuda").manual_seed(E + inter)
    offs, counts = _offsets(E)
    R = int(offs[-1])
    assert _tile(R, E, 2 * inter, hidden, True, True) == (160, cols)
    x = torch.randn(R, hidden, generator=g, device="cuda").bfloat16()
    w1 = (0.1 * torch.randn(E, hidden, 2 * inter, generator=g, device="cuda")).bfloat16()
    wp = torch.rand(R, generator=g, device="cuda")
    act, fc1, _ = K.fc1_swiglu(x, None, w1, offs.cuda(), wp, R, "swiglu", 1.0, None, 7.0, save_fc1=True,
                               fc1_dtype=fmt)
    torch.cuda.synchronize()
    for e in range(E):
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


@pytest.mark.parametrize("E,inter,cols", [(100, 256, 256), (100, 512, 512), (13, 128, 256)])
def test_stream_fp8_save(E, inter, cols):
    """Codes and scales of an FP8 save, in both epilogue passes: exactly the
    quantized bf16 save, which narrows the same fp32 sums."""
    from mega_moe.ops import _kernels as K

    hidden = 256
    g = torch.Generator(device="cuda").manual_seed(E + inter)
    offs, _ = _offsets(E)
    R = int(offs[-1])
    assert _tile(R, E, 2 * inter, hidden, True, True) == (160, cols)
    x = torch.randn(R, hidden, generator=g, device="cuda").bfloat16()
    w1 = (0.1 * torch.randn(E, hidden, 2 * inter, generator=g, device="cuda")).bfloat16()
    wp = torch.rand(R, generator=g, device="cuda")
    args = (x, None, w1, offs.cuda(), wp, R, "swiglu", 1.0, None, 7.0)
    act, fc1, _ = K.fc1_swiglu(*args, save_fc1=True, fc1_dtype="bf16")
    act8, fc8, scale = K.fc1_swiglu(*args, save_fc1=True, fc1_dtype="fp8")
    torch.cuda.synchronize()
    codes, scales = O.quantize_fc1(fc1.float().cpu(), "fp8")
    assert torch.equal(act8, act) and torch.equal(scale.cpu(), scales)
    assert torch.equal(fc8.cpu().view(torch.uint8), codes.view(torch.uint8))
