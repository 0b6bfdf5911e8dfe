"""A token's output does not depend on the size of the call or on what is saved
(GPU): every row-GEMM tile sums an element's products over ascending K, so all
tile heights and widths give the same bits. Exact comparisons."""

import pytest
import torch

import mega_moe
from mega_moe.bench_configs import CaseSpec, make_inputs

pytestmark = pytest.mark.gpu


# rows of expert 0, experts: one round of the narrow tiles, the 256- and (n a
# multiple of 512) 512-column tiles, and 256 x 256 tiles (148 rows on average)
@pytest.mark.parametrize("k", [64, 320, 1088])  # 1088: the register-staged 256 x 256 tiles
@pytest.mark.parametrize("n_contig", [True, False])
@pytest.mark.parametrize("n", [384, 512, 768])
def test_row_gemm(k, n_contig, n):
    from mega_moe.ops import _kernels as K

    g = torch.Generator(device="cuda").manual_seed(n + k)
    shared = 100  # rows of expert 0 that every call has
    a0 = torch.randn(shared, k, generator=g, device="cuda").bfloat16()
    b0 = torch.randn((k, n) if n_contig else (n, k), generator=g, device="cuda").bfloat16()
    out = []
    for E, more in ((1, 0), (8, 0), (60, 0), (300, 0), (3, 500)):
        R = shared + more + (E - 1) * 20
        a = torch.randn(R, k, generator=g, device="cuda").bfloat16()
        a[:shared] = a0
        b = torch.randn((E,) + tuple(b0.shape), generator=g, device="cuda").bfloat16()
        b[0] = b0
        bl = b if n_contig else b.transpose(1, 2)
        offs = torch.tensor([0] + [shared + more + 20 * e for e in range(E)], dtype=torch.int32, device="cuda")
        c = K.grouped_gemm(a, None, b, bl.stride(0), bl.stride(2), bl.stride(1), offs, R, n, k)
        out.append(c[:shared].clone())
    for i, c in enumerate(out[1:]):
        assert torch.equal(c, out[0]), i + 1


@pytest.mark.parametrize("hidden,inter,experts,top_k", [(2048, 768, 128, 8), (512, 384, 12, 4), (256, 128, 4, 2)])
@pytest.mark.parametrize("act", ["swiglu", "situglu", "clamp_swiglu"])
def test_layer(hidden, inter, experts, top_k, act):
    tokens = 200 * experts // top_k  # 200 rows for each expert: 256 x 256 tiles
    inp = make_inputs(CaseSpec("bits", tokens, hidden, inter, experts, top_k, "softmax_topk", True), device="cuda",
                      seed=6, weight_scale=0.1)

    def op(fmt="bf16"):
        cfg = mega_moe.MoEForwardConfig(activation=act, save_fc1_dtype=fmt)
        return mega_moe.FusedMoEForward(None, max_tokens_per_rank=tokens, hidden_size=hidden, top_k=top_k,
                                        num_experts=experts, config=cfg)

    serve = op()
    full = serve.forward(inp["x"], inp["selected"], inp["gate_up"], inp["down"], inp["rw"])
    saving = [op(fmt) for fmt in ("bf16", "fp16", "fp8")]
    for n in (1, 5, 32, tokens // 4, tokens // 2, tokens):
        args = (inp["x"][:n], inp["selected"][:n], inp["gate_up"], inp["down"], inp["rw"][:n])
        assert torch.equal(serve.forward(*args), full[:n]), n
        for o in saving:
            assert torch.equal(o.forward(*args, return_saved=True)[0], full[:n]), (n, o.config.save_fc1_dtype)
