"""Weight gradients of ragged experts beside rows that hold infinities and NaN
(GPU): the rows after an expert's last one, another expert's or, with dropped
routes, never written, take no part in its gradient."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# rows per expert choose the kernel: persistent, 64-row K steps, register-staged (with
# Q read through a buffer descriptor, or gathered by address)
@pytest.mark.parametrize("counts,n1,n2", [
    ([70, 1, 33, 50], 512, 256), ([500, 333, 1, 800], 256, 512), ([500, 333], 128, 384),
    ([2100, 2049, 2177, 2500], 256, 512), ([2112, 9000, 1, 0, 64, 4099], 512, 256),
])
@pytest.mark.parametrize("gather", ["none", "p", "pq"])
def test_rows_past_the_end(counts, n1, n2, gather):
    from mega_moe.ops import _kernels as K

    g = torch.Generator(device="cuda").manual_seed(sum(counts))
    E = len(counts)
    offs = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).int()
    n, cap = int(offs[-1]), int(offs[-1]) + 100  # 100 capacity rows hold no route
    p = torch.randn(cap, n1, generator=g, device="cuda").bfloat16()
    q = torch.randn(cap, n2, generator=g, device="cuda").bfloat16()
    straight = torch.arange(cap, device="cuda").int()
    prow = torch.randperm(cap, generator=g, device="cuda").int() if "p" in gather else straight
    qrow = torch.randperm(cap, generator=g, device="cuda").int() if "q" in gather else straight
    for bad, lo, hi in ((float("nan"), n, cap), (float("inf"), int(offs[1]), int(offs[2]))):
        p[prow[lo:hi].long()] = bad  # never-written rows; all of expert 1
        q[qrow[lo:hi].long()] = bad
    c = K.grouped_wgrad(p, prow if "p" in gather else None, q, qrow if "q" in gather else None, offs.cuda(), n1, n2,
                        max_rows=cap)
    torch.cuda.synchronize()
    for e in range(E):
        r0, r1 = int(offs[e]), int(offs[e + 1])
        if e == 1:
            continue
        pe, qe = p[prow[r0:r1].long()].float(), q[qrow[r0:r1].long()].float()
        ref, mag = pe.t() @ qe, pe.abs().t() @ qe.abs()
        err = (c[e].float() - ref).abs()
        # fp32 sums in two orders, one bf16 rounding
        assert bool((err <= 2.0 ** -8 * ref.abs() + (r1 - r0) * 2.0 ** -23 * mag).all()), (e, counts[e])


@pytest.mark.parametrize("tokens,experts,top_k", [(60, 4, 2), (3000, 8, 2), (4700, 2, 1)])
@pytest.mark.parametrize("fmt", ["bf16", "fp8"])
def test_layer_with_drops_over_nan_memory(tokens, experts, top_k, fmt):
    """Forward and backward with dropped routes give the same finite results
    whatever the memory of their buffers held before."""
    import mega_moe
    from mega_moe.bench_configs import CaseSpec, make_inputs

    inp = make_inputs(CaseSpec("drops", tokens, 512, 256, experts, top_k, "softmax_topk", True), device="cuda", seed=9,
                      weight_scale=0.1)
    sel = inp["selected"].clone()
    sel[torch.rand(sel.shape, generator=torch.Generator().manual_seed(1)) < 0.1] = -1
    names = ("grad_hidden", "grad_routing_weights", "grad_gate_up", "grad_fc2")
    got = []
    for fill in (0.0, float("nan")):
        op = mega_moe.FusedMoEForward(None, max_tokens_per_rank=tokens, hidden_size=512, top_k=top_k,
                                      num_experts=experts, config=mega_moe.MoEForwardConfig(save_fc1_dtype=fmt))
        held = [torch.full((n,), fill, device="cuda") for n in [1 << 22] * 16 + [1 << 18] * 32 + [1 << 12] * 64 + [64] * 64]
        del held  # the allocator hands this memory out again
        out, saved = op.forward(inp["x"], sel, inp["gate_up"], inp["down"], inp["rw"], return_saved=True)
        grads = mega_moe.moe_backward_triton(saved, inp["dy"])
        got.append([out.clone()] + [grads[n].clone() for n in names])
        del out, saved, grads, op
    for name, a, b in zip(("out",) + names, *got):
        assert bool(torch.isfinite(b).all()) and torch.equal(a, b), name
