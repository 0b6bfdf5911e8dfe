"""The one-call forward and backward give the bits of the staged entry points
(which a stage timer selects), and saved tensors that are not as the forward
wrote them take the staged calls (GPU)."""

import pytest
import torch

import mega_moe
from mega_moe.bench_configs import CaseSpec, make_inputs
from mega_moe.ops import backward as B
from mega_moe.runtime.timing import StageTimer

pytestmark = pytest.mark.gpu

GRADS = ("grad_hidden", "grad_routing_weights", "grad_fc2", "grad_gate_up", "grad_swiglu", "grad_fc1_output",
         "grad_gate")
TABLES = ("expert_counts", "split_size_cum_per_expert", "route_to_send", "fc1_output")


def _op(spec, fmt):
    cfg = mega_moe.MoEForwardConfig(save_fc1_dtype=fmt, activation="situglu", situ_beta=2, situ_linear_beta=3.0)
    return mega_moe.FusedMoEForward(None, max_tokens_per_rank=spec.tokens, hidden_size=spec.hidden, top_k=spec.top_k,
                                    num_experts=spec.experts, config=cfg)


@pytest.mark.parametrize("spec", [
    CaseSpec("one_token", 1, 256, 128, 4, 2, "softmax_topk", True),
    CaseSpec("ragged", 333, 512, 384, 12, 4, "zipf", True),
    CaseSpec("rows256", 1200, 256, 256, 4, 2, "softmax_topk", True),
], ids=lambda s: s.name)
@pytest.mark.parametrize("fmt", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("recompute", ["0", "1"])
@pytest.mark.parametrize("contiguous_down", [False, True])
def test_one_call_equals_staged(spec, fmt, recompute, contiguous_down, monkeypatch):
    monkeypatch.setenv("MOE_SAVED_RECOMPUTE", recompute)
    inp = make_inputs(spec, device="cuda", seed=3, weight_scale=0.1)
    sel = inp["selected"].clone()
    sel[0, -1] = -1
    down = inp["down"].contiguous() if contiguous_down else inp["down"]
    args = (inp["x"], sel, inp["gate_up"], down, inp["rw"])
    one, staged = _op(spec, fmt), _op(spec, fmt)
    staged.stage_timer = StageTimer()
    o1, s1 = one.forward(*args, return_saved=True)
    o2, s2 = staged.forward(*args, return_saved=True)
    assert B._one_call(s1, inp["dy"], inp["x"], s1["_tiles"])
    g1, g2 = mega_moe.moe_backward_triton(s1, inp["dy"]), mega_moe.moe_backward_triton(s2, inp["dy"])
    torch.cuda.synchronize()
    n = int(s1["split_size_cum_per_expert"][-1])
    assert torch.equal(o1, o2)
    valid = {"fc1_output": n, "grad_swiglu": n, "grad_fc1_output": n, "grad_gate": n}
    bits = lambda t: t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t  # noqa: E731
    for k in TABLES:
        assert torch.equal(bits(s1[k][:valid.get(k)]), bits(s2[k][:valid.get(k)])), k
    for k in GRADS:
        assert torch.equal(g1[k][:valid.get(k)], g2[k][:valid.get(k)]), k
    assert torch.equal(one.forward(*args), staged.forward(*args))  # nothing saved: tables in scratch


def test_changed_saves_take_the_staged_calls():
    spec = CaseSpec("changed", 64, 256, 128, 4, 2, "softmax_topk", True)
    inp = make_inputs(spec, device="cuda", seed=4, weight_scale=0.1)
    _, saved = _op(spec, "bf16").forward(inp["x"], inp["selected"], inp["gate_up"], inp["down"], inp["rw"],
                                         return_saved=True)
    ref = mega_moe.moe_backward_triton(saved, inp["dy"])
    rows = torch.empty(saved["fc1_output"].shape[0], 512, dtype=torch.bfloat16, device="cuda")
    rows[:, :256] = saved["fc1_output"]
    saved["fc1_output"] = rows[:, :256]  # strided rows: accepted by the staged entry points
    assert not B._one_call(saved, inp["dy"], inp["x"], saved["_tiles"])
    got = mega_moe.moe_backward_triton(saved, inp["dy"])
    for k in GRADS:
        assert torch.equal(got[k], ref[k]), k
    saved["fc1_output"] = saved["fc1_output"].float()
    with pytest.raises(TypeError):
        mega_moe.moe_backward_triton(saved, inp["dy"])


def test_replaced_offsets_are_read():
    spec = CaseSpec("replaced", 300, 256, 128, 4, 2, "softmax_topk", True)
    inp = make_inputs(spec, device="cuda", seed=5, weight_scale=0.1)
    got = []
    for drop_lists in (False, True):
        _, saved = _op(spec, "bf16").forward(inp["x"], inp["selected"], inp["gate_up"], inp["down"], inp["rw"],
                                             return_saved=True)
        moved = saved["split_size_cum_per_expert"].clone()
        moved[1] -= 1  # the first expert's last row counts as the second's
        saved["split_size_cum_per_expert"] = moved
        if drop_lists:
            del saved["_tiles"]
        got.append(mega_moe.moe_backward_triton(saved, inp["dy"]))
    for k in GRADS:
        assert torch.equal(got[0][k], got[1][k]), k


def test_one_call_holds_no_workspaces():
    spec = CaseSpec("held", 64, 256, 128, 4, 2, "softmax_topk", True)
    inp = make_inputs(spec, device="cuda", seed=6, weight_scale=0.1)
    op = _op(spec, "bf16")
    args = (inp["x"], inp["selected"], inp["gate_up"], inp["down"], inp["rw"])
    op.forward(*args)
    _, saved = op.forward(*args, return_saved=True)
    mega_moe.moe_backward_triton(saved, inp["dy"])
    assert op._workspaces.nbytes() == 0  # the passes bring their own scratch
    op.build_routing_plan(inp["selected"])
    assert op._workspaces.nbytes() > 0
