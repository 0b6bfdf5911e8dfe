"""The backward runs its row GEMMs on the saved M-tile lists only beside the
offsets they were cut from; with offsets replaced, trimmed or edited, each GEMM
cuts its own (CPU: the kernels are replaced by recorders)."""

import copy

import pytest
import torch

from mega_moe.ops import backward as B
from mega_moe.ops._saved import MoESaved
from mega_moe.runtime import routing

T, K_, H, F, E = 6, 2, 128, 128, 4
R = T * K_


def _saved():
    offsets = torch.tensor([0, 3, 3, 8, 12], dtype=torch.int32)
    tables = routing.RouteTables(R, E, K_, "cpu", True, with_tiles=False)
    tables.offsets, tables.tiles = offsets, torch.zeros(256, dtype=torch.uint8)
    bf = torch.bfloat16
    return MoESaved(
        batch_size=T, topk=K_, hidden_dim=H, ffn_dim=F, total_routes=R, experts_per_rank=E, activation="swiglu",
        situ_beta=1.0, situ_linear_beta=None, clamp_limit=7.0, hidden_states=torch.zeros(T, H, dtype=bf),
        gate_up_weight=torch.zeros(E, H, 2 * F, dtype=bf), down_weight=torch.zeros(E, H, F, dtype=bf),
        fc1_output=torch.zeros(R, 2 * F, dtype=bf), swiglu_out_weighted=torch.zeros(R, F, dtype=bf),
        recv_weights_sorted=torch.zeros(R), split_size_cum_per_expert=offsets, expert_counts=offsets.diff(),
        send_token_indices=torch.zeros(R, dtype=torch.int32), route_to_send=torch.zeros(R, dtype=torch.int32),
        _tiles=tables.tiles, _tiles_key=tables.tiles_key() if hasattr(tables, "tiles_key") else None)


def _run(saved, monkeypatch):
    """The tile lists, offsets and capacities that the backward's row GEMMs get."""
    seen = []

    def gemm(a, a_rows, b, se, sn, sk, offsets, max_rows, n, k, pool=None, tiles=None):
        seen.append((tiles, offsets, max_rows))
        return torch.zeros(max_rows, n, dtype=torch.bfloat16)

    monkeypatch.setattr(B.K, "grouped_gemm", gemm)
    monkeypatch.setattr(B.K, "swiglu_bwd", lambda ga, fc1, w, offsets, rows, **kw: (
        torch.zeros(rows, 2 * F, dtype=torch.bfloat16), torch.zeros(rows, dtype=torch.bfloat16)))
    monkeypatch.setattr(B.K, "grouped_wgrad", lambda p, pr, q, qr, offsets, n1, n2, **kw: torch.zeros(
        E, n1, n2, dtype=torch.bfloat16))
    monkeypatch.setattr(B.K, "combine_bwd", lambda dx, r2s, t, k, dscale: (torch.zeros(t, H), torch.zeros(t, k)))
    B.moe_backward_triton(saved, torch.zeros(T, H, dtype=torch.bfloat16))
    assert len(seen) == 2
    return seen


def test_unchanged_saves_keep_their_lists(monkeypatch):
    s = _saved()
    s["recv_expert_offsets"], s["plan_send_bucket_starts"]  # reading the derived keys changes nothing
    assert all(t is s["_tiles"] for t, _, _ in _run(s, monkeypatch))


def _replace(s):
    s["split_size_cum_per_expert"] = torch.tensor([0, 4, 4, 8, 12], dtype=torch.int32)


def _edit(s):
    s["split_size_cum_per_expert"][1] = 4


def _edit_view(s):
    s["plan_send_bucket_starts"].add_(0)


def _trim(s):  # the tables without the last expert's rows
    s["split_size_cum_per_expert"] = s["split_size_cum_per_expert"].clamp(max=8)
    s["total_routes"] = 8


def _fewer_rows(s):
    s["total_routes"] = 8


def _copied(s):
    s["split_size_cum_per_expert"] = s["split_size_cum_per_expert"].clone()


def _no_key(s):
    del s["_tiles_key"]


@pytest.mark.parametrize("change", [_replace, _edit, _edit_view, _trim, _fewer_rows, _copied, _no_key])
def test_changed_saves_drop_their_lists(change, monkeypatch):
    s = _saved()
    change(s)
    for tiles, offsets, rows in _run(s, monkeypatch):
        assert tiles is None and offsets is s["split_size_cum_per_expert"] and rows == s["total_routes"]


def test_copies_and_inference_tensors(monkeypatch):
    c = copy.deepcopy(_saved())  # lists, key and offsets copied together, or the lists are dropped
    assert all(t is None or t is c["_tiles"] for t, _, _ in _run(c, monkeypatch))
    with torch.inference_mode():
        s = _saved()
    assert all(t is None for t, _, _ in _run(s, monkeypatch))
