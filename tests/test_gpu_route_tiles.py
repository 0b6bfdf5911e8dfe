"""Routing in one launch and the M-tile lists it writes (GPU): units of 2048
routes, the switch above 32768 routes from recounting in every workgroup to a
count table, from that to a scanned table, and the switch at 1024 experts to
the large-expert kernels."""

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # (T, k, E, all routes to one expert)
    (1, 1, 1, False),
    (1, 8, 128, False),
    (63, 1, 5, False),
    (2047, 1, 31, False),
    (2048, 1, 1024, False),
    (2049, 1, 1023, True),
    (4096, 8, 32, False),    # 32768 routes: the last recounting size
    (16384, 2, 8, True),     # the same, repeated ids in every wavefront
    (2049, 1, 1, True),
    (32769, 1, 33, False),   # the first size with a count table
    (32769, 1, 511, False),
    (32769, 1, 512, False),
    (32769, 1, 1, True),     # 1024 rows of the table at a time, 17 units
    (34817, 1, 1000, True),
    (8192, 16, 896, False),
    (39900, 16, 600, False),
    (41000, 16, 600, False),
    (83000, 16, 500, True),
    (120000, 16, 600, False),  # 938 units: summed; the next ones are scanned
    (131073, 16, 600, False),
    (131073, 16, 600, True),
    (300, 3, 1025, False),
]


def _lists(buf, max_rows, E, offsets):
    """(device list, expected list) of both tile heights."""
    off = 0
    for bm in (160, 256):
        cap = max_rows // bm + min(E, max_rows)
        words = buf[off:off + 16 + 16 * cap].view(torch.int32).cpu().numpy()
        n = int(words[0])
        want = [(e, r, min(r + bm, int(offsets[e + 1])), 0) for e in range(E)
                for r in range(int(offsets[e]), int(offsets[e + 1]), bm)]
        assert len(want) <= cap
        yield words[4:4 + 4 * n].reshape(-1, 4), np.array(want, np.int32).reshape(-1, 4)
        off += (32 + 16 * cap + 255) // 256 * 256


@pytest.mark.parametrize("T,k,E,hot", CASES)
def test_route_tiles(T, k, E, hot):
    from mega_moe import _lib
    from mega_moe.runtime.routing import route

    rng = np.random.default_rng(T + E)
    sel = np.full((T, k), E // 2, np.int32) if hot else rng.integers(0, E, size=(T, k)).astype(np.int32)
    sel[rng.random((T, k)) < 0.1] = -1
    dev = torch.from_numpy(sel).cuda()
    rw = torch.rand(T, k, device="cuda")
    ws = torch.empty(int(_lib.load().mm_route_workspace_bytes(T * k, E)), dtype=torch.uint8, device="cuda")
    t = route(dev, E, rw, ws, with_tiles=True)
    torch.cuda.synchronize()
    ref = O.route(sel, E, k)
    nv = int(ref["offsets"][-1])
    assert t.offsets.cpu().numpy().tolist() == ref["offsets"].tolist()
    assert t.counts.cpu().numpy().tolist() == ref["counts"].tolist()
    assert np.array_equal(t.send_route[:nv].cpu().numpy(), ref["send_route"])
    assert np.array_equal(t.send_token[:nv].cpu().numpy(), ref["send_token"])
    assert np.array_equal(t.route_to_send.cpu().numpy(), ref["route_to_send"])
    assert torch.equal(t.weight_perm[:nv].cpu(), rw.cpu().reshape(-1)[torch.from_numpy(ref["send_route"]).long()])
    for got, want in _lists(t.tiles, T * k, E, ref["offsets"]):
        assert np.array_equal(got, want)
