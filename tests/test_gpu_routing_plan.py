"""The merged routing chain (af3_routing_plan: one or three launches for at most
1024 experts) at the edges of its dispatch: batches of exactly and one past the
one-block limit, chunk edges of the three-launch form, the smallest and largest
expert and slot counts, dropped ids, and logits with equal, -0, infinite and NaN
entries; every index, tile map and work order bit-exact."""
import ctypes

import pytest
import torch

from agent_factory_3_amd import _capi
from agent_factory_3_amd import routing as R
from oracle import routing as O
from tests._tol import check_close
from tests.test_gpu_routing import _check

pytestmark = pytest.mark.gpu


def _orders(ed, n_rows, E):
    """The work order of each size the plan made, against its definition."""
    hist = ed.hist.cpu().tolist()
    for bm, order in ed.gemm_order.items():
        full = [(b << 16) | e for e in range(E) for b in range(hist[e] // bm)]
        tails = sorted([e for e in range(E) if hist[e] % bm], key=lambda e: (-(hist[e] % bm), e))
        want = full + [((hist[e] // bm) << 16) | e for e in tails]
        want += [-1] * (R.max_tiles(n_rows, E, bm) - len(want))
        assert order.cpu().tolist() == want


@pytest.mark.parametrize("T,E,K,topk", [
    (1, 1, 1, True), (1, 2, 2, False), (1, 1024, 4, False), (15, 1024, 16, False), (64, 256, 16, True),
    (255, 32, 4, True), (256, 128, 4, True), (257, 128, 4, True), (1024, 32, 4, False), (1025, 32, 4, False),
    (256, 32, 16, False), (257, 3, 2, True), (512, 1024, 3, False), (700, 257, 4, True), (40, 1000, 5, True),
    (2049, 33, 7, True), (513, 128, 16, False), (8191, 64, 1, False),
])
def test_plan_matches_oracle(dev, T, E, K, topk):
    g = torch.Generator().manual_seed(T * 7 + E + K)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    if topk:
        out, ref = R.routing(logits.to(dev), K), O.routing_topk(logits, K)
    else:
        ids = torch.rand(T, E, generator=g).topk(K, dim=1).indices.to(torch.int32)   # unsorted slots
        out, ref = R.routing_replay(logits.to(dev), ids.to(dev), K), O.routing_replay(logits, ids, K)
    _check(*out, ref)
    _orders(out[0].expt_data, T * K, E)


# the prefix over chunks in its own launch: just past the one-block limit, experts past whole blocks of 16, more
# chunks than a block's segments hold in one round; the most counts the scan kernel takes along
@pytest.mark.parametrize("T,E,K", [(2049, 1024, 4), (2048, 1024, 4), (16385, 128, 4), (16384, 128, 4), (9000, 250, 1),
                                   (140000, 17, 4)])
def test_plan_prefix_over_many_chunks(dev, T, E, K):
    g = torch.Generator().manual_seed(T + E)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    ids = torch.rand(T, E, generator=g).topk(K, dim=1).indices.to(torch.int32)
    out, ref = R.routing_replay(logits.to(dev), ids.to(dev), K), O.routing_replay(logits, ids, K)
    _check(*out, ref)
    _orders(out[0].expt_data, T * K, E)


@pytest.mark.parametrize("T,E,K", [(40, 5, 2), (1021, 200, 4), (30000, 70, 4)])
def test_plan_maps_of_any_block_size(dev, T, E, K):
    """Maps and orders for every block size the call takes, past the sizes one sorting pass of the tails holds and
    with experts of many tiles, some of them idle."""
    g = torch.Generator().manual_seed(E)
    pref = torch.rand(E, generator=g) ** 6 + 1e-9
    pref[::3] = 1e-12
    ids = torch.stack([torch.multinomial(pref, K, replacement=False, generator=g) for _ in range(T)]).to(torch.int32)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    bms = (1, 7, 32, 512, 513, 1300, 3000, 64)
    lib, ld, idd = _capi.load(), logits.to(dev), ids.to(dev)
    mt = max(R.max_tiles(T * K, E, bm) for bm in bms)
    n = int(lib.af3_routing_plan_workspace_bytes(T, E, K, 0))
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device=dev)
    hist, topk, gate, offs = (torch.empty(m, dtype=torch.int32, device=dev) for m in (E, T * K, T * K, E + 1))
    gs = torch.empty(T * K, dtype=torch.bfloat16, device=dev)
    pad = torch.empty(len(bms), E + 1, dtype=torch.int32, device=dev)
    maps, orders = (torch.empty(len(bms), mt, dtype=torch.int32, device=dev) for _ in range(2))
    _capi.call("af3_routing_plan", ld.data_ptr(), E, idd.data_ptr(), 0, T, E, K, gs.data_ptr(), hist.data_ptr(),
               topk.data_ptr(), gate.data_ptr(), offs.data_ptr(), (ctypes.c_int32 * len(bms))(*bms), len(bms),
               len(bms), mt, pad.data_ptr(), maps.data_ptr(), orders.data_ptr(), ws.data_ptr(), n,
               _capi.stream_of(torch.device(dev)))
    h = torch.bincount(ids.reshape(-1).long(), minlength=E)
    assert torch.equal(hist.cpu(), h.to(torch.int32))
    for i, bm in enumerate(bms):
        want_pad, want_map = O.expt_data(h, bm, mt)
        assert torch.equal(pad[i].cpu(), want_pad) and torch.equal(maps[i].cpu(), want_map), bm
        full = [(b << 16) | e for e in range(E) for b in range(int(h[e]) // bm)]
        tails = sorted([e for e in range(E) if int(h[e]) % bm], key=lambda e: (-(int(h[e]) % bm), e))
        want = full + [((int(h[e]) // bm) << 16) | e for e in tails]
        got = orders[i].cpu().tolist()
        assert got[:len(want)] == want and all(v == -1 for v in got[len(want):]), bm


@pytest.mark.parametrize("T", [40, 1100])  # one block, three launches
def test_plan_drops_out_of_range_ids(dev, T):
    E, K = 12, 4
    g = torch.Generator().manual_seed(T)
    ids = torch.randint(-2, E + 2, (T, K), generator=g, dtype=torch.int32)   # repeats and dropped ids
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    rd, gi, si = R.routing_replay(logits.to(dev), ids.to(dev), K)
    flat = ids.reshape(-1)
    valid = (flat >= 0) & (flat < E)
    order = torch.sort(torch.where(valid, flat, E), stable=True).indices
    n = int(valid.sum())
    assert torch.equal(gi.src_indx.cpu()[:n], order[:n].to(torch.int32))
    assert (gi.src_indx.cpu()[n:] == -1).all() and (rd.gate_scal.cpu()[n:] == 0).all()
    want = torch.full((T * K,), -1, dtype=torch.int32)
    want[order[:n]] = torch.arange(n, dtype=torch.int32)
    assert torch.equal(gi.dst_indx.cpu(), want)
    assert torch.equal(rd.expt_hist.cpu(), torch.bincount(flat[valid].long(), minlength=E).to(torch.int32))
    assert int(rd.expt_data.token_offs_raw.cpu()[-1]) == n


@pytest.mark.parametrize("T", [33, 400])  # top-k inside the one-block plan, and in its own launch
def test_plan_topk_special_logits(dev, T):
    E, K = 48, 4
    g = torch.Generator().manual_seed(T)
    logits = torch.randint(-2, 3, (T, E), generator=g).to(torch.bfloat16)    # many ties
    logits[logits == 0] = -0.0
    logits[torch.rand(T, E, generator=g) < 0.3] = 0.0                        # -0 and +0 tie
    logits[torch.rand(T, E, generator=g) < 0.1] = float("-inf")
    logits[torch.rand(T, E, generator=g) < 0.1] = float("nan")               # sorts last
    out = R.routing(logits.to(dev), K)
    ref = O.routing_topk(logits, K)
    _check(*out, ref)
    logits[0] = float("-inf")
    logits[0, 5] = 1.0
    assert torch.equal(R.routing(logits.to(dev), K)[1].src_indx.cpu(), O.routing_topk(logits, K)["topk_indx"])


def test_outputs_change_in_place_on_their_own(dev, monkeypatch):
    """The index tensors share a buffer, not a version: one may change between forward and backward."""
    monkeypatch.setattr(R, "GAMMA_GRAD", True)
    g = torch.Generator().manual_seed(3)
    logits = torch.randn(70, 32, generator=g).to(torch.bfloat16).to(dev)
    w = torch.randn(280, generator=g).to(torch.bfloat16).to(dev)
    grads = []
    for change in (False, True):
        lg = logits.clone().requires_grad_(True)
        rd, gi, _ = R.routing(lg, 4)
        if change:
            gi.dst_indx.fill_(-1)
            rd.expt_data.token_offs_raw.zero_()
            assert [t._version for t in (gi.src_indx, rd.expt_hist)] == [0, 0]
        rd.gate_scal.backward(w)
        grads.append(lg.grad)
    assert torch.equal(grads[0], grads[1]) and grads[0].abs().sum() > 0


def test_kept_histogram_keeps_nothing_else(dev):
    """A histogram kept for statistics holds its E counts alive, not the routing's index buffer."""
    logits = torch.randn(2000, 32, device=dev).to(torch.bfloat16)
    assert R.routing(logits, 4)[0].expt_hist.untyped_storage().nbytes() == 4 * 32


def test_entry_points_agree(dev):
    """af3_routing_replay / _topk / _replay_noalloc give the plan's outputs."""
    for T, E, K in ((50, 32, 4), (3000, 128, 4)):
        g = torch.Generator().manual_seed(T)
        logits = torch.randn(T, E, generator=g).to(torch.bfloat16).to(dev)
        rd, gi, si = R.routing(logits, K)
        ids, _ = O.topk_ids(logits.cpu(), K)
        ids = ids.to(dev)
        ws_n = _capi.workspace_bytes(T, E, K)
        ws = torch.empty(ws_n, dtype=torch.uint8, device=dev)
        for name in ("af3_routing_topk", "af3_routing_replay", "af3_routing_replay_noalloc"):
            o = [torch.empty(n, dtype=torch.int32, device=dev) for n in (E, T * K, T * K, E + 1)]
            gs = torch.empty(T * K, dtype=torch.bfloat16, device=dev)
            idp = () if name.endswith("topk") else (ids.data_ptr(),)
            tail = () if name.endswith("noalloc") else (ws.data_ptr(), ws_n)
            _capi.call(name, logits.data_ptr(), E, *idp, T, E, K, gs.data_ptr(), *[t.data_ptr() for t in o], *tail,
                       _capi.stream_of(torch.device(dev)))
            assert torch.equal(o[0], rd.expt_hist) and torch.equal(o[1], gi.src_indx)
            assert torch.equal(o[2], gi.dst_indx) and torch.equal(o[3], rd.expt_data.token_offs_raw)


@pytest.mark.parametrize("T,E,K", [(8191, 64, 1), (300, 32, 1), (4096, 32, 2), (512, 1024, 3), (1403, 257, 3),
                                   (1100, 128, 4), (700, 256, 16)])
def test_workspace_is_not_exceeded(dev, T, E, K):
    """Every entry point stays within a workspace of exactly the queried size (bytes behind it unchanged)."""
    g = torch.Generator().manual_seed(T + E + K)
    logits = torch.randn(T, E, generator=g).to(torch.bfloat16)
    ids = torch.rand(T, E, generator=g).topk(K, dim=1).indices.to(torch.int32)
    lib = _capi.load()
    ld, idd = logits.to(dev), ids.to(dev)
    for name in ("af3_routing_topk", "af3_routing_replay", "af3_routing_plan"):
        for topk in (0, 1):
            if (name.endswith("topk") and not topk) or (name.endswith("replay") and topk):
                continue
            ref = O.routing_topk(logits, K) if topk else O.routing_replay(logits, ids, K)
            plan = name.endswith("plan")
            n = int(lib.af3_routing_plan_workspace_bytes(T, E, K, topk)) if plan else _capi.workspace_bytes(T, E, K)
            ws = torch.full((2 * n + (1 << 20),), 0xA5, dtype=torch.uint8, device=dev)   # room behind the workspace
            o = [torch.empty(m, dtype=torch.int32, device=dev) for m in (E, T * K, T * K, E + 1)]
            gs = torch.empty(T * K, dtype=torch.bfloat16, device=dev)
            outs = (gs.data_ptr(), *[t.data_ptr() for t in o])
            tail = (ws.data_ptr(), n, _capi.stream_of(torch.device(dev)))
            if plan:
                mt = R.max_tiles(T * K, E, 128)
                pad = torch.empty(E + 1, dtype=torch.int32, device=dev)
                maps = torch.empty(2, mt, dtype=torch.int32, device=dev)
                _capi.call(name, ld.data_ptr(), E, idd.data_ptr(), topk, T, E, K, *outs, (ctypes.c_int32 * 1)(128), 1,
                           1, mt, pad.data_ptr(), maps[0].data_ptr(), maps[1].data_ptr(), *tail)
            else:
                _capi.call(name, ld.data_ptr(), E, *(() if topk else (idd.data_ptr(),)), T, E, K, *outs, *tail)
            torch.cuda.synchronize()
            assert (ws[n:] == 0xA5).all(), name
            assert torch.equal(o[1].cpu(), ref["topk_indx"]) and torch.equal(o[0].cpu(), ref["hist"].to(torch.int32))
            assert torch.equal(o[2].cpu(), ref["gate_indx"])


@pytest.mark.parametrize("T,H,E", [(1, 64, 1), (63, 128, 33), (64, 320, 64), (65, 384, 65), (129, 2880, 129),
                                   (200, 2880, 256), (31, 448, 128), (300, 576, 32)])
def test_router_ring_edges(dev, T, H, E):
    """Row, column and k-step edges of the ring (fewer k-steps than stages included)."""
    g = torch.Generator().manual_seed(T + H + E)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w = (torch.randn(E, H, generator=g) * H ** -0.5).to(torch.bfloat16)
    got = R.router_logits_hip(x.to(dev), w.to(dev), None)
    ref, mag = O.router_logits(x, w, None)
    check_close(got, ref, mag=mag, n=H, what=f"router T={T} H={H} E={E}")


@pytest.mark.parametrize("H", [64, 128, 192, 512, 2048])
@pytest.mark.parametrize("E", [8, 33, 128, 160, 193, 256])
def test_router_past_one_block_per_cu(dev, H, E):
    """More than 256 blocks take two or three stages and other column paddings: the same sums, so the logits of
    the first 256 blocks are those of a smaller batch, bit for bit."""
    T = 256 * 64 + 65
    g = torch.Generator().manual_seed(H + E)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    w = (torch.randn(E, H, generator=g) * H ** -0.5).to(torch.bfloat16).to(dev)
    b = torch.randn(E, generator=g).to(torch.bfloat16).to(dev)
    got = R.router_logits_hip(x, w, b)
    assert torch.equal(got[:16384], R.router_logits_hip(x[:16384], w, b))
    assert torch.equal(got[16000:], R.router_logits_hip(x[16000:], w, b))
