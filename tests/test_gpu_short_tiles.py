"""The short-tile grouped GEMMs (32- / 64-row maps, tile_cfg 27 / 29) against the
128-row kernels, bit for bit (same fragments, same order of the sums): tile edges
of every expert row count, column tails, the smallest reduction, scale bytes that
take the integer conversion, every operand form moe_rows accepts; and the choice
of the map."""
import pytest
import torch

from agent_factory_3_amd import quantization as Q
from agent_factory_3_amd import routing as R

pytestmark = pytest.mark.gpu

HIST = [0, 1, 31, 32, 33, 0, 63, 64, 65, 96, 129, 5]


def _routing(dev, hist, k=1, short=(32, 64)):
    """Expert-sorted rows with the given counts and every map the kernels take."""
    h = torch.tensor(hist, dtype=torch.int32, device=dev)
    n = sum(hist)
    old = R.BLOCK_MS
    R.BLOCK_MS = short + old
    try:
        ed = R.compute_expt_data(h, len(hist), n)
        for bm in R.BLOCK_MS[:-1]:
            R.gemm_order_for(ed, bm)
    finally:
        R.BLOCK_MS = old
    return R.RoutingData(None, h, len(hist), k, ed), n


def _both(monkeypatch, bm, fn):
    monkeypatch.setattr(Q, "FWD_SHORT_ROWS", ())
    monkeypatch.setattr(Q, "DX_SHORT_ROWS", ())
    ref = fn()
    monkeypatch.setattr(Q, "FWD_SHORT_ROWS", ((1 << 30, bm),))
    monkeypatch.setattr(Q, "DX_SHORT_ROWS", ((1 << 30, bm),))
    calls = []
    orig = Q._capi.try_call
    monkeypatch.setattr(Q._capi, "try_call", lambda name, *a: calls.append(a[18]) or orig(name, *a))
    call = Q._capi.call
    monkeypatch.setattr(Q._capi, "call", lambda name, *a: (calls.append(a[18]) if name == "af3_moe_gemm" else None)
                        or call(name, *a))
    got = fn()
    monkeypatch.setattr(Q._capi, "try_call", orig)
    monkeypatch.setattr(Q._capi, "call", call)
    assert calls and all(c == bm for c in calls), calls     # the launches took the short map
    return got, ref


@pytest.mark.parametrize("bm", [32, 64])
@pytest.mark.parametrize("trans,N,K,r,form", [
    (False, 64, 320, 0, "plain"), (False, 576, 640, 16, "gather"), (False, 320, 2880, 32, "swiglu"),
    (False, 512, 960, 8, "odd"), (False, 192, 320, 0, "gamma32"), (False, 256, 640, 0, "untiled"),
    (True, 64, 64, 0, "plain"), (True, 576, 704, 16, "gather"), (True, 320, 1440 + 32, 32, "swiglu"),
    (True, 512, 128, 8, "odd"), (True, 192, 64, 0, "gamma32"), (True, 2880, 192, 0, "untiled"),
])
def test_short_tiles_equal_the_128_row_kernels(dev, monkeypatch, bm, trans, N, K, r, form):
    g = torch.Generator().manual_seed(N + K + bm)
    E = len(HIST)
    rd, n = _routing(dev, HIST)
    rows, cols = (K, N) if trans else (N, K)
    blocks = torch.randint(0, 256, (E, rows, cols // 32, 16), generator=g, dtype=torch.uint8)
    scales = torch.randint(118, 123, (E, rows, cols // 32), generator=g, dtype=torch.uint8)
    if form == "odd":
        for e, v in ((1, 0), (3, 1), (6, 254), (8, 255), (10, 253)):
            scales[e, rows // 2, 0] = v
    blocks, scales = blocks.to(dev), scales.to(dev)
    bias = (torch.randn(E, N, generator=g)).to(torch.bfloat16).to(dev) if not trans else None
    gam = torch.rand(n, generator=g).to(dev)
    gam = gam if form == "gamma32" else None if form == "plain" else gam.to(torch.bfloat16)
    L = torch.randn(n, r, generator=g).to(torch.bfloat16).to(dev) if r else None
    B = (torch.randn(*((E, r, N) if trans else (E, N, r)), generator=g) * 0.1).to(torch.bfloat16).to(dev) if r else None
    gather = None
    if form == "gather":
        x = torch.randn(n // 2, K + 64, generator=g).to(torch.bfloat16).to(dev)[:, :K]    # strided rows
        idx = torch.randint(0, n // 2, (n,), generator=g, dtype=torch.int32).to(dev)
        gather = R.GatherIndx(idx, idx)
    else:
        x = torch.randn(n, K, generator=g).to(torch.bfloat16).to(dev)
    kw = dict(lora_l=L, lora_b=B)
    if form not in ("plain", "untiled"):
        kw.update(dict(s_tiled=Q.mxfp4_tile_dx_scales(scales)) if trans else dict(w_tiled=Q.mxfp4_tile_fwd(blocks)))
    if form == "swiglu":
        gu = (torch.randn(n, 2 * N, generator=g) * 3).to(torch.bfloat16).to(dev)
        kw["swiglu"] = ("bwd", gu, 1.702, 7.0) if trans else ("fwd", 1.702, 7.0)
    got, ref = _both(monkeypatch, bm,
                     lambda: Q.moe_rows(x, blocks, scales, bias, rd, gather, gam, trans, **kw))
    got, ref = (got, ref) if isinstance(got, tuple) else ((got,), (ref,))
    for a, b in zip(got, ref):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("E,rows", [(4, 4), (40, 4), (12, 300)])  # fewer m-tiles than the spread order's limit, more
def test_short_tiles_work_orders(dev, monkeypatch, E, rows):
    g = torch.Generator().manual_seed(E)
    hist = [rows if e % 3 else 0 for e in range(E)]
    rd, n = _routing(dev, hist)
    N, K = 1152, 320
    blocks = torch.randint(0, 256, (E, N, K // 32, 16), generator=g, dtype=torch.uint8).to(dev)
    scales = torch.randint(118, 123, (E, N, K // 32), generator=g, dtype=torch.uint8).to(dev)
    x = torch.randn(n, K, generator=g).to(torch.bfloat16).to(dev)
    dy = torch.randn(n, N, generator=g).to(torch.bfloat16).to(dev)
    for bm in (32, 64):
        got, ref = _both(monkeypatch, bm, lambda: Q.moe_rows(x, blocks, scales, None, rd))
        assert torch.equal(got, ref)
        got, ref = _both(monkeypatch, bm, lambda: Q.moe_rows(dy, blocks, scales, None, rd, trans_w=True))
        assert torch.equal(got, ref)


def test_map_choice(dev):
    """Few rows per expert and whole k-groups take the short maps, everything else the 128-row one."""
    logits = torch.randn(200, 32, device=dev).to(torch.bfloat16)
    ed = R.routing(logits, 4)[0].expt_data                       # 25 rows per expert
    assert Q._short_block_m(ed, 800, 32, 5760, 2880, False, True) == 64
    assert Q._short_block_m(ed, 800, 32, 2880, 5760, True, True) == 64
    assert Q._short_block_m(ed, 400, 32, 5760, 2880, False, True) == 32
    assert Q._short_block_m(ed, 400, 32, 5760, 384, False, True) == 0        # K % 320
    assert Q._short_block_m(ed, 400, 32, 5760, 3200, False, True) == 0       # K > 3072
    assert Q._short_block_m(ed, 400, 32, 96, 2880, True, True) == 0          # N % 64
    assert Q._short_block_m(ed, 400, 32, 5760, 2880, False, False) == 0      # 64-bit offsets
    assert Q._short_block_m(ed, 1 << 20, 32, 5760, 2880, False, True) == 0
    big = R.routing(torch.randn(8000, 16, device=dev).to(torch.bfloat16), 4)[0].expt_data     # 2000 rows per expert
    assert 32 not in big.block_pid_map and Q._short_block_m(big, 100, 16, 5760, 2880, False, True) == 0


@pytest.mark.parametrize("trans,rows,want", [(False, 24, 32), (False, 25, 64), (False, 48, 64), (False, 49, 0),
                                             (True, 18, 32), (True, 19, 64), (True, 32, 64), (True, 33, 0)])
def test_map_choice_at_its_lines(trans, rows, want):
    ed = R.ExptData(None, None, block_pid_map={32: 0, 64: 0}, gemm_order={32: 0, 64: 0})
    for E in (32, 128):
        assert Q._short_block_m(ed, rows * E, E, 2880, 2880, trans, True) == want


@pytest.mark.parametrize("off", [1, 8])
def test_scales_at_an_unaligned_address(dev, monkeypatch, off):
    """The short forward copies 16-byte runs of scales: at any other address the call keeps the general
    kernel's result, plain and (unfused: None) with SwiGLU; the input gradient takes them anywhere."""
    g = torch.Generator().manual_seed(off)
    E, N, K = len(HIST), 192, 320
    rd, n = _routing(dev, HIST)
    blocks = torch.randint(0, 256, (E, N, K // 32, 16), generator=g, dtype=torch.uint8).to(dev)
    scales = torch.randint(118, 123, (E, N, K // 32), generator=g, dtype=torch.uint8)
    store = torch.zeros(scales.numel() + 16, dtype=torch.uint8, device=dev)
    s = store[off:off + scales.numel()].view(scales.shape)
    s.copy_(scales)
    x = torch.randn(n, K, generator=g).to(torch.bfloat16).to(dev)
    dy = torch.randn(n, N, generator=g).to(torch.bfloat16).to(dev)
    al = scales.to(dev)
    y, ref = Q.moe_rows(x, blocks, s, None, rd), Q.moe_rows(x, blocks, al, None, rd)
    # the same exact products (K of them) in another order of the fp32 sum, then one bf16 rounding each
    w = Q.mxfp4_to_bf16(blocks, al).float().abs()
    mag = torch.cat([x[a:a + h].float().abs() @ w[e].t() for e, (a, h) in
                     enumerate(zip([sum(HIST[:i]) for i in range(E)], HIST))])
    assert ((y.float() - ref.float()).abs() <= 2 * K * 2.0 ** -24 * mag + 2.0 ** -7 * ref.float().abs()).all()
    assert Q.moe_rows(x, blocks, s, None, rd, swiglu=("fwd", 1.702, 7.0)) is None
    monkeypatch.setattr(Q, "DX_SHORT_ROWS", ((1 << 30, 64),))
    assert torch.equal(Q.moe_rows(dy, blocks, s, None, rd, trans_w=True),
                       Q.moe_rows(dy, blocks, al, None, rd, trans_w=True))


@pytest.mark.parametrize("r", [16, 32])
@pytest.mark.parametrize("trans_b,K", [(0, 64), (0, 576), (0, 2880), (1, 128), (1, 1472)])
def test_lora_rows_32_row_map(dev, monkeypatch, r, trans_b, K):
    """The 32-row LoRA row product: bit-equal to the 128-row one on every tile edge (fewer k-steps than
    ring stages included), with and without a gather."""
    g = torch.Generator().manual_seed(K + r)
    E = len(HIST)
    rd, n = _routing(dev, HIST)
    ed = rd.expt_data
    x = torch.randn(n, K + 8, generator=g).to(torch.bfloat16).to(dev)[:, :K]
    wl = torch.randn(*((E, K, r) if trans_b else (E, r, K)), generator=g).to(torch.bfloat16).to(dev)
    idx = torch.randint(0, 2 * n, (n,), generator=g, dtype=torch.int32).to(dev)
    for gather, k in ((None, 1), (idx, 2)):
        out = []
        for lim in (0, 1 << 20):
            monkeypatch.setattr(Q, "LORA_SHORT_TILES", lim)
            out.append(Q._lora_rows(x, gather, k, wl, trans_b, 0.5, ed, r, K))
        assert torch.equal(out[0], out[1])
