"""The weight-streaming grouped GEMMs (xtu_stream_gate_up / xtu_stream_down)
against the dequantized-fp32 oracle: every row-tile count and its remainders,
K of one partial round up to several, all formats and tile heights, y in
sorted and in flat pair order, and the layer calls that take them."""
import numpy as np
import pytest
import torch

from helpers import (bf16_tensor_to_bits, check_close, dense_to_numpy, make_dense_layer,
                     oracle_layer, random_routing)
from xtu_moe_amd import _lib
from xtu_moe_amd import formats as F
from xtu_moe_amd import layer as L
from xtu_moe_amd.layer import ExpertWeights, _p, _stream, moe_forward

pytestmark = pytest.mark.gpu

FMTS = [F.FMT_MXFP4, F.FMT_NVFP4, F.FMT_FP8, F.FMT_BF16]
# rows per expert: the edges of 16-row MFMA tiles and of each tile height
ROWS = [1, 15, 16, 17, 0, 33, 48, 49, 64, 65, 80, 96, 97, 128, 129]


def _weights(fmt, E, NS, H, I, seed):
    d = make_dense_layer(fmt, E + NS, H, I, seed=seed)
    return d, ExpertWeights.from_dense(fmt, d["w13"], d["s13"], d["w2"], d["s2"], d["gs13"],
                                       d["gs2"], n_shared=NS, device="cuda")


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("bm", [16, 64, 128])
@pytest.mark.parametrize("H,I", [(256, 128), (768, 384)])
def test_row_tile_edges(fmt, bm, H, I):
    if bm > _lib.call("xtu_stream_max_tile_m", fmt):
        pytest.skip("taller than this format's tiles")
    _row_tile_edges(fmt, bm, H, I, 0)


@pytest.mark.parametrize("bm", [64, 128])
@pytest.mark.parametrize("H,I", [(256, 128), (768, 384)])
def test_bf16_wide_items_row_tile_edges(bm, H, I):
    """From 512 items on BF16 takes four panels per wave in both passes (a grid
    bound past the tiles: the surplus workgroups leave)."""
    _row_tile_edges(F.FMT_BF16, bm, H, I, -(-512 // min(I // 128, H // 256)))


def _row_tile_edges(fmt, bm, H, I, min_tiles):
    print(f"stream fmt={fmt} bm={bm} H={H} I={I} min_tiles={min_tiles}", flush=True)
    E = len(ROWS)
    ids = np.repeat(np.arange(E, dtype=np.int32), ROWS)
    rng = np.random.default_rng(bm + H)
    rng.shuffle(ids)
    T = len(ids)
    ids = ids[:, None].copy()
    wts = rng.random((T, 1)).astype(np.float32) + 0.5
    d, W = _weights(fmt, E, 0, H, I, seed=H + I)
    x = torch.randn((T, H), generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    xd, idd, wd = x.cuda(), torch.from_numpy(ids).cuda(), torch.from_numpy(wts).cuda()
    seg = L.segmentation(T, 1, E, 0, bm, torch.device("cuda")).run(idd, wd)
    lo, hi = seg.tile_range_ptrs(0, E)
    max_tiles = max(seg.max_tiles, min_tiles)
    act = torch.full((T, I), float("nan"), dtype=torch.bfloat16, device="cuda")
    _lib.call("xtu_stream_gate_up", fmt, _p(xd), T, _p(seg.sorted_tok), H, I, _p(W.w13),
              _p(W.s13), _p(W.gs13), 0, 0, 0, _p(seg.seg_start), _p(seg.tile_expert),
              _p(seg.tile_row0), lo, hi, bm, max_tiles, _p(act), 2.0, 1.0, 0.0, _stream())
    ys = []
    for pair_of in (0, _p(seg.sorted_pair)):
        y = torch.full((T, H), float("nan"), device="cuda")
        _lib.call("xtu_stream_down", fmt, _p(act), H, I, _p(W.w2), _p(W.s2), _p(W.gs2), 0, 0, 0,
                  _p(seg.seg_start), _p(seg.tile_expert), _p(seg.tile_row0), lo, hi, bm,
                  max_tiles, pair_of, _p(y), _stream())
        ys.append(y)
    torch.cuda.synchronize()
    assert torch.equal(ys[0][seg.inv.long()], ys[1])
    out = (ys[1] * wd).cpu().numpy()
    ref = oracle_layer(fmt, dense_to_numpy(fmt, d), bf16_tensor_to_bits(x), ids, wts, E, 0, H, I,
                       limit=2.0)
    check_close(out, ref, bf16_out=False, what=f"stream fmt={fmt} bm={bm}")


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("T", [12, 40, 200])
def test_layer_takes_them(fmt, T):
    """Auto dispatch: a decode batch past the staged rows, a batch of short
    tiles and one of tall ones, with shared experts, invalid ids, dropped zero
    weights and a slot map."""
    E, NS, I, K = 128, 1, 512, 8
    H = 2048 if T <= L.DECODE_MAX_TOKENS else 256   # 12 rows of 2048 are past the staged rows
    d, W = _weights(fmt, E, NS, H, I, seed=7)
    ids, wts = random_routing(T, K, E, seed=T, invalid_frac=0.05, zero_frac=0.05)
    x = torch.randn((T, H), generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    if T > L.DECODE_MAX_TOKENS:
        want = {F.FMT_FP8: 64, F.FMT_BF16: 128}.get(fmt, 16 if T == 40 else 64)
        assert L.stream_tile_m(fmt, T, K, E, NS, H, I) == want
    else:
        n = L.decode_max_tiles(T * (K + NS), min(E, T * K) + NS)
        assert L.decode_stream_gate_up(fmt, T, H, I, n)
        assert L.decode_stream_down(fmt, H, I, n) == (fmt != F.FMT_BF16)
    perm = torch.randperm(E + NS, generator=torch.Generator().manual_seed(1))
    Wp = ExpertWeights(fmt, H, I, E, NS, *[None if t is None else t[perm.cuda()].contiguous()
                                           for t in (W.w13, W.s13, W.w2, W.s2, W.gs13, W.gs2)])
    smap = torch.argsort(perm).to(torch.int32).cuda()
    for t in L._BUF_CACHE.values():   # a row the kernels leave out shows up
        if t.is_floating_point():
            t.fill_(float("nan"))
    out = moe_forward(x.cuda(), torch.from_numpy(ids).cuda(), torch.from_numpy(wts).cuda(), Wp,
                      slot_map=smap, out_dtype=torch.float32)
    torch.cuda.synchronize()
    ref = oracle_layer(fmt, dense_to_numpy(fmt, d), bf16_tensor_to_bits(x), ids, wts, E, NS, H, I)
    check_close(out.cpu().numpy(), ref, bf16_out=False, what=f"stream layer fmt={fmt} T={T}")


@pytest.mark.parametrize("bm", [16, 64, 128])
@pytest.mark.parametrize("H,I", [(256, 128), (768, 384)])
def test_int8_rows_equal_the_expanded_planes(bm, H, I):
    """Codes expanded in registers: bitwise the integer GEMM over the expanded
    planes, with scale spreads of 0..3 and rows marked for the fallback (their
    columns are zero sums in both)."""
    E = len(ROWS)
    fmt = F.FMT_MXFP4
    ids = np.repeat(np.arange(E, dtype=np.int32), ROWS)
    rng = np.random.default_rng(bm + I)
    rng.shuffle(ids)
    T = len(ids)
    d, _ = _weights(fmt, E, 0, H, I, seed=H)
    for k in ("s13", "s2"):   # spread 0..3 per row, a few rows past it
        s = d[k].to(torch.int32)
        s = 120 + torch.randint(0, 4, s.shape, generator=torch.Generator().manual_seed(3))
        s[:, 5::37, 0] = 131
        d[k] = s.to(torch.uint8)
    W = ExpertWeights.from_dense(fmt, d["w13"], d["s13"], d["w2"], d["s2"], n_shared=0,
                                 device="cuda")
    w13_8, em13, w2_8, em2 = W.int8_planes()
    x = torch.randn((T, H), generator=torch.Generator().manual_seed(T)).to(torch.bfloat16).cuda()
    idd = torch.from_numpy(ids[:, None].copy()).cuda()
    wd = torch.ones((T, 1), device="cuda")
    st = _stream()
    dev = x.device
    a8 = torch.empty((T, H), dtype=torch.int8, device=dev)
    cr = torch.empty(T, dtype=torch.int32, device=dev)
    _lib.call("xtu_i8_quant_rows", _p(x), T, H, _p(a8), _p(cr), st)
    acts, ys = [], []
    for b in (128, bm):
        seg = L.segmentation(T, 1, E, 0, b, dev)
        seg.run(idd, wd)
        lo, hi = seg.tile_range_ptrs(0, E)
        act = torch.full((T, I), float("nan"), dtype=torch.bfloat16, device=dev)
        a8a = torch.empty((T, I), dtype=torch.int8, device=dev)
        cra = torch.empty(T, dtype=torch.int32, device=dev)
        y = torch.full((T, H), float("nan"), device=dev)
        tiles = (_p(seg.seg_start), _p(seg.tile_expert), _p(seg.tile_row0), lo, hi)
        if not acts:
            _lib.call("xtu_i8_gemm_gate_up", _p(a8), _p(cr), _p(seg.sorted_tok), H, I, _p(w13_8),
                      _p(em13), 0, *tiles, seg.max_tiles, _p(act), 0, 2.0, 1.0, 0.0, st)
        else:
            _lib.call("xtu_stream_i8_gate_up", _p(a8), _p(cr), T, _p(seg.sorted_tok), H, I,
                      _p(W.w13), _p(W.s13), _p(em13), 0, *tiles, b, seg.max_tiles, _p(act), 2.0,
                      1.0, 0.0, st)
        _lib.call("xtu_i8_quant_rows", _p(act), T, I, _p(a8a), _p(cra), st)
        if not acts:
            _lib.call("xtu_i8_gemm_down", _p(a8a), _p(cra), H, I, _p(w2_8), _p(em2), 0, *tiles,
                      seg.max_tiles, _p(y), 0, st)
        else:
            _lib.call("xtu_stream_i8_down", _p(a8a), _p(cra), H, I, _p(W.w2), _p(W.s2), _p(em2),
                      0, *tiles, b, seg.max_tiles, _p(y), st)
        acts.append(act)
        ys.append(y)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(ys[0]).all())
    assert torch.equal(acts[0], acts[1]) and torch.equal(ys[0], ys[1])
