"""The layer's dispatch rules (host code only): which kernels a decode batch
takes, at shapes on each side of a line."""
import pytest
import torch

from xtu_moe_amd import layer as L
from xtu_moe_amd.formats import FMT_BF16, FMT_FP8, FMT_MXFP4, FMT_NVFP4


def _gate_up_streams(fmt, T, E, NS, H, I, K):
    tiles = L.decode_max_tiles(T * (K + NS), min(E, T * K) + NS)
    return L.decode_stream_gate_up(fmt, T, H, I, tiles)


@pytest.mark.parametrize("fmt,T,H,want", [
    # 4-bit weights: the decode kernel as long as its fast form holds (T <= 4),
    # however many bytes of rows it stages
    (FMT_MXFP4, 3, 7168, False), (FMT_MXFP4, 4, 7168, False), (FMT_MXFP4, 5, 7168, True),
    (FMT_NVFP4, 3, 7168, False), (FMT_NVFP4, 4, 8192, False), (FMT_NVFP4, 5, 7168, True),
    # FP8: no fast form at H = 7168; at 4096 up to T = 8
    (FMT_FP8, 3, 7168, True), (FMT_FP8, 8, 4096, False), (FMT_FP8, 9, 4096, True),
    # BF16: past 40 KB of rows at H = 2048, and where K is not whole rounds
    (FMT_BF16, 10, 2048, False), (FMT_BF16, 11, 2048, True), (FMT_BF16, 3, 4096, False),
    (FMT_BF16, 16, 8192, False), (FMT_BF16, 3, 5120, True), (FMT_BF16, 5, 7168, True)])
def test_decode_gate_up_streams_past_the_fast_form(fmt, T, H, want):
    assert _gate_up_streams(fmt, T, 256, 1, H, 2048, 8) == want


@pytest.mark.parametrize("fmt,I,want", [(FMT_MXFP4, 768, True), (FMT_MXFP4, 1024, False),
                                        (FMT_FP8, 768, True), (FMT_FP8, 896, False),
                                        (FMT_NVFP4, 512, True), (FMT_NVFP4, 640, False),
                                        (FMT_BF16, 512, False)])
def test_decode_down_streams_at_a_short_k(fmt, I, want):
    assert L.decode_stream_down(fmt, 2048, I, 64) == want
    assert not L.decode_stream_down(fmt, 2048, I, 16)   # 256 work items


@pytest.mark.parametrize("T,K,NS,E,H,I,fused", [
    # 13 to 24 active experts of MXFP4 at a short K: the separate down where it
    # writes pair order, the fused one where it cannot (K = 7; three shared)
    (2, 8, 0, 128, 2048, 768, False), (2, 8, 1, 256, 2048, 512, False),
    (2, 7, 3, 256, 2048, 512, True), (2, 6, 3, 256, 2048, 512, True),
    (2, 8, 1, 256, 2048, 2048, True), (1, 10, 1, 512, 2048, 512, True)])
def test_fused_down_leaves_only_for_the_down_in_pair_order(T, K, NS, E, H, I, fused):
    active = min(E, T * K) + NS
    by_pair = L.down_by_pair(K, NS, torch.bfloat16)
    assert by_pair == (K in L.COMBINE_BY_PAIR_K and NS <= 2)
    assert L.decode_fused_down_use(FMT_MXFP4, T, T * (K + NS), H, I, active, E + NS,
                                   by_pair=by_pair) == fused


def test_down_by_pair_switch(monkeypatch):
    monkeypatch.setenv(L.DOWN_BY_PAIR_ENV, "0")
    assert not L.down_by_pair(8, 1, torch.bfloat16)
    monkeypatch.delenv(L.DOWN_BY_PAIR_ENV)
    assert not L.down_by_pair(8, 1, torch.float16)


@pytest.mark.parametrize("T,K,E,NS,small", [(64, 16, 1024, 0, True), (341, 3, 1024, 0, True),
                                            (341, 3, 1025, 0, False), (2, 4, 2047, 0, False),
                                            (2, 4, 3, 1, False), (1, 3, 3, 1, True),
                                            (2, 17, 64, 0, False), (64, 16, 1024, 1, False)])
def test_small_segmentation_takes_what_its_entry_takes(T, K, E, NS, small):
    """At most 1024 experts and K <= E besides the pair and bucket limits."""
    assert L.segmentation(T, K, E, NS, 16, "cpu", stream=0).small == small


@pytest.mark.parametrize("wl,T,i8,kernel", [
    ("ds-v3-mxfp4-decode", 4, False, "decode_gate_up_kernel"),
    ("ds-v3-mxfp4-decode", 8, False, "stream_gemm_kernel"),
    ("ds-v3-mxfp4-prefill", 8192, False, "mx_pair_gemm_kernel"),
    ("qwen3-next-int8", 8192, True, "stream_gemm_kernel"),
    ("qwen3-next-nvfp4", 4, False, "decode_gate_up_kernel"),
    ("mixtral-tiny-bf16", 128, False, "moe_gemm_kernel")])
def test_bench_times_the_gate_up_the_layer_takes(wl, T, i8, kernel):
    bench = pytest.importorskip("bench")
    c = bench.WORKLOADS[wl]
    fmt = {"mxfp4": FMT_MXFP4, "nvfp4": FMT_NVFP4, "bf16": FMT_BF16}[c["fmt"]]
    name, bm, tiles = bench.gate_up_choice(fmt, T, c["E"], c["NS"], c["H"], c["I"], c["K"], i8, None)
    assert name == kernel
    if T <= L.DECODE_MAX_TOKENS:
        assert (bm, tiles) == (L.DECODE_TILE, L.decode_max_tiles(
            T * (c["K"] + c["NS"]), min(c["E"], T * c["K"]) + c["NS"]))


def test_streaming_leaves_planes_past_32_bit_offsets():
    """One expert's gate/up plane of 2 GiB: the kernels with 64-bit plane
    offsets keep it (2 I H bytes of FP8, I H of MXFP4 codes)."""
    big, fits = 1 << 16, (1 << 16) - 128
    assert L.stream_tile_m(FMT_FP8, 64, 2, 8, 0, 16384, fits) == 64
    assert L.stream_tile_m(FMT_FP8, 64, 2, 8, 0, 16384, big) == 0
    assert L.stream_i8_tile_m(64, 2, 8, 32768, fits) == 64
    assert L.stream_i8_tile_m(64, 2, 8, 32768, big) == 0
