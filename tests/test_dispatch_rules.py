"""The layer's dispatch rules (host code only): which kernels a decode batch
takes, at shapes on each side of a line."""
import pytest

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
    # FP8: no fast form at H = 7168; at 4096 up to five staged rows
    (FMT_FP8, 3, 7168, True), (FMT_FP8, 5, 4096, False), (FMT_FP8, 6, 4096, True),
    (FMT_BF16, 10, 2048, False), (FMT_BF16, 11, 2048, True)])
def test_decode_gate_up_streams_past_the_fast_form(fmt, T, H, want):
    assert _gate_up_streams(fmt, T, 256, 1, H, 2048, 8) == want


@pytest.mark.parametrize("fmt,I,want", [(FMT_MXFP4, 768, True), (FMT_MXFP4, 1024, False),
                                        (FMT_FP8, 768, True), (FMT_FP8, 896, False),
                                        (FMT_NVFP4, 512, True), (FMT_NVFP4, 640, False),
                                        (FMT_BF16, 512, False)])
def test_decode_down_streams_at_a_short_k(fmt, I, want):
    assert L.decode_stream_down(fmt, 2048, I, 64) == want
    assert not L.decode_stream_down(fmt, 2048, I, 16)   # 256 work items
