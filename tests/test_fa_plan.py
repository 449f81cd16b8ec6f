"""The prefill's plan as its workspace query shows it (host code: needs the built library, no GPU)."""
import ctypes

import pytest

H, KV = 16, 2


def _bytes(max_t, T):
    import moex_amd
    f = ctypes.CDLL(moex_amd.LIB_PATH).moex_attn_workspace_bytes
    f.restype, f.argtypes = ctypes.c_size_t, [ctypes.c_int] * 4
    return f(H, KV, max_t, T)


@pytest.mark.parametrize("max_t,T,pieces", [
    (320, 65, False), (320, 213, False), (320, 300, False),                  # the device would split at no position
    (384, 150, False), (448, 213, False), (512, 300, False), (512, 400, False),  # only the heavier token tiles
    (384, 65, True), (448, 150, True), (512, 213, True), (576, 300, True),   # every token tile, at the last positions
    (8192, 213, True), (262144, 1024, True), (262144, 1025, False),          # half a full grid is the last that splits
])
def test_small_caches_keep_pairs(max_t, T, pieces):
    """Key pieces take a workspace of T * H * pieces * 1040 bytes; a chunk in a cache too small for them to pay has none."""
    images = KV * ((max_t + 31) // 32) * 37632
    least = 2 * T * H * 1040
    assert (_bytes(max_t, T) - images >= least) == pieces
