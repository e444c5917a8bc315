"""What calls ask of their callers' memory (sizes only: no GPU)."""
import ctypes as C

from hibana_amd import _lib


def test_the_layer_from_its_rows_asks_for_logits_only_where_it_makes_them():
    lib = _lib.lib()
    ex = _lib.HbW3Experts(256, 256, 256, 256, 0, 0, 512, 0, 2048, 512, 2048, 1)
    up256 = lambda v: (v + 255) // 256 * 256  # noqa: E731
    for m, made in [(1, True), (64, True), (65, False), (2048, False)]:
        extra = lib.hb_w3_moe_layer_rows_workspace_bytes(m, 10, C.byref(ex), 1, 512) - lib.hb_w3_moe_workspace_bytes(m, 10, C.byref(ex), 1)
        assert extra == (up256(m * 512 * 2) if made else 0) + 2 * up256(m * 10 * 4), m


def test_the_dense_product_asks_for_what_its_cut_shares():
    lib = _lib.lib()
    assert lib.hb_nvfp4_gemm_room_bytes(64, 25600, 5120) == 0  # every tile a workgroup's own
    assert lib.hb_nvfp4_gemm_room_bytes(16, 1024, 12800) == 0 and lib.hb_nvfp4_gemm_room_bytes(17, 1024, 12800) > 4096
    assert lib.hb_tune(b"nvfp4_tile_ks", 3) == 0
    try:
        assert lib.hb_nvfp4_gemm_room_bytes(64, 25600, 5120) > 4096  # a forced cut has its room
    finally:
        lib.hb_tune(b"nvfp4_tile_ks", 0)
