"""Which kernels a call takes: rules that the kernel libraries decide on the host (for 256 compute units where there is no GPU to ask)."""
import pytest
import torch

from mini_inference_engine_amd.kernels import library, modules  # noqa: F401
from mini_inference_engine_amd.kernels.hip_backend import HipBackend


# rows, columns, K and whether the own tile makes q/k/v with the rotation behind it faster than the library: few compute units over a long K, and more of them or a shorter one
@pytest.mark.parametrize("case", [(129, 768, 3072, False), (129, 640, 2560, False), (300, 768, 4096, False), (192, 1280, 5120, False), (129, 896, 8192, False),
                                  (256, 768, 3072, True), (350, 768, 4096, True), (129, 768, 2048, True), (129, 2560, 2048, True), (2048, 2560, 2048, True),
                                  (512, 6144, 4096, True), (2048, 6144, 4096, False)])
def test_rotated_products_on_own_tiles_where_they_gain(case):
    M, N, K, gains = case
    lib = library.load("tile_gemm_bf16")
    assert bool(lib.mie_tile_gemm_rope_gains(M, N, K)) == gains
    assert lib.mie_tile_gemm_tile(M, N, K) > 0 or not gains


# rows, columns, K and whether the own tile adds into the stream faster than the library: few workgroups over a long K, the widest
# tile on three quarters of the chip, the widest tiles of many columns over a short K, and each one's other side
@pytest.mark.parametrize("case", [(129, 1024, 2048, False), (256, 1024, 3072, False), (192, 1536, 1536, False), (256, 1024, 1024, True), (300, 1024, 3072, True),
                                  (1536, 4096, 4096, False), (1500, 4096, 14336, False), (768, 8192, 8192, False), (1700, 4096, 4096, True),
                                  (2048, 4096, 14336, True), (600, 8192, 2048, False), (1024, 8192, 2048, False), (1024, 8192, 8192, True),
                                  (129, 2048, 2048, True), (512, 2048, 2048, True), (1132, 2048, 5632, True), (2048, 2048, 5632, True), (4096, 8192, 1024, False)])
def test_added_products_on_own_tiles_where_they_gain(case):
    M, N, K, gains = case
    lib = library.load("tile_gemm_bf16")
    assert bool(lib.mie_tile_gemm_add_gains(M, N, K)) == gains
    assert lib.mie_tile_gemm_tile(M, N, K) > 0 or not gains


@pytest.mark.parametrize("case", [(2048, 4096, 14336, 0), (2047, 4096, 14336, 0), (1792, 4096, 14336, 8), (2048, 4096, 11008, 8), (2048, 4096, 4096, 8)])
def test_added_products_read_weights_ahead_where_a_step_gains_by_it(case):
    M, N, K, ahead = case
    lib = library.load("tile_gemm_bf16")
    assert lib.mie_tile_gemm_tile(M, N, K) == 256128, "the only tile that such products take"
    assert lib.mie_tile_gemm_add_ahead(M, N, K) == ahead


# single tokens, portions, tokens of the longest, query and kv heads, splits: as many single workgroups as compute units and one more, and
# more portions than a grid of the portions' own kernel has rows for
@pytest.mark.parametrize("case", [(64, 1, 40, 32, 4, 1, True), (65, 1, 40, 32, 4, 1, False), (16, 1, 40, 32, 4, 4, True), (17, 1, 40, 32, 4, 4, False),
                                  (1, 65535, 2, 4, 1, 1, True), (1, 65536, 2, 4, 1, 1, False), (1, 1, 0, 32, 4, 1, False), (0, 1, 40, 32, 4, 1, False)])
def test_steps_whose_attention_is_one_launch(case):
    lib = library.load("prefill_attention_bf16", ("-DHEAD_DIM=64",))
    assert bool(lib.mie_step_attention_takes(*case[:-1])) == case[-1]
    assert not library.load("prefill_attention_bf16", ("-DHEAD_DIM=128",)).mie_step_attention_takes(*case[:-1])


# rows, columns, K and the parts that a long K is added in: one workgroup a compute unit, two of three to five parts, never two of two parts
@pytest.mark.parametrize("case", [(129, 2048, 5632, 8), (512, 4096, 14336, 2), (384, 4096, 14336, 5), (385, 4104, 4096, 3), (300, 8192, 4096, 0), (384, 8192, 14336, 0),
                                  (512, 6144, 8192, 0), (256, 8192, 4096, 2), (513, 4096, 4096, 0), (512, 8192, 4096, 0), (300, 4096, 4032, 0)])
def test_parts_of_a_long_k(case):
    M, N, K, units = case
    o = HipBackend.__new__(HipBackend)
    o.true_fp32 = False
    x, w = (torch.empty(n, K, dtype=torch.bfloat16, device="meta") for n in (M, N))
    assert o._tile_split(x, w, None) == units
