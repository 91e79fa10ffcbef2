"""The kernels that the GEMM entry points choose by shape, at shapes where the rule was measured on both
sides (figures beside the rules in csrc/gemm_fp8.hip and csrc/gemm_w8a16.hip). No GPU: the choice of 256 compute
units."""
import pytest

F16, BF16, F32 = 0, 1, 2
ROWS16, TILE32, ROW1 = 50, 26, 51


@pytest.fixture(scope="module")
def lib():
  from cache_dit_amd import _native
  if not _native.is_built():
    pytest.skip("libcdit_hip.so not built")
  return _native.load()


@pytest.mark.parametrize("M,N,K,want", [
    # long K on few columns: the 16-row kernel splits K over four wavefronts
    (9, 576, 14608, ROWS16), (8, 2048, 12288, ROWS16), (4, 2048, 15360, ROWS16), (2, 4096, 15360, ROWS16),
    (9, 1024, 3072, ROWS16), (16, 1024, 12288, ROWS16),
    # a last batch of its steps that is nearly empty
    (9, 256, 3200, TILE32), (16, 384, 8736, TILE32),
    # longer K: a later batch of the 16-row kernel costs less
    (16, 832, 9600, ROWS16), (16, 2304, 9344, ROWS16), (13, 3184, 6272, ROWS16), (16, 2112, 4096, TILE32),
    # K remainders: up to 11 rows, rows that start on 64-byte boundaries, some 20 workgroups and fewer
    (9, 416, 2224, ROWS16), (11, 2016, 2448, ROWS16), (12, 320, 2144, ROWS16), (16, 288, 5280, ROWS16),
    (10, 1120, 7232, ROWS16), (14, 1600, 2752, ROWS16), (15, 528, 4544, TILE32), (16, 944, 11024, TILE32),
    # many columns
    (16, 9216, 3072, TILE32), (16, 18432, 5120, TILE32), (8, 18432, 3072, TILE32), (4, 9216, 5120, TILE32),
    (2, 18432, 3072, ROWS16), (2, 9216, 5120, TILE32), (1, 9216, 3072, ROW1), (1, 9216, 4112, ROWS16)])
def test_few_rows(lib, M, N, K, want):
  for dtype in (F16, BF16, F32):
    assert lib.cdit_debug_gemm_choice(0, M, N, K, dtype) == want


@pytest.mark.parametrize("M,N,K,want", [
    # rows beyond 16384 elements are quantized in the GEMM's kernel where they fit its LDS
    (2, 16192, 16512, 1), (2, 22592, 17472, 1), (3, 7936, 18688, 1), (2, 9216, 5120, 2),
    # codes of more than 48 KiB in every workgroup's LDS
    (8, 256, 6128, 1), (8, 256, 6144, 2), (8, 256, 6464, 2), (6, 256, 8384, 2), (4, 2304, 12480, 2),
    (2, 2816, 15360, 1), (4, 2304, 12272, 1), (1, 9216, 3072, 1), (8, 3072, 3072, 1),
    (16, 9216, 3072, 2), (16, 3072, 3072, 2), (8, 2048, 12288, 2), (17, 64, 64, 2)])
def test_launches_of_few_rows(lib, M, N, K, want):
  assert lib.cdit_debug_linear_launches(M, N, K) == want


@pytest.mark.parametrize("M,N,K,tiles", [
    (300, 3072, 2224, True),
    # five and four tiles per CU (K remainders, K of one or two steps) and beyond
    (160, 8192, 400, True), (161, 8192, 400, False),
    (144, 8032, 1680, False), (128, 8192, 1680, True), (72, 11840, 8992, False), (898, 1088, 11536, False),
    (160, 8192, 256, True), (161, 8192, 256, False),
    # few columns, of which some XCDs get twice as many as others
    (2240, 288, 15136, False), (1366, 576, 3920, False), (1366, 576, 784, True), (1199, 704, 4160, True),
    (1199, 704, 6160, False)])
def test_tiles_of_more_than_16_rows(lib, M, N, K, tiles):
  for dtype in (F16, BF16, F32):
    assert (lib.cdit_debug_gemm_choice(0, M, N, K, dtype) == TILE32) == tiles


@pytest.mark.parametrize("M,N,K,want", [
    # whole steps that one round of a tile covers
    (77, 3072, 4096, 39), (303, 640, 4736, 38), (203, 3392, 4992, 33), (96, 8192, 3072, 34), (97, 8192, 3072, 34),
    (1579, 352, 12032, 33), (1631, 480, 9600, 33), (1806, 304, 3840, 33), (639, 1168, 3200, 33), (1848, 400, 1024, 33),
    (2280, 320, 1408, 33), (2048, 320, 1408, 33)])
def test_tiles_of_one_round(lib, M, N, K, want):
  for dtype in (F16, BF16, F32):
    if dtype != F32 or K > 1024:
      assert lib.cdit_debug_gemm_choice(0, M, N, K, dtype) == want


@pytest.mark.parametrize("M,N,K,want", [
    # fp32 outputs of short K
    (1848, 400, 1024, TILE32), (1107, 592, 384, TILE32), (96, 8192, 1024, TILE32), (97, 8192, 1024, 17), (2416, 288, 896, 17),
    (4608, 3072, 1024, 18)])
def test_fp32_outputs_of_short_k(lib, M, N, K, want):
  assert lib.cdit_debug_gemm_choice(0, M, N, K, F32) == want


@pytest.mark.parametrize("M,N,K,want", [
    # 32 x 32 tiles, and in place of 80 x 48 where no XCD has more than two of them per CU
    (35, 320, 384, 38), (35, 320, 512, 38), (49, 7072, 384, TILE32), (1440, 480, 512, 33), (1440, 480, 640, 33),
    (426, 1616, 512, 33), (52, 6704, 1408, TILE32), (102, 4096, 1280, TILE32), (52, 6704, 3200, 33), (67, 7552, 1152, 33), (49, 12032, 1152, 33),
    (773, 320, 384, 38), (632, 1216, 1280, 33), (2032, 256, 2688, 33), (2028, 256, 384, 26),
    # 128 x 96
    (1037, 2304, 512, 18), (2209, 1120, 1024, 18), (531, 4368, 512, 37), (361, 7936, 1280, 37), (494, 4576, 384, 37), (587, 3968, 384, 37),
    # 96 x 96 in place of one round of 64 x 128
    (838, 1984, 14720, 17), (178, 9216, 4480, 17), (1221, 1408, 13568, 17), (5283, 304, 2560, 36), (446, 4416, 7424, 36),
    (316, 5600, 14464, 36), (1163, 1648, 13568, 36), (1265, 1216, 5888, 36), (638, 2944, 6528, 36), (2959, 608, 3328, 17), (2600, 656, 1792, 36), (5283, 304, 5120, 36)])
def test_where_other_tiles_are_better(lib, M, N, K, want):
  for dtype in (F16, BF16, F32):
    if dtype != F32 or K > 1024:
      assert lib.cdit_debug_gemm_choice(0, M, N, K, dtype) == want


@pytest.mark.parametrize("M,N,K,want", [
    # a round of 256 x 192 tiles not in place of two of 64 x 128 for many rows, short K or columns in eights
    (5417, 736, 1408, 17), (1590, 2560, 1664, 17), (1069, 3648, 1152, 17), (277, 11264, 6528, 17), (409, 9120, 4736, 17),
    (447, 8880, 8832, 15), (1065, 3744, 6528, 15), (282, 12144, 11008, 15),
    # two of 128 x 128
    (361, 11184, 10752, 18), (374, 11120, 3840, 15)])
def test_fp16_and_fp32_outputs_of_two_rounds(lib, M, N, K, want):
  for dtype in (F16, F32):
    assert lib.cdit_debug_gemm_choice(0, M, N, K, dtype) == want


@pytest.mark.parametrize("M,N,K,want", [
    # 256 x 128 tiles between one round of 128 x 128 and two of 256 x 192, not in their place
    (1357, 4464, 2224, 19), (3261, 7280, 1040, 15), (5499, 3440, 1296, 15), (1678, 12080, 4000, 15), (947, 5216, 3728, 16),
    (2269, 7248, 1344, 16), (4608, 3072, 3056, 14), (256, 12288, 2992, 18)])
def test_tiles_for_k_remainders(lib, M, N, K, want):
  assert lib.cdit_debug_gemm_choice(0, M, N, K, BF16) == want


@pytest.mark.parametrize("M,N,K,want", [
    # tiles of which one round covers the problem
    (2257, 272, 15680, 25), (2346, 288, 3392, 25), (2277, 272, 1408, 25), (1738, 272, 2944, 25),
    (158, 4800, 14400, 12), (152, 4768, 6320, 12), (89, 2768, 12144, 13), (91, 3008, 10656, 23), (146, 3520, 11392, 25), (254, 2896, 7744, 26), (42, 11008, 9536, 25),
    (245, 2560, 1664, 25), (299, 2368, 3328, 26), (77, 3072, 4096, 21), (154, 5056, 2560, 26),
    # a round of 256 x 192 tiles or two of 128 x 128
    (616, 12224, 8064, 11), (1152, 6624, 11392, 11), (630, 12288, 4800, 8), (878, 6928, 13424, 8),
    # where other tiles are better than one round
    (94, 2752, 1216, 13), (94, 3008, 1216, 23), (124, 2752, 1216, 24), (254, 1152, 1056, 23), (103, 3008, 672, 13), (127, 3072, 4160, 24), (43, 6032, 2064, 13), (43, 6032, 4288, 23),
    (284, 976, 13104, 13), (200, 1968, 704, 24), (20, 8832, 1088, 13), (20, 8832, 2496, 24), (492, 1216, 1344, 25), (98, 5568, 1136, 13), (123, 6112, 1312, 26),
    (57, 8208, 1424, 26), (178, 8160, 14896, 12), (177, 6144, 13952, 12), (248, 5376, 6016, 27), (1051, 2336, 8304, 11),
    (1391, 1888, 5984, 29), (41, 5776, 9040, 13), (41, 5776, 9024, 23), (107, 3456, 2752, 24), (115, 3456, 2752, 24), (159, 5312, 14336, 12),
    (159, 5312, 4096, 26), (284, 6048, 13088, 28), (284, 6048, 13120, 28),
    (2489, 256, 1248, 25), (1626, 304, 816, 24), (1151, 256, 12976, 23), (282, 928, 4272, 13), (96, 2976, 896, 23),
    (1331, 2256, 576, 29),
    # shorter K
    (1524, 288, 256, 13), (53, 6016, 320, 13), (127, 5584, 192, 13),
    # up to 16 rows
    (5, 7952, 2944, 50), (5, 9216, 3072, 21), (6, 7952, 2944, 22), (16, 18432, 5120, 13), (16, 3072, 3072, 50),
    (2, 18432, 3072, 51), (1, 9216, 3072, 51), (16, 18432, 3136, 13)])
def test_weight_only(lib, M, N, K, want):
  assert lib.cdit_debug_gemm_choice(1, M, N, K, BF16) == want
