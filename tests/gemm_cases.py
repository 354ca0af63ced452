"""Shapes that steer the GEMM dispatcher into every kernel variant, shared by the CPU coverage test and the GPU
parity tests, plus the full-size shapes of the benchmark configurations.

A *variant* is one compiled code path: the kernel, its token-tile height, whether it writes split-K partial sums,
for the decode kernel how many 128-channel groups a workgroup walks, for the wave-split decode kernel how many waves
share a workgroup's K, whether a wave's share takes one turn of its four-slot register ring ("one_round") or several and
whether the workgroup owns one 16-channel tile or two, for the wave-split tile and the large-M kernels whether K ends on a
128-byte block.  `variant_of` maps a plan (sglang_amd._lib.gemm_plan) to such a key.
"""

# ---- FP8 (M, N, K); K % 16 != 0 means unaligned rows (byte-granular loader)
FP8_ROUTE_SHAPES = [
    # decode kernel (M <= 16, K % 128 == 0, N % 128 == 0): whole-K and split, 1 / 2 / 3+ channel groups per workgroup,
    # an uneven last workgroup (16640 = 130 groups), short last K ranges (4480 = 35 blocks, 2176 = 17 blocks)
    (1, 128, 128), (3, 256, 512), (16, 2048, 7168), (13, 18432, 7168), (13, 66560, 1152), (16, 16640, 4480), (15, 33280, 2176),
    (5, 66048, 512), (2, 133120, 384),
    # wave-split decode kernel (few tokens or a small weight, K of at least 8 blocks; N % 16 == 0 is enough): 8 waves with one
    # round (K = 4096) and two (K = 7168, 4480 = 35 blocks: a ragged second round), 4 waves with many rounds (K = 18432) and
    # with one (N % 128 != 0 at short K), ragged N (576, 1088), every token count class
    (1, 512, 4096), (4, 1536, 7168), (2, 7168, 2048), (2, 36864, 7168), (1, 512, 18432), (12, 48, 1152), (1, 512, 7168), (1, 16640, 4480),
    # ... and two channel tiles per workgroup (N / 32 >= 200 and three tokens or more, or K beyond 64 blocks): both wave counts,
    # one round and several, an uneven split of the K blocks over the waves (2176 = 17 blocks), N % 32 == 0 but N % 128 != 0
    (16, 7168, 2048), (9, 33280, 2176), (7, 16640, 4096), (7, 33280, 4096), (3, 36864, 7168), (6, 16640, 4480), (1, 7168, 18432), (16, 7168, 18432),
    (5, 6432, 1280),
    (5, 48, 128), (16, 16, 256),  # a single K block (three of the four waves have nothing to add), a single workgroup
    # three-stage mid-M kernel: 64 / 128 token tiles x 256 / 192 / 128 channel tiles, whole-K and split, ragged M, K blocks per
    # range = 1, 2, 0 mod 3
    (48, 16384, 2048), (33, 16384, 2176), (40, 65536, 512), (200, 16384, 2048), (100, 32768, 640), (130, 8192, 7168),
    (250, 8192, 7296), (100, 16384, 3584), (500, 4096, 14336),
    # the same kernel with 256-channel tiles and a K split (long K, many channels), and with 128-channel tiles
    (65, 7168, 18432), (24, 36864, 14336), (100, 36864, 640), (40, 4096, 7168), (300, 4096, 7168), (1000, 4096, 2048),
    (400, 4096, 16384), (100, 65536, 512), (130, 4096, 7168),
    # decode sizes on the mid-M kernel (4 .. 16 tokens, one round of unsplit tiles): instead of the wave-split kernel with
    # 192-channel tiles, instead of the split streaming kernel with 128- and 256-channel tiles
    (4, 36864, 7168), (13, 36864, 7168), (16, 24576, 1536), (14, 32768, 2048), (16, 49152, 2048),
    # K blocks left over after whole trips over the stages that no shape above has: 64 x 192 (four stages) 3; 128 x 128 (four) 2 and
    # 3; 128 x 192 and 128 x 256 (three) 0
    (20, 36864, 896), (100, 32768, 768), (100, 32768, 896), (100, 36864, 768), (300, 16384, 768),
    # small tiles with more workgroups than CUs: 64 x 192 and 128 x 128
    (135, 49152, 1024), (198, 36864, 1024),
    # 192-channel tiles (a wave's three channel tiles are 64 channels apart): whole-K and split, a ragged last tile
    (100, 36864, 512), (20, 36864, 1024), (130, 3072, 7168), (300, 3072, 14336), (130, 1000, 896),
    # 256 x 256 two-phase and 256 x 128 pipelined kernels, K a multiple of 128 and not
    # (the pipelined kernel is left K that is no multiple of 128: the mid-M and two-phase kernels take the rest)
    (4096, 4352, 512), (4000, 4300, 400), (4096, 2178, 256), (4000, 2100, 272), (4096, 2176, 256),
    # generic kernel: every token-tile height, aligned and byte-granular loads, whole-K and split
    (7, 1088, 512), (16, 576, 7168), (7, 1096, 512), (16, 584, 7168), (1, 1088, 3884), (17, 384, 2304), (20, 256, 264), (33, 512, 512), (64, 128, 3884),
    (50, 300, 520), (127, 128, 4096), (130, 640, 896), (1500, 640, 1000), (130, 200, 300), (2048, 4224, 264),
    # between 17 and 1024 tokens only K % 128 != 0 (or unaligned rows) leaves the mid-M kernel to the generic one
    (20, 256, 2064), (33, 256, 272), (100, 256, 400), (100, 640, 2064),
    # 128-channel tiles with a ragged last channel tile; a handful of channels; a single K block
    (50, 3000, 4224), (40, 8, 1024), (100, 16, 4096), (1000, 8, 128),
]

# ---- INT8 (M, N, K): the operator requires K % 16 == 0 and N % 8 == 0
INT8_ROUTE_SHAPES = [
    (16, 128, 512), (1, 6144, 4096), (1, 16640, 4480), (9, 33280, 2176), (16, 7168, 18432), (7, 33280, 4096),
    (5, 66048, 512), (2, 133120, 384),
    # a dozen tokens or more on the mid-M kernel where one round of unsplit 64-token tiles fills the chip (128- and 256-channel tiles)
    (16, 28672, 512), (13, 36864, 1024), (12, 24576, 2304), (8, 24576, 5760),  # (eight tokens where K has more than 44 blocks)
    (400, 6144, 896),  # 128 x 128 tiles (four stages) with three K blocks left after whole trips
    (20, 8192, 4096), (40, 65536, 512), (200, 16384, 2048), (200, 32768, 1024), (300, 4096, 14336), (130, 8192, 7168),
    (100, 16384, 3584), (500, 4096, 14336),
    # the mid-M kernel's 128-channel tiles (and 128 x 256 with a K split): ragged M, a ragged last channel tile
    (700, 6144, 14336), (100, 6144, 7168), (100, 28672, 512), (40, 6144, 14336), (20, 2048, 4096), (20, 4096, 1024),
    (33, 12288, 14336),  # 64 x 256 tiles with a K split
    # the 128 x 256 tile is the two-phase 128-token kernel: whole K and split, ragged M (200, 300, 700), K steps 0, 1, 2 mod 3
    (130, 8192, 1024), (250, 16384, 1152), (256, 28672, 4096),
    (50, 3000, 4224), (40, 8, 1024), (100, 16, 4096), (1000, 8, 128),
    (4096, 4096, 512), (4000, 4088, 1024),
    (1, 16, 512), (1, 24, 512), (3, 48, 1152), (5, 48, 128), (16, 16, 256), (17, 136, 1024), (64, 1024, 512), (100, 4096, 1024), (128, 16384, 512), (2048, 4224, 272),
    # between 17 and 1024 tokens only K % 128 != 0 leaves the mid-M kernel to the generic one
    (20, 256, 2064), (33, 256, 272), (100, 256, 400), (100, 640, 2064),
]

# ---- every variant that each of the four GEMMs runs, with a small shape that reaches it ("fp8": block scales, "fp8_ue8m0": packed
# exponents, "fp8_scaled": one scale per token and channel).  Found by asking the plan queries for 5.6 million random shapes
# of 1 .. 5000 tokens, N up to 320000 and K up to 19000; tests/test_gemm_routes_cpu.py checks that other random shapes add none.
VARIANT_SHAPES = {
    "fp8": {
        ("resident", "kb2"): (450, 16472, 256), ("resident", "kb3"): (452, 16528, 384), ("resident", "kb4"): (449, 16424, 512), ("resident", "kb5"): (450, 16504, 640), ("resident", "kb6"): (449, 16520, 768),
        ("decode", "split", "gpw1"): (13, 20864, 1536), ("decode", "split", "gpw3+"): (13, 66176, 1152),
        ("decode", "whole", "gpw1"): (1, 16512, 128), ("decode", "whole", "gpw2"): (1, 65664, 128),
        ("decode", "whole", "gpw3+"): (2, 133376, 128), ("decode_wavesplit", "w4", "one_round", "two_tiles"): (3, 6400, 1024),
        ("decode_wavesplit", "w4", "one_round"): (1, 16, 1024), ("decode_wavesplit", "w4", "rounds", "two_tiles"): (1, 7936, 17664),
        ("decode_wavesplit", "w4", "rounds"): (1, 10544, 13312), ("decode_wavesplit", "w8", "one_round", "two_tiles"): (3, 16512, 3840),
        ("decode_wavesplit", "w8", "one_round"): (1, 16512, 3840), ("decode_wavesplit", "w8", "rounds", "two_tiles"): (3, 12416, 8064),
        ("decode_wavesplit", "w8", "rounds"): (1, 13312, 7552), ("dma3", 128, "split", "bn128", "deep"): (2761, 8, 7424),
        ("dma3", 128, "split", "bn192"): (71, 8272, 12160), ("dma3", 128, "split"): (67, 8280, 13056),
        ("dma3", 128, "whole", "bn128", "deep"): (4238, 584, 512), ("dma3", 128, "whole", "bn192"): (97, 32896, 128),
        ("dma3", 128, "whole"): (289, 16408, 128), ("dma3", 160, "split", "bn128", "deep"): (2456, 8, 14080),
        ("dma3", 160, "split", "bn192"): (129, 11264, 11648), ("dma3", 160, "whole", "bn128", "deep"): (130, 24696, 128),
        ("dma3", 160, "whole", "bn192"): (129, 32896, 128), ("dma3", 192, "split", "bn128"): (4210, 8, 5504),
        ("dma3", 192, "whole", "bn128"): (484, 8344, 128), ("dma3", 256, "split", "bn128"): (4112, 264, 12800),
        ("dma3", 256, "whole", "bn128"): (641, 10760, 128), ("dma3", 64, "split", "bn128", "deep"): (674, 8, 14848),
        ("dma3", 64, "split", "bn128"): (1874, 8, 8576), ("dma3", 64, "split", "bn192", "deep"): (722, 264, 14208),
        ("dma3", 64, "split"): (1832, 200, 10240), ("dma3", 64, "whole", "bn128", "deep"): (49, 4112, 128),
        ("dma3", 64, "whole", "bn128"): (65, 16472, 128), ("dma3", 64, "whole", "bn192", "deep"): (17, 32880, 128),
        ("dma3", 64, "whole"): (129, 12832, 128), ("dma3", 96, "split", "bn128", "deep"): (1618, 8, 9472),
        ("dma3", 96, "split", "bn192", "deep"): (2893, 272, 8192), ("dma3", 96, "split"): (258, 4096, 10240),
        ("dma3", 96, "whole", "bn128", "deep"): (66, 25216, 384), ("dma3", 96, "whole", "bn192", "deep"): (65, 32896, 128),
        ("dma3", 96, "whole"): (194, 16518, 128), ("generic", 128, "aligned", "split"): (68, 8, 960),
        ("generic", 128, "aligned", "whole"): (66, 8, 16), ("generic", 128, "bytes", "split"): (68, 8, 1038),
        ("generic", 128, "bytes", "whole"): (65, 8, 26), ("generic", 16, "aligned", "split"): (1, 8, 912),
        ("generic", 16, "aligned", "whole"): (1, 8, 16), ("generic", 16, "bytes", "split"): (1, 8, 907),
        ("generic", 16, "bytes", "whole"): (1, 8, 17), ("generic", 256, "aligned", "split"): (1052, 6688, 928),
        ("generic", 256, "bytes", "split"): (1114, 7024, 922), ("generic", 256, "bytes", "whole"): (1025, 6792, 17),
        ("generic", 32, "aligned", "split"): (17, 8, 960), ("generic", 32, "aligned", "whole"): (17, 8, 32),
        ("generic", 32, "bytes", "split"): (20, 8, 983), ("generic", 32, "bytes", "whole"): (17, 8, 18),
        ("generic", 64, "aligned", "split"): (33, 8, 912), ("generic", 64, "aligned", "whole"): (33, 8, 32),
        ("generic", 64, "bytes", "split"): (39, 8, 941), ("generic", 64, "bytes", "whole"): (33, 8, 18),
        ("pingpong", "kfull"): (223, 49272, 128), ("pingpong", "ktail"): (1323, 11460, 16), ("pipelined", "ktail"): (1094, 6576, 16),
        ("wavesplit_tile", 16, 8, "kfull"): (5, 1120, 8320), ("wavesplit_tile", 16, 16, "kfull"): (17, 8, 128), ("wavesplit_tile", 16, 32, "kfull"): (97, 579, 128),
        ("wavesplit_tile", 16, 64, "kfull"): (65, 2728, 128), ("wavesplit_tile", 32, 16, "kfull"): (81, 680, 128),
        ("wavesplit_tile", 32, 32, "kfull"): (49, 2064, 128), ("wavesplit_tile", 32, 64, "kfull"): (49, 4137, 128),
        ("wavesplit_tile", 48, 16, "kfull"): (194, 616, 128), ("wavesplit_tile", 48, 32, "kfull"): (193, 1223, 128),
        ("wavesplit_tile", 64, 32, "kfull"): (49, 4358, 128), ("wavesplit_tile", 64, 64, "kfull"): (1637, 291, 512),
    },
    "fp8_ue8m0": {
        ("resident", "kb2"): (450, 16472, 256), ("resident", "kb3"): (452, 16528, 384), ("resident", "kb4"): (449, 16424, 512), ("resident", "kb5"): (450, 16504, 640), ("resident", "kb6"): (449, 16520, 768),
        ("decode", "split", "gpw1"): (13, 20864, 1536), ("decode", "split", "gpw3+"): (13, 66176, 1152),
        ("decode", "whole", "gpw1"): (1, 16512, 128), ("decode", "whole", "gpw2"): (1, 65664, 128),
        ("decode", "whole", "gpw3+"): (2, 133376, 128), ("decode_wavesplit", "w4", "one_round", "two_tiles"): (3, 6400, 1024),
        ("decode_wavesplit", "w4", "one_round"): (1, 16, 1024),
         ("decode_wavesplit", "w8", "one_round", "two_tiles"): (3, 16512, 3840),
        ("decode_wavesplit", "w8", "one_round"): (1, 16512, 3840),
         ("dma3", 128, "split", "bn128", "deep"): (2761, 8, 7424),
        ("dma3", 128, "split", "bn192"): (71, 8272, 12160), ("dma3", 128, "split"): (67, 8280, 13056),
        ("dma3", 128, "whole", "bn128", "deep"): (4238, 584, 512), ("dma3", 128, "whole", "bn192"): (97, 32896, 128),
        ("dma3", 128, "whole"): (289, 16408, 128), ("dma3", 160, "split", "bn128", "deep"): (2456, 8, 14080),
        ("dma3", 160, "split", "bn192"): (129, 11264, 11648), ("dma3", 160, "whole", "bn128", "deep"): (130, 24696, 128),
        ("dma3", 160, "whole", "bn192"): (129, 32896, 128), ("dma3", 192, "split", "bn128"): (4210, 8, 5504),
        ("dma3", 192, "whole", "bn128"): (484, 8344, 128), ("dma3", 256, "split", "bn128"): (4112, 264, 12800),
        ("dma3", 256, "whole", "bn128"): (641, 10760, 128), ("dma3", 64, "split", "bn128", "deep"): (674, 8, 14848),
        ("dma3", 64, "split", "bn128"): (1874, 8, 8576), ("dma3", 64, "split", "bn192", "deep"): (722, 264, 14208),
        ("dma3", 64, "split"): (1832, 200, 10240), ("dma3", 64, "whole", "bn128", "deep"): (49, 4112, 128),
        ("dma3", 64, "whole", "bn128"): (65, 16472, 128), ("dma3", 64, "whole", "bn192", "deep"): (17, 32880, 128),
        ("dma3", 64, "whole"): (129, 12832, 128), ("dma3", 96, "split", "bn128", "deep"): (1618, 8, 9472),
        ("dma3", 96, "split", "bn192", "deep"): (2893, 272, 8192), ("dma3", 96, "split"): (258, 4096, 10240),
        ("dma3", 96, "whole", "bn128", "deep"): (66, 25216, 384), ("dma3", 96, "whole", "bn192", "deep"): (65, 32896, 128),
        ("dma3", 96, "whole"): (194, 16518, 128), ("generic", 16, "aligned", "split", "unpacked"): (1, 8, 1024),
        ("generic", 16, "aligned", "whole", "unpacked"): (1, 8, 128), ("pingpong", "kfull"): (223, 49272, 128),
        ("wavesplit_tile", 16, 8, "kfull"): (5, 1120, 8320), ("wavesplit_tile", 16, 16, "kfull"): (17, 8, 128), ("wavesplit_tile", 16, 32, "kfull"): (97, 579, 128),
        ("wavesplit_tile", 16, 64, "kfull", "unpacked"): (7, 12824, 7808), ("wavesplit_tile", 16, 64, "kfull"): (65, 2728, 128),
        ("wavesplit_tile", 32, 16, "kfull"): (81, 680, 128), ("wavesplit_tile", 32, 32, "kfull"): (49, 2064, 128),
        ("wavesplit_tile", 32, 64, "kfull"): (49, 4137, 128), ("wavesplit_tile", 48, 16, "kfull"): (194, 616, 128),
        ("wavesplit_tile", 48, 32, "kfull"): (193, 1223, 128), ("wavesplit_tile", 64, 32, "kfull"): (49, 4358, 128),
        ("wavesplit_tile", 64, 64, "kfull"): (1637, 291, 512),
    },
    "fp8_scaled": {
        ("resident", "kb2"): (481, 16904, 256), ("resident", "kb3"): (484, 16496, 384), ("resident", "kb4"): (486, 16760, 512), ("resident", "kb5"): (486, 16584, 640), ("resident", "kb6"): (513, 16392, 768),
        ("decode", "split", "gpw1"): (13, 20864, 1536), ("decode", "split", "gpw3+"): (13, 66176, 1152),
        ("decode", "whole", "gpw1"): (1, 16512, 128), ("decode", "whole", "gpw2"): (1, 65664, 128),
        ("decode", "whole", "gpw3+"): (2, 133376, 128), ("decode_wavesplit", "w4", "one_round", "two_tiles"): (3, 6400, 1024),
        ("decode_wavesplit", "w4", "one_round"): (1, 16, 1024),
         ("decode_wavesplit", "w8", "one_round", "two_tiles"): (3, 16512, 3840),
        ("decode_wavesplit", "w8", "one_round"): (1, 16512, 3840),
         ("dma3", 128, "split", "bn128", "deep"): (3348, 8, 6272),
        ("dma3", 128, "split", "bn192"): (71, 8272, 12160), ("dma3", 128, "split"): (67, 8280, 13056),
        ("dma3", 128, "whole", "bn128", "deep"): (194, 12416, 640), ("dma3", 128, "whole", "bn192"): (194, 16528, 128),
        ("dma3", 128, "whole"): (196, 24704, 128), ("dma3", 160, "split", "bn128", "deep"): (2716, 8, 10752),
        ("dma3", 160, "split", "bn192"): (313, 5480, 18432), ("dma3", 160, "whole", "bn128", "deep"): (130, 24696, 128),
        ("dma3", 160, "whole", "bn192"): (289, 16408, 128), ("dma3", 192, "split", "bn128"): (4174, 8, 15488),
        ("dma3", 192, "whole", "bn128"): (161, 24608, 128), ("dma3", 256, "split", "bn128"): (211, 8312, 17664),
        ("dma3", 256, "whole", "bn128"): (4677, 1544, 128), ("dma3", 64, "split", "bn128", "deep"): (674, 8, 14848),
        ("dma3", 64, "split", "bn128"): (2462, 8, 6528), ("dma3", 64, "split", "bn192", "deep"): (871, 280, 11648),
        ("dma3", 64, "split"): (17, 17024, 8320), ("dma3", 64, "whole", "bn128", "deep"): (194, 616, 128),
        ("dma3", 64, "whole", "bn128"): (65, 16472, 128), ("dma3", 64, "whole", "bn192", "deep"): (17, 32880, 128),
        ("dma3", 64, "whole"): (17, 57344, 512), ("dma3", 96, "split", "bn128", "deep"): (3334, 8, 5248),
        ("dma3", 96, "split", "bn192", "deep"): (2958, 264, 9344), ("dma3", 96, "split"): (263, 4136, 16640),
        ("dma3", 96, "whole", "bn128", "deep"): (65, 18944, 512), ("dma3", 96, "whole", "bn192", "deep"): (65, 32896, 128),
        ("dma3", 96, "whole"): (261, 16488, 128), ("generic", 128, "aligned", "split"): (65, 6016, 16688),
        ("generic", 128, "aligned", "whole"): (708, 2816, 16), ("generic", 16, "aligned", "split"): (1, 8, 1024),
        ("generic", 16, "aligned", "whole"): (1, 8, 128),
        ("generic", 32, "aligned", "split"): (17, 9656, 10480), ("generic", 32, "aligned", "whole"): (26, 50944, 16),
        ("generic", 64, "aligned", "split"): (33, 6016, 16688), ("generic", 64, "aligned", "whole"): (34, 33648, 16),
        ("pingpong", "kfull"): (193, 49640, 128), ("pingpong", "ktail"): (1555, 9984, 16), ("pipelined", "ktail"): (1094, 6576, 16),
        ("wavesplit_tile", 16, 8, "kfull"): (5, 1120, 8320), ("wavesplit_tile", 16, 16, "kfull"): (17, 8, 128), ("wavesplit_tile", 16, 16, "ktail"): (1, 8, 16),
        ("wavesplit_tile", 16, 32, "kfull"): (129, 456, 128), ("wavesplit_tile", 16, 32, "ktail"): (100, 592, 16),
        ("wavesplit_tile", 16, 64, "kfull"): (33, 4104, 384), ("wavesplit_tile", 16, 64, "ktail"): (172, 1352, 16),
        ("wavesplit_tile", 32, 16, "kfull"): (81, 680, 128), ("wavesplit_tile", 32, 16, "ktail"): (85, 712, 16),
        ("wavesplit_tile", 32, 32, "kfull"): (50, 2104, 384), ("wavesplit_tile", 32, 32, "ktail"): (100, 1408, 16),
        ("wavesplit_tile", 32, 64, "kfull"): (17, 8320, 768), ("wavesplit_tile", 32, 64, "ktail"): (195, 1664, 16),
        ("wavesplit_tile", 48, 16, "kfull"): (193, 616, 256), ("wavesplit_tile", 48, 16, "ktail"): (162, 768, 16),
        ("wavesplit_tile", 48, 32, "kfull"): (903, 272, 512), ("wavesplit_tile", 48, 32, "ktail"): (199, 1224, 16),
        ("wavesplit_tile", 64, 32, "kfull"): (53, 4240, 896), ("wavesplit_tile", 64, 32, "ktail"): (248, 1432, 16),
        ("wavesplit_tile", 64, 64, "kfull"): (1816, 264, 2176), ("wavesplit_tile", 64, 64, "ktail"): (323, 1536, 16),
    },
    "int8": {
        ("resident", "kb2"): (481, 16904, 256), ("resident", "kb3"): (484, 16496, 384), ("resident", "kb4"): (486, 16760, 512), ("resident", "kb5"): (542, 16592, 640), ("resident", "kb6"): (577, 20496, 768),
        ("decode", "whole", "gpw1"): (1, 16512, 128), ("decode", "whole", "gpw2"): (1, 65664, 128),
        ("decode", "whole", "gpw3+"): (2, 133376, 128), ("decode_wavesplit", "w4", "one_round"): (1, 16, 1024),
         ("decode_wavesplit", "w8", "one_round"): (1, 16512, 3840),
         ("dma3", 128, "split", "bn128", "deep"): (2796, 8, 5760),
        ("dma3", 128, "split", "bn192"): (198, 5448, 12288), ("dma3", 128, "split"): (329, 4352, 18560),
        ("dma3", 128, "whole", "bn128", "deep"): (194, 12416, 640), ("dma3", 128, "whole", "bn192"): (194, 16528, 128),
        ("dma3", 128, "whole"): (1295, 10760, 128), ("dma3", 160, "split", "bn128", "deep"): (2456, 8, 14080),
        ("dma3", 160, "split", "bn192"): (313, 5480, 18432), ("dma3", 160, "whole", "bn128", "deep"): (130, 24696, 128),
        ("dma3", 160, "whole", "bn192"): (289, 16408, 128), ("dma3", 192, "split", "bn128"): (3076, 264, 16640),
        ("dma3", 192, "whole", "bn128"): (484, 8344, 128), ("dma3", 256, "split", "bn128"): (208, 8568, 16512),
        ("dma3", 256, "whole", "bn128"): (4677, 1544, 128), ("dma3", 64, "split", "bn128", "deep"): (674, 8, 14848),
        ("dma3", 64, "split", "bn128"): (2462, 8, 6528), ("dma3", 64, "split", "bn192", "deep"): (792, 136, 17280),
        ("dma3", 64, "split"): (17, 5848, 17408), ("dma3", 64, "whole", "bn128", "deep"): (194, 616, 128),
        ("dma3", 64, "whole", "bn128"): (65, 16472, 128), ("dma3", 64, "whole", "bn192", "deep"): (17, 33280, 512),
        ("dma3", 64, "whole"): (12, 33096, 128), ("dma3", 96, "split", "bn128", "deep"): (1606, 8, 12928),
        ("dma3", 96, "split", "bn192", "deep"): (2958, 264, 9344), ("dma3", 96, "split"): (263, 4136, 16640),
        ("dma3", 96, "whole", "bn128", "deep"): (65, 18944, 512), ("dma3", 96, "whole", "bn192", "deep"): (65, 32896, 128),
        ("dma3", 96, "whole"): (389, 10904, 128), ("generic", 128, "aligned", "split"): (65, 6016, 16688),
        ("generic", 128, "aligned", "whole"): (708, 2816, 16), ("generic", 16, "aligned", "split"): (1, 8, 1024),
        ("generic", 16, "aligned", "whole"): (1, 8, 128),
        ("generic", 256, "aligned", "whole"): (1094, 6576, 16), ("generic", 32, "aligned", "split"): (17, 9656, 10480),
        ("generic", 32, "aligned", "whole"): (26, 50944, 16), ("generic", 64, "aligned", "split"): (33, 6016, 16688),
        ("generic", 64, "aligned", "whole"): (34, 33648, 16), ("pingpong", "kfull"): (223, 49272, 128),
        ("pingpong128", "whole"): (196, 24704, 128), ("wavesplit_tile", 16, 8, "kfull"): (5, 1120, 8320), ("wavesplit_tile", 16, 16, "kfull"): (17, 8, 128),
        ("wavesplit_tile", 16, 16, "ktail"): (1, 8, 16), ("wavesplit_tile", 16, 32, "kfull"): (129, 456, 128),
        ("wavesplit_tile", 16, 32, "ktail"): (100, 592, 16), ("wavesplit_tile", 16, 64, "kfull"): (33, 4104, 384),
        ("wavesplit_tile", 16, 64, "ktail"): (172, 1352, 16), ("wavesplit_tile", 32, 16, "kfull"): (81, 680, 128),
        ("wavesplit_tile", 32, 16, "ktail"): (85, 712, 16), ("wavesplit_tile", 32, 32, "kfull"): (50, 2104, 384),
        ("wavesplit_tile", 32, 32, "ktail"): (100, 1408, 16), ("wavesplit_tile", 32, 64, "kfull"): (17, 8320, 768),
        ("wavesplit_tile", 32, 64, "ktail"): (195, 1664, 16), ("wavesplit_tile", 48, 16, "kfull"): (193, 616, 256),
        ("wavesplit_tile", 48, 16, "ktail"): (162, 768, 16), ("wavesplit_tile", 48, 32, "kfull"): (903, 272, 512),
        ("wavesplit_tile", 48, 32, "ktail"): (199, 1224, 16), ("wavesplit_tile", 64, 32, "kfull"): (53, 4240, 896),
        ("wavesplit_tile", 64, 32, "ktail"): (248, 1432, 16), ("wavesplit_tile", 64, 64, "kfull"): (1816, 264, 2176),
        ("wavesplit_tile", 64, 64, "ktail"): (323, 1536, 16),
    },
}
# Shapes that ran the register wave-split kernel in several turns or the streaming kernel before the wave-split tile took them over: one to
# three K blocks for its eight waves, 16 and 128 channels, and the weights from 100 million on
TAKEN_OVER_SHAPES = [(1, 16, 128), (1, 128, 128), (3, 6432, 128), (2, 48, 256), (16, 272, 384), (9, 128, 1152), (1, 7936, 17664), (1, 10544, 13312),
                     (3, 12416, 8064), (1, 13312, 7552)]
FP8_REQUIRED_VARIANTS = set(VARIANT_SHAPES["fp8"])
INT8_REQUIRED_VARIANTS = set(VARIANT_SHAPES["int8"])

# The mid-M tiles run a ring of LDS stages over the K blocks: (M, N) at which K alone does not move an unsplit tile away for every
# remainder of the K blocks over its stages.  (tile, stages) -> (M, N)
MID_TILE_SWEEPS = {
    "fp8": {(64, 128, 3): (97, 24584), (64, 128, 6): (33, 8392), (64, 192, 4): (17, 32816), (64, 256, 3): (129, 13232), (96, 128, 5): (65, 24744), (96, 192, 4): (67, 32824), (96, 256, 3): (258, 16632), (128, 128, 4): (97, 24584), (128, 192, 3): (97, 33024), (128, 256, 3): (290, 16848), (160, 128, 4): (132, 25544), (160, 192, 3): (131, 33032), (192, 128, 3): (322, 12296), (256, 128, 3): (652, 10768)},
    "fp8_scaled": {(64, 128, 3): (65, 16520), (64, 128, 6): (49, 4232), (64, 192, 4): (17, 32816), (64, 256, 3): (129, 18672), (96, 128, 5): (65, 18584), (96, 192, 4): (67, 32824), (96, 256, 3): (258, 16632), (128, 128, 4): (97, 24584), (128, 192, 3): (97, 33024), (128, 256, 3): (195, 25208), (160, 128, 4): (132, 25544), (160, 192, 3): (131, 33032), (192, 128, 3): (165, 24840), (256, 128, 3): (1163, 6432)},
    "int8": {(64, 128, 3): (17, 32816), (64, 128, 6): (49, 4232), (64, 192, 4): (17, 32816), (64, 256, 3): (17, 36832), (96, 128, 5): (65, 18584), (96, 192, 4): (67, 32824), (96, 256, 3): (258, 16632), (128, 128, 4): (97, 24584), (128, 192, 3): (97, 33024), (128, 256, 3): (1312, 10760), (160, 128, 4): (132, 25544), (160, 192, 3): (131, 33032), (192, 128, 3): (322, 12296), (256, 128, 3): (1163, 6432)},
}

# ---- what the one-call linears do: (quantizer, kernel, channel tile of a fused or wave-split kernel, waves or channel groups, K split),
# with a shape that reaches it; where a kind is not named, all of "block", "ue8m0", "token_fp8" and "int8" do it there
LINEAR_SHAPES = [(1, 128, 128), (15, 128, 1408), (8, 34176, 1536), (2, 18432, 7424), (1, 16, 1024), (1, 29104, 3456), (3, 6400, 1024), (3, 28288, 3584),
                 (13, 25728, 1280), (2, 22400, 6784), (13, 33024, 1152), (2, 33216, 7168), (13, 49536, 1152), (1, 16, 2176), (2, 4144, 2176),
                 (9, 8320, 1024), (1, 16, 128), (4, 12528, 8064), (3, 6720, 128), (3, 13760, 7424), (16, 16, 2688), (16, 4336, 2688),
                 (15, 8336, 2816), (1, 8320, 128), (15, 16, 1280), (12, 16896, 128), (5, 4864, 28800), (3, 14208, 7168), (9, 128, 1152), (17, 16, 128),
                 (1, 8, 128), (1, 8, 1024), (1, 66304, 128), (5, 27904, 8192), (3, 78208, 256), (1, 131328, 128), (11, 16, 1920), (2, 23872, 3840),
                 (2, 33472, 4096), (1, 80768, 3328), (3, 17408, 3840), (5, 17920, 3840), (13, 20864, 1536), (13, 65664, 1152), (1, 16512, 128),
                 (7, 32512, 1792), (15, 28160, 1024), (5, 19392, 4096),
                 (17, 2816, 7168), (15, 2104, 2816), (3, 256, 6400), (12, 136, 15872)]
# Above decode sizes, the wave-split tiles that quantize their tokens: (tokens x channels, whether a thread has more than four pieces of eight
# values, five with 32 tokens), each with a last tile of a few tokens or channels; some of the four linears run the tile named
QUANT_TILE_SHAPES = {((16, 16), False): (143, 24, 640), ((16, 16), True): (49, 16, 1664), ((16, 32), False): (83, 688, 640),
                     ((16, 32), True): (76, 968, 1408), ((16, 64), False): (54, 2656, 384), ((16, 64), True): (110, 1168, 1152),
                     ((32, 32), False): (21, 5200, 896), ((32, 32), True): (18, 7064, 1152), ((32, 64), False): (139, 2304, 640),
                     ((32, 64), True): (23, 9392, 896)}
# Grouped calls by the rows of each expert: (name, rows, N, K, small tile that runs)
GROUPED_SHAPES = [
    ("decode_like", [1, 0, 3, 1, 0, 0, 2, 8, 1, 1, 0, 5, 16, 1, 2, 1], 512, 7168, "16x64"),
    ("one_token", [1], 256, 128, "16x16"),
    ("empty_experts_around_a_big_one", [0, 0, 700, 0, 1, 0], 384, 512, "32x64"),
    ("prefill_like", [130, 257, 128, 64, 511, 129, 300, 200], 768, 1024, "64x128"),
    ("tile_edges", [64, 65, 63, 128, 127, 129, 1, 256], 256, 256, "16x64"),
    ("many_small", [3] * 300, 128, 256, "64x128"),
    ("large_experts", [1000, 513, 384, 2], 512, 512, "64x128"),
    ("ragged_channels", [40, 90, 17], 200, 384, "16x16"),
    ("decode_like_wide", [1, 0, 3, 1, 0, 0, 2, 8, 1, 1, 0, 5, 16, 1, 2, 1], 1664, 7168, "64x128"),
    ("empty_experts_around_a_big_one_wide", [0, 0, 700, 0, 1, 0], 1280, 512, "64x128"),
    ("tile_edges_wide", [64, 65, 63, 128, 127, 129, 1, 256], 1024, 256, "64x256"),
    ("large_experts_wide", [1000, 513, 384, 2], 640, 512, "64x128"),
    ("ragged_channels_wide", [40, 90, 17], 4424, 384, "64x128"),
]
# Grouped calls: experts (uneven: some without a row, one with many), stacked rows, N, K, and the kernel and small tile that run
GROUPED_FORMS = [
    (40, 1240, 2056, 128, "grouped_dma3", "64x256"), (2, 3254, 328, 384, "grouped_dma3", "64x128"),
    (16, 16, 64, 384, "grouped_wavesplit", "16x16"), (8, 209, 416, 128, "grouped_wavesplit", "16x32"), (40, 29, 392, 1152, "grouped_wavesplit", "16x64"),
    (5, 56, 1240, 128, "grouped_wavesplit", "32x32"), (40, 492, 272, 128, "grouped_wavesplit", "32x64"), (40, 1798, 136, 128, "grouped_wavesplit", "64x64"),
    (24, 1574, 128, 128, "grouped_wavesplit", "16x64"), (16, 1613, 224, 128, "grouped_wavesplit", "64x64"), (3, 545, 1544, 1152, "grouped_dma3", "64x128"),
    (40, 29, 2056, 128, "grouped_dma3", "64x128"),  # (more workgroups than CUs: two share one)
    (24, 1233, 2056, 384, "grouped_dma3", "128x256"), (16, 2075, 2056, 384, "grouped_dma3", "128x256"),
    (1, 1695, 2056, 640, "grouped_dma3", "128x128"), (24, 3078, 768, 2048, "grouped_dma3", "128x128"),
    (2, 5548, 2056, 384, "grouped_pingpong+grouped_dma3", "128x256")]

# K in parts of blocks (one scale per token and channel, INT8): (shape, mid-M tile and LDS stages that run), every tile from three blocks on,
# fewer blocks than stages among them; and K of two blocks
RAGGED_TILE_SHAPES = [
    ((17, 17208, 272), (64, 128, 6)), ((17, 36192, 272), (64, 128, 3)), ((17, 36192, 400), (64, 192, 4)), ((33, 17208, 656), (64, 128, 6)),
    ((20, 16392, 6160), (64, 128, 6)), ((17, 45656, 304), (64, 192, 4)), ((396, 8888, 1456), (64, 256, 3)), ((71, 18736, 400), (96, 128, 5)),
    ((70, 33408, 272), (96, 192, 4)), ((272, 16456, 288), (96, 256, 3)), ((97, 24888, 928), (128, 128, 4)), ((207, 17048, 288), (128, 192, 3)),
    ((215, 25152, 272), (128, 256, 3)), ((133, 24744, 352), (160, 128, 4)), ((136, 35040, 272), (160, 192, 3)), ((331, 12432, 368), (192, 128, 3)),
    ((667, 10824, 272), (256, 128, 3)),
    ((3275, 528, 240), (64, 128, 3)), ((2002, 400, 176), (64, 128, 6)), ((1802, 2192, 144), (96, 192, 4)), ((389, 10920, 208), (96, 256, 3)),
    ((193, 16752, 240), (128, 192, 3)), ((3051, 2344, 192), (128, 256, 3)), ((3471, 1168, 160), (160, 128, 4)), ((3703, 1560, 160), (160, 192, 3)),
    ((490, 8408, 224), (192, 128, 3)), ((3279, 2336, 144), (256, 128, 3)),
]
# The same on weights of 100 million bytes and more whose rows lie a multiple of 128 bytes apart all the same: loaded as a stream.  (shape,
# kernel and its tile)
STREAMED_RAGGED_SHAPES = [
    ((14, 23168, 4320), ("dma3", 64, 128)), ((25, 32224, 3104), ("dma3", 64, 128)), ((10, 46304, 2160), ("dma3", 64, 192)),
    ((33, 35752, 2800), ("dma3", 64, 192)), ((2, 57024, 1760), ("dma3", 64, 256)), ((50, 53480, 1872), ("dma3", 64, 256)),
    ((2, 9080, 11088), ("wavesplit_tile", 16, 16)), ((6, 18664, 5360), ("wavesplit_tile", 16, 32)), ((2, 16032, 6240), ("wavesplit_tile", 16, 64)),
]

# Every kernel of the wave-split tile that quantizes its tokens: (kinds, tokens x channels of the tile, at most so many pieces of eight values a
# thread, K in whole blocks or in parts, weights cached or of 100 million bytes and more, which are loaded as a stream), and a shape.
# (K in parts streams where the rows' pitch is a multiple of 128 all the same.)
QUANT_TILE_KERNELS = [
    ("token_fp8 int8", 16, 16, 2, "parts", "cached", (17, 40, 48)),
    ("token_fp8 int8", 16, 16, 4, "parts", "cached", (18, 40, 528)),
    ("token_fp8 int8", 16, 16, 10, "parts", "cached", (18, 40, 1088)),
    ("token_fp8 int8", 16, 32, 2, "parts", "cached", (50, 1032, 48)),
    ("token_fp8 int8", 16, 32, 4, "parts", "cached", (173, 392, 544)),
    ("token_fp8 int8", 16, 32, 10, "parts", "cached", (133, 464, 1104)),
    ("token_fp8 int8", 16, 64, 2, "parts", "cached", (162, 760, 144)),
    ("token_fp8 int8", 16, 64, 4, "parts", "cached", (199, 656, 528)),
    ("token_fp8 int8", 16, 64, 10, "parts", "cached", (257, 496, 1040)),
    ("token_fp8 int8", 32, 32, 5, "parts", "cached", (66, 1688, 48)),
    ("token_fp8 int8", 32, 32, 10, "parts", "cached", (401, 600, 656)),
    ("token_fp8 int8", 32, 64, 5, "parts", "cached", (98, 2312, 48)),
    ("block ue8m0 token_fp8 int8", 16, 8, 2, "whole", "cached", (2, 40, 3072)),
    ("block ue8m0 token_fp8 int8", 16, 8, 4, "whole", "cached", (3, 2040, 3200)),
    ("block ue8m0 token_fp8 int8", 16, 8, 10, "whole", "cached", (5, 200, 3328)),
    ("block ue8m0 token_fp8 int8", 16, 16, 2, "whole", "cached", (17, 40, 128)),
    ("block ue8m0 token_fp8 int8", 16, 16, 4, "whole", "cached", (17, 40, 640)),
    ("block ue8m0 token_fp8 int8", 16, 16, 10, "whole", "cached", (18, 40, 1152)),
    ("block ue8m0 token_fp8 int8", 16, 32, 2, "whole", "cached", (114, 520, 128)),
    ("block ue8m0 token_fp8 int8", 16, 32, 4, "whole", "cached", (133, 456, 640)),
    ("block ue8m0 token_fp8 int8", 16, 32, 10, "whole", "cached", (131, 456, 1152)),
    ("block ue8m0 token_fp8 int8", 16, 64, 2, "whole", "cached", (194, 624, 256)),
    ("block ue8m0 token_fp8 int8", 16, 64, 4, "whole", "cached", (227, 552, 640)),
    ("block ue8m0 token_fp8 int8", 16, 64, 10, "whole", "cached", (217, 616, 1152)),
    ("block ue8m0 token_fp8 int8", 32, 32, 5, "whole", "cached", (307, 400, 128)),
    ("block ue8m0 token_fp8 int8", 32, 32, 10, "whole", "cached", (371, 664, 768)),
    ("block ue8m0 token_fp8 int8", 32, 64, 5, "whole", "cached", (194, 1256, 640)),
    ("block ue8m0", 32, 64, 10, "whole", "cached", (300, 840, 768)),
    ("token_fp8 int8", 16, 16, 4, "parts", "streamed", (1, 9640, 10864)),
    ("token_fp8 int8", 16, 32, 2, "parts", "streamed", (1, 17040, 5920)),
    ("token_fp8 int8", 16, 32, 4, "parts", "streamed", (1, 7192, 13936)),
    ("token_fp8 int8", 16, 32, 10, "parts", "streamed", (2, 6920, 14624)),
    ("token_fp8 int8", 16, 64, 2, "parts", "streamed", (3, 69552, 1440)),
    ("token_fp8 int8", 16, 64, 4, "parts", "streamed", (1, 11160, 9072)),
    ("token_fp8 int8", 16, 64, 10, "parts", "streamed", (2, 11312, 8880)),
    ("block ue8m0 token_fp8 int8", 16, 32, 2, "whole", "streamed", (1, 16848, 6912)),
    ("block ue8m0 token_fp8 int8", 16, 32, 4, "whole", "streamed", (1, 7600, 13312)),
    ("block ue8m0 token_fp8 int8", 16, 32, 10, "whole", "streamed", (2, 7448, 13440)),
    ("block ue8m0 token_fp8 int8", 16, 64, 2, "whole", "streamed", (3, 39064, 2560)),
    ("block ue8m0 token_fp8 int8", 16, 64, 4, "whole", "streamed", (3, 20616, 4864)),
    ("block ue8m0 token_fp8 int8", 16, 64, 10, "whole", "streamed", (2, 8592, 11648)),
    ("block ue8m0 token_fp8 int8", 16, 16, 4, "whole", "streamed", (1, 11184, 13312)),
    ("block ue8m0 token_fp8 int8", 16, 16, 10, "whole", "streamed", (1, 2504, 40576)), ("token_fp8 int8", 16, 16, 10, "parts", "streamed", (1, 3760, 27040)),
]
# Linears that quantize their tokens in the one launch when they are called eagerly, and the launches of a captured call: (linear, shape, launches).
# us in a graph with one launch and with two:
CAPTURED_LINEARS = [
    ("ue8m0", (173, 256, 2048), 2),  # 6.7, 5.5
    ("ue8m0", (185, 640, 1536), 2),  # 6.6, 5.65
    ("int8", (121, 384, 1536), 2),  # 6.5, 5.6
    ("block", (48, 768, 2048), 2),  # 6.6, 5.8
    ("token_fp8", (168, 768, 1280), 2),  # 7.0, 6.0
    ("block", (46, 512, 1280), 1),  # 5.1, 5.3
    ("ue8m0", (669, 384, 640), 1),  # 4.3, 6.8
    ("token_fp8", (69, 384, 768), 1),  # 4.2, 5.3
    ("int8", (103, 768, 768), 1),  # 4.35, 5.6
    ("block", (89, 2560, 1024), 1),  # 5.5, 5.7
    # K in parts of blocks at decode sizes
    ("int8", (13, 1152, 2784), 2),  # 7.6, 6.3
    ("int8", (9, 640, 4384), 2),  # 7.9, 6.7
    ("token_fp8", (15, 640, 2016), 2),  # 6.25, 5.6
    ("int8", (3, 768, 10432), 1),  # 8.8, 9.4
    ("token_fp8", (4, 6016, 8352), 1),  # 16.3, 17.1
    ("int8", (14, 8320, 1504), 1),  # 7.8, 7.8
]
QUANT_PIECES = {16: (2, 4, 10), 32: (5, 10)}  # by the tile's tokens


def quant_tile_kernel(plan: dict, M: int, N: int, K: int, padded: bool = True):
    """The kernel of QUANT_TILE_KERNELS that a linear with this plan runs, None where its tokens are quantized elsewhere."""
    if plan["quantizer"] != "fused" or plan["kernel"] != "wavesplit_tile":
        return None
    pieces = -(-min(M, plan["bm"]) * -(-K // 128) * 16 // 512)
    streams = plan["bm"] >= M and M <= 16 and N * K >= 1e8 and (padded or K % 128 == 0)
    return (plan["bm"], plan["bn"], next(p for p in QUANT_PIECES[plan["bm"]] if pieces <= p), "parts" if K % 128 else "whole",
            "streamed" if streams else "cached")


def linear_variant_of(plan: dict, M: int):
    if M > 16:
        return (plan["quantizer"], "above decode sizes")
    k, fused = plan["kernel"], plan["quantizer"] == "fused"
    return (plan["quantizer"], k, plan["bn"] if fused or k in ("wavesplit_tile", "decode_wavesplit") else 0,
            min(3, plan["groups_per_wg"]) if k == "decode" else plan["groups_per_wg"], plan["splits"] > 1)


# ---- the benchmark configurations at full size: name -> (K, N)
DSV3_MLP = {"gate_up": (7168, 36864), "down": (18432, 7168)}
DSV3_MLA = {"q_a": (7168, 1536), "kv_a": (7168, 576), "q_b": (1536, 24576), "kv_b": (512, 32768)}
LLAMA3_8B = {"qkv": (4096, 6144), "gate_up": (4096, 28672), "down": (14336, 4096)}

FP8_DECODE_CONFIG = [(M, N, K) for M in (1, 8, 32, 128) for (K, N) in DSV3_MLP.values()]
FP8_PREFILL_CONFIG = [(4096, N, K) for (K, N) in list(DSV3_MLP.values()) + list(DSV3_MLA.values())]
INT8_CONFIG = [(M, N, K) for M in (1, 256, 4096) for (K, N) in LLAMA3_8B.values()]


def variant_of(plan: dict, K: int):
    """What a plan runs, as a key; "unpacked": behind the launch that expands packed exponents to fp32 scales."""
    if plan.get("exponents") == "unpacked":
        return variant_of({**plan, "exponents": "mfma"}, K) + ("unpacked",)
    k = plan["kernel"]
    sp = "split" if plan["splits"] > 1 else "whole"
    if k == "decode":
        g = plan["groups_per_wg"]
        return (k, sp, f"gpw{g}" if g < 3 else "gpw3+")
    if k == "decode_wavesplit":  # waves per workgroup; one turn of the wave's four-slot ring or several
        waves = plan["groups_per_wg"]
        key = (k, f"w{waves}", "rounds" if -(-K // 128) > 4 * waves else "one_round")
        return key + ("two_tiles",) if plan["bn"] == 32 else key  # 32 channels per workgroup (FP8) or 16
    if k == "wavesplit_tile":
        return (k, plan["bm"], plan["bn"], "kfull" if K % 128 == 0 else "ktail")
    if k == "pingpong128":
        return (k, sp)
    if k == "resident":  # a kernel for each number of K blocks
        return (k, f"kb{K // 128}")
    if k == "dma3":  # "deep": more than three LDS stages (small tiles when every workgroup has a CU to itself, FP8)
        key = (k, plan["bm"], sp) if plan["bn"] == 256 else (k, plan["bm"], sp, f"bn{plan['bn']}")
        return key + ("deep",) if plan["stages"] > 3 else key
    if k in ("pingpong", "pipelined"):
        return (k, "kfull" if K % 128 == 0 else "ktail")
    return (k, plan["bm"], "aligned" if plan["aligned"] else "bytes", sp)


def plan_for(kind: str, M: int, N: int, K: int) -> dict:
    from sglang_amd import _lib

    return _lib.gemm_plan(kind, M, N, K, aligned=(K % 16 == 0))
