"""Sizes (m, n, k) by the kernel that they are meant for; test_matmul_plans.py asks the library whether they reach it, the GPU tests
run them."""

# The weight-streaming kernel with bf16 activations, K in steps of 512: strips of every height, with and without K slices
STREAMED_BF16 = [
    (1, 36, 512), (16, 100, 1024), (17, 8188, 1024), (32, 28, 2048),            # strips of 32 rows: ragged, none full
    (16, 8212, 1024), (33, 12276, 1024), (100, 616, 6656),                      # 48: one row more than 256 strips of 32 hold
    (65, 8212, 1024), (128, 12300, 1024), (64, 14332, 512),                     # 64, and one round of them exceeded
    (16, 4100, 4096), (64, 4092, 4096), (31, 500, 8192), (128, 2044, 8192),     # narrow strips over K slices
    (16, 16388, 1024), (33, 1232, 6656), (128, 28764, 512), (17, 2152, 6656),   # 112 and 128
]
# The same with any other K, by the plain call or with a workspace
STREAMED_BF16_ANY_K = [
    (1, 36, 256), (16, 100, 320), (17, 260, 448), (33, 64, 576), (5, 132, 704),     # one to eleven groups of 64
    (16, 8196, 960), (64, 16388, 1088), (65, 28, 1472), (128, 8252, 1984),          # strips of 32, 64, 128
    (5, 2880, 2880), (45, 2880, 2880), (100, 2880, 2880), (31, 516, 14272), (128, 1028, 4160),
]
# ... with f32 or f16 activations, K in steps of 512, N of 4, in passes of 64 rows.  Ragged last strips, one strip more than a round of
# 256 holds, K slices of narrow strips, several passes
STREAMED_F32_F16 = [
    (6, 36, 512), (16, 8188, 1024), (17, 8196, 1024), (32, 12284, 1024), (33, 12292, 512), (64, 16388, 512), (16, 4100, 4096),
    (31, 2044, 4096), (64, 500, 8192), (65, 28, 1024), (128, 4092, 1024), (15, 616, 6656), (45, 3320, 2560), (129, 1020, 2048),
    (1024, 28, 1024), (1025, 28, 1024),
]
# The kernel for several f32 or f16 rows: tiles of 128, 192, 224 and 256 weight rows, over K slices and not, that end one row past a
# tile or one before it, odd N, whole groups of four blocks and a remainder.  By the call with a workspace, as the operators make it
ROWS = {
    "f32": [(45, 1151, 256), (45, 1153, 288), (45, 2881, 2912), (300, 10943, 256), (20, 6529, 544), (485, 9601, 576), (512, 14335, 1056),
            (20, 12319, 800), (300, 6145, 2080), (400, 14591, 256), (20, 8193, 800)],
    "f16": [(45, 1793, 256), (45, 2047, 544), (45, 2881, 2912), (300, 10943, 256), (20, 8447, 800), (485, 9601, 576), (400, 12319, 288),
            (20, 9857, 1184), (512, 14335, 1056), (400, 12289, 256), (20, 11521, 1184)],
}
