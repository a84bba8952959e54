"""Shapes that the GEMM's rules send to each output tile, at ragged edges and with a K tail (imported by the
GPU tests that run them and by the CPU test that pins the rules' answers on 256 compute units)."""
T256, T256x192, T256x128, T128, T128_PAIR, T64x128, T128x64, T64, T32x64 = range(9)
CUS = 256

# tile: M, N, K of a product that runs on it unsplit (with an MN-major A the 32-row tiles become 64-row ones)
PLAIN = {T256x128: (2352, 1712, 336), T128: (3600, 528, 336), T128_PAIR: (2320, 3216, 336), T64x128: (528, 3280, 336),
         T128x64: (3296, 272, 336), T64: (2864, 144, 336), T32x64: (48, 1056, 336)}
# tile: M, N, K, splits
SPLIT = {T256x128: (672, 2976, 3024, 3), T128: (336, 2720, 3344, 3), T64x128: (272, 1824, 3120, 3),
         T128x64: (144, 1808, 3280, 4), T64: (16, 1200, 6096, 6), T32x64: (16, 4096, 14336, 4)}
# tile: tokens, inputs, hidden of an FP32 SwiGLU block whose dgate|dup product (two outputs) runs on it
TWO_OUTPUTS = {T256: (336, 1040, 3872), T256x128: (336, 528, 3600), T128: (336, 272, 3296), T128_PAIR: (336, 3280, 1168),
               T64x128: (352, 192, 4000), T128x64: (336, 144, 2864), T64: (336, 16, 16)}
# tile: KV heads, query rows, keys, width of a materialized attention whose dK and dV run on it as a pair
PAIR = {T256x128: (4, 16, 1888, 256), T128: (16, 80, 384, 256), T128_PAIR: (32, 80, 128, 256), T64x128: (64, 80, 32, 240),
        T128x64: (2, 80, 2080, 144), T64: (1, 80, 32, 192)}
# tile: M, N, K of a fused-epilogue product (residual, SwiGLU forward and backward)
EPILOGUE = {T256x128: (3632, 1056, 336), T128_PAIR: (3600, 544, 336), T64x128: (3296, 288, 336), T64: (144, 224, 336)}
# tile: tokens, heads (Hq, Hkv), hidden of the fused QKV projection
QKV = {T128_PAIR: (528, 27, 1, 336), T64x128: (200, 6, 1, 336)}
# padded linear: logical rows, inputs, outputs; tiles of y, dx and dw, all stored through the cropped epilogue
CROPPED = {(1777, 2001, 3003): (T256x128, T128, T256x128), (2345, 331, 1703): (T256x128, None, None),
           (3595, 331, 517): (T128, None, None), (2311, 331, 3205): (T128_PAIR, None, None), (517, 331, 3277): (T64x128, None, None),
           (3283, 331, 269): (T128x64, None, None)}
# F32 matmul: A, B shapes; tile edge and splits of the product, dA and dB
F32 = {((4, 1000, 1024), (1024, 1000)): ((128, 1), (128, 1), (128, 4)), ((4, 999, 1023), (1023, 1004)): ((128, 1), (128, 1), (128, 4)),
       ((4, 1000, 1024), (1024, 1001)): ((128, 1), (128, 1), (128, 4)), ((4, 1001, 1021), (1021, 1003)): ((128, 1), (128, 1), (128, 4)),
       ((4, 1000, 1021), (4, 1021, 1003)): ((128, 1), (128, 1), (128, 1)), ((2049, 509), (509, 2047)): ((64, 1), (128, 7), (128, 4)),
       ((3000, 17, 33), (3000, 33, 21)): ((64, 1), (64, 1), (64, 1)), ((31, 4097), (4097, 33)): ((64, 16), (64, 1), (64, 1))}
