"""Problems that run on the smallest tiles of the blocked GEMM, K-contiguous operands, on 256 compute units: not few enough results for their K for the
kernel whose waves share K.  Operand kind (0 16-bit / 1 int8 / 2 fp8), layout pair, rung, m, n, k, bytes per element of D."""
CASES = [(0, 0, "Tiny", 528, 528, 208, 4), (1, 0, "Tiny", 160, 96, 224, 4), (2, 0, "Tiny", 416, 32, 224, 4), (0, 0, "Tiny", 512, 640, 192, 4),
         (0, 0, "Tiny64", 128, 128, 64, 4), (1, 0, "Tiny", 384, 128, 384, 4), (2, 0, "Tiny", 512, 256, 384, 4)]
