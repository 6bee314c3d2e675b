"""Problems that run on wide waves, four waves of 128 x 128 or 128 x 64 results, on 256 compute units: operand kind (0 16-bit / 1 int8),
layout pair (0 both K-contiguous / 1 A only / 2 B only / 3 neither), rung, m, n, bytes of K, bytes per element of D."""

# C and D in 16 and 8 bits: partly filled tiles with a last row, column and stage of every kind, whole 256 x 128 and 256 x 256 tiles
NARROW_C = [(0, 0, "Wide", 1040, 6000, 416, 2), (0, 0, "Wide", 528, 7184, 4128, 2), (0, 1, "Wide", 1808, 3088, 1312, 2),
            (1, 0, "Wide", 1040, 6000, 416, 1), (1, 1, "Wide", 528, 7184, 1312, 1), (0, 0, "Wide", 1536, 3584, 768, 2),
            (0, 1, "Wide", 2560, 2560, 768, 2), (1, 0, "Wide", 1536, 3584, 1024, 1), (0, 0, "Big", 2048, 7168, 3072, 2),
            (0, 1, "Big", 2048, 7168, 3072, 2), (0, 2, "Big", 2048, 7168, 3072, 2), (1, 0, "Big", 2048, 7168, 3072, 1),
            (1, 1, "Big", 2048, 7168, 3072, 1), (1, 2, "Big", 2048, 7168, 3072, 1), (1, 3, "Big", 2048, 7168, 3072, 1)]

# rows of a 32-bit D 32 KiB apart: waves of two runs of rows, in whole tiles, in half tiles of a last round, and in partly filled ones
RUNS_OF_ROWS = [(0, 0, "Wide", 768, 8192, 4096, 4), (0, 1, "Wide", 784, 8192, 2080, 4), (0, 0, "Wide", 784, 8192, 1312, 4),
                (1, 0, "Wide", 784, 8192, 1312, 4), (1, 1, "Wide", 784, 8192, 4128, 4), (0, 0, "Big", 2560, 8192, 3072, 4),
                (0, 1, "Big", 4096, 8192, 3072, 4), (0, 2, "Big", 5120, 8192, 3072, 4), (1, 0, "Big", 4096, 8192, 3072, 4),
                (1, 1, "Big", 2560, 8192, 3072, 4), (1, 2, "Big", 4096, 8192, 3072, 4), (1, 3, "Big", 5120, 8192, 3072, 4)]
