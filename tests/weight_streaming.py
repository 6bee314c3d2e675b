"""Problems of the weight-streaming kernel that has all of A in LDS, on 256 compute units (beyond 32 columns per unit): operand kind (0 16-bit /
1 int8 / 2 fp8), K steps that it fetches together, m, n, bytes of K.  16 and 32 rows; last workgroups (of 64 columns) of 16, 32 and 48
columns and whole ones."""
CASES = [(kind, steps, m, n, k_bytes)
         for kind in range(3)
         for steps, m, n, k_bytes in [(2, 16, 8208, 1024), (4, 16, 8272, 2048), (2, 16, 10256, 3072), (8, 16, 8256, 4096), (8, 16, 8224, 8192),
                                      (2, 32, 8208, 1024), (4, 32, 8272, 2048), (2, 32, 8240, 3072), (8, 32, 10256, 4096)]]

# 16-bit operands, route, m, n, k
HALF = [("Skinny8", 16, 8208, 2048), ("Skinny4", 32, 8272, 1024), ("Skinny8", 32, 8208, 2048), ("Sliced", 32, 352, 4096), ("Sliced", 48, 1040, 4096)]
# 8-bit operands, slices of K over workgroups: m, n, k
SLICED = [(48, 352, 8192), (48, 1040, 5120), (32, 352, 6144), (16, 352, 9216)]
# operand kind, route, m, n, k
REPLAYED = [(1, "Skinny2", 16, 8208, 1024), (2, "Skinny4", 32, 8272, 2048), (1, "Sliced", 48, 352, 5120)]
