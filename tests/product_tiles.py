"""Shapes that reach every tile of the matrix-product kernel, whole and with K
splits, in both weight layouts: (operator, layout, tile rows, tile columns, rows
scaled by a pass first) -> (M, K, N) of a whole launch and of a K-split one.
Every shape has a partial row tile, a partial column tile and a partial last
chunk of 64 k, the whole ones K long enough for the unrolled loop of whole
chunks.  STAGED: the same for operands that are not 16-byte aligned.
tests/test_plans.py holds them to the plan, tests/test_gpu_gemm.py runs them."""

NK, KN = 0, 1
TILES = {
    ("linear", NK, 32, 64, False): ((17, 856, 24), (5, 1448, 24)),
    ("linear", NK, 32, 128, False): ((2049, 888, 200), (90, 6504, 3208)),
    ("linear", NK, 64, 128, False): ((2049, 848, 472), (2049, 1504, 208)),
    ("linear", NK, 128, 128, False): ((2049, 856, 912), (2049, 2144, 392)),
    ("linear", NK, 128, 192, False): ((2049, 840, 1936), (2049, 3088, 920)),
    ("linear", NK, 128, 256, False): ((2049, 880, 2936), (2049, 4376, 984)),
    ("linear", NK, 256, 256, False): ((2049, 848, 3920), (2049, 6248, 1928)),
    ("linear", KN, 32, 64, False): ((17, 856, 24), (5, 1288, 24)),
    ("linear", KN, 32, 128, False): ((2049, 888, 200), (2049, 3488, 72)),
    ("linear", KN, 64, 128, False): ((2049, 864, 392), (2049, 2096, 200)),
    ("linear", KN, 128, 128, False): ((2049, 856, 912), (2049, 2568, 416)),
    ("linear", KN, 128, 192, False): ((2049, 840, 1936), (2049, 2440, 944)),
    ("linear", KN, 128, 256, False): ((2049, 880, 2936), (2049, 3400, 1000)),
    ("linear", KN, 256, 256, False): ((2049, 848, 3920), (2049, 4952, 1968)),
    ("rmsnorm_linear", NK, 32, 64, False): ((250, 880, 528), (17, 856, 24)),
    ("rmsnorm_linear", NK, 32, 128, False): ((250, 840, 2080), (250, 1416, 1104)),
    ("rmsnorm_linear", NK, 64, 128, False): ((250, 848, 4112), (250, 1240, 2056)),
    ("rmsnorm_linear", NK, 128, 128, True): ((300, 840, 24), (257, 904, 24)),
    ("rmsnorm_linear", NK, 128, 192, True): ((2049, 840, 1936), (2049, 3088, 920)),
    ("rmsnorm_linear", NK, 128, 256, True): ((2049, 880, 2936), (2049, 4376, 984)),
    ("rmsnorm_linear", NK, 256, 256, True): ((2049, 848, 3920), (2049, 6248, 1928)),
    ("rmsnorm_linear", KN, 32, 64, False): ((250, 840, 664), (17, 856, 24)),
    ("rmsnorm_linear", KN, 32, 128, False): ((250, 840, 2080), (250, 1320, 728)),
    ("rmsnorm_linear", KN, 64, 128, False): ((250, 848, 4112), (250, 1488, 1376)),
    ("rmsnorm_linear", KN, 128, 128, True): ((1300, 880, 24), (300, 840, 24)),
    ("rmsnorm_linear", KN, 128, 192, True): ((2049, 840, 1936), (2049, 2440, 944)),
    ("rmsnorm_linear", KN, 128, 256, True): ((2049, 880, 2936), (2049, 3400, 1000)),
    ("rmsnorm_linear", KN, 256, 256, True): ((2049, 848, 3920), (2049, 4952, 1968)),
    ("gated_mlp", NK, 32, 128, False): ((2049, 856, 40), (17, 856, 24)),
    ("gated_mlp", NK, 64, 128, False): ((2049, 888, 200), (2049, 4272, 24)),
    ("gated_mlp", NK, 128, 128, False): ((2049, 848, 472), (2049, 2096, 200)),
    ("gated_mlp", NK, 128, 256, False): ((2049, 848, 984), (2049, 4152, 480)),
    ("gated_mlp", NK, 256, 256, False): ((2049, 840, 1936), (2049, 5096, 976)),
    ("gated_mlp", KN, 32, 128, False): ((2049, 856, 40), (17, 856, 24)),
    ("gated_mlp", KN, 64, 128, False): ((2049, 888, 200), (2049, 3760, 24)),
    ("gated_mlp", KN, 128, 128, False): ((2049, 848, 472), (2049, 2520, 200)),
    ("gated_mlp", KN, 128, 256, False): ((2049, 848, 984), (2049, 2952, 472)),
    ("gated_mlp", KN, 256, 256, False): ((2049, 840, 1936), (2049, 4112, 1000)),
}

STAGED = {
    ("linear", NK, 32, 128): ((250, 344, 24), (65, 1464, 24)),
    ("linear", NK, 64, 128): ((2049, 328, 440), (2049, 1632, 208)),
    ("linear", KN, 32, 128): ((250, 344, 24), (5, 1376, 24)),
    ("linear", KN, 64, 128): ((2049, 328, 440), (2049, 1864, 200)),
    ("rmsnorm_linear", NK, 32, 128): ((250, 344, 24), (65, 736, 24)),
    ("rmsnorm_linear", NK, 64, 128): ((2049, 328, 440), (2049, 3408, 24)),
    ("rmsnorm_linear", KN, 32, 128): ((250, 344, 24), (100, 664, 24)),
    ("rmsnorm_linear", KN, 64, 128): ((2049, 328, 440), (2049, 3408, 24)),
    ("gated_mlp", NK, 32, 128): ((250, 344, 24), (65, 736, 24)),
    ("gated_mlp", NK, 64, 128): ((2049, 352, 224), (2049, 1704, 72)),
    ("gated_mlp", KN, 32, 128): ((250, 344, 24), (65, 736, 24)),
    ("gated_mlp", KN, 64, 128): ((2049, 352, 224), (2049, 3728, 24)),
}
