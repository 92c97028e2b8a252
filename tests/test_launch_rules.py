"""Which instance the any-width and bf16 kernels' shape rules pick, without a GPU:
the shapes that test_gpu_widths runs reach every compiled instance on 256 CUs.
Digits as in csrc/mx4_kernels.h: waves along M and N, 32 x 32 tiles a wave along M
and N, K slices; for the skinny kernel chunks a wave and tiles a workgroup."""
import ctypes

import pytest

# (kind, bf16 x): {(m, rows of the weights, k): digits}
GEMM_SHAPES = {
    ("exact", True): {
        (33, (12300,), 288): 22111, (700, (500,), 288): 22112, (100, (700,), 544): 22113, (70, (2100,), 1600): 22114,
        (200, (18500,), 288): 22231, (260, (3000,), 8224): 22234, (65, (8500,), 288): 24111, (65, (3000,), 8224): 24114,
        (65, (18500,), 288): 24121, (33, (6300,), 8224): 42124, (385, (12300,), 288): 24221, (33, (12300,), 8224): 24224,
        (33, (130, 65), 544): 22113, (65, (4200, 65), 288): 22111, (200, (18500, 65), 288): 22231, (65, (8500, 65), 288): 24111,
        (65, (18500, 65), 288): 24121, (385, (12300, 65), 288): 24221, (33, (6300, 65), 8224): 42124},
    ("exact", False): {
        (33, (6300,), 288): 22112, (100, (700,), 544): 22113, (70, (1500,), 1600): 22114, (65, (8500,), 416): 14211,
        (65, (6300,), 288): 14212, (65, (3000,), 416): 14214, (200, (8500,), 288): 14221, (65, (8500,), 288): 14223,
        (129, (12300,), 288): 22221, (33, (8500,), 288): 22223, (33, (12300,), 288): 22233, (129, (18500,), 288): 22231,
        (33, (130, 65), 544): 22113, (65, (4200, 65), 288): 22111, (65, (8500, 65), 288): 14211, (1030, (130, 65), 416): 14214,
        (65, (18500, 65), 288): 14221, (33, (6300, 65), 416): 22224, (33, (12300, 65), 1056): 22233,
        (129, (18500, 65), 288): 22231},
    ("bf16", True): {
        (65, (2100,), 328): 42111, (65, (4200,), 1032): 42113, (33, (4200,), 1032): 24114, (129, (8500,), 136): 24111,
        (129, (12300,), 136): 42121, (65, (8500,), 2056): 42123, (260, (12300,), 136): 24221, (200, (8500,), 4104): 24223,
        (33, (2100, 65), 136): 42111, (129, (8500, 65), 136): 24111, (260, (12300, 65), 136): 24221,
        (129, (12300, 65), 136): 42121},
    ("bf16", False): {
        (33, (4200,), 136): 22111, (300, (1000,), 1032): 22113, (65, (2100,), 1032): 24114, (65, (3000,), 328): 24113,
        (65, (8500,), 136): 24111, (129, (12300,), 136): 42121, (65, (6300,), 1032): 42124, (20000, (50,), 136): 42111,
        (33, (4200, 65), 136): 22111, (65, (8500, 65), 136): 24111, (129, (12300, 65), 136): 42121},
}
GEMM_INSTANCES = {("exact", True): {2211, 2223, 2411, 2412, 2422, 4212}, ("exact", False): {2211, 2222, 2223, 1422, 1421},
                  ("bf16", True): {4212, 2411, 4211, 2422}, ("bf16", False): {4212, 2411, 4211, 2211}}

# (MXFP4, bf16 x, m, rows of the weights, k): digits
SKINNY_SHAPES = {
    (True, True, 5, (40, 9), 96): 11, (True, True, 5, (4780, 9), 992): 12, (True, True, 16, (9580, 9), 224): 14,
    (True, True, 9, (40, 9), 1632): 21, (True, True, 7, (4780, 9), 1600): 22, (True, True, 7, (4200, 16), 3264): 42,
    (True, True, 29, (40, 9), 96): 11, (True, True, 29, (4780, 9), 992): 12, (True, True, 20, (9580, 9), 224): 14,
    (True, True, 32, (40, 9), 1632): 21, (True, True, 29, (4780, 9), 1600): 22, (True, True, 17, (9580, 9), 2080): 24,
    (True, False, 5, (40, 9), 1632): 11, (True, False, 12, (4780, 9), 992): 12, (True, False, 16, (9580, 9), 1120): 14,
    (True, False, 29, (40, 9), 1632): 11, (True, False, 17, (3180, 9), 992): 12, (True, False, 29, (4780, 9), 1120): 14,
    (False, True, 5, (40, 9), 1608): 11, (False, True, 7, (17000, 600), 1608): 12, (False, True, 29, (40, 9), 1608): 11,
    (False, True, 20, (4780, 9), 136): 12, (False, True, 29, (5000, 9), 2056): 22,
    (False, False, 5, (40, 9), 1608): 11, (False, False, 12, (4780, 9), 1032): 12, (False, False, 16, (9580, 9), 1128): 14,
    (False, False, 29, (40, 9), 1608): 11, (False, False, 17, (3180, 9), 1032): 12, (False, False, 29, (4780, 9), 1128): 14,
}
SKINNY_INSTANCES = {(True, True, False): {11, 12, 14, 21, 22, 42}, (True, True, True): {11, 12, 14, 21, 22, 24},
                    (True, False, False): {11, 12, 14}, (True, False, True): {11, 12, 14},
                    (False, True, False): {11, 12}, (False, True, True): {11, 12, 22},
                    (False, False, False): {11, 12, 14}, (False, False, True): {11, 12, 14}}


@pytest.fixture(scope="module")
def lib():
    import mx4hip

    return ctypes.CDLL(str(mx4hip.LIB_PATH))


def gemm_rule(lib, kind, x_bf16, m, rows, k):
    fn = getattr(lib, f"mx4_rule_gemm_{kind}")
    u32 = ctypes.c_uint32
    fn.restype, fn.argtypes = u32, [ctypes.POINTER(u32), u32, u32, u32, ctypes.c_bool, ctypes.c_int, ctypes.c_uint64]
    return fn((u32 * len(rows))(*rows), len(rows), m, k, x_bf16, 256, 32 << 20)


def skinny_rule(lib, fp4, x_bf16, m, tiles, k):
    fn = lib.mx4_rule_skinny_any
    u32 = ctypes.c_uint32
    fn.restype, fn.argtypes = u32, [ctypes.c_bool, ctypes.c_bool, u32, u32, u32, ctypes.c_int]
    return fn(fp4, x_bf16, m, k, tiles, 256)


@pytest.mark.parametrize("kind,x_bf16", list(GEMM_SHAPES))
def test_gemm_shapes_reach_every_instance(lib, kind, x_bf16):
    seen = {True: set(), False: set()}
    for (m, rows, k), want in GEMM_SHAPES[kind, x_bf16].items():
        assert gemm_rule(lib, kind, x_bf16, m, rows, k) == want, (m, rows, k)
        assert m > 32 and k % (32 if kind == "exact" else 8) == 0 and (kind == "bf16" or k % 128 != 0)
        seen[len(rows) > 1].add(want // 10)
    assert seen[False] == GEMM_INSTANCES[kind, x_bf16]
    if kind == "exact":  # (a group has a kernel of its own)
        assert seen[True] == GEMM_INSTANCES[kind, x_bf16]


def test_skinny_shapes_reach_every_instance(lib):
    seen = {key: set() for key in SKINNY_INSTANCES}
    for (fp4, x_bf16, m, rows, k), want in SKINNY_SHAPES.items():
        tiles = sum((n + 15) // 16 for n in rows)
        assert skinny_rule(lib, fp4, x_bf16, m, tiles, k) == want, (fp4, x_bf16, m, rows, k)
        seen[fp4, x_bf16, m > 16].add(want)
    assert seen == SKINNY_INSTANCES


def test_rules_pick_compiled_instances_only(lib):
    """Over a grid of shapes, nothing outside the compiled instances."""
    for kind, x_bf16 in GEMM_SHAPES:
        for m in (33, 64, 77, 130, 300, 1000, 5000):
            for n in (1, 64, 300, 2000, 9000, 50000):
                for k in (32, 160, 1600, 4288, 12320):
                    for rows in ((n,), (n, 40), (n, n, 7, 64)):
                        got = gemm_rule(lib, kind, x_bf16, m, rows, k)
                        assert got // 10 in GEMM_INSTANCES[kind, x_bf16] and 1 <= got % 10 <= 4, (kind, x_bf16, m, rows, k, got)
    for (fp4, x_bf16, many), known in SKINNY_INSTANCES.items():
        for m in (17, 29, 32) if many else (2, 7, 16):
            for tiles in (1, 100, 256, 257, 300, 512, 513, 1024, 1025, 1500, 9000):
                for k in (32, 992, 1024, 1600, 2048, 2080, 3264, 12320, 100000):
                    assert skinny_rule(lib, fp4, x_bf16, m, tiles, k) in known, (fp4, x_bf16, m, tiles, k)
