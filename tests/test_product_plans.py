"""The rule by which products of more than 64 rows choose their tiles, asked of the kernel library as its launcher asks it."""
import random

from llm_rs_amd.csrc import build as native

# (rows, features, k, epilogue, rows of a tile, parts): where the plan chosen was measured against all others
MEASURED = [(2032, 2048, 2048, 2, 128, 1), (2032, 2048, 8192, 2, 128, 1), (2032, 3072, 2048, 0, 256, 1), (2048, 4096, 14336, 2, 256, 1), (1024, 4096, 14336, 2, 256, 2),
            (900, 3072, 2048, 0, 128, 1), (700, 2048, 8192, 2, 256, 4), (200, 16384, 2048, 3, 128, 1), (450, 16384, 2048, 3, 256, 1)]


def test_plans_are_the_measured_ones():
    lib = native.load_hip()
    for M, N, K, epi, rows, parts in MEASURED:
        assert lib.llmrs_gemm_mid_plan(M, N, K, epi) == 100 * parts + rows // 128, (M, N, K, epi)


def test_plans_have_room_and_no_empty_part():
    lib = native.load_hip()
    room = lib.llmrs_gemm_workspace_floats
    room.restype = __import__("ctypes").c_long
    rng = random.Random(1)
    for _ in range(4000):
        M, N, K = rng.randint(1, 5000), rng.choice([rng.randint(1, 30000), 1024 * rng.randint(1, 16)]), 8 * rng.randint(1, 1800) if rng.random() < 0.3 else 64 * rng.randint(1, 240)
        for epi in range(4):
            plan = lib.llmrs_gemm_mid_plan(M, N, K, epi)
            if M <= 64 or K % 64:
                assert plan == 0
            if plan == 0:
                continue
            parts, nk = plan // 100, K // 64
            assert plan % 100 in (1, 2) and 1 <= parts <= 16 and (parts - 1) * -(-nk // parts) < nk
            assert room(M, N, K) >= (parts * M * N if parts > 1 else 0)
            if N % 4 == 0 and 4 <= N <= 16384:
                assert lib.llmrs_gemm_norms_whole(M, N, K) and room(M, N, K) > 0
