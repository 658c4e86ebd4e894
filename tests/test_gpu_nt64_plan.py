"""K ranges of the FP64 force bias are planned for the loads that the launch takes: 16 bytes
a lane (row tiles up to 64) where every n N is even, 4 bytes (up to 48 rows, more cost
per chunk) where one is odd.  The rule restated (us and bandwidth as in k_nt64.hip)
against a new context's default."""

import math

import pytest

pytestmark = pytest.mark.gpu


def _ranges(N, X, na, nb, W):
    tallest, over, whole = (4, 0.25, 4.0) if na * N % 2 == 0 and nb * N % 2 == 0 else (3, 0.75, 6.0)
    chunks = -(-na * N // 16) + -(-nb * N // 16)

    def cost(blocks, rm, each):
        rounds = -(-W // (16 * rm)) * blocks / 256.0
        return (math.ceil(rounds) if rounds < whole else rounds) * (each + 2.0) * (rm + over)

    best, least = 1, None
    for ks in range(1, 17):
        if 2 * ks > max(chunks, 2):
            break
        blocks, each = -(-X // 128) * ks, float(-(-chunks // ks))
        rows = 1
        for rm in range(2, tallest + 1):
            if cost(blocks, rm, each) < 0.999 * cost(blocks, rows, each):
                rows = rm
        t = cost(blocks, rows, each) + W * X * 32.0 / 4.4e12 / 0.43e-6 * ks
        if least is None or t < 0.98 * least:
            best, least = ks, t
    return best


@pytest.mark.parametrize("case", [(24, 72, 5, 5, 10), (101, 505, 9, 9, 33), (151, 600, 15, 13, 300),
                                  (199, 800, 17, 17, 512), (200, 800, 17, 17, 512), (255, 1275, 25, 25, 71),
                                  (255, 1275, 24, 24, 71), (301, 1000, 31, 29, 600)])
def test_default_ranges(case):
    import torch

    from ipie_amd import _lib

    N, X, na, nb, W = case
    print(f"[case] K ranges {case}", flush=True)
    ctx = _lib.Context(N, X, na, nb, W, device=torch.device("cuda", 0))
    assert ctx.tune_get("fb_split")[0] == _ranges(*case)
