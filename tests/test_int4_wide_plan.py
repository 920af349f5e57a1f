"""int4_plan (int4_gemm_plan.hpp, built here for the host): what it hands to the launcher exists, covers the product and stays within the
scratch that callers have."""
import random

from test_int4_gemm_plan import RING, WIDE, planner  # noqa: F401


def test_plans_cover_the_product(planner):  # noqa: F811
    rng, kinds = random.Random(1), set()
    for i in range(20000):
        m, n, kt, cus = rng.randint(17, 2300), int(64 * 2000 ** rng.random()), rng.randint(1, 128), 256 if i % 4 else rng.randint(1, 320)
        one, second, col, splits, per = planner(m, n, kt, cus)
        if cus == 256:
            kinds.add((one, splits > 1, second >= 0))
        assert one in RING or one in WIDE, (m, n, kt)  # tiles the launcher has
        assert second == -1 or second in WIDE, (m, n, kt)
        assert one == (1 if m <= 32 else 2) if m <= 64 else one != 1
        assert second < 0 or (0 < col < n and col % 16 == 0 and splits == 1), (m, n, kt)
        assert splits >= 1 and splits * per >= kt > (splits - 1) * per, (m, n, kt)
        assert splits == 1 or splits * m * n * 4 + m * kt * 256 <= 31 << 20, (m, n, kt)
    assert {(16, False, False), (19, False, False), (0, False, False), (0, True, False), (2, True, False), (1, True, False), (19, False, True)} <= kinds
