"""Slots dealt to numbers of parts that are no powers of two, and to as many as there can be: the lookups of test_gpu_pool_parts at
those lengths (sums exact in 32 bits in any order)."""
import pytest

import test_gpu_pool_parts as parts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lens", [
    (16, [3200, 3201, 4800, 4801]),          # 2, 3, 3, 4 parts
    (8, [6401, 8001, 11200, 11201, 20803]),  # 5, 6, 7, 8, 14: with spread signs from the second on
    (4, [1601] * 33 + [160001])])            # 2 each, 101
@pytest.mark.parametrize("kind", ["few signs", "distinct", "long examples"])
def test_numbers_of_parts(tn, oracle, dim, lens, kind):
    parts.test_parts_of_slots(tn, oracle, dim, lens, kind)


def test_most_parts(tn, oracle):
    parts.test_parts_of_slots(tn, oracle, 3, [3_280_000], "few signs")  # 2050, of which there are 2048
