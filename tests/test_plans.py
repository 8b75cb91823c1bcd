"""Bounds of the work-sharing rules (csrc/plans.h) over the sizes of the entry
points, on the CPU: the partial results a plan writes fit what its launch asked
for, and split counts stay within what the second passes are built for."""
import os
import random
import re

import pytest

import plans


def _sizes(count):
    rng = random.Random(20260812)
    for _ in range(count):
        m = int(2 ** rng.uniform(0, 17))
        k = 4 * int(2 ** rng.uniform(0, 12))
        n = 4 * int(2 ** rng.uniform(0, 12))
        yield m, k, n


@pytest.mark.parametrize("cus", [1, 80, 256, 304])
def test_linear_partial_sums_fit_their_buffer(cus):
    for m, k, n in list(_sizes(1500)) + [(2600, 3072, 768), (3458, 4096, 1024), (866, 3072, 768)]:
        f = plans.linear_form(m, k, n, cus)
        floats, most = f.splits * m * n, max(f.provided, f.splits) * m * n
        assert 1 <= f.splits <= 8 and (f.provided > 1 or f.splits == 1), (m, k, n, f)
        assert f.tiles == -(-m // f.tm) * -(-n // f.tn)
        # the work buffer holds `most`; the fixed scratch takes a call only if all fits
        assert floats <= most
        if f.splits > 1 and f.provided * m * n <= plans.MAX_PARTIAL_FLOATS:
            assert most <= plans.MAX_PARTIAL_FLOATS, (m, k, n, f)
        # every split runs at least four stages of 32 k
        assert f.splits == 1 or f.splits * 4 <= -(-k // 32)


def test_attention_partial_results_fit_their_buffer():
    rng = random.Random(20260812)
    for _ in range(1500):
        s, n = int(2 ** rng.uniform(0, 9)), int(2 ** rng.uniform(0, 15))
        f = plans.attention_form(s, n)
        assert f.waves in (4, 8) and 1 <= f.splits <= min(8, -(-n // 64))
        assert f.provided > 1 or f.splits == 1, (s, n, f)


def test_the_fixed_scratch_is_the_plans_limit():
    """The allocation-free entry point's array is as large as the most that a plan
    takes beyond what callers provide for, by definition and not by chance."""
    src = open(os.path.join(plans._CSRC, "linear_api.hip")).read()
    assert re.search(r"kScratchFloats = static_cast<size_t>\(vk::kMaxPartialFloats\);", src)
    launch = open(os.path.join(plans._CSRC, "linear.hip")).read()
    assert "VK_UNSUPPORTED_IF(most * mn > partial_floats" in launch


def test_the_gpu_tests_reach_the_forms_they_name():
    """Shapes of the GPU tests against the rules: a change of their constants that
    moves a shape to another form is seen here."""
    attention = pytest.importorskip("test_gpu_attention_split")
    linear = pytest.importorskip("test_gpu_linear_split")
    for table in (linear.FORM_OF, linear.SHAPE_FORM):
        for (m, k, n), form in table.items():
            assert tuple(plans.linear_form(m, k, n)[:3]) == form, (m, k, n)
    assert {f[:2] for f in linear.FORM_OF.values()} == {(64, 64), (64, 128), (128, 128), (128, 256)}
    for table in (attention.FORM_OF, attention.SIZE_FORM):
        for (s, n), form in table.items():
            assert tuple(plans.attention_form(s, n)[:2]) == form, (s, n)
    assert {(w, sp > 1) for w, sp in attention.FORM_OF.values()} == {(4, False), (4, True),
                                                                     (8, False), (8, True)}
