"""Which chunks of a projection finish their plaintexts' transform inside the product: only those where that
was measured to be no slower than encoding the plaintexts whole."""

import pytest

from holmes_amd.context import CKKSContext


class Fp64:
    rows_mac = True


@pytest.mark.parametrize("inputs,giants,limbs,pays", [
    (1, 4, 1, False), (1, 4, 2, False), (1, 16, 1, True), (1, 9, 1, False), (1, 8, 2, True), (1, 7, 2, False),
    (1, 4, 3, True), (1, 6, 3, True), (1, 5, 17, False), (1, 3, 17, False), (1, 16, 17, True),
    (2, 8, 1, False), (2, 8, 3, False), (2, 12, 3, False), (2, 16, 3, True), (2, 20, 2, False), (2, 24, 2, True),
    (2, 8, 4, True), (2, 7, 4, True), (2, 12, 4, True),
    (2, 6, 6, False), (2, 6, 8, True), (2, 9, 17, False), (2, 4, 17, False), (2, 16, 17, True),
    (3, 16, 17, False)])
def test_rule(inputs, giants, limbs, pays):
    assert CKKSContext.rows_mac_pays(Fp64(), inputs, giants, limbs) is pays


def test_only_contexts_that_have_the_kernel():
    class Wide:
        rows_mac = False

    assert CKKSContext.rows_mac_pays(Wide(), 1, 16, 17) is False
