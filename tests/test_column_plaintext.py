"""Plaintext rows that lack the transform's row pass (CKKSContext.encode(..., row_pass=False)) hold doubles, and
only the product that finishes them takes them: every other operation on plaintexts refuses both the
object and its tensor."""

import pytest

torch = pytest.importorskip("torch")

from holmes_amd import fhe  # noqa: E402
from holmes_amd.context import Cipher, CipherState, CKKSContext  # noqa: E402

N, LIMBS = 8, 2


class Recorder:
    """A context that records which product a call reaches."""

    N = N

    def __init__(self):
        self.calls = []

    def q_prime_idx(self, limbs):
        return list(range(limbs))

    def empty(self, *shape):
        return torch.zeros(shape, dtype=torch.uint64)

    def poly_op(self, op, *args, **kwargs):
        self.calls.append("poly_op")

    def _mac(self, name, c0, c1, pts, limbs, giants):
        self.calls.append((name, pts.dtype))
        return torch.zeros((2, giants, c0[0].shape[0], limbs, N), dtype=torch.uint64)

    def bsgs_mac(self, c0, c1, pts, limbs, giants, prime_idx=None):
        return self._mac("bsgs_mac", c0, c1, pts, limbs, giants)

    def bsgs_mac_rows(self, c0, c1, pts, limbs, giants):
        return self._mac("bsgs_mac_rows", c0, c1, pts, limbs, giants)


def _cipher():
    cv = [torch.zeros((1, LIMBS, N), dtype=torch.uint64) for _ in range(2)]
    return Cipher(cv, CipherState(LIMBS, 1, 2.0**10), slots=N // 2)


def _columns():
    return fhe.ColumnPlaintext(torch.zeros((1, LIMBS, N), dtype=torch.float64), CipherState(LIMBS, 1, 2.0**10),
                               slots=N // 2)


@pytest.mark.parametrize("op", [lambda ct, pt, ctx: fhe.homo_mul_pt(ct, pt, ctx),
                                lambda ct, pt, ctx: fhe.homo_add_pt(ct, pt, ctx),
                                lambda ct, pt, ctx: fhe.grouped_pairwise_mac(ct, pt, 1, ctx)],
                         ids=["homo_mul_pt", "homo_add_pt", "grouped_pairwise_mac"])
def test_other_operations_refuse_column_rows(op):
    ctx = Recorder()
    with pytest.raises(AttributeError, match="hoisted_mac_sum"):
        op(_cipher(), _columns(), ctx)
    assert ctx.calls == []


def test_the_product_takes_each_form_to_its_own_kernel():
    ct = _cipher()
    whole = torch.zeros((1, LIMBS, N), dtype=torch.uint64)
    for pts, want in ((_columns(), ("bsgs_mac_rows", torch.float64)),
                      (fhe.Plaintext(whole, CipherState(LIMBS, 1, 2.0**10), slots=N // 2), ("bsgs_mac", torch.uint64)),
                      (whole, ("bsgs_mac", torch.uint64))):
        ctx = Recorder()
        out = fhe.hoisted_mac_sum(ct, [0], pts, 1, 1, ctx, baby_rotations=(ct,))
        assert ctx.calls == [want]
        assert out.state.scale_degree == 2


def test_the_tensors_are_told_apart_by_type():
    doubles, words = (torch.zeros((1, LIMBS, N), dtype=d) for d in (torch.float64, torch.uint64))
    with pytest.raises(ValueError, match="uint64"):
        CKKSContext._check_poly(doubles, LIMBS, N)
    with pytest.raises(ValueError, match="float64"):
        CKKSContext._check_poly(words, LIMBS, N, torch.float64)
