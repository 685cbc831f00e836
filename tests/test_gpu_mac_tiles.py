"""GPU parity of the multiply-accumulate's two kernels where their tiles end: the matrix-core kernel's
16 giants x 16 columns x 16 babies (full, one short, one more, several chunks of babies), the VALU
kernel's tiles of 1 to 4 inputs x 8 giants, and the rows the vector loads cannot take, bit-exact against
the oracle on both prime widths."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module", params=["50-bit", "59/60-bit"])
def env(request):
    from holmes_amd import fhe
    from holmes_amd.context import CKKSContext

    bits = dict(dcrt_bits=50, first_mod=50) if request.param == "50-bit" else dict(dcrt_bits=59, first_mod=60)
    ctx = CKKSContext(fhe.CKKSContextSpec(depth=3, dnum=2, seed=5, **bits))
    return ctx, O.OracleContext(16, ctx.L, ctx.K, ctx.alpha, ctx.primes)


def _residues(rng, shape, q):
    return rng.integers(0, 2**62, size=shape, dtype=np.uint64) % q


def _check(env, ni, nb, G, limbs, offset=0):
    ctx, orc = env
    rng = np.random.default_rng(1000 * ni + 10 * nb + G)
    q = np.array(ctx.primes[:limbs], dtype=np.uint64).reshape(1, limbs, 1)
    pts = _residues(rng, (G * nb, limbs, ctx.N), q)
    babies = _residues(rng, (nb, 2, ni, limbs, ctx.N), q.reshape(1, 1, 1, limbs, 1))
    # every product at its largest, and zeros
    pts[:, :, :3] = np.array([p - 1 for p in ctx.primes[:limbs]], dtype=np.uint64).reshape(1, limbs, 1)
    babies[..., :2] = np.array([p - 1 for p in ctx.primes[:limbs]], dtype=np.uint64).reshape(1, 1, 1, limbs, 1)
    babies[..., 2] = 0
    buf = torch.zeros(pts.size + 2, dtype=torch.uint64, device="cuda")
    buf.view(torch.int64)[offset:offset + pts.size].copy_(torch.from_numpy(pts.view(np.int64)).reshape(-1))
    tp = buf[offset:offset + pts.size].view(pts.shape)
    bt = torch.from_numpy(babies).cuda()
    res = ctx.bsgs_mac([bt[b, 0] for b in range(nb)], [bt[b, 1] for b in range(nb)], tp, limbs, G).cpu().numpy()
    for i in range(ni):
        want = orc.bsgs_mac(limbs, nb, G, pts, np.ascontiguousarray(babies[:, :, i]))
        assert np.array_equal(res[:, :, i], want), f"input {i}"


@pytest.mark.parametrize("ni,nb,G,limbs", [(8, 16, 16, 2), (7, 15, 15, 1), (5, 16, 32, 1), (15, 31, 30, 1),
                                           (9, 48, 17, 1), (16, 64, 16, 1), (13, 33, 27, 1)])
def test_matrix_core_tiles(env, ni, nb, G, limbs):
    _check(env, ni, nb, G, limbs)


@pytest.mark.parametrize("ni,nb,G,limbs", [(1, 9, 8, 2), (2, 3, 9, 1), (3, 8, 7, 1), (4, 2, 16, 1), (5, 8, 8, 1),
                                           (10, 7, 1, 1)])
def test_vector_tiles(env, ni, nb, G, limbs):
    _check(env, ni, nb, G, limbs)


@pytest.mark.parametrize("ni,nb,G,limbs", [(16, 16, 25, 1), (13, 16, 16, 2), (12, 16, 32, 1), (16, 36, 16, 1),
                                           (16, 40, 31, 1), (8, 14, 16, 3)])
def test_matrix_core_tiles_with_partial_tiles(env, ni, nb, G, limbs):
    """Shapes that both widths' rules send to the matrix-core kernel (three quarters of the tiles' volume
    real) whose last tile of giants, of columns or step of babies is partly empty."""
    up = lambda v: -(-v // 16) * 16  # noqa: E731
    assert 4 * G * 2 * ni * nb >= 3 * up(G) * up(2 * ni) * up(nb)
    _check(env, ni, nb, G, limbs)


@pytest.mark.parametrize("ni,nb,G,limbs", [(10, 3, 9, 1), (10, 5, 4, 1), (11, 3, 5, 1), (12, 2, 8, 1), (14, 2, 3, 1)])
def test_vector_tiles_of_many_inputs(env, ni, nb, G, limbs):
    """More than two input tiles: of 2 or 4 by the giants, of 4 full and one short, of 3."""
    _check(env, ni, nb, G, limbs)


def test_rows_that_are_not_16_byte_aligned(env):
    """A shape of the matrix-core kernel whose plaintexts start at an odd word."""
    _check(env, 8, 16, 16, 1, offset=1)


@pytest.mark.parametrize("ni,nb,G,limbs", [(1, 16, 32, 2), (1, 1, 1, 1), (2, 5, 17, 1), (2, 16, 7, 1), (1, 64, 5, 1)])
def test_row_pass_inside_the_product(env, ni, nb, G, limbs):
    """Plaintexts with the column pass only, finished inside the product, against encoding them whole
    (bit-exact against the oracle in test_gpu_bsgs); the wide path refuses them."""
    from holmes_amd import _native as nat

    ctx, _ = env
    gen = torch.Generator(device="cuda").manual_seed(nb * 100 + G)
    re, im = (torch.randn(G * nb, ctx.max_slots, dtype=torch.float64, device="cuda", generator=gen) for _ in range(2))
    scale = float(ctx.rescale_divisor_at(2))
    if not ctx.rows_mac:
        with pytest.raises(nat.NativeError):
            ctx.encode(re, scale, limbs, values_im=im, row_pass=False)
        return
    q = torch.tensor([int(p) for p in ctx.primes[:limbs]], dtype=torch.int64, device="cuda")[:, None]
    x = torch.randint(0, 1 << 62, (nb, 2, ni, limbs, ctx.N), dtype=torch.int64, device="cuda", generator=gen)
    x.remainder_(q)
    x[..., :2] = q - 1
    x = x.view(torch.uint64)
    b0, b1 = [x[b, 0] for b in range(nb)], [x[b, 1] for b in range(nb)]
    want = ctx.bsgs_mac(b0, b1, ctx.encode(re, scale, limbs, values_im=im), limbs, G)
    got = ctx.bsgs_mac_rows(b0, b1, ctx.encode(re, scale, limbs, values_im=im, row_pass=False), limbs, G)
    assert torch.equal(got.view(torch.int64), want.view(torch.int64))
    with pytest.raises(nat.NativeError):
        ctx.bsgs_mac_rows([ctx.zeros(3, 1, ctx.N)], [ctx.zeros(3, 1, ctx.N)], ctx.zeros(1, 1, ctx.N), 1, 1)


def test_rows_without_their_row_pass_are_told_apart(env):
    """encode(row_pass=False) gives float64: each product refuses the other's plaintexts."""
    ctx, _ = env
    if not ctx.rows_mac:
        return
    re = torch.randn(4, ctx.max_slots, dtype=torch.float64, device="cuda")
    whole, cols = ctx.encode(re, 2.0**40, 1), ctx.encode(re, 2.0**40, 1, row_pass=False)
    assert (whole.dtype, cols.dtype) == (torch.uint64, torch.float64)
    x = [ctx.zeros(1, 1, ctx.N)]
    with pytest.raises(ValueError, match="uint64"):
        ctx.bsgs_mac(x, x, cols, 1, 4)
    with pytest.raises(ValueError, match="float64"):
        ctx.bsgs_mac_rows(x, x, whole, 1, 4)
    with pytest.raises(ValueError, match="float64"):
        ctx.encode(re, 2.0**40, 1, row_pass=False, out=whole)


@pytest.mark.parametrize("D,lanes,shift,B,base,G", [(96, 4, 0, 1, 0, 3), (96, 8, 5, 7, 2, 2), (64, 1, 0, 9, 1, 2),
                                                    (1, 2, 3, 17, 0, 1)])
def test_packed_baby_chunks(env, D, lanes, shift, B, base, G):
    """The packer's groups of 8 baby steps: alone, one short, one more, rows shorter than a group."""
    ctx, _ = env
    W = np.random.default_rng(B).standard_normal((D, D))
    got = ctx.pack_diagonals(torch.from_numpy(W).cuda(), lanes=lanes, lane_shift=shift, baby_steps=B,
                             giant_base=base, giant_count=G).cpu().numpy()
    assert np.array_equal(got, O.pack_diagonals(W, lanes, shift, B, base, G, ctx.max_slots))


@pytest.mark.parametrize("D,lanes,shift,B,base,G", [(96, 8, 5, 1, 3, 2), (96, 4, 7, 2, 1, 3), (64, 8, 0, 3, 0, 2),
                                                    (96, 2, 11, 4, 2, 2), (64, 4, 3, 5, 0, 2), (64, 1, 0, 8, 1, 1)])
def test_packed_baby_groups(env, D, lanes, shift, B, base, G):
    """The packer's groups of 1, 2, 4 and 8 baby steps a thread, full and one over."""
    test_packed_baby_chunks(env, D, lanes, shift, B, base, G)
