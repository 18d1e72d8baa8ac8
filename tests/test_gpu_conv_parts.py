"""The bfloat16-parts form of the convolution (conv_kernel.h): blocks of 32 and of 64 pairs, forced
by ssc_conv_tuning where the rule would take the float form, against sums in 64 bits."""
import numpy as np
import pytest
import torch

from test_gpu_parity import random_voxels, rel_l2

pytestmark = pytest.mark.gpu

FLOAT, BLOCKS = 1 | 1024, {32: 1 | 4096, 64: 1 | 2048}
# A sum of K * Cin products in 32 bits, each rounded once or twice: a few 2^-24 of its norm.
TOL = 5e-7


def _rulebook(n, grid, k, s, seed, device):
    from ss_conv.sp_ops.ops import get_indice_pairs
    idx = torch.from_numpy(random_voxels(np.random.default_rng(seed), 2, grid, n)).to(device)
    return (idx.shape[0],) + tuple(get_indice_pairs(idx, 2, [grid] * 3, k, s, k // 2))


def _reference(x, w, pairs, num, n_out, inverse):
    ref = torch.zeros(n_out, w.shape[-2] if inverse else w.shape[-1], dtype=torch.float64)
    w = w.reshape(-1, *w.shape[-2:]).cpu().double()
    x, pairs, a = x.cpu().double(), pairs.cpu().long(), int(inverse)
    for k, m in enumerate(num.cpu().tolist()):
        f = w[k].t() if inverse else w[k]
        ref.index_add_(0, pairs[k, 1 - a, :m], x[pairs[k, a, :m]] @ f)
    return ref


def _conv(x, w, pairs, num, n_out, inverse, flags):
    """One call under a tuning setting; the input gradient of x with `inverse`."""
    from ss_conv import _ext
    try:
        assert _ext._lib.ssc_conv_tuning(flags) == 0
        if not inverse:
            return _ext.indice_conv_fp32(x, w, pairs, num, n_out, 0, 0)
        k, ci, co = w.shape[0] * w.shape[1] * w.shape[2], w.shape[3], w.shape[4]
        return _ext._conv_any(x, w, w, (ci * co, 1, co), pairs, pairs, num, k, co, ci, n_out, True,
                              False)
    finally:
        _ext._lib.ssc_conv_tuning(1)


# voxels, grid, kernel, stride, channels in and out: no row block full and none, one row, tiles of
# several row blocks and their remainders, two and three chunks (the last half used or partly),
# column blocks with one to four groups, several tiles to a range
CASES = [(1, 6, 3, 1, 64, 64), (5, 6, 3, 1, 64, 16), (70, 8, 3, 1, 128, 72), (400, 10, 3, 2, 64, 128),
         (900, 12, 3, 1, 124, 48), (1500, 16, 3, 1, 64, 100), (900, 12, 3, 1, 188, 80),
         (2500, 16, 3, 1, 256, 136), (300, 8, 5, 1, 64, 64), (9000, 24, 3, 1, 64, 30)]


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("case", CASES)
def test_parts_match_sums_in_64_bits(case, blk, device):
    n, grid, k, s, ci, co = case
    print("case", case, blk, flush=True)
    n_in, o_idx, pairs, num = _rulebook(n, grid, k, s, 5, device)
    n_out = o_idx.shape[0]
    g = torch.Generator().manual_seed(n)
    w = torch.randn(k, k, k, ci, co, generator=g).to(device)
    for inverse, rows, out_rows, c in ((False, n_in, n_out, ci), (True, n_out, n_in, co)):
        x = torch.randn(rows, c, generator=g).to(device)
        y = _conv(x, w, pairs, num, out_rows, inverse, BLOCKS[blk])
        ref = _reference(x, w, pairs, num, out_rows, inverse)
        err = rel_l2(y.cpu().numpy(), ref.numpy())
        old = rel_l2(_conv(x, w, pairs, num, out_rows, inverse, FLOAT).cpu().numpy(), ref.numpy())
        assert err < TOL and err <= max(1.05 * old, 1e-7), (inverse, err, old)
        assert torch.equal(y, _conv(x, w, pairs, num, out_rows, inverse, BLOCKS[blk]))


@pytest.mark.parametrize("blk", [32, 64])
def test_parts_by_the_rule(blk, device):
    """Sizes at which the rule itself takes the form: the same bits as when it is forced."""
    n, grid, co = {32: (12000, 32, 64), 64: (14000, 20, 128)}[blk]
    n_in, o_idx, pairs, num = _rulebook(n, grid, 3, 1, 6, device)
    x = torch.randn(n_in, 64, device=device)
    w = torch.randn(3, 3, 3, 64, co, device=device)
    y = _conv(x, w, pairs, num, o_idx.shape[0], False, 1)
    assert torch.equal(y, _conv(x, w, pairs, num, o_idx.shape[0], False, BLOCKS[blk]))
    assert not torch.equal(y, _conv(x, w, pairs, num, o_idx.shape[0], False, FLOAT))


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("what", ["inf", "nan", "both", "large", "tiny", "subnormal", "filter inf",
                                  "filter subnormal", "filter large"])
def test_parts_cannot(what, blk, device):
    """Elements that parts do not add up to, and sums that are not finite or next to nothing: the
    workgroup that meets one works its rows out with float instructions."""
    n_in, o_idx, pairs, num = _rulebook(700, 12, 3, 1, 7, device)
    n_out = o_idx.shape[0]
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(n_in, 64, generator=g), torch.randn(3, 3, 3, 64, 72, generator=g)
    some = torch.rand(n_in, 64, generator=g) < 2e-3
    if what in ("inf", "both"):
        x[some] = float("inf")
    if what == "both":
        x[torch.rand(n_in, 64, generator=g) < 2e-3] = -float("inf")
    if what == "nan":
        x[some] = float("nan")
    if what == "large":  # rounds to an infinity as a bfloat16
        x[some] = 3.4e38
        w *= 1e-3
    if what == "tiny":  # sums below 2^-95 that are not zero
        x *= 2.0 ** -70
        w *= 2.0 ** -40
    if what == "subnormal":  # bits below 2^-133, next to nothing but times 2^100
        x *= 2.0 ** -125
        w *= 2.0 ** 100
    if what == "filter inf":
        w[1, 1, 2, 5, 7] = float("inf")
    if what == "filter subnormal":
        x *= 2.0 ** 100
        w *= 2.0 ** -125
    if what == "filter large":
        w[0, 1, 2, 5, 7] = -3.4e38
        x *= 1e-3
    x, w = x.to(device), w.to(device)
    y = _conv(x, w, pairs, num, n_out, False, BLOCKS[blk]).cpu().double()
    old = _conv(x, w, pairs, num, n_out, False, FLOAT).cpu().double()
    assert torch.equal(torch.isnan(y), torch.isnan(old))
    assert torch.equal(torch.isinf(y) * y.sign(), torch.isinf(old) * old.sign())
    fine = torch.isfinite(old)
    ref = _reference(x, w, pairs, num, n_out, False)
    if fine.all():
        assert rel_l2(y.numpy(), ref.numpy()) < TOL
    else:
        assert (~fine).any() and rel_l2(y[fine].numpy(), old[fine].numpy()) < TOL


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("ci,co", [(128, 64), (512, 72)])
def test_second_walk_is_no_further_off(ci, co, blk, device):
    """Rows that are worked out again because others of their workgroup are not finite: against
    64 bits no further off than the float form's."""
    n_in, o_idx, pairs, num = _rulebook(3000, 16, 3, 1, 9, device)
    n_out = o_idx.shape[0]
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(n_in, ci, generator=g), torch.randn(3, 3, 3, ci, co, generator=g)
    x[::100, 3] = float("inf")
    x, w = x.to(device), w.to(device)
    y = _conv(x, w, pairs, num, n_out, False, BLOCKS[blk]).cpu()
    old = _conv(x, w, pairs, num, n_out, False, FLOAT).cpu()
    ref = _reference(x, w, pairs, num, n_out, False)
    fine = torch.isfinite(ref)
    assert torch.equal(fine, torch.isfinite(y)) and 0.1 < fine.float().mean() < 0.99
    err, was = (rel_l2(v[fine].numpy(), ref[fine].numpy()) for v in (y, old))
    assert err <= 1.05 * was, (err, was)


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("where", ["rows", "filters", "scaled"])
def test_parts_hold_every_bit(where, blk, device):
    """Elements with bits down to the last one of a float, and sums far below those of ordinary
    layers, are no reason to leave the form (whose sums differ from the float form's in their last
    bits), and lose nothing in it."""
    n_in, o_idx, pairs, num = _rulebook(700, 12, 3, 1, 7, device)
    n_out = o_idx.shape[0]
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(n_in, 64, generator=g), torch.randn(3, 3, 3, 64, 72, generator=g)
    plain = _conv(x.to(device), w.to(device), pairs, num, n_out, False, BLOCKS[blk])
    if where == "scaled":  # elements with bits below 2^-133, sums of 2^-100
        for a, b in ((-105, 0), (0, -105), (-52, -53)):
            y = _conv((x * 2.0 ** a).to(device), (w * 2.0 ** b).to(device), pairs, num, n_out, False,
                      BLOCKS[blk])
            assert torch.equal(y * 2.0 ** 105, plain), (a, b)
        return
    some = torch.rand((n_in, 64) if where == "rows" else w.shape, generator=g) < 0.01
    (x if where == "rows" else w)[some] = 0.0
    none = _conv(x.to(device), w.to(device), pairs, num, n_out, False, BLOCKS[blk])
    assert not torch.equal(none, _conv(x.to(device), w.to(device), pairs, num, n_out, False, FLOAT))
    (x if where == "rows" else w)[some] = 2.0 ** -130 * 1.2345  # next to nothing beside the others
    assert torch.equal(none, _conv(x.to(device), w.to(device), pairs, num, n_out, False, BLOCKS[blk]))
    # rows (columns) of nothing but such elements, far from where the others' sums are
    (x if where == "rows" else w.view(-1, 72))[::2] = 2.0 ** -148 * torch.randint(1, 1 << 20, (64 if where == "rows" else 72,), generator=g)
    if where == "filters":
        w[:] = w.view(-1, 72)[0]
        x = x.abs()
    y = _conv(x.to(device), w.to(device), pairs, num, n_out, False, BLOCKS[blk]).cpu()
    ref = _reference(x, w, pairs, num, n_out, False)
    assert ((y.double() - ref).norm(dim=1) <= TOL * ref.norm(dim=1) + 64 * 27 * 2.0 ** -150).all()


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("odd", [False, True])
def test_parts_with_epilogue(blk, odd, device):
    """Batch norm and gate on the way out, also where the rows are worked out a second time."""
    from ss_conv import _ext
    from ss_conv.activation import Activation
    from ss_conv.batchnorm import BatchNorm
    from ss_conv.convolution import Convolution
    from ss_conv.fused import ConvBatchNormActivation
    from ss_conv.sp_ops.tensor import SparseTensor
    rs = [(8, 0), (8, 1), (8, 2), (8, 3)]
    gated = rs + [(24, 0)]
    torch.manual_seed(4)
    block = ConvBatchNormActivation(Convolution([(16, 0), (16, 1)], gated, 3, padding=1), BatchNorm(gated),
                                    Activation(rs, (torch.relu, torch.sigmoid))).to(device).eval()
    idx = torch.from_numpy(random_voxels(np.random.default_rng(8), 2, 16, 1500)).to(device)
    x = torch.randn(idx.shape[0], 64, device=device)
    if odd:
        x[3, 5] = 2.0 ** -130 * 1.2345
    got = []
    for flags in (BLOCKS[blk], FLOAT):
        try:
            assert _ext._lib.ssc_conv_tuning(flags) == 0
            with torch.no_grad():
                got.append(block(SparseTensor(x, idx, [16] * 3, 2)).features.cpu().numpy())
        finally:
            _ext._lib.ssc_conv_tuning(1)
    assert rel_l2(got[0], got[1]) < 2e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_gradients_nobody_asks_for(dtype, device):
    """A convolution whose input, or whose filters, need no gradient: the other one's bits do not
    change and nothing is returned in its place."""
    from ss_conv.sp_ops.functional import SparseConvFunction
    n_in, o_idx, pairs, num = _rulebook(700, 12, 3, 1, 7, device)
    x = torch.randn(n_in, 64, device=device).to(dtype)
    w = (torch.randn(3, 3, 3, 64, 72, device=device) / 40).to(dtype)
    dy = torch.randn(o_idx.shape[0], 72, device=device).to(dtype)
    got = {}
    for want in ((True, True), (True, False), (False, True)):
        a, b = [t.clone().requires_grad_(need) for t, need in zip((x, w), want)]
        SparseConvFunction.apply(a, b, pairs, num, o_idx.shape[0]).backward(dy)
        got[want] = a.grad, b.grad
    assert got[True, False][1] is None and got[False, True][0] is None
    assert torch.equal(got[True, False][0], got[True, True][0])
    assert torch.equal(got[False, True][1], got[True, True][1])
