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


# rulebooks other than a regular one in key order: stride, submanifold, transposed, what else
OTHERS = {"stride 3": (3, 0, 0, ""), "stride 4": (4, 0, 0, ""), "submanifold": (1, 1, 0, ""),
          "transposed": (2, 0, 1, ""), "rows in any order": (1, 0, 0, "rows"),
          "pairs in any order": (1, 0, 0, "pairs"), "two ranges": (1, 0, 0, 128),
          "second split": (1, 0, 0, 32)}


@pytest.mark.parametrize("blk", [32, 64])
@pytest.mark.parametrize("what", list(OTHERS))
def test_parts_over_other_rulebooks(what, blk, device):
    """Strides whose offsets have few pairs, submanifold and transposed rulebooks, input rows and
    pairs in any order, two ranges of rows to a workgroup and the second split of the work: both
    directions against sums in 64 bits."""
    from ss_conv.sp_ops.ops import get_indice_pairs
    s, subm, transpose, more = OTHERS[what]
    rng = np.random.default_rng(11)
    idx = random_voxels(rng, 2, 24, 6000)
    if more == "rows":
        idx = idx[rng.permutation(len(idx))]
    idx = torch.from_numpy(idx).to(device)
    o_idx, pairs, num = get_indice_pairs(idx, 2, [24] * 3, 3, s, 1, 1, 0, bool(subm), bool(transpose))
    if more == "pairs":  # a tensor the library knows nothing of, each offset's pairs shuffled
        pairs = pairs.clone()
        for k, m in enumerate(num.cpu().tolist()):
            pairs[k, :, :m] = pairs[k, :, torch.from_numpy(rng.permutation(m)).to(device)]
    flags = BLOCKS[blk] | (more if isinstance(more, int) else 0)
    g = torch.Generator().manual_seed(2)
    w = torch.randn(3, 3, 3, 64, 72, generator=g).to(device)
    n_in, n_out = idx.shape[0], o_idx.shape[0]
    for inverse, rows, out_rows, c in ((False, n_in, n_out, 64), (True, n_out, n_in, 72)):
        x = torch.randn(rows, c, generator=g).to(device)
        y = _conv(x, w, pairs, num, out_rows, inverse, flags)
        assert rel_l2(y.cpu().numpy(), _reference(x, w, pairs, num, out_rows, inverse).numpy()) < TOL
        assert torch.equal(y, _conv(x, w, pairs, num, out_rows, inverse, flags))
        if c == 64:  # (whole chunks: the form is taken)
            assert not torch.equal(y, _conv(x, w, pairs, num, out_rows, inverse, FLOAT))


def _without_plans(st):
    """The same rows and rulebook under a record without plans: they are built from the pairs."""
    from ss_conv import _ext
    from ss_conv.sp_ops.tensor import SparseTensor
    t = SparseTensor(st.features, st.indices, st.spatial_shape, st.batch_size)
    t.indice_dict, t.plan_dict = st.indice_dict, {}
    pairs, meta = st.indice_dict["a"][2], st.plan_dict["a"]
    pairs._ssc_meta = _ext.RulebookMeta(pairs._version, meta.canonical, pairs_ref=pairs, kind=meta.kind)
    return t


def test_layer_over_a_rulebook_from_a_file(device):
    """A sparse tensor saved whole and loaded again: its rulebook serves a layer as before."""
    import io
    from ss_conv.sp_ops.conv import SparseConvolution
    from ss_conv.sp_ops.tensor import SparseTensor
    torch.manual_seed(1)
    layer = SparseConvolution(3, 64, 64, 3, padding=1, bias=False, indice_key="a").to(device).eval()
    idx = torch.from_numpy(random_voxels(np.random.default_rng(4), 2, 20, 8000)).to(device)
    st = SparseTensor(torch.randn(idx.shape[0], 64, device=device), idx, [20] * 3, 2)
    with torch.no_grad():
        y = layer(st)
        file = io.BytesIO()
        torch.save((st, layer), file)
        file.seek(0)
        st2, layer2 = torch.load(file, weights_only=False)
        assert len(st2.plan_dict["a"].plans) == 0 < len(st.plan_dict["a"].plans)
        z = layer2(st2)
        assert rel_l2(z.features.cpu().numpy(), y.features.cpu().numpy()) < TOL
        assert torch.equal(z.features, layer(_without_plans(st)).features)


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
@pytest.mark.parametrize("what", ["inf", "nan", "both", "large", "tiny", "tinier", "subnormal", "filter inf",
                                  "filter subnormal", "filter large"])
def test_parts_cannot(what, blk, device):
    """Elements too large for the scaled parts, and sums that are not finite or next to nothing: the
    workgroup that meets one works its rows out with float instructions.  Elements and sums that
    only the scale keeps in reach of the parts."""
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
    if what == "large":  # an infinity as a scaled bfloat16
        x[some] = 3.4e38
        w *= 1e-3
    if what == "tiny":  # sums of 2^-110, whose parts' products are not rounded thanks to the scale
        x *= 2.0 ** -70
        w *= 2.0 ** -40
    if what == "tinier":  # sums some of which are below 2^-126 and not zero
        x *= 2.0 ** -64
        w *= 2.0 ** -62
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
@pytest.mark.parametrize("odd", [None, "inf", "nan", "large", "filter inf", "gate inf", "gate large"])
def test_parts_with_epilogue(blk, odd, device):
    """Batch norm and gate on the way out, also where the rows are worked out a second time: sums
    that are not finite, in a column that is stored and in a gate's, which relu and sigmoid may
    hide (an infinity's parts are an infinity and NaNs)."""
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
    with torch.no_grad():
        w = block.conv.eval_weight(x)
        if odd in ("inf", "nan"):
            x[::200, 5] = float(odd)
        if odd == "large":  # an infinity once scaled, the sums are none
            x[::200, 5] = 3e38
            w *= 1e-3
        if odd == "filter inf":
            w[1, 1, 2, 7, 40] = float("inf")
        if odd == "gate inf":
            w[1, 1, 2, 7, 128 + 3] = float("inf")
        if odd == "gate large":
            w[1, 1, 2, 7, 128 + 3] = 3e38
            x *= 1e-3
    got = []
    for flags in (BLOCKS[blk], FLOAT):
        try:
            assert _ext._lib.ssc_conv_tuning(flags) == 0
            with torch.no_grad():
                got.append(block(SparseTensor(x, idx, [16] * 3, 2)).features.cpu())
        finally:
            _ext._lib.ssc_conv_tuning(1)
    assert torch.equal(torch.isnan(got[0]), torch.isnan(got[1]))
    assert torch.equal(torch.isinf(got[0]) * got[0].sign(), torch.isinf(got[1]) * got[1].sign())
    fine = torch.isfinite(got[1]) & (got[1].abs() < 1e4)
    assert fine.float().mean() > 0.3 and rel_l2(got[0][fine].numpy(), got[1][fine].numpy()) < 2e-6
    huge = torch.isfinite(got[1]) & ~fine
    if odd in (None, "large"):
        assert bool(huge.any()) == (odd == "large")
    if huge.any():
        assert rel_l2(got[0][huge].double().numpy(), got[1][huge].double().numpy()) < 2e-6


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
