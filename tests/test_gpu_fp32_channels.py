"""fp32 networks whose channels differ in magnitude.  A channel may be scaled by a power of two on its
way out of a layer and back on its way into the next: batch norm and ReLU commute with it, every
product stays the same number, and sums in fp32 do not change by a bit.  Direct fp32 towers hold their
operands as two halves, relative to the largest of a board and of an output channel, so such
networks are where they could lose what fp32 holds."""
import copy

import numpy as np
import pytest

from helpers import conv3x3_f64, rel_l2, tower_f64

pytestmark = pytest.mark.gpu


def spread(net, inputs, stream, mids):
    """net with channel c of every layer's output times 2^exponent: `inputs` of the planes
    (which the caller scales), `stream` of the residual stream, mids[b] inside block b."""
    def p2(e):
        return np.ldexp(np.float32(1.0), np.asarray(e, np.int32)).astype(np.float32)

    out = copy.deepcopy(net)
    for l in range(net.n_layers):
        before = inputs if l == 0 else stream if l % 2 else mids[l // 2 - 1]
        after = mids[l // 2] if l % 2 else stream
        out.conv_w[l] = (net.conv_w[l] * p2(after)[:, None, None, None] *
                         p2(-np.asarray(before))[None, :, None, None]).astype(np.float32)
        out.bn_mean[l] = net.bn_mean[l] * p2(after)
        out.conv_b[l] = net.conv_b[l] * p2(after)
    out.pol_conv_w = (net.pol_conv_w.reshape(2, -1) * p2(-np.asarray(stream))).astype(np.float32)
    out.val_conv_w = (net.val_conv_w.reshape(1, -1) * p2(-np.asarray(stream))).astype(np.float32)
    return out


def make_pipe(pkg, netgen, net, max_batch, precision=0):
    w, _ = netgen.prepare(net)
    pipe = pkg.HIPScheduler(precision, max_batch)
    pipe.initialize(net.filters)
    pipe.push_weights(6, 18, net.filters, w)
    return pipe


def is_direct(pkg, pipe, x):
    import torch
    n = len(x)
    d_in = torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda()
    pol, val = torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")
    torch.cuda.synchronize()
    _, cnt = pipe.profile_forward(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr())
    return cnt[pkg.K_IN] == 0


def exponents(case, filters, blocks, rng):
    zero = np.zeros(filters, int)
    planes = np.zeros(18, int)
    mids = [zero] * blocks
    steps = np.array([-24, 0, 24])
    if case == "inside":
        return planes, zero, [rng.choice(steps, filters) for _ in mids], True
    if case == "stream":
        return planes, rng.choice(steps, filters), mids, True
    if case == "any":
        return planes, rng.integers(-30, 31, filters), [rng.integers(-30, 31, filters) for _ in mids], True
    if case == "planes":
        return rng.integers(-30, 31, 18), zero, mids, True
    if case == "one":        # one channel far below all others, one far above
        e = zero.copy()
        e[3], e[filters - 2] = -40, 20
        return planes, e, [e[::-1].copy() for _ in mids], True
    assert case == "extreme"   # further apart than exponents are moved: the Winograd kernels
    return planes, zero, [rng.choice(np.array([-60, 0, 50]), filters) for _ in mids], False


@pytest.mark.parametrize("case", ["inside", "stream", "any", "planes", "one", "extreme"])
@pytest.mark.parametrize("filters,maxb", [(64, 8), (64, 150), (128, 12), (200, 9), (256, 40), (512, 2)])
def test_channels_of_any_magnitude(pkg, netgen, case, filters, maxb):
    """Raw planes against a float64 network, from float planes and from planes in bits, and by the
    forward without allocations.  The bound: twice the error of the handle whose channels are alike,
    and half a unit of the last place of fp32 for the rest."""
    print("case: channels %s, %d filters, handle of %d" % (case, filters, maxb), flush=True)
    import torch
    blocks, n = 2, min(maxb, 3)
    net = netgen.make_network(blocks, filters, 8100 + filters)
    rng = np.random.default_rng(8200 + filters)
    planes, stream, mids, direct = exponents(case, filters, blocks, rng)
    x = netgen.synthetic_inputs(n, seed=8101)
    y = (x * np.ldexp(1.0, planes)[None, :, None]).astype(np.float32)
    want = tower_f64(net, x)
    plain, pipe = make_pipe(pkg, netgen, net, maxb), make_pipe(pkg, netgen, spread(net, planes, stream, mids), maxb)
    base, got = plain.forward_batch(x), pipe.forward_batch(y)
    for i in range(n):
        for k, name in enumerate(("pol", "val")):
            alike, err = rel_l2(base[k][i], want[name][i]), rel_l2(got[k][i], want[name][i])
            # (the Winograd kernels round more than the direct ones: the bound of test_gpu_parity)
            assert err <= (2 * alike + 2.0 ** -24 if direct else 1e-5), (i, name, err, alike)
    assert is_direct(pkg, pipe, y) == direct
    if filters <= 256:
        d_in = torch.from_numpy(y).cuda()
        pol, val = torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")
        torch.cuda.synchronize()
        pipe.forward_batch_device_noalloc(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr())
        pipe.sync()
        assert np.array_equal(pol.cpu().numpy(), got[0]) and np.array_equal(val.cpu().numpy(), got[1])
    if case != "planes":   # (the queue sends 0/1 planes as bits)
        one = pipe.forward(y[n - 1])
        assert np.array_equal(one[0], got[0][n - 1]) and np.array_equal(one[1], got[1][n - 1])
    pipe.close()
    plain.close()


def test_parts_of_a_network_that_share_nothing(pkg, netgen):
    """Two halves of the channels that no filter joins, one of them 2^24 below the other, and heads that
    read that one alone: its precision is its own."""
    print("case: two halves", flush=True)
    filters, half, n = 128, 64, 3
    net = netgen.make_network(2, filters, 8300)
    for l in range(1, net.n_layers):
        net.conv_w[l][:half, half:] = 0.0
        net.conv_w[l][half:, :half] = 0.0
    net.pol_conv_w[:, :half] = 0.0
    net.val_conv_w[:, :half] = 0.0
    low = np.where(np.arange(filters) < half, 0, -24)
    x = netgen.synthetic_inputs(n, seed=8301)
    want = tower_f64(net, x)
    for maxb in (3, 40):
        plain, pipe = make_pipe(pkg, netgen, net, maxb), make_pipe(
            pkg, netgen, spread(net, np.zeros(18, int), low, [low, low]), maxb)
        base, got = plain.forward_batch(x), pipe.forward_batch(x)
        for i in range(n):
            for k, name in enumerate(("pol", "val")):
                alike, err = rel_l2(base[k][i], want[name][i]), rel_l2(got[k][i], want[name][i])
                assert err <= 2 * alike + 2.0 ** -24, (maxb, i, name, err, alike)
        assert is_direct(pkg, pipe, x)
        pipe.close()
        plain.close()


@pytest.mark.parametrize("filters,maxb,layer", [(64, 8, 0), (64, 8, 2), (128, 40, 1), (128, 40, 2)])
def test_layer_with_channels_of_any_magnitude(pkg, netgen, orc, filters, maxb, layer):
    """One layer of such a network, every stage in the caller's units: Y against a float64
    convolution with every channel in its own unit (bound of test_fp32_direct_convolution), M and V against
    the oracle's stages."""
    print("case: layer %d, %d filters of %d" % (layer, filters, maxb), flush=True)
    n = 2
    rng = np.random.default_rng(8400 + layer)
    net = netgen.make_network(1, filters, 8401)
    planes, stream, mid = rng.integers(-20, 21, 18), rng.integers(-30, 31, filters), rng.integers(-30, 31, filters)
    s = spread(net, planes, stream, [mid])
    before, after = [(planes, stream), (stream, mid), (mid, stream)][layer]
    a = np.abs(rng.standard_normal((n, len(before), 361)))
    a = (a * np.ldexp(1.0, before)[None, :, None]).astype(np.float32)
    r = None
    if layer == 2:
        r = np.abs(rng.standard_normal((n, filters, 361)))
        r = (r * np.ldexp(1.0, after)[None, :, None]).astype(np.float32)
    pipe = make_pipe(pkg, netgen, s, maxb)
    assert is_direct(pkg, pipe, netgen.synthetic_inputs(n, seed=1))
    V, M, Y = pipe.debug_layer(layer, a, r)
    conv = conv3x3_f64(a.reshape(n, -1, 19, 19), s.conv_w[layer]).reshape(n, filters, 361)
    scale = 1.0 / np.sqrt(s.bn_var[layer].astype(np.float64) + 1e-5)
    want = scale[None, :, None] * (conv - s.bn_mean[layer].astype(np.float64)[None, :, None])
    want = np.maximum(0.0, want + (0.0 if r is None else r.astype(np.float64)))
    bound = 2.0 * 2.0 ** -24 * (9 * filters * 3 / 32) ** 0.5 + 2.0 ** -22
    own = np.ldexp(1.0, -np.asarray(after))[None, :, None]
    assert rel_l2(Y * own, want * own) <= bound
    w, _ = netgen.prepare(s)
    U = np.asarray(w.m_conv_weights[layer], np.float32).reshape(36, len(before), filters)
    back = np.ldexp(1.0, -np.asarray(before))
    for i in range(n):
        Vr = orc.transform_in(a[i], len(before))
        Mr = orc.sgemm(U, Vr, len(before), filters)
        Vr, Mr = Vr.reshape(36, -1, 25), Mr.reshape(36, -1, 25)
        assert rel_l2(V[i] * back[None, :, None], Vr * back[None, :, None]) <= 1e-5
        assert rel_l2(M[i] * own[0], Mr * own[0]) <= 1e-5
    pipe.close()


@pytest.mark.parametrize("precision,filters,maxb", [(0, 64, 4), (0, 128, 40), (1, 128, 40)])
@pytest.mark.parametrize("size", [1e-40, 1e-42, 3e-36, 1e-30])
def test_dead_channels_keep_the_direct_kernels(pkg, netgen, precision, filters, maxb, size):
    """Output channels whose filters have decayed to nearly nothing, below the smallest normal number
    among them, change neither the results nor the kernels of the others."""
    print("case: dead channels of %g, precision %d, %d filters" % (size, precision, filters), flush=True)
    n = 3
    net = netgen.make_network(2, filters, 8500)
    rng = np.random.default_rng(8501)
    for l, k in ((0, 3), (1, 5), (2, 7), (3, 9), (4, 1)):
        net.conv_w[l][k] = (rng.standard_normal(net.conv_w[l][k].shape) * size).astype(np.float32)
    net.bn_mean[1][5] = 0.0      # a channel that is dead altogether
    net.bn_mean[0][3] = 0.0
    net.bn_var[3][9] = 0.0       # ... and one with the statistics of such a channel
    x = netgen.synthetic_inputs(n, seed=8502)
    want = tower_f64(net, x)
    pipe = make_pipe(pkg, netgen, net, maxb, precision)
    assert is_direct(pkg, pipe, x)
    pol, val = pipe.forward_batch(x)
    tol = 1e-5 if precision == 0 else 2e-2
    for i in range(n):
        assert rel_l2(pol[i], want["pol"][i]) <= tol and rel_l2(val[i], want["val"][i]) <= tol, i
    pipe.close()


@pytest.mark.parametrize("filters,maxb", [(64, 8), (128, 40)])
@pytest.mark.parametrize("far", [24, 48])
def test_planes_in_bits_are_those_in_floats(pkg, netgen, filters, maxb, far):
    """A plane that is empty in every position, whose filters are 2^far times all others': it sets the
    factors of the input planes and nothing else.  Positions sent as bits and as floats give the same
    planes, with the precision of the network whose filters are alike."""
    print("case: empty plane, %d filters of %d, 2^%d" % (filters, maxb, far), flush=True)
    import torch
    n = 3
    net = netgen.make_network(2, filters, 8600)
    zero = np.zeros(filters, int)
    low = spread(net, np.zeros(18, int), zero - far, [zero, zero])
    low.conv_w[0][:, 17] *= np.float32(2.0 ** far)
    x = netgen.synthetic_inputs(n, seed=8601)
    assert not x[:, 17].any()
    x[1, 16] = 0.0
    want = tower_f64(net, x)
    plain, pipe = make_pipe(pkg, netgen, net, maxb), make_pipe(pkg, netgen, low, maxb)
    base, bits = plain.forward_batch(x), pipe.forward_batch(x)
    d_in = torch.from_numpy(x).cuda()
    pol, val = torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")
    torch.cuda.synchronize()
    pipe.forward_batch_device(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr())
    pipe.sync()
    assert is_direct(pkg, pipe, x)
    for i in range(n):
        one = pipe.forward(x[i])
        for k, (name, floats) in enumerate((("pol", pol), ("val", val))):
            assert np.array_equal(floats.cpu().numpy()[i], bits[k][i]), (i, name)
            assert np.array_equal(one[k], bits[k][i]), (i, name)
            alike, err = rel_l2(base[k][i], want[name][i]), rel_l2(bits[k][i], want[name][i])
            assert err <= 2 * alike + 2.0 ** -24, (i, name, err, alike)
    pipe.close()
    plain.close()


@pytest.mark.parametrize("filters,maxb", [(64, 8), (128, 40)])
@pytest.mark.parametrize("scale,mean", [(1.0, 1e8), (2.0 ** 24, 1e3), (2.0 ** 24, -1e-30)])
def test_channels_that_look_larger_than_they_are(pkg, netgen, filters, maxb, scale, mean):
    """Channels whose batch norm says that they are 2^20 and more above the others, and that never fire
    (or, with filters to match, are alike): the others keep their precision."""
    print("case: scale %g mean %g, %d filters of %d" % (scale, mean, filters, maxb), flush=True)
    n = 3
    net = netgen.make_network(2, filters, 8700)
    where = ((0, 3), (1, 5), (2, 7), (3, 9), (4, 1))
    for l, k in where:
        net.bn_mean[l][k] = mean
        if mean < 0:
            net.conv_w[l][k] *= np.float32(1.0 / scale)
    x = netgen.synthetic_inputs(n, seed=8701)
    w, _ = netgen.prepare(net)
    for l, k in where:
        w.m_batchnorm_stddevs[l] = np.array(w.m_batchnorm_stddevs[l], np.float32)
        w.m_batchnorm_stddevs[l][k] = scale
    # the same in float64: what never fires is zero whatever its scale; else the scale in the filters
    same = copy.deepcopy(net)
    for l, k in where:
        same.bn_var[l][k] = 1.0 - 1e-5
        if mean < 0:
            same.conv_w[l][k] *= np.float32(scale)
            same.bn_mean[l][k] *= scale
    want = tower_f64(same, x)
    pipe = pkg.HIPScheduler(pkg.FP32, maxb)
    pipe.initialize(filters)
    pipe.push_weights(6, 18, filters, w)
    assert is_direct(pkg, pipe, x)
    plain = make_pipe(pkg, netgen, same, maxb)
    base, got = plain.forward_batch(x), pipe.forward_batch(x)
    for i in range(n):
        for k, name in enumerate(("pol", "val")):
            alike, err = rel_l2(base[k][i], want[name][i]), rel_l2(got[k][i], want[name][i])
            assert err <= 2 * alike + 2.0 ** -24, (i, name, err, alike)
    pipe.close()
    plain.close()
