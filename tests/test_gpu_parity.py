"""Parity of the HIP path (through the C ABI) with the CPU oracle on identical
seeded networks and inputs.  Tolerances:
  fp32: policy probabilities and value within 1e-4 max abs; raw planes rel-L2 <= 1e-5
  fp16: policy within 2e-2, value within 2e-2; raw planes rel-L2 <= 2e-2
Deep random-init networks saturate softmax/tanh, so the raw 1x1 planes and the
logits are compared relatively as well.
"""
import threading

import numpy as np
import pytest

from helpers import max_abs, rel_l2

pytestmark = pytest.mark.gpu


def make_pipes(pkg, netgen, orc, blocks, filters, seed, precision, max_batch, winograd=False):
    """winograd: one Winograd position of layer 1 is scaled, which no 3x3 filter can express, so
    that a network of either precision runs the Winograd kernels whatever its width."""
    net = netgen.make_network(blocks, filters, seed)
    w, h = netgen.prepare(net)
    w_ref, h_ref = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    if winograd:
        for ws in (w, w_ref):
            u = np.array(ws.m_conv_weights[1], np.float32).reshape(36, filters, filters)
            u[14] *= 1.25
            ws.m_conv_weights[1] = u
    ref = orc.OraclePipe()
    ref.initialize(filters)
    ref.push_weights(6, 18, filters, w_ref)
    pipe = pkg.HIPScheduler(precision, max_batch)
    pipe.initialize(filters)
    pipe.push_weights(6, 18, filters, w)
    pipe.push_heads(h)
    return net, pipe, ref, h_ref


@pytest.mark.parametrize("precision,winograd", [(0, False), (0, True), (1, False), (1, True)])
@pytest.mark.parametrize("filters,n", [(8, 3), (64, 3), (192, 3), (192, 30), (128, 3), (128, 40),
                                       (256, 3), (256, 16), (256, 20), (256, 40)])
def test_single_layer_stages(pkg, netgen, orc, precision, winograd, filters, n):
    """V, M and Y of one convolution layer against the oracle's stages, for the input
    layer (18 planes) and a residual-tower layer with a skip connection.  The M stage is
    the check the reference's tuner makes of every GEMM it times, against a plain sgemm
    (reference src/Tuner.cpp:262-301).  A layer is a direct convolution: Y is what a forward
    computes, V and M come from its filters by the tiled kernels.  With filters that are no 3x3
    ones (winograd) all three are the stages of such a network's forward; in fp32, 128 and 256
    filters then put the streaming GEMM under it, at 3 boards (one 32-row block per work-group)
    and at 40 (several blocks per work-group, a last block of 8 rows)."""
    print("case: single_layer precision=%d filters=%d n=%d" % (precision, filters, n), flush=True)
    net, pipe, ref, _ = make_pipes(pkg, netgen, orc, 1, filters, 40 + filters, precision,
                                   max(4, n), winograd)
    rng = np.random.default_rng(filters)
    tol = 1e-5 if precision == 0 else 4e-3
    # layer 0 on real input planes
    x = netgen.synthetic_inputs(n, seed=3)
    V, M, Y = pipe.debug_layer(0, x)
    for i in range(n):
        Vr = orc.transform_in(x[i], 18)
        Mr = orc.sgemm(ref.U[0], Vr, 18, filters)
        Yr = orc.batchnorm(orc.transform_out(Mr, filters), ref.mean[0], ref.scale[0])
        assert rel_l2(V[i], Vr) <= tol, ("V layer0", i)
        assert rel_l2(M[i], Mr) <= tol, ("M layer0", i)
        assert rel_l2(Y[i], Yr) <= tol, ("Y layer0", i)
    # layer 2 (second conv of the block) with a residual input
    a = np.abs(rng.standard_normal((n, filters, 361))).astype(np.float32)
    r = np.abs(rng.standard_normal((n, filters, 361))).astype(np.float32)
    if precision == 1:  # make the inputs exactly representable in half precision
        a = a.astype(np.float16).astype(np.float32)
        r = r.astype(np.float16).astype(np.float32)
    V, M, Y = pipe.debug_layer(2, a, r)
    for i in range(n):
        Vr = orc.transform_in(a[i], filters)
        Mr = orc.sgemm(ref.U[2], Vr, filters, filters)
        Yr = orc.batchnorm(orc.transform_out(Mr, filters), ref.mean[2], ref.scale[2], r[i])
        assert rel_l2(V[i], Vr) <= tol, ("V layer2", i)
        assert rel_l2(M[i], Mr) <= tol, ("M layer2", i)
        assert rel_l2(Y[i], Yr) <= 2 * tol, ("Y layer2", i)
    pipe.close()


def check_outputs(pkg, orc, pipe, ref, h_ref, x, precision, idx=None, all_raw=False):
    """Raw planes, logits, policy and value of the HIP pipe against the oracle.

    The reference's answer is itself only defined up to its BLAS back-end's summation
    order (OpenBLAS / Eigen / MKL builds exist).  On random-init networks the logits
    reach 1e3..1e8, so a last-ulp change of the planes can move a non-saturated
    probability by more than 1e-4.  Each position is therefore also evaluated with the
    oracle's second sgemm provider; where the two oracle runs disagree by more than a
    fifth of the tolerance, the position is reported as ill-conditioned (with the gap
    between its two largest logits) and compared at 10x their disagreement instead.  At
    most one position of a case may take that route.  Raw planes and logits are always
    compared at the strict relative tolerance, for every position checked; with all_raw
    the raw planes of every position of the batch are (the oracle runs them on all host
    threads), whatever idx selects for the head outputs.  Every position checked must also
    pass the engine's own run-time self-check (Network::compare_net_outputs, reference
    src/Network.cpp:666-691): the L2 norm over the 362 policy entries and the winrate
    (1 + value) / 2 at most 0.2, with no relaxation for ill-conditioned positions."""
    raw_tol = 1e-5 if precision == 0 else 2e-2
    p_tol = 1e-4 if precision == 0 else 2e-2
    policy, value, logits, pol, val = pipe.evaluate_batch(x, want_raw=True)
    worst = dict(pol=0.0, val=0.0, logits=0.0, policy=0.0, value=0.0, ill_conditioned=0,
                 engine_selfcheck=0.0)
    if all_raw:
        import os
        rp_all, rv_all, _ = ref.forward_many(x, threads=min(16, os.cpu_count() or 1))
        for i in range(x.shape[0]):
            e_pol, e_val = rel_l2(pol[i], rp_all[i]), rel_l2(val[i], rv_all[i])
            assert e_pol <= raw_tol and e_val <= raw_tol, ("raw planes", i, e_pol, e_val)
            worst["pol"] = max(worst["pol"], e_pol)
            worst["val"] = max(worst["val"], e_val)
    have_blas = orc.use_openblas() != "builtin"
    orc.use_builtin()
    for i in (range(x.shape[0]) if idx is None else idx):
        rp, rv = ref.forward(x[i])
        hd = orc.heads(h_ref, rp, rv)
        tol_i = p_tol
        if have_blas:
            orc.use_openblas()
            rp2, rv2 = ref.forward(x[i])
            orc.use_builtin()
            hd2 = orc.heads(h_ref, rp2, rv2)
            noise = max(max_abs(hd["policy"], hd2["policy"]), abs(hd["value"] - hd2["value"]))
            if noise > p_tol / 5:
                worst["ill_conditioned"] += 1
                tol_i = max(p_tol, 10 * noise)
                top = np.sort(hd["logits"])[-2:]
                print("ill-conditioned position %d: top-2 logit gap %.4g, oracle back ends "
                      "differ by %.3g, compared at %.3g" % (i, float(top[1] - top[0]), noise,
                                                            tol_i), flush=True)
        worst["pol"] = max(worst["pol"], rel_l2(pol[i], rp))
        worst["val"] = max(worst["val"], rel_l2(val[i], rv))
        e_l = rel_l2(logits[i], hd["logits"])
        worst["logits"] = max(worst["logits"], e_l)
        assert e_l <= raw_tol, ("logits", i, e_l)
        e_p = max_abs(policy[i], hd["policy"])
        e_v = abs(float(value[i]) - hd["value"])
        worst["policy"] = max(worst["policy"], e_p)
        worst["value"] = max(worst["value"], e_v)
        assert e_p <= tol_i and e_v <= tol_i, (i, e_p, e_v, tol_i)
        d = np.asarray(policy[i], np.float64) - np.asarray(hd["policy"], np.float64)
        e_engine = float(np.sqrt(np.sum(d * d) + (0.5 * (float(value[i]) - hd["value"])) ** 2))
        worst["engine_selfcheck"] = max(worst["engine_selfcheck"], e_engine)
        assert e_engine <= 0.2, ("engine self-check bar", i, e_engine)
        assert abs(float(policy[i].sum()) - 1.0) < 1e-4
    print("parity", worst, flush=True)
    assert worst["pol"] <= raw_tol and worst["val"] <= raw_tol, worst
    assert worst["ill_conditioned"] <= 1, worst
    return worst


@pytest.mark.parametrize("blocks,filters,batch,precision", [
    (1, 8, 3, 0),       # the shape of the reference's test network (1 block x 8 filters)
    (6, 128, 1, 0),     # the smallest benchmark configuration: 6x128 fp32 batch 1
    (15, 192, 8, 0),    # 15x192 fp32 batch 8
    (1, 8, 3, 1),
    (6, 128, 4, 1),     # the same small net in fp16: the non-saturated fp16 check
    (2, 96, 5, 1),
])
def test_forward_parity(pkg, netgen, orc, blocks, filters, batch, precision):
    print("case: forward %dx%d b%d precision=%d" % (blocks, filters, batch, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, blocks, filters, 1000 + blocks, precision,
                                       batch)
    x = netgen.synthetic_inputs(batch, seed=blocks * 7 + filters)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, precision)
    pipe.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("batch", [72, 64, 52, 41, 36, 35, 33, 32, 24, 21, 18, 17, 16, 10, 9, 8, 2, 1])
def test_forward_parity_wide_batches(pkg, netgen, orc, precision, batch):
    """256 filters at batch sizes on both sides of changes of kernel shape (fp32: the streaming
    GEMM with 1 to 8 blocks of 32 tile rows per work-group; fused transform: 64 channels per
    work-group from 21 boards, 32 from 17, 16 below; fp16: the direct convolution's tiles), in both
    precisions, including batches whose tile count is not a multiple of any tile height."""
    print("case: wide 3x256 b%d precision=%d" % (batch, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 3, 256, 3000, precision, batch)
    x = netgen.synthetic_inputs(batch, seed=batch)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, precision,
                  idx=sorted({0, min(1, batch - 1), batch // 2, batch - 1}))
    pipe.close()


@pytest.mark.parametrize("blocks,filters,batch", [(20, 256, 32), (40, 256, 64), (15, 192, 16),
                                                  (10, 128, 24)])
def test_forward_parity_deep_fp16(pkg, netgen, orc, blocks, filters, batch):
    """Deep fp16 towers: the two large fp16 benchmark configurations (20x256 batch 32, 40x256
    batch 64) at full size, and 15x192 and 10x128, under per-layer activation scales: raw planes of
    every position of the batch against the oracle, head outputs of three of them."""
    print("case: deep fp16 %dx%d b%d" % (blocks, filters, batch), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, blocks, filters, 2000 + blocks,
                                       pkg.FP16, batch)
    x = netgen.synthetic_inputs(batch, seed=blocks)
    s = pipe.act_scales()
    print("act scales: first %s last %s" % (s[:3], s[-3:]), flush=True)
    assert np.all(s >= 1.0) and np.all(np.log2(s) == np.round(np.log2(s)))
    check_outputs(pkg, orc, pipe, ref, h_ref, x, pkg.FP16, idx=[0, batch // 2, batch - 1],
                  all_raw=True)
    pipe.close()


def test_forward_parity_deep_fp16_with_plain_half_storage(pkg, netgen, orc):
    """40x256 at batch 64 with batch-norm statistics that keep the activations O(1) through
    all 40 blocks, as a trained network's do: the activation scales then come out as 1 for
    every layer, i.e. plain half-precision storage as in the reference's half pipeline, the
    heads are not saturated, and policy and value of all 64 positions are held to the fp16
    tolerance where it bites (no position may take the ill-conditioned route here)."""
    from helpers import normalise_network
    print("case: deep fp16, normalised 40x256 b64", flush=True)
    blocks, filters, batch = 40, 256, 64
    net = normalise_network(netgen.make_network(blocks, filters, 2100),
                            netgen.synthetic_inputs(4, seed=2101))
    w, h = netgen.prepare(net)
    w_ref, h_ref = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    ref = orc.OraclePipe()
    ref.initialize(filters)
    ref.push_weights(6, 18, filters, w_ref)
    pipe = pkg.HIPScheduler(pkg.FP16, batch)
    pipe.initialize(filters)
    pipe.push_weights(6, 18, filters, w)
    pipe.push_heads(h)
    s = pipe.act_scales()
    print("act scales: min %g max %g" % (s.min(), s.max()), flush=True)
    assert np.all(s == 1.0), s
    x = netgen.synthetic_inputs(batch, seed=2102)
    worst = check_outputs(pkg, orc, pipe, ref, h_ref, x, pkg.FP16, all_raw=True)
    assert worst["ill_conditioned"] == 0, worst
    # not a saturated case: the mean policy maximum is far from one-hot, values spread
    policy, value, _ = pipe.evaluate_batch(x)
    print("policy max: mean %.3f; |value|: mean %.3f max %.3f"
          % (policy.max(axis=1).mean(), np.abs(value).mean(), np.abs(value).max()), flush=True)
    assert policy.max(axis=1).mean() < 0.9 and np.abs(value).mean() < 0.95
    pipe.close()


def test_failed_push_weights_leaves_the_handle_unchanged(pkg, netgen, orc):
    """push_weights is all or nothing.  An fp16 push whose calibration cannot settle (a
    layer with an infinite batch-norm scale: its activations are infinite at any scale) fails
    after the filters of every layer went up; the handle must then refuse forwards exactly as
    before any push, and accept a second push with good weights, whose results are right."""
    print("case: failed push_weights", flush=True)
    net = netgen.make_network(2, 64, 71)
    w, h = netgen.prepare(net)
    bad = pkg.ForwardPipeWeights()
    bad.__dict__.update(w.__dict__)
    bad.m_batchnorm_stddevs = [v.copy() for v in w.m_batchnorm_stddevs]
    bad.m_batchnorm_stddevs[3][:] = np.inf
    x = netgen.synthetic_inputs(3, seed=72)
    pipe = pkg.HIPScheduler(pkg.FP16, 4)
    pipe.initialize(64)
    with pytest.raises(pkg.LzhipError):
        pipe.push_weights(6, 18, 64, bad)
    with pytest.raises(ValueError, match="push_weights has not been called"):
        pipe.forward_batch(x)
    import torch
    d = torch.zeros(3, 18, 361, device="cuda")
    o1, o2 = torch.zeros(3, 722, device="cuda"), torch.zeros(3, 361, device="cuda")
    with pytest.raises(ValueError, match="push_weights has not been called"):
        pipe.forward_batch_device_noalloc(3, d.data_ptr(), o1.data_ptr(), o2.data_ptr())
    pipe.push_weights(6, 18, 64, w)            # accepted: the failed push left nothing behind
    pol, val = pipe.forward_batch(x)
    w_ref, _ = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    ref = orc.OraclePipe()
    ref.initialize(64)
    ref.push_weights(6, 18, 64, w_ref)
    for i in range(3):
        rp, rv = ref.forward(x[i])
        assert rel_l2(pol[i], rp) <= 2e-2 and rel_l2(val[i], rv) <= 2e-2
    pipe.close()


def test_golden_fixtures_on_device(pkg, netgen):
    import os
    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "tower_golden.npz"))
    for tag in ("b1f8", "b2f16"):
        blocks, filters, seed = [int(v) for v in g[tag + "_cfg"]]
        net = netgen.make_network(blocks, filters, seed)
        w, h = netgen.prepare(net)
        for precision, raw_tol, p_tol in ((pkg.FP32, 1e-5, 1e-4), (pkg.FP16, 2e-2, 2e-2)):
            pipe = pkg.HIPScheduler(precision, 4)
            pipe.initialize(filters)
            pipe.push_weights(6, 18, filters, w)
            pipe.push_heads(h)
            policy, value, logits, pol, val = pipe.evaluate_batch(g[tag + "_x"], want_raw=True)
            assert rel_l2(pol, g[tag + "_pol"]) <= raw_tol
            assert rel_l2(val, g[tag + "_val"]) <= raw_tol
            assert max_abs(policy, g[tag + "_policy"]) <= p_tol
            assert max_abs(value, g[tag + "_value"]) <= p_tol
            pipe.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_reference_weights_file_on_device(pkg, netgen, orc, precision):
    """The weights file of the reference's own unit tests (1 block x 8 filters, loaded
    through the text-format reader) against the oracle: 8 filters exercise the padding of
    the channel dimension to 64 with real weights."""
    import os
    print("case: reference weights file precision=%d" % precision, flush=True)
    net = netgen.load_weights(os.path.join(os.path.dirname(__file__), "golden", "0k.txt.gz"))
    w, h = netgen.prepare(net)
    w_ref, h_ref = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    ref = orc.OraclePipe()
    ref.initialize(net.filters)
    ref.push_weights(6, 18, net.filters, w_ref)
    pipe = pkg.HIPScheduler(precision, 8)
    pipe.initialize(net.filters)
    pipe.push_weights(6, 18, net.filters, w)
    pipe.push_heads(h)
    check_outputs(pkg, orc, pipe, ref, h_ref, netgen.synthetic_inputs(8, seed=31), precision)
    pipe.close()


def test_handle_created_from_a_weights_file(pkg, netgen, orc, tmp_path):
    """lzhip_create_from_file (reading, Winograd transform, bias folding, push of tower and
    heads in one call) gives bit for bit what the Python reader plus push_weights/push_heads
    give, for the reference's own test file (gzip) and for a seeded 2-block net written as
    format 2 in plain text; the heads it pushed serve `heads=None`, and format 2 turns the
    value round for white."""
    import os
    print("case: create from file", flush=True)
    x = netgen.synthetic_inputs(5, seed=41)
    ref_file = os.path.join(os.path.dirname(__file__), "golden", "0k.txt.gz")
    net2 = netgen.make_network(2, 24, 43)
    net2.value_head_not_stm = True
    v2_file = str(tmp_path / "v2.txt")
    netgen.save_weights(net2, v2_file)
    for path in (ref_file, v2_file):
        net = netgen.load_weights(path)
        w, h = netgen.prepare(net)
        a = pkg.HIPScheduler(pkg.FP32, 8)
        a.initialize(net.filters)
        a.push_weights(6, 18, net.filters, w)
        a.push_heads(h)
        b = pkg.HIPScheduler.from_file(path, pkg.FP32, 8)
        assert (b.filters, b.n_layers) == (net.filters, net.n_layers)
        pa, pb = a.forward_batch(x), b.forward_batch(x)
        assert np.array_equal(pa[0], pb[0]) and np.array_equal(pa[1], pb[1])
        ea, eb = a.evaluate_batch(x), b.evaluate_batch(x)
        assert np.array_equal(ea[0], eb[0]) and np.array_equal(ea[1], eb[1])
        # callers above forward(): the heads pushed from the file, and the format-2 flag
        boards = np.full((1, 361), pkg.EMPTY, np.uint8)
        boards[0, 72] = pkg.BLACK
        pol_a, win_a = a.get_output(h, boards, pkg.WHITE, 2)
        pol_b, win_b = b.get_output(None, boards, pkg.WHITE, 2)
        assert np.array_equal(pol_a, pol_b)
        want = 1.0 - win_a if net.value_head_not_stm else win_a
        assert abs(win_b - want) < 1e-7
        a.close()
        b.close()


@pytest.mark.parametrize("precision,winograd", [(0, False), (0, True), (1, False)])
@pytest.mark.parametrize("filters,maxb", [(64, 8), (128, 40), (192, 16), (192, 40), (256, 40)])
def test_batch_composition_does_not_change_results(pkg, netgen, orc, precision, winograd, filters, maxb):
    """A position evaluated alone, in a partial batch and in a full batch gives
    bit-identical planes: points and rows of the GEMM are independent, and a network's layers run
    one kernel family at every batch (whatever the tile shapes, blocks per work-group or channel
    groups the batch selects, a value is summed in the same order).  With filters that are no 3x3
    ones (winograd) fp32 at 192 filters takes the streaming GEMM in handles of up to 16 positions
    and the tiled one in larger ones."""
    print("case: batch composition %d filters precision=%d" % (filters, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, filters, 77, precision, maxb, winograd)
    x = netgen.synthetic_inputs(maxb, seed=5)
    pol_all, val_all = pipe.forward_batch(x)
    for lo, hi in ((2, 5), (4, 5), (0, min(17, maxb)), (1, min(34, maxb)), (0, 1)):
        pol, val = pipe.forward_batch(x[lo:hi])
        assert np.array_equal(pol_all[lo:hi], pol) and np.array_equal(val_all[lo:hi], val), (lo, hi)
    # a larger batch after a smaller one (stale rows in the padded tile range)
    pol_b, val_b = pipe.forward_batch(x)
    assert np.array_equal(pol_all, pol_b) and np.array_equal(val_all, val_b)
    with pytest.raises(ValueError):
        pipe.forward_batch(np.zeros((maxb + 1, 18, 361), np.float32))
    pipe.close()


def test_scheduler_concurrent_requests(pkg, netgen, orc):
    """Many threads call forward() at once: each gets its own position's result,
    identical to the batch executor's, and the batches fill."""
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 78, pkg.FP32, 8)
    x = netgen.synthetic_inputs(24, seed=6)
    pol_ref = np.concatenate([pipe.forward_batch(x[i:i + 8])[0] for i in range(0, 24, 8)])
    out = [None] * 24
    pipe.reset_stats()

    def work(i):
        for rep in range(3):
            out[i] = pipe.forward(x[i])

    th = [threading.Thread(target=work, args=(i,)) for i in range(24)]
    [t.start() for t in th]
    [t.join() for t in th]
    for i in range(24):
        assert np.array_equal(out[i][0], pol_ref[i])
    st = pipe.stats()
    assert st["requests"] == 72 and st["halted"] == 0
    assert st["max_batch_seen"] <= 8 and st["batches"] < 72
    pipe.close()


def test_drain_and_resume(pkg, netgen, orc):
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, 8, 79, pkg.FP32, 4)
    x = netgen.synthetic_inputs(1, seed=7)[0]
    pipe.forward(x)
    pipe.drain()
    with pytest.raises(pkg.NetworkHaltException):
        pipe.forward(x)
    pipe.resume()
    pol, val = pipe.forward(x)
    rp, rv = ref.forward(x)
    assert rel_l2(pol, rp) < 1e-5
    assert pipe.stats()["halted"] == 1
    pipe.close()


@pytest.mark.parametrize("winograd", [False, True])
def test_device_resident_forward_and_profile(pkg, netgen, orc, winograd):
    """The device-pointer entry point (what the bench times) gives the same planes as
    the host entry point, and the per-kernel timing hook reports every launch."""
    import torch
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 80, pkg.FP16, 4, winograd)
    x = netgen.synthetic_inputs(4, seed=8)
    pol_h, val_h = pipe.forward_batch(x)
    d_in = torch.from_numpy(x).cuda()
    d_pol = torch.zeros(4, 722, device="cuda")
    d_val = torch.zeros(4, 361, device="cuda")
    torch.cuda.synchronize()
    pipe.forward_batch_device(4, d_in.data_ptr(), d_pol.data_ptr(), d_val.data_ptr())
    pipe.sync()
    assert np.array_equal(d_pol.cpu().numpy(), pol_h) and np.array_equal(d_val.cpu().numpy(), val_h)
    ms, cnt = pipe.profile_forward(4, d_in.data_ptr(), d_pol.data_ptr(), d_val.data_ptr())
    # 2 blocks = 5 conv layers: 5 GEMMs, 4 fused out->in transforms, 1 plain of each; as direct
    # convolutions (counted with the GEMMs) one launch a layer
    assert list(cnt) == ([1, 1, 5, 1, 1, 4] if winograd else [1, 0, 5, 0, 1, 0])
    assert np.array_equal(ms > 0, cnt > 0) and np.all(ms < 50)
    rp, rv = ref.forward(x[3])
    assert rel_l2(pol_h[3], rp) <= 2e-2 and rel_l2(val_h[3], rv) <= 2e-2
    assert np.array_equal(d_pol.cpu().numpy(), pol_h)
    pipe.close()


def test_lanes_run_side_by_side_with_equal_results(pkg, netgen, orc):
    """Forwards of different batches enqueued on the handle's two lanes, many in a row with no
    synchronisation between them, give bit for bit what each batch gives alone on lane 0;
    host-buffer calls from four threads (more than there are lanes) likewise.  A lane that does not
    exist is refused."""
    import threading
    import torch
    print("case: lanes", flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 3, 128, 81, pkg.FP16, 16)
    assert pipe.lanes() == 3      # up to batch 48; two above
    xa = netgen.synthetic_inputs(16, seed=21)
    xb = netgen.synthetic_inputs(11, seed=22)
    want_a = pipe.forward_batch(xa)
    want_b = pipe.forward_batch(xb)
    d_a, d_b = torch.from_numpy(xa).cuda(), torch.from_numpy(xb).cuda()
    pol = [torch.zeros(16, 722, device="cuda") for _ in range(2)]
    val = [torch.zeros(16, 361, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    for rep in range(6):
        pipe.forward_batch_device(16, d_a.data_ptr(), pol[0].data_ptr(), val[0].data_ptr(), lane=0)
        pipe.forward_batch_device(11, d_b.data_ptr(), pol[1].data_ptr(), val[1].data_ptr(), lane=1)
    pipe.sync()
    assert np.array_equal(pol[0].cpu().numpy(), want_a[0])
    assert np.array_equal(val[0].cpu().numpy(), want_a[1])
    assert np.array_equal(pol[1].cpu().numpy()[:11], want_b[0])
    assert np.array_equal(val[1].cpu().numpy()[:11], want_b[1])
    # the roles swapped: lane 1 takes the batch lane 0 had
    pipe.forward_batch_device(16, d_a.data_ptr(), pol[1].data_ptr(), val[1].data_ptr(), lane=1)
    pipe.forward_batch_device(11, d_b.data_ptr(), pol[0].data_ptr(), val[0].data_ptr(), lane=0)
    pipe.sync()
    assert np.array_equal(pol[1].cpu().numpy(), want_a[0])
    assert np.array_equal(pol[0].cpu().numpy()[:11], want_b[0])
    # the third lane, alone and beside the others
    for rep in range(3):
        pipe.forward_batch_device(11, d_b.data_ptr(), pol[0].data_ptr(), val[0].data_ptr(), lane=0)
        pipe.forward_batch_device(16, d_a.data_ptr(), pol[1].data_ptr(), val[1].data_ptr(), lane=2)
    pipe.sync()
    assert np.array_equal(pol[1].cpu().numpy(), want_a[0])
    assert np.array_equal(val[1].cpu().numpy(), want_a[1])
    assert np.array_equal(pol[0].cpu().numpy()[:11], want_b[0])
    for lane in (3, -1):
        with pytest.raises(ValueError):
            pipe.forward_batch_device(4, d_a.data_ptr(), pol[0].data_ptr(), val[0].data_ptr(),
                                      lane=lane)

    bad = []
    def caller(x, want):
        for _ in range(8):
            got = pipe.forward_batch(x)
            if not (np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])):
                bad.append(1)
    th = [threading.Thread(target=caller, args=(xa, want_a)),
          threading.Thread(target=caller, args=(xb, want_b)),
          threading.Thread(target=caller, args=(xa[:5], (want_a[0][:5], want_a[1][:5]))),
          threading.Thread(target=caller, args=(xb[:2], (want_b[0][:2], want_b[1][:2])))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    # against the oracle as well, so that "equal" is not "equally wrong"
    for i in (0, 10):
        rp, rv = ref.forward(xb[i])
        assert rel_l2(want_b[0][i], rp) <= 2e-2 and rel_l2(want_b[1][i], rv) <= 2e-2
    pipe.close()
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, 64, 82, pkg.FP16, 52)
    assert pipe.lanes() == 2
    pipe.close()


def test_graph_replays_match_stream_launches(pkg, netgen, orc):
    """The forward is replayed from a captured HIP graph.  Replays of several graphs
    (different batch sizes and buffers), with other work and synchronisations in between,
    must reproduce the first results bit for bit, and match a pipe that launches every
    kernel on the stream (the default; graphs are enabled with LZHIP_GRAPH=1)."""
    import os
    import torch
    _, plain, _, _ = make_pipes(pkg, netgen, orc, 3, 64, 81, pkg.FP16, 8)
    os.environ["LZHIP_GRAPH"] = "1"
    try:
        net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 3, 64, 81, pkg.FP16, 8)
    finally:
        del os.environ["LZHIP_GRAPH"]
    x = netgen.synthetic_inputs(8, seed=9)
    want8 = plain.forward_batch(x)
    want3 = plain.forward_batch(x[:3])
    d_in = torch.from_numpy(x).cuda()
    d_pol = torch.zeros(8, 722, device="cuda")
    d_val = torch.zeros(8, 361, device="cuda")
    for rep in range(4):
        got8 = pipe.forward_batch(x)                      # graph (8, internal buffers)
        assert np.array_equal(got8[0], want8[0]) and np.array_equal(got8[1], want8[1]), rep
        got3 = pipe.forward_batch(x[:3])                  # graph (3, internal buffers)
        assert np.array_equal(got3[0], want3[0]) and np.array_equal(got3[1], want3[1]), rep
        d_pol.zero_()
        torch.cuda.synchronize()
        pipe.forward_batch_device(8, d_in.data_ptr(), d_pol.data_ptr(), d_val.data_ptr())
        pipe.sync()                                       # graph (8, caller buffers)
        assert np.array_equal(d_pol.cpu().numpy(), want8[0]), rep
        assert np.array_equal(d_val.cpu().numpy(), want8[1]), rep
        policy, value, _ = pipe.evaluate_batch(x[:5])     # eager head kernel after a graph
        assert policy.shape == (5, 362)
    pipe.close()
    plain.close()


@pytest.mark.parametrize("precision,winograd,filters,maxb,batches", [
    (1, False, 256, 32, (1, 5, 8, 9, 16, 17, 20, 21, 23, 32)),
    (1, False, 192, 42, (1, 7, 10, 15, 21, 22, 37, 42)),
    (1, False, 128, 64, (1, 8, 9, 18, 32, 33, 36, 44, 45, 64)),
    (0, False, 256, 32, (1, 5, 8, 9, 16, 17, 20, 21, 23, 32)),
    (0, False, 192, 16, (1, 5, 9, 15, 16)),
    (0, False, 128, 64, (1, 8, 9, 18, 32, 33, 36, 44, 45, 64)),
    (0, True, 256, 32, (1, 5, 8, 9, 16, 17, 20, 21, 23, 32)),
    (0, True, 192, 16, (1, 5, 9, 15, 16)),
    (0, True, 128, 64, (1, 8, 9, 18, 32, 33, 36, 44, 45, 64)),
])
def test_busy_lanes_and_tile_layouts_give_the_same_bits(pkg, netgen, orc, precision, winograd, filters,
                                                        maxb, batches):
    """Every batch on one lane alone, and on all lanes at once with many forwards in a row and no
    synchronisation, gives the same bits; so does, where filters are no 3x3 ones (winograd), an fp32
    handle that keeps V and M of the tower's layers in two arrays (LZHIP_INPLACE=0) beside the
    default that keeps them in one; and the result agrees with the oracle."""
    import os
    import torch
    print("case: busy lanes, %d filters precision=%d" % (filters, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 4, filters, 3100, precision, maxb, winograd)
    pipes = [pipe]
    if winograd:
        os.environ["LZHIP_INPLACE"] = "0"
        try:
            pipes.append(make_pipes(pkg, netgen, orc, 4, filters, 3100, precision, maxb, winograd)[1])
        finally:
            del os.environ["LZHIP_INPLACE"]
    x = netgen.synthetic_inputs(maxb, seed=3101)
    for n in batches:
        want = pipe.forward_batch(x[:n])
        for other in pipes[1:]:
            got = other.forward_batch(x[:n])
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), n
    nb = batches[4]
    want = pipe.forward_batch(x[:nb])
    tol = 1e-5 if precision == 0 else 2e-2
    rp, rv = ref.forward(x[7])
    assert rel_l2(want[0][7], rp) <= tol and rel_l2(want[1][7], rv) <= tol
    # every lane at once, many forwards in a row without synchronisation
    d_in = torch.from_numpy(x).cuda()
    for p in pipes:
        outs = [(torch.zeros(nb, 722, device="cuda"), torch.zeros(nb, 361, device="cuda"))
                for _ in range(p.lanes())]
        torch.cuda.synchronize()
        for rep in range(8):
            for k, (pol, val) in enumerate(outs):
                p.forward_batch_device(nb, d_in.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
        p.sync()
        for pol, val in outs:
            assert np.array_equal(pol.cpu().numpy(), want[0])
            assert np.array_equal(val.cpu().numpy(), want[1])
    for p in pipes:
        p.close()


@pytest.mark.parametrize("precision,filters", [(1, 256), (0, 256), (0, 384), (1, 384)])
def test_random_batches_on_all_lanes_match_the_plain_forward(pkg, netgen, orc, precision, filters):
    """A seeded sequence of 400 forwards of random batches (1 to 32 boards) dealt to
    random lanes with no synchronisation between them -- so that consecutive forwards of a lane
    change between tiles, and between having the device alone and sharing it -- gives, forward by
    forward, the bits of another handle that runs one batch at a time."""
    import torch
    print("case: random batches on all lanes, %d filters precision=%d" % (filters, precision), flush=True)
    maxb = 32
    net, plain, ref, h_ref = make_pipes(pkg, netgen, orc, 3, filters, 3300, precision, maxb)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 3, filters, 3300, precision, maxb)
    x = netgen.synthetic_inputs(maxb, seed=3301)
    want = {}
    rng = np.random.default_rng(3302)
    plan = [(int(rng.integers(1, maxb + 1)), int(rng.integers(0, pipe.lanes()))) for _ in range(400)]
    for n, _ in plan:
        if n not in want:
            want[n] = plain.forward_batch(x[:n])
    d_in = torch.from_numpy(x).cuda()
    outs = [(torch.zeros(maxb, 722, device="cuda"), torch.zeros(maxb, 361, device="cuda"))
            for _ in plan]
    torch.cuda.synchronize()
    for i, (n, lane) in enumerate(plan):
        pipe.forward_batch_device(n, d_in.data_ptr(), outs[i][0].data_ptr(), outs[i][1].data_ptr(),
                                  lane=lane)
        if i % 97 == 96:
            pipe.sync()           # now and then a forward finds the device empty
    pipe.sync()
    for i, (n, lane) in enumerate(plan):
        assert np.array_equal(outs[i][0].cpu().numpy()[:n], want[n][0]), (i, n, lane)
        assert np.array_equal(outs[i][1].cpu().numpy()[:n], want[n][1]), (i, n, lane)
    pipe.close()
    plain.close()


def test_error_behaviour_on_device(pkg, netgen):
    """Calls out of order and arguments out of range are refused with an error code and a
    message, never executed: forward before push_weights, push_weights twice, an even layer
    count, wrong tensor sizes, empty and oversized batches, bad precision/batch/filter
    arguments at creation, device heads before push_heads.  The pipe keeps working
    afterwards."""
    print("case: error behaviour", flush=True)
    net = netgen.make_network(1, 64, 5)
    w, h = netgen.prepare(net)
    x = netgen.synthetic_inputs(3, seed=2)
    pipe = pkg.HIPScheduler(pkg.FP32, 2)
    pipe.initialize(64)
    with pytest.raises(ValueError):
        pipe.forward_batch(x[:1])                      # no weights yet
    with pytest.raises(ValueError):
        pipe.push_weights(6, 18, 32, w)                # filter count differs from initialize
    bad = pkg.ForwardPipeWeights()
    bad.__dict__.update(w.__dict__)
    bad.m_conv_weights = w.m_conv_weights[:2]          # two layers: not 1 + 2*blocks
    bad.m_batchnorm_means = w.m_batchnorm_means[:2]
    bad.m_batchnorm_stddevs = w.m_batchnorm_stddevs[:2]
    with pytest.raises(ValueError):
        pipe.push_weights(6, 18, 64, bad)
    pipe.push_weights(6, 18, 64, w)
    with pytest.raises(ValueError):
        pipe.push_weights(6, 18, 64, w)                # twice
    with pytest.raises(ValueError):
        pipe.forward_batch(x)                          # 3 > max_batch 2
    with pytest.raises(ValueError):
        pipe.forward_batch(np.zeros((0, 18, 361), np.float32))
    with pytest.raises(ValueError):
        pipe.forward(np.zeros(100, np.float32))
    with pytest.raises(ValueError):
        pipe.evaluate_batch(x[:1])                     # device heads not pushed
    pol, val = pipe.forward_batch(x[:2])
    assert np.isfinite(pol).all() and np.isfinite(val).all()
    assert b"" == pkg.lib().lzhip_last_error()[:0]
    pipe.close()
    for args in ((pkg.FP32, 0), (pkg.FP32, 5000), (7, 4)):
        p = pkg.HIPScheduler(*args)
        with pytest.raises((ValueError, pkg.LzhipError)):
            p.initialize(64)
    p = pkg.HIPScheduler(pkg.FP32, 2)
    with pytest.raises((ValueError, pkg.LzhipError)):
        p.initialize(0)
    for prec, filters in ((pkg.FP32, 576), (pkg.FP16, 576), (pkg.FP16, 1100)):
        p = pkg.HIPScheduler(prec, 2)
        with pytest.raises(ValueError):
            p.initialize(filters)                      # no GEMM pipeline for this width
    p = pkg.HIPScheduler(pkg.FP32, 2, device=99)
    with pytest.raises(pkg.LzhipError):
        p.initialize(64)


@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("filters,batch", [(128, 1), (128, 9), (128, 30), (128, 52), (128, 72),
                                           (192, 2), (192, 16), (192, 17), (192, 40), (192, 64)])
def test_streaming_gemm_at_narrower_widths(pkg, netgen, orc, filters, batch, precision):
    """Nets whose filters are no 3x3 ones.  fp32 nets of 128 filters, and of 192 in handles of up to
    16 positions, run the streaming GEMM with 4 and 6 wavefronts per work-group (256 filters: 8);
    larger handles of 192 filters the tiled one, and so do fp16 nets at the same sizes.  The
    batches take different numbers of blocks per work-group, with tile counts that are not
    multiples of the 32-row block."""
    print("case: streaming width %d b%d precision=%d" % (filters, batch, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 5100 + filters, precision,
                                       batch, winograd=True)
    x = netgen.synthetic_inputs(batch, seed=filters + batch)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, precision,
                  idx=sorted({0, batch // 2, batch - 1}))
    pipe.close()


@pytest.mark.parametrize("filters,batch", [(640, 4), (768, 3), (896, 2), (1024, 12), (1024, 8),
                                           (384, 28), (448, 30), (320, 52)])
def test_fp16_widths_on_the_tiled_gemm(pkg, netgen, orc, filters, batch):
    """fp16 widths on the tiled GEMM kernels, where a network's filters are no 3x3 ones or its
    handle is too large for direct convolution: the widest ones -- 10, 12, 14 and 16 k-slices, at
    1024 filters the one-pass 256x256 tile (from 11 boards) and the 128x64 tile below it -- and
    widths at batches that take the 128x128 persistent and the 128x64 tiles."""
    print("case: fp16 width %d b%d" % (filters, batch), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 5000 + filters, pkg.FP16,
                                       batch, winograd=True)
    x = netgen.synthetic_inputs(batch, seed=filters + batch)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, pkg.FP16, idx=[0, batch - 1])
    pipe.close()


@pytest.mark.parametrize("precision,winograd", [(0, False), (0, True), (1, False)])
@pytest.mark.parametrize("filters,batch", [(384, 6), (512, 44), (320, 3)])
def test_other_widths(pkg, netgen, orc, precision, winograd, filters, batch):
    """Widths other than the benchmark's: direct convolution in fp32, and in fp16 at 384 and 320
    filters; the tiled GEMM's 8 k-slices in fp16 at 512; and where filters are no 3x3 ones
    (winograd) its 12, 16 and 10 k-slices in fp32, with its large tile at 512 filters."""
    print("case: width %d b%d precision=%d" % (filters, batch, precision), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 4000 + filters, precision,
                                       batch, winograd)
    x = netgen.synthetic_inputs(batch, seed=filters)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, precision, idx=[0, batch - 1])
    pipe.close()


def test_bit_packed_and_float_requests_agree(pkg, netgen, orc):
    """Queued requests whose planes hold only 0 and 1 travel one bit per value; any other
    value sends the request down the float path.  Both must give bit-for-bit what the
    batch executor gives for the same planes handed over as floats."""
    print("case: bit-packed requests", flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 91, pkg.FP32, 4)
    x = netgen.synthetic_inputs(4, seed=12)
    x[1, 3, 17] = 0.25          # not a 0/1 plane
    x[2, 16, :] = 1.0
    x[3, 17, 360] = 1.0         # the very last value: the partial last word
    pol, val = pipe.forward_batch(x)
    for i in range(4):
        p1, v1 = pipe.forward(x[i])
        assert np.array_equal(p1, pol[i]) and np.array_equal(v1, val[i]), i
    policy, value, _ = pipe.evaluate_batch(x)
    for i in (0, 1, 3):
        pe, ve = pipe.forward_eval(x[i])
        assert np.abs(pe - policy[i]).max() <= 1e-6 and abs(ve - value[i]) <= 1e-6, i
    pipe.close()


def test_fp16_range_beyond_the_calibration_positions(pkg, netgen, orc):
    """Stored activations are scaled at push_weights from 8 synthetic positions (target
    maximum 16) and clamped at 2040 on storage, by the fused and the unfused output
    transform alike.  Planes 64 times larger than anything the calibration saw still sit
    inside that range and agree with the oracle; planes 4096 times larger run into the clamp
    and must come out finite, with a policy that sums to one; and a single layer whose
    outputs exceed the clamp stores exactly min(y, 2040)."""
    print("case: fp16 range", flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 3, 128, 6100, pkg.FP16, 4)
    x = netgen.synthetic_inputs(4, seed=61)
    big = (64.0 * x).astype(np.float32)
    policy, value, logits, pol, val = pipe.evaluate_batch(big, want_raw=True)
    for i in range(4):
        rp, rv = ref.forward(big[i])
        assert rel_l2(pol[i], rp) <= 2e-2 and rel_l2(val[i], rv) <= 2e-2, i
    huge = (4096.0 * x).astype(np.float32)
    policy, value, logits, pol, val = pipe.evaluate_batch(huge, want_raw=True)
    assert np.isfinite(pol).all() and np.isfinite(val).all() and np.isfinite(logits).all()
    assert np.isfinite(policy).all() and np.isfinite(value).all()
    assert np.allclose(policy.sum(axis=1), 1.0, atol=1e-3)
    # one layer through the unfused kernel, inputs chosen so that many outputs pass 2040
    rng = np.random.default_rng(62)
    # (inputs stay inside the stored range themselves, so that V = B^T d B stays in half range)
    a = np.minimum(np.abs(rng.standard_normal((2, 128, 361))) * 600.0, 2000.0)
    a = a.astype(np.float16).astype(np.float32)
    V, M, Y = pipe.debug_layer(1, a)
    clipped = 0
    for i in range(2):
        Vr = orc.transform_in(a[i], 128)
        Mr = orc.sgemm(ref.U[1], Vr, 128, 128)
        Yr = orc.batchnorm(orc.transform_out(Mr, 128), ref.mean[1], ref.scale[1])
        want = np.minimum(Yr, 2040.0)
        clipped += int((Yr > 2040.0).sum())
        assert Y[i].max() <= 2040.0
        assert rel_l2(Y[i], want) <= 4e-3
    assert clipped > 100, clipped
    pipe.close()


@pytest.mark.parametrize("filters,batches", [
    (256, (1, 2, 3, 5, 6, 8, 9, 17, 18, 34, 35, 71)),
    (192, (1, 3, 4, 7, 8, 11, 12, 22, 23, 45, 46)),
    (128, (1, 5, 6, 11, 12, 17, 34, 35, 68, 69)),
])
def test_direct_convolution_tiles(pkg, netgen, orc, filters, batches):
    """fp16 towers of 128, 192 and 256 filters: one layer with a skip connection at batches on
    both sides of every change of tile, whole batch against a float32 convolution."""
    import torch
    import torch.nn.functional as F
    maxb = max(batches)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6600 + filters, pkg.FP16, maxb)
    rng = np.random.default_rng(filters)
    a = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    r = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    y = F.conv2d(torch.from_numpy(a.reshape(maxb, filters, 19, 19)), torch.from_numpy(net.conv_w[2]),
                 padding=1).numpy().reshape(maxb, filters, 361)
    want = np.maximum(0.0, ref.scale[2][None, :, None] * (y - ref.mean[2][None, :, None]) + r)
    for n in batches:
        print("case: direct convolution, %d filters, %d boards" % (filters, n), flush=True)
        got = pipe.debug_layer(2, a[:n], r[:n])[2]
        for i in range(n):
            assert rel_l2(got[i], want[i]) <= 2e-3, (n, i)
    pipe.close()


@pytest.mark.parametrize("filters,maxb,batches", [
    (64, 11, (1, 11)), (64, 17, (12, 17)), (64, 22, (1, 18, 22)),
    (64, 137, (11, 12, 22, 23, 34, 35, 68, 69, 102, 103, 136, 137)),
    (128, 5, (1, 5)), (128, 8, (6, 8)), (128, 11, (9, 11)),
    (192, 3, (1, 3)), (192, 5, (4, 5)), (192, 7, (1, 6, 7)), (192, 44, (44,)),
    (256, 2, (1, 2)), (256, 4, (3, 4)), (256, 5, (1, 5)),
    (384, 1, (1,)), (384, 2, (2,)), (384, 3, (1, 3)), (384, 45, (1, 5, 6, 11, 12, 17, 18, 22, 23, 44, 45)),
    (320, 2, (1, 2)), (320, 3, (3,)), (320, 4, (1, 4)), (320, 55, (3, 6, 7, 13, 20, 21, 27, 28, 55)),
    (448, 1, (1,)), (448, 2, (2,)), (448, 3, (1, 3)), (448, 9, (1, 4, 5, 9)),
    (512, 1, (1,)), (512, 2, (1, 2)), (512, 8, (1, 4, 5, 8)),
    (640, 6, (1, 3, 4, 6)), (768, 5, (5,)), (1024, 4, (1, 2, 3, 4)),
    # widths that are padded to a multiple of 64
    (24, 12, (1, 12)), (100, 5, (1, 5)), (100, 70, (12, 17, 18, 35, 52, 69, 70)),
    (200, 2, (1, 2)), (200, 36, (6, 9, 17, 18, 26, 35, 36)), (330, 4, (1, 4)),
])
def test_direct_convolution_of_small_handles_and_other_widths(pkg, netgen, orc, filters, maxb, batches):
    """fp16 towers whose handle is small enough for the convolution that deals its sum to the
    wavefronts (three tiles, both ends of each), and the tiles of 64 filters, of more than 256 and
    of padded widths: one layer with a skip connection against a float32 convolution."""
    import torch
    import torch.nn.functional as F
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6650 + filters, pkg.FP16, maxb)
    rng = np.random.default_rng(filters + maxb)
    a = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    r = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    y = F.conv2d(torch.from_numpy(a.reshape(maxb, filters, 19, 19)), torch.from_numpy(net.conv_w[2]),
                 padding=1).numpy().reshape(maxb, filters, 361)
    want = np.maximum(0.0, ref.scale[2][None, :, None] * (y - ref.mean[2][None, :, None]) + r)
    for n in batches:
        print("case: %d filters, %d boards of %d" % (filters, n, maxb), flush=True)
        got = pipe.debug_layer(2, a[:n], r[:n])[2]
        for i in range(n):
            assert rel_l2(got[i], want[i]) <= 2e-3, (n, i)
    pipe.close()


@pytest.mark.parametrize("filters,maxb,direct", [
    (64, 200, True), (100, 40, True), (256, 64, True), (320, 64, True), (384, 45, True),
    (448, 9, True), (448, 10, False), (512, 8, True), (512, 9, False), (640, 6, True),
    (640, 7, False), (768, 5, True), (768, 6, False), (1024, 4, True), (1024, 5, False)])
def test_which_handles_convolve_directly(pkg, netgen, orc, filters, maxb, direct):
    """fp16 handles of up to 384 filters, and wider ones whose largest batch makes no more than
    one tile of 96 points x 64 filters per compute unit, run one kernel per layer; the others run
    the Winograd kernels.  Both agree with the oracle, also for one position on the handle."""
    import torch
    print("case: kernels of %d filters, handles of %d" % (filters, maxb), flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6680 + filters, pkg.FP16, maxb)
    x = netgen.synthetic_inputs(maxb, seed=6681)
    d_in = torch.from_numpy(x).cuda()
    pol, val = torch.zeros(maxb, 722, device="cuda"), torch.zeros(maxb, 361, device="cuda")
    torch.cuda.synchronize()
    _, cnt = pipe.profile_forward(maxb, d_in.data_ptr(), pol.data_ptr(), val.data_ptr())
    assert (cnt[pkg.K_IN] == 0) == direct, list(cnt)
    one_pol, one_val = pipe.forward_batch(x[:1])
    assert np.array_equal(pol.cpu().numpy()[0], one_pol[0])
    assert np.array_equal(val.cpu().numpy()[0], one_val[0])
    for i in {0, maxb - 1}:
        rp, rv = ref.forward(x[i])
        assert rel_l2(pol.cpu().numpy()[i], rp) <= 2e-2, i
        assert rel_l2(val.cpu().numpy()[i], rv) <= 2e-2, i
    pipe.close()


def test_winograd_filters_of_no_3x3_filter(pkg, netgen, orc):
    """Winograd-domain filters that are not the transform of any 3x3 filter have no direct
    form: such a network runs through the Winograd kernels and agrees with the oracle."""
    net = netgen.make_network(1, 128, 6700)
    w, h = netgen.prepare(net)
    w_ref, h_ref = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    rng = np.random.default_rng(6701)
    for ws in (w, w_ref):
        ws.m_conv_weights[1] = (rng.standard_normal(36 * 128 * 128) * 0.04).astype(np.float32).reshape(36, 128, 128)
        rng = np.random.default_rng(6701)
    ref = orc.OraclePipe()
    ref.initialize(128)
    ref.push_weights(6, 18, 128, w_ref)
    pipe = pkg.HIPScheduler(pkg.FP16, 5)
    pipe.initialize(128)
    pipe.push_weights(6, 18, 128, w)
    x = netgen.synthetic_inputs(5, seed=67)
    pol, val = pipe.forward_batch(x)
    for i in range(5):
        rp, rv = ref.forward(x[i])
        assert rel_l2(pol[i], rp) <= 2e-2 and rel_l2(val[i], rv) <= 2e-2, i
    pipe.close()


@pytest.mark.parametrize("filters,maxb,batches", [
    # sums dealt to the wavefronts: the tiles of 16 and of 32 channels, both ends of each
    (64, 45, (1, 22, 23, 33, 34, 45)), (128, 11, (1, 5, 6, 8, 9, 11)), (192, 7, (1, 2, 3, 5, 6, 7)),
    (256, 5, (1, 2, 3, 4, 5)), (320, 4, (1, 2, 3, 4)), (384, 3, (1, 2, 3)), (448, 3, (1, 2, 3)),
    (512, 2, (1, 2)),
    # ... and of 64 channels
    (64, 34, (24, 34)), (128, 22, (11, 12, 17, 18, 22)), (192, 15, (7, 8, 11, 12, 15)),
    (256, 11, (5, 6, 8, 9, 11)), (320, 6, (4, 5, 6)), (384, 5, (3, 4, 5)), (448, 4, (3, 4)),
    (512, 4, (3, 4)),
    # the other tiles on both sides of every change
    (64, 137, (1, 22, 23, 34, 68, 69, 136, 137)), (128, 70, (1, 11, 12, 17, 34, 35, 68, 69, 70)),
    (192, 46, (1, 7, 8, 11, 22, 23, 45, 46)), (256, 36, (1, 5, 6, 8, 9, 17, 34, 35, 36)),
    (384, 24, (1, 3, 6, 11, 12, 23, 24)), (512, 18, (1, 4, 5, 9, 17, 18)),
    # more than a round of every tile
    (192, 121, (91, 121)), (256, 69, (69,)), (320, 28, (28,)),
    # 64 points by 64 channels
    (64, 46, (34, 35, 45, 46)), (128, 24, (17, 18, 22, 23, 24)), (192, 17, (11, 12, 15, 16, 17)),
    (256, 13, (8, 9, 11, 12, 13)), (384, 8, (5, 6, 7, 8)),
    # 128 points: 64 and 128 channels
    (64, 103, (90, 91, 102, 103)), (128, 91, (44, 46, 90, 91)), (192, 61, (16, 30, 31, 60, 61)),
    (256, 46, (20, 22, 23, 45, 46)), (384, 31, (13, 14, 15, 30, 31)),
    # widths that are padded to a multiple of 64
    (24, 46, (1, 46)), (100, 12, (1, 12)), (200, 6, (1, 6)),
])
def test_fp32_direct_convolution(pkg, netgen, orc, filters, maxb, batches):
    """fp32 towers of 3x3 filters: one layer with a skip connection against a float64 convolution.
    The bound is what fp32 sums of 9 * filters products show (rounding of a partial sum per 32
    products and part: 2^-24 sqrt(9 * filters * 3 / 32) at most, times two for what the matrix
    instruction drops); boards of very different magnitude side by side keep their own scale."""
    import torch
    import torch.nn.functional as F
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6900 + filters, pkg.FP32, maxb)
    rng = np.random.default_rng(filters + maxb)
    a = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float32)
    r = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float32)
    size = 10.0 ** rng.integers(-12, 13, maxb).astype(np.float32)   # one magnitude a board
    size[0] = 1.0
    a *= size[:, None, None]
    r *= size[:, None, None]
    y = F.conv2d(torch.from_numpy(a.reshape(maxb, filters, 19, 19)).double(),
                 torch.from_numpy(net.conv_w[2]).double(), padding=1).numpy().reshape(maxb, filters, 361)
    scale, mean = ref.scale[2].astype(np.float64), ref.mean[2].astype(np.float64)
    want = np.maximum(0.0, scale[None, :, None] * (y - mean[None, :, None]) + r)
    bound = 2.0 * 2.0 ** -24 * (9 * filters * 3 / 32) ** 0.5 + 2.0 ** -22
    for n in batches:
        print("case: fp32, %d filters, %d boards of %d" % (filters, n, maxb), flush=True)
        got = pipe.debug_layer(2, a[:n], r[:n])[2]
        for i in range(n):
            assert rel_l2(got[i], want[i]) <= bound, (n, i, rel_l2(got[i], want[i]), bound)
    pipe.close()


@pytest.mark.parametrize("filters,batches", [
    (64, (90, 91, 103, 136, 137, 181, 182)), (128, (45, 46, 90, 91)), (192, (22, 23, 30, 31, 60, 61)),
    (256, (20, 22, 23, 45, 46)), (384, (12, 14, 15, 30, 31)), (320, (14, 17, 18, 25)),
])
def test_direct_convolution_tiles_of_128_points(pkg, netgen, orc, filters, batches):
    """fp16 tiles of 128 points by 64 and by 128 channels on both sides of every change: one layer with a
    skip connection, whole batch against a float32 convolution, and a position's bits in the
    smallest and in the largest batch."""
    import torch
    import torch.nn.functional as F
    maxb = max(batches)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6620 + filters, pkg.FP16, maxb)
    rng = np.random.default_rng(filters)
    a = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    r = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float16).astype(np.float32)
    y = F.conv2d(torch.from_numpy(a.reshape(maxb, filters, 19, 19)), torch.from_numpy(net.conv_w[2]),
                 padding=1).numpy().reshape(maxb, filters, 361)
    want = np.maximum(0.0, ref.scale[2][None, :, None] * (y - ref.mean[2][None, :, None]) + r)
    one = pipe.debug_layer(2, a[:1], r[:1])[2]
    for n in batches:
        print("case: direct convolution, %d filters, %d boards" % (filters, n), flush=True)
        got = pipe.debug_layer(2, a[:n], r[:n])[2]
        assert np.array_equal(got[0], one[0])
        for i in range(n):
            assert rel_l2(got[i], want[i]) <= 2e-3, (n, i)
    pipe.close()


@pytest.mark.parametrize("filters,batches", [
    (64, (1, 5, 6, 8, 9)), (128, (1, 2, 3, 4, 5)), (192, (1, 2, 3)), (256, (1, 2, 3)),
    (320, (1, 2)), (384, (1, 2)), (448, (1, 2)), (512, (1, 2)),
    (24, (1, 5, 6)), (200, (1, 2)),           # padded to 64 and 256
    # a wavefront's 16 channels of tiles of 48 and of 64 points
    (64, (34, 35, 45, 46)), (128, (17, 18, 22, 23)), (192, (11, 12, 15, 16)), (256, (8, 9, 11, 12)),
    (384, (5, 6, 7, 8)), (512, (4, 5, 6)),
    # more than a round of every tile, for a forward with the device to itself
    (128, (136, 137, 181, 182)), (192, (90, 91, 120, 121, 136, 137)), (256, (68, 69, 90, 91, 137)),
    (384, (45, 46, 60, 61)), (320, (27, 28, 36, 37)),
])
def test_direct_convolution_tiles_of_16_channels(pkg, netgen, orc, filters, batches):
    """The same for the tiles of 16 channels, of small handles and of a wavefront: both sides of
    every change to the next one."""
    test_direct_convolution_tiles_of_128_points(pkg, netgen, orc, filters, batches)


@pytest.mark.parametrize("filters,batches", [
    (128, (1, 11, 12, 14)), (192, (1, 2, 3, 5, 7)), (192, (1, 7, 8, 9)), (256, (1, 2, 3, 5)), (256, (1, 5, 6, 7)),
    (128, (15,)), (192, (10,)), (256, (8,)),     # the first handles that no longer deal out their sums
])
def test_sums_dealt_to_more_wavefronts(pkg, netgen, orc, filters, batches):
    """Handles whose layers deal their sum to the wavefronts, up to tiles of 80 points: each tile against a
    float32 convolution, and on several lanes, where a wavefront has two shares of the sum, the bits of one lane."""
    test_direct_convolution_tiles_of_128_points(pkg, netgen, orc, filters, batches)
    test_layers_replayed_on_several_lanes(pkg, netgen, orc, filters, pkg.FP16, batches)


@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("filters,batches", [
    # 80x128 to 160x128 and 192x128 points by channels, the last batch of each and the first of the next
    (256, (23, 28, 29, 34, 35, 39, 40, 45, 46, 51, 52, 56, 57)),
    (128, (46, 56, 57, 68, 69, 79, 80, 90, 91, 102, 103, 113, 114)),
    (384, (15, 18, 19, 22, 23, 26, 27, 30, 31, 33, 34, 37, 38)),
    (192, (31, 37, 38)), (320, (19, 22, 23)),       # 160x64
    (256, (70, 81, 100)),                           # more than a round
])
def test_direct_convolution_tiles_in_steps_of_16_points(pkg, netgen, orc, precision, filters, batches):
    """Tiles whose four wavefronts stand side by side, and 160x64, on both sides of every change, with the
    bounds of the tests above."""
    if precision == pkg.FP16:
        test_direct_convolution_tiles_of_128_points(pkg, netgen, orc, filters, batches)
    else:
        test_fp32_direct_convolution(pkg, netgen, orc, filters, max(batches), batches)


@pytest.mark.parametrize("filters,last", [(24, 16), (64, 16), (128, 16), (192, 16), (256, 16), (512, 16)])
def test_first_layer_from_the_callers_planes(pkg, netgen, orc, filters, last):
    """fp16 batches whose first layer reads the planes as floats, up to the last that does and the next one, which
    packs them: the same bits, with values that are not 0 and 1 and some beyond the stored range."""
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 7150 + filters, pkg.FP16, last + 1)
    x = netgen.synthetic_inputs(last + 1, seed=7151)
    rng = np.random.default_rng(7152)
    x.reshape(last + 1, -1)[:] += rng.standard_normal(x.shape).reshape(last + 1, -1).astype(np.float32) * 0.1
    x.reshape(last + 1, -1)[:, ::997] = 7e4
    print("case: first layer, %d filters, %d boards" % (filters, last), flush=True)
    pol, val = pipe.forward_batch(x)
    for n in (1, 2, 9, last):
        p, v = pipe.forward_batch(x[:n])
        assert np.array_equal(p, pol[:n]) and np.array_equal(v, val[:n]), n
    pipe.close()


@pytest.mark.parametrize("filters,maxb,batches", [
    (64, 46, (45, 46)), (64, 45, (1, 5, 6, 8, 9, 11, 12, 22, 23, 34, 35, 45)),
    (192, 15, (1, 7, 8, 11, 12, 15)), (320, 6, (1, 4, 5, 6)), (384, 5, (1, 3, 4, 5)),
])
def test_fp32_tiles_dealt_to_wavefronts(pkg, netgen, orc, filters, maxb, batches):
    """fp32 tiles whose blocks are dealt to two or three wavefronts, the smallest and the largest batch of each,
    with the bounds of the test above; position 0 has the same bits in all of them, also on several lanes."""
    test_fp32_direct_convolution(pkg, netgen, orc, filters, maxb, batches)
    test_layers_replayed_on_several_lanes(pkg, netgen, orc, filters, pkg.FP32, batches)


@pytest.mark.parametrize("filters,maxb", [(128, 40), (192, 16), (192, 40), (256, 9), (384, 28), (512, 44)])
def test_fp32_filters_of_no_3x3_filter(pkg, netgen, orc, filters, maxb):
    """fp32 networks whose filters are no 3x3 ones run the Winograd kernels: the streaming GEMM, the
    tiled ones, and one position on the handle with the same bits."""
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, filters, 6950 + filters, pkg.FP32, maxb,
                                       winograd=True)
    x = netgen.synthetic_inputs(maxb, seed=6951)
    check_outputs(pkg, orc, pipe, ref, h_ref, x, 0, idx=[0, maxb - 1])
    pol, val = pipe.forward_batch(x)
    one_pol, one_val = pipe.forward_batch(x[:1])
    assert np.array_equal(pol[0], one_pol[0]) and np.array_equal(val[0], one_val[0])
    pipe.close()


def test_fp32_range_and_values_that_are_no_numbers(pkg, netgen, orc):
    """fp32 planes of any magnitude, an infinity and a NaN among them: planes 1e30 and 1e-30 times
    the engine's agree with the oracle's at the same magnitudes, and an infinity or a NaN in one
    position leaves the other positions of the batch as they are."""
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 6960, pkg.FP32, 4)
    x = netgen.synthetic_inputs(4, seed=6961)
    want = pipe.forward_batch(x)
    for factor in (1e30, 1e-30, 3e-3):
        big = (factor * x).astype(np.float32)
        pol, val = pipe.forward_batch(big)
        for i in range(4):
            rp, rv = ref.forward(big[i])
            assert rel_l2(pol[i], rp) <= 1e-5 and rel_l2(val[i], rv) <= 1e-5, (factor, i)
    for bad in (np.inf, np.nan, -np.inf):
        y = x.copy()
        y[1].reshape(-1)[5] = bad
        pol, val = pipe.forward_batch(y)
        for i in (0, 2, 3):
            assert np.array_equal(pol[i], want[0][i]) and np.array_equal(val[i], want[1][i]), (bad, i)
    pipe.close()


@pytest.mark.parametrize("filters,maxb,batches", [
    (64, 8, (1, 8)), (192, 8, (1, 2, 3, 8)), (256, 5, (1, 2, 3, 5)), (320, 4, (1, 2, 4)), (384, 3, (1, 2, 3)),
    (448, 3, (1, 3)), (512, 4, (1, 2, 3, 4)), (512, 9, (1, 4, 9)),
])
def test_fp32_largest_planes_in_the_last_tile(pkg, netgen, orc, filters, maxb, batches):
    """fp32 layers whose results are 1e6 times larger in their last channel: read with the scale of the other
    tiles' peaks they would leave fp16's range.  The bound is that of planes of any magnitude above."""
    net = netgen.make_network(1, filters, 6970 + filters)
    for layer in (0, 1):
        net.conv_w[layer][-1] *= 1e6
    w, h = netgen.prepare(net)
    w_ref, h_ref = netgen.prepare(net, orc.winograd_transform_f, orc.process_bn_var)
    ref = orc.OraclePipe()
    ref.initialize(filters)
    ref.push_weights(6, 18, filters, w_ref)
    pipe = pkg.HIPScheduler(pkg.FP32, maxb)
    pipe.initialize(filters)
    pipe.push_weights(6, 18, filters, w)
    x = netgen.synthetic_inputs(maxb, seed=6971)
    for n in batches:
        print("case: fp32 peaks, %d filters, %d boards of %d" % (filters, n, maxb), flush=True)
        pol, val = pipe.forward_batch(x[:n])
        for i in {0, n - 1}:
            rp, rv = ref.forward(x[i])
            assert rel_l2(pol[i], rp) <= 1e-5 and rel_l2(val[i], rv) <= 1e-5, (n, i)
    pipe.close()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 100])
def test_heads_at_the_edges_of_their_tiles(pkg, netgen, orc, n):
    """The fully connected heads work on tiles of 32 positions by 32 outputs, and sixteen
    partial sums meet for each output.  Against float64 from the raw planes of the same call; a
    sum of K products and a bias in fp32, in any order, is within (K + 4) 2^-24 of the sum of
    the magnitudes (two of the four roundings are the batch norm's)."""
    print("case: heads n=%d" % n, flush=True)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 1, 32, 7100, pkg.FP32, 100)
    x = netgen.synthetic_inputs(n, seed=71)
    policy, value, logits, pol, val = pipe.evaluate_batch(x, want_raw=True)

    def fc(a, w, b):
        w = np.asarray(w, np.float64).reshape(len(b), -1)
        bound = (a.shape[1] + 4) * 2.0 ** -24 * (np.abs(a) @ np.abs(w).T + np.abs(b))
        return a @ w.T + b, bound

    def bn(a, mean, scale, per):
        mean, scale = (np.repeat(np.asarray(v, np.float64), per) for v in (mean, scale))
        return np.maximum(0.0, scale * (a.astype(np.float64) - mean))

    h = h_ref
    p = bn(pol, h.bn_pol_mean, h.bn_pol_scale, 361)
    want, bound = fc(p, h.ip_pol_w, np.asarray(h.ip_pol_b, np.float64))
    assert (np.abs(logits - want) <= bound).all(), (np.abs(logits - want) / bound).max()
    e = np.exp(logits.astype(np.float64) - logits.max(axis=1, keepdims=True))
    assert np.abs(policy - e / e.sum(axis=1, keepdims=True)).max() <= 1e-5
    v = bn(val, h.bn_val_mean, h.bn_val_scale, 361)
    hid, hb = fc(v, h.ip1_val_w, np.asarray(h.ip1_val_b, np.float64))
    hid = np.maximum(0.0, hid)
    out, ob = fc(hid, h.ip2_val_w, np.asarray(h.ip2_val_b, np.float64))
    ob = ob + hb @ np.abs(np.asarray(h.ip2_val_w, np.float64)).reshape(-1, 1)
    # (tanh has slope at most 1; its own error is a few units of the last place of 1)
    assert (np.abs(value - np.tanh(out[:, 0])) <= ob[:, 0] + 4 * 2.0 ** -24).all()
    pipe.close()


@pytest.mark.parametrize("filters,precision,sizes", [
    (64, 1, (1, 3, 20)), (128, 1, (2, 20, 21)), (192, 1, (8, 9)), (256, 1, (1, 5, 6)), (64, 0, (1, 8, 9)),
    (64, 1, tuple(range(1, 13))),
])
def test_layers_replayed_on_several_lanes(pkg, netgen, orc, filters, precision, sizes):
    """Small forwards on two and on three lanes in turn: their layers are one launch of a graph from
    the eighth use of a batch size on.  Every forward, with new planes each and work of the
    program's own between them, gives the bits of another handle that runs one batch at a time; so do
    more batch sizes than a lane keeps graphs of, and calls from three threads."""
    import threading
    import torch
    print("case: replayed layers, %d filters, precision %d" % (filters, precision), flush=True)
    maxb = max(max(sizes), 2)
    net, plain, ref, h_ref = make_pipes(pkg, netgen, orc, 2, filters, 7300, precision, maxb)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, filters, 7300, precision, maxb)
    rounds = 14 if len(sizes) < 4 else 10
    x = netgen.synthetic_inputs(maxb + rounds, seed=7301)
    want = {(n, r): plain.forward_batch(x[r:r + n]) for n in sizes for r in range(rounds)}
    dev = torch.from_numpy(x).cuda()
    for lanes in (2, pipe.lanes()):
        for n in sizes:
            outs = []
            for r in range(rounds):
                for k in range(lanes):
                    p, v = torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")
                    torch.cuda.synchronize()
                    d = dev[r:r + n].contiguous()
                    torch.cuda.synchronize()
                    pipe.forward_batch_device(n, d.data_ptr(), p.data_ptr(), v.data_ptr(), lane=k)
                    outs.append((r, d, p, v))
                if r % 5 == 4:
                    pipe.sync()
            pipe.sync()
            for r, _, p, v in outs:
                assert np.array_equal(p.cpu().numpy(), want[n, r][0]), (lanes, n, r)
                assert np.array_equal(v.cpu().numpy(), want[n, r][1]), (lanes, n, r)
    wrong = []

    def caller(n):
        for r in range(rounds):
            pol, val = pipe.forward_batch(x[r:r + n])
            if not (np.array_equal(pol, want[n, r][0]) and np.array_equal(val, want[n, r][1])):
                wrong.append((n, r))

    th = [threading.Thread(target=caller, args=(sizes[i % len(sizes)],)) for i in range(3)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert not wrong, wrong
    pipe.close()
    plain.close()


def lzhip_events(call):
    """Names of this library's kernels that call() ran, and how many graphs it launched."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    names = [e.name for e in p.events()]
    return [n for n in names if "lzhip" in n], sum("GraphLaunch" in n for n in names)


def test_frequent_batch_sizes_are_replayed_whatever_came_first(pkg, netgen, orc):
    """Twenty batch sizes, some of them often enough for a graph each, before the one that is then used
    throughout: that one is replayed all the same, and gives the bits of the plain launches."""
    import torch
    print("case: layer graphs of frequent sizes", flush=True)
    maxb, lanes = 24, 2
    net, plain, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 7400, pkg.FP16, maxb)
    net, pipe, ref, h_ref = make_pipes(pkg, netgen, orc, 2, 64, 7400, pkg.FP16, maxb)
    x = netgen.synthetic_inputs(maxb, seed=7401)
    d_in = torch.from_numpy(x).cuda()
    outs = [(torch.zeros(maxb, 722, device="cuda"), torch.zeros(maxb, 361, device="cuda"))
            for _ in range(lanes)]
    torch.cuda.synchronize()

    def forwards(n, reps):
        for _ in range(reps):
            for k, (pol, val) in enumerate(outs):
                pipe.forward_batch_device(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
        pipe.sync()

    for n in range(1, 21):
        forwards(n, 3 if n <= 10 else 10)
    for n, reps in ((22, 12), (24, 40)):
        forwards(n, reps)
        want = plain.forward_batch(x[:n])
        for _ in range(3):
            kernels, graphs = lzhip_events(lambda: forwards(n, 2))
            assert graphs == 2 * lanes and len(kernels) == 2 * lanes * 7, (n, graphs, len(kernels))
            for pol, val in outs:
                assert np.array_equal(pol.cpu().numpy()[:n], want[0]), n
                assert np.array_equal(val.cpu().numpy()[:n], want[1]), n
    for n in range(1, 21):   # as frequent as those: more sizes than a lane has graphs
        forwards(n, 60)
        want = plain.forward_batch(x[:n])
        for pol, val in outs:
            assert np.array_equal(pol.cpu().numpy()[:n], want[0]), n
            assert np.array_equal(val.cpu().numpy()[:n], want[1]), n
    pipe.close()
    plain.close()


@pytest.mark.parametrize("precision,filters,n", [(1, 256, 70), (0, 128, 17), (1, 64, 20)])
def test_graph_replays_run_the_kernels_of_the_lanes_in_use(pkg, netgen, orc, precision, filters, n):
    """With LZHIP_GRAPH=1, forwards on one lane and then on several run the kernels that plain
    launches would: which tiles a layer takes follows the lanes in use, not those at the first call."""
    import os
    import torch
    print("case: graphs and lanes, %d filters precision=%d" % (filters, precision), flush=True)
    _, plain, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 7500, precision, n)
    os.environ["LZHIP_GRAPH"] = "1"
    try:
        _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 7500, precision, n)
    finally:
        del os.environ["LZHIP_GRAPH"]
    x = netgen.synthetic_inputs(n, seed=7501)
    want = plain.forward_batch(x)
    d_in = torch.from_numpy(x).cuda()
    outs = [(torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda"))
            for _ in range(plain.lanes())]
    torch.cuda.synchronize()

    def forwards(p, lanes, reps):
        for _ in range(reps):
            for k, (pol, val) in enumerate(outs[:lanes]):
                p.forward_batch_device(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
        p.sync()

    for lanes in (1, 2, plain.lanes(), 1):
        ran = []
        for p in (plain, pipe):
            forwards(p, lanes, 3)
            ran.append(sorted(lzhip_events(lambda: forwards(p, lanes, 4))[0]))
            for pol, val in outs[:lanes]:
                assert np.array_equal(pol.cpu().numpy(), want[0])
                assert np.array_equal(val.cpu().numpy(), want[1])
        assert len(ran[0]) == 4 * lanes * 5 and ran[0] == ran[1], (lanes, ran)
    pipe.close()
    plain.close()


@pytest.mark.parametrize("maxb,n", [(11, 6), (11, 8), (45, 8), (45, 36), (45, 45)])
def test_fp32_tiles_of_64_filters_on_three_lanes(pkg, netgen, orc, maxb, n):
    """Three fp32 forwards of 64 filters side by side take tiles of 48 points on fewer wavefronts, or in place of 64
    points, than a forward alone: other kernels and the same bits."""
    import torch
    print("case: three lanes, 64 filters, %d boards of %d" % (n, maxb), flush=True)
    _, plain, _, _ = make_pipes(pkg, netgen, orc, 1, 64, 7600, pkg.FP32, maxb)
    _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, 64, 7600, pkg.FP32, maxb)
    assert pipe.lanes() == 3
    x = netgen.synthetic_inputs(n, seed=7601)
    want = plain.forward_batch(x)
    d_in = torch.from_numpy(x).cuda()
    outs = [(torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")) for _ in range(3)]
    torch.cuda.synchronize()

    def forwards(lanes):
        for k, (pol, val) in enumerate(outs[:lanes]):
            pipe.forward_batch_device(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
        pipe.sync()

    ran = {}
    for lanes in (1, 3):
        for _ in range(3):
            forwards(lanes)
        for pol, val in outs[:lanes]:
            pol.zero_(), val.zero_()
        torch.cuda.synchronize()
        ran[lanes] = set(lzhip_events(lambda: forwards(lanes))[0])
        for pol, val in outs[:lanes]:
            assert np.array_equal(pol.cpu().numpy(), want[0]) and np.array_equal(val.cpu().numpy(), want[1]), lanes
    assert ran[1] and ran[3] - ran[1], ran
    pipe.close()
    plain.close()


@pytest.mark.parametrize("precision,filters,n,tiles", [
    (1, 320, 20, "aab"), (1, 192, 33, "aab"),       # 160x64 points by channels, or 192x64
    (1, 128, 46, "abb"), (1, 256, 24, "abb"), (1, 384, 17, "abb"),      # 80x128, or 192x64
    (0, 256, 24, "aab"), (0, 256, 30, "abb"), (0, 384, 17, "aab"), (0, 192, 33, "aaa"),
    (1, 256, 70, "ab"), (1, 192, 91, "ab"), (0, 256, 70, "ab"),         # more than a round
])
def test_large_tiles_on_one_lane_and_beside_others(pkg, netgen, orc, precision, filters, n, tiles):
    """Forwards on one, two and three lanes give the same bits.  `tiles` has a letter for each number of lanes: equal
    letters run the same kernels, others do not."""
    import torch
    print("case: large tiles beside others, %d filters, %d boards, precision %d" % (filters, n, precision), flush=True)
    _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 7700, precision, n)
    assert pipe.lanes() == len(tiles)
    x = [netgen.synthetic_inputs(n, seed=7701 + k) for k in range(len(tiles))]
    d_in = [torch.from_numpy(v).cuda() for v in x]
    outs = [(torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")) for _ in tiles]
    torch.cuda.synchronize()

    def forward(planes, lane):
        pol, val = outs[lane]
        pipe.forward_batch_device(n, d_in[planes].data_ptr(), pol.data_ptr(), val.data_ptr(), lane=lane)

    want = []
    for k in range(len(tiles)):
        for _ in range(3):
            forward(k, 0)
        pipe.sync()
        want.append([o.cpu().numpy() for o in outs[0]])
    ran = []
    for lanes in range(1, len(tiles) + 1):
        for _ in range(3):
            for k in range(lanes):
                forward(k, k)
        pipe.sync()
        for pol, val in outs:
            pol.zero_(), val.zero_()
        torch.cuda.synchronize()
        ran.append(set(lzhip_events(lambda: [forward(k, k) for k in range(lanes)] + [pipe.sync()])[0]))
        for k in range(lanes):
            assert all(np.array_equal(o.cpu().numpy(), w) for o, w in zip(outs[k], want[k])), (lanes, k)
    for i in range(len(tiles)):
        for j in range(i):
            assert ran[i] and (ran[i] == ran[j]) == (tiles[i] == tiles[j]), (i + 1, j + 1, ran)
    pipe.close()


@pytest.mark.parametrize("filters,maxb,sizes", [
    (128, 17, (1, 16)), (384, 17, (1, 9, 16)), (448, 9, (1, 9)), (512, 8, (1, 8)), (1024, 4, (1, 4)),
])
def test_first_layer_kernel_against_packed_planes(pkg, netgen, orc, filters, maxb, sizes):
    """Direct fp16 networks of all widths: a forward alone convolves the caller's planes in one launch, forwards side by side
    pack them first, and planes of 0 and 1 from host memory travel as bits.  Same bits from all three, with other values
    and some beyond the stored range from the first two."""
    import torch
    _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 7800 + filters, pkg.FP16, maxb)
    rng = np.random.default_rng(7801)
    for n in sizes:
        print("case: first layer, %d filters, %d boards of %d" % (filters, n, maxb), flush=True)
        stones = netgen.synthetic_inputs(n, seed=7802)
        other = stones + rng.standard_normal(stones.shape).astype(np.float32) * 0.1
        other.reshape(n, -1)[:, ::997] = 7e4
        for x, bits in ((stones, True), (other, False)):
            d_in = torch.from_numpy(x).cuda()
            outs = [(torch.zeros(n, 722, device="cuda"), torch.zeros(n, 361, device="cuda")) for _ in range(2)]
            torch.cuda.synchronize()

            def forwards(lanes):
                for k, (pol, val) in enumerate(outs[:lanes]):
                    pipe.forward_batch_device(n, d_in.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
                pipe.sync()

            got = []
            for lanes in (1, 2):
                for _ in range(3):
                    forwards(lanes)
                for pol, val in outs:
                    pol.zero_(), val.zero_()
                torch.cuda.synchronize()
                ran = lzhip_events(lambda: forwards(lanes))[0]
                first = sum("conv3x3_first_k" in e for e in ran)
                packs = sum("pack_input_k" in e for e in ran)
                assert (first, packs) == ((1, 0) if lanes == 1 else (0, 2)), (n, lanes, ran)
                got += [[o.cpu().numpy() for o in outs[k]] for k in range(lanes)]
            if bits:
                got.append(pipe.forward_batch(x))
            for other_way in got[1:]:
                assert all(np.array_equal(a, b) for a, b in zip(got[0], other_way)), n
            assert np.isfinite(got[0][0]).all() and np.abs(got[0][0]).max() > 0
    pipe.close()


@pytest.mark.parametrize("filters,maxb,batches", [
    # sums dealt to the wavefronts: every tile of a handle
    (64, 45, (5, 6, 8, 9, 11, 12, 22, 23, 34, 35, 45)), (128, 23, (4, 5, 8, 11, 12, 22, 23)),
    (192, 15, (3, 7, 8, 11, 12, 15)), (256, 11, (2, 5, 6, 8, 11)), (320, 6, (2, 4, 5, 6)), (384, 5, (2, 3, 4, 5)),
    (512, 4, (2, 3, 4)),
    # and not: small tiles, steps of 16 points by 128 channels, 160x64, more than a round
    (64, 182, (22, 35, 68, 91, 137, 182)), (128, 114, (17, 34, 46, 57, 68, 80, 91, 103, 114)),
    (192, 91, (11, 16, 22, 31, 38, 61, 91)), (256, 70, (8, 12, 17, 23, 29, 35, 40, 46, 52, 57, 70)),
    (320, 28, (9, 13, 19, 23, 28)), (384, 38, (5, 8, 15, 19, 23, 27, 31, 34, 38)),
])
def test_fp32_tiles_give_a_position_the_same_bits(pkg, netgen, orc, filters, maxb, batches):
    """One layer of an fp32 handle with a skip connection: the first position of every batch, and the last one, whose tile
    is the ragged one, have the bits that they have alone, whatever tile the batch takes and however large
    the boards beside them are."""
    _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 7900 + filters, pkg.FP32, maxb)
    rng = np.random.default_rng(filters + maxb)
    a = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float32)
    r = np.abs(rng.standard_normal((maxb, filters, 361))).astype(np.float32)
    size = 10.0 ** rng.integers(-12, 13, maxb).astype(np.float32)
    a *= size[:, None, None]
    r *= size[:, None, None]
    first = pipe.debug_layer(2, a[:1], r[:1])[2]
    for n in batches:
        print("case: fp32 bits, %d filters, %d boards of %d" % (filters, n, maxb), flush=True)
        got = pipe.debug_layer(2, a[:n], r[:n])[2]
        last = pipe.debug_layer(2, a[n - 1:n], r[n - 1:n])[2]
        assert np.array_equal(got[0], first[0]) and np.array_equal(got[n - 1], last[0]), n
    pipe.close()


@pytest.mark.parametrize("filters,batches", [(192, (1, 3, 7)), (256, (1, 2, 5))])
def test_sum_of_64_channels_is_one_chain(pkg, netgen, orc, filters, batches):
    """fp16 layers of 192 and 256 filters, handles that deal their sums: 64 input channels are summed one k-step after
    the other, by whichever wavefronts, so that a network's outputs stay what they are.  Channels 0 to 31 bring 1.5 * 2^24,
    where fp32 has steps of 2; channels 32 to 63 then bring 0.5 in each of nine steps, which is lost nine times (summed
    apart they would be 4); the next 64 channels take the first sum away."""
    net = netgen.make_network(1, filters, 8000 + filters)
    w2 = np.zeros_like(net.conv_w[2])
    w2[:, 0, 1, 1], w2[:, 64, 1, 1] = 4096.0, -4096.0
    w2[:, 32] = 0.5
    net.conv_w[2] = w2
    net.bn_mean[2][:], net.bn_var[2][:] = -1.0, 1.0
    w, _ = netgen.prepare(net)
    pipe = pkg.HIPScheduler(pkg.FP16, max(batches))
    pipe.initialize(filters)
    pipe.push_weights(6, 18, filters, w)
    for n in batches:
        print("case: one chain, %d filters, %d boards" % (filters, n), flush=True)
        a = np.zeros((n, filters, 361), np.float32)
        a[:, 0], a[:, 64], a[:, 32] = 6144.0, 6144.0, 1.0
        got = pipe.debug_layer(2, a, np.zeros_like(a))[2].reshape(n, filters, 19, 19)[:, :, 1:18, 1:18]
        assert np.abs(got - 1.0).max() <= 2.0 ** -10, (n, got.min(), got.max())
    pipe.close()


@pytest.mark.parametrize("filters,handles", [(128, (12, 14)), (192, (8, 9)), (256, (6, 7))])
def test_handles_past_the_dealt_sums_have_the_bits_of_large_ones(pkg, netgen, orc, filters, handles):
    """fp16 handles whose largest batch is just past 64 points x 32 channels on every unit give the bits of a handle of 32."""
    print("case: handles of %s, %d filters" % (handles, filters), flush=True)
    x = netgen.synthetic_inputs(max(handles), seed=8101)
    _, large, _, _ = make_pipes(pkg, netgen, orc, 2, filters, 8100, pkg.FP16, 32)
    for maxb in handles:
        _, pipe, _, _ = make_pipes(pkg, netgen, orc, 2, filters, 8100, pkg.FP16, maxb)
        for n in (1, maxb):
            want, got = large.forward_batch(x[:n]), pipe.forward_batch(x[:n])
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), (maxb, n)
        pipe.close()
    large.close()


@pytest.mark.parametrize("precision,filters,n,like", [(1, 384, 53, 59), (0, 384, 53, 59), (1, 256, 81, 89)])
def test_no_third_round_of_the_smallest_tiles(pkg, netgen, orc, precision, filters, n, like):
    """Three rounds of 80x128 points by channels are slower than two of 128x128, which a forward of a few boards more takes."""
    import torch
    print("case: rounds, %d filters, %d and %d boards, precision %d" % (filters, n, like, precision), flush=True)
    _, pipe, _, _ = make_pipes(pkg, netgen, orc, 1, filters, 8200, precision, like)
    d_in = torch.from_numpy(netgen.synthetic_inputs(like, seed=8201)).cuda()
    outs = {b: (torch.zeros(b, 722, device="cuda"), torch.zeros(b, 361, device="cuda")) for b in (n, like)}
    torch.cuda.synchronize()

    def forward(b):
        pipe.forward_batch_device(b, d_in.data_ptr(), outs[b][0].data_ptr(), outs[b][1].data_ptr())
        pipe.sync()

    ran = {}
    for b in outs:
        forward(b)
        ran[b] = set(lzhip_events(lambda: forward(b))[0])
    assert ran[n] and ran[n] == ran[like], ran
    for a, b in zip(outs[n], outs[like]):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy()[:n])
    pipe.close()


@pytest.mark.parametrize("filters,n,like", [(384, 38, 122), (256, 57, 187)])
def test_no_more_rounds_of_smaller_tiles(pkg, netgen, orc, filters, n, like):
    """Five rounds of 112x128 or seven of 80x128 are slower than three of 192x128, the tile of a full round."""
    test_no_third_round_of_the_smallest_tiles(pkg, netgen, orc, pkg.FP16, filters, n, like)
