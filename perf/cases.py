"""What the speed of this library is measured on: evaluations of Go positions through the
public entry points of the package, from one position on one thread to large batches on the
device, in both precisions and at the widths and depths Leela Zero networks come in.

`listed()` are fixed cases, `draw(rng)` gives more of the same ranges; `prepare` makes what a
program holds before the call, `run` is one pass, `work` what the pass cannot do without.
"""
import importlib
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

lz = importlib.import_module("leela-zero_amd")

WIDTHS = (64, 128, 192, 256, 384)
LARGEST_FP16 = (40, 256, 200)     # blocks, filters, positions of the largest listed cases
LARGEST_FP32 = (40, 256, 64)


def _case(name, kind, blocks, filters, precision, n, **more):
    c = {"name": name, "kind": kind, "blocks": blocks, "filters": filters,
         "precision": precision, "n": n, "max_batch": n, "lanes": 1}
    c.update(more)
    return c


def listed():
    return [
        # One search thread, the smallest benchmark network in single precision: an engine on a
        # small net, where the latency of one blocking evaluation is everything.
        _case("queue_6x128_fp32_1", "queue", 6, 128, "fp32", 1),
        # One search thread on a strong net in half precision, with the engine's default
        # --batchsize 5: analysis of single positions.
        _case("queue_20x256_fp16_1", "queue", 20, 256, "fp16", 1, max_batch=5),
        # The root of a search averaged over the 8 symmetries, heads on the calling thread.
        _case("average_15x192_fp16_8", "average", 15, 192, "fp16", 8),
        # The 15x192 benchmark configuration: single precision, batch 8, host arrays, heads.
        _case("host_15x192_fp32_8", "host", 15, 192, "fp32", 8),
        # Analysis of a game record: an odd number of positions in one call, host arrays, heads.
        _case("host_10x128_fp16_37", "host", 10, 128, "fp16", 37),
        # 16 search threads behind the queue at max batch 32: the search configuration.
        _case("callers_40x256_fp16_16", "callers", 40, 256, "fp16", 16, max_batch=32),
        # A small batch of a small net, already on the device.
        _case("tower_10x128_fp16_5", "tower", 10, 128, "fp16", 5),
        # The 20x256 benchmark configuration, one batch after the other.
        _case("tower_20x256_fp16_32", "tower", 20, 256, "fp16", 32),
        # The headline configuration: batches of 64 on two lanes side by side.
        _case("tower_40x256_fp16_64x2", "tower", 40, 256, "fp16", 64, lanes=2),
        # The same network in single precision.
        _case("tower_40x256_fp32_64", "tower", 40, 256, "fp32", 64),
        # A network wider than the published ones, ragged batch.
        _case("tower_10x384_fp16_44", "tower", 10, 384, "fp16", 44),
        # Many games played at once on one card: the largest batch.
        _case("tower_40x256_fp16_200", "tower", 40, 256, "fp16", 200),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("queue", "average", "host", "host", "callers", "tower", "tower", "tower"))
    precision = rng.choice(("fp16", "fp16", "fp32"))
    filters = rng.choice(WIDTHS)
    blocks = _log_int(rng, 3, 40)
    most = 200 if precision == "fp16" else 64
    lanes, max_batch = 1, None
    if kind == "queue":
        n, max_batch = 1, rng.choice((1, 5, 16, 32))
    elif kind == "average":
        n = 8
    elif kind == "host":
        n = _log_int(rng, 1, 64)
    elif kind == "callers":
        n = _log_int(rng, 2, 32)
        max_batch = rng.choice((n, 32))
    else:
        n, lanes = _log_int(rng, 1, most), rng.choice((1, 2))
    b, f, m = LARGEST_FP16 if precision == "fp16" else LARGEST_FP32
    while blocks * filters * filters * n * lanes * _rounds(kind) > b * f * f * m:
        blocks -= 1
    c = _case("", kind, blocks, filters, precision, n, lanes=lanes)
    c["max_batch"] = max_batch or n
    del c["name"]
    return c


def _rounds(kind):
    """Evaluations each caller makes in a pass."""
    return 4 if kind == "callers" else 1


# --- what a program keeps: the network on the device --------------------------------------

_kept = {}      # the one handle in use (a program holds one network), by its description


def _weights(blocks, filters):
    """A network as a pipe receives it, with the statistics of a trained one: He-normal 3x3
    filters in Winograd form, batch norm that gives the second convolution of a block a small
    share of the residual stream, heads that do not saturate."""
    g = torch.Generator(device="cuda").manual_seed(1000 * blocks + filters)

    def normal(*shape, var=1.0):
        return torch.randn(shape, generator=g, device="cuda") * var ** 0.5

    def host(t):
        return t.float().cpu().numpy()

    s2 = 2.0 ** 0.5
    G = torch.tensor([[1, 0, 0], [-2 / 3, -s2 / 3, -1 / 3], [-2 / 3, s2 / 3, -1 / 3],
                      [1 / 6, s2 / 6, 1 / 3], [1 / 6, -s2 / 6, 1 / 3], [0, 0, 1]],
                     dtype=torch.float64, device="cuda")
    GG = torch.kron(G, G).float()               # [36][9]: u = G f G^T, both row-major
    w = lz.ForwardPipeWeights()
    for l in range(1 + 2 * blocks):
        cin = lz.INPUT_CHANNELS if l == 0 else filters
        f = normal(9, cin * filters, var=2.0 / (9 * cin))
        w.m_conv_weights.append(host(GG @ f).reshape(36, cin, filters))
        w.m_conv_biases.append(np.zeros(filters, np.float32))
        w.m_batchnorm_means.append(host(normal(filters, var=0.01)))
        share = 0.15 if l >= 2 and l % 2 == 0 else 1.0
        w.m_batchnorm_stddevs.append(host(share * (0.8 + 0.4 * torch.rand(
            filters, generator=g, device="cuda"))))
    w.m_conv_pol_w, w.m_conv_pol_b = host(normal(2, filters, var=1.0 / filters)), np.zeros(2, np.float32)
    w.m_conv_val_w, w.m_conv_val_b = host(normal(filters, var=1.0 / filters)), np.zeros(1, np.float32)
    h = lz.HeadWeights()
    h.bn_pol_mean, h.bn_pol_scale = np.zeros(2, np.float32), np.ones(2, np.float32)
    h.ip_pol_w, h.ip_pol_b = host(normal(362, 722, var=1.0 / 722)), np.zeros(362, np.float32)
    h.bn_val_mean, h.bn_val_scale = np.zeros(1, np.float32), np.ones(1, np.float32)
    h.ip1_val_w, h.ip1_val_b = host(normal(256, 361, var=2.0 / 361)), np.zeros(256, np.float32)
    h.ip2_val_w, h.ip2_val_b = host(normal(256, var=0.5 / 256)), np.zeros(1, np.float32)
    return w, h


def _network(case):
    key = (case["blocks"], case["filters"], case["precision"], case["max_batch"])
    if key not in _kept:
        _kept.clear()
        w, h = _weights(case["blocks"], case["filters"])
        pipe = lz.HIPScheduler(lz.FP16 if case["precision"] == "fp16" else lz.FP32,
                               case["max_batch"])
        pipe.initialize(case["filters"])
        pipe.push_weights(6, lz.INPUT_CHANNELS, case["filters"], w)
        pipe.push_heads(h)
        _kept[key] = pipe
    return _kept[key]


# --- positions ------------------------------------------------------------------------------

def _stones(n, seed):
    """n x 8 boards: each point own with probability 0.2, the opponent's with 0.2."""
    u = np.random.default_rng(seed).random((n, 8, lz.NPTS), dtype=np.float32)
    return u < 0.2, (u >= 0.2) & (u < 0.4)


def _planes(n, seed):
    own, opp = _stones(n, seed)
    x = np.zeros((n, lz.INPUT_CHANNELS, lz.NPTS), np.float32)
    x[:, 0:8], x[:, 8:16], x[:, 16] = own, opp, 1.0
    return x


def prepare(case, seed):
    n, lanes = case["n"], case["lanes"]
    s = {"kind": case["kind"], "pipe": _network(case), "n": n}
    if case["kind"] == "average":
        own, opp = _stones(1, seed)
        s["boards"] = np.where(own[0], lz.BLACK, np.where(opp[0], lz.WHITE, lz.EMPTY)).astype(np.uint8)
    elif case["kind"] == "tower":
        s["in"] = [torch.from_numpy(_planes(n, seed + 7919 * k)).cuda() for k in range(lanes)]
        s["pol"] = [torch.zeros(n, lz.POL_SIZE, device="cuda") for _ in range(lanes)]
        s["val"] = [torch.zeros(n, lz.VAL_SIZE, device="cuda") for _ in range(lanes)]
    elif case["kind"] == "callers":
        s["x"] = _planes(n * _rounds("callers"), seed)
        s["pool"] = ThreadPoolExecutor(n)
    else:
        s["x"] = _planes(n, seed)
    return s


def _caller(pipe, x):
    return [pipe.forward(p) for p in x]


def run(s):
    pipe, n = s["pipe"], s["n"]
    if s["kind"] == "queue":            # a search thread: one blocking request
        return pipe.forward(s["x"][0])
    if s["kind"] == "average":          # Network::get_output with the average over symmetries
        return pipe.get_output_average(None, s["boards"], lz.BLACK)
    if s["kind"] == "host":             # a whole batch from host arrays, heads on the device
        policy, value, logits = pipe.evaluate_batch(s["x"])
        return policy, 0.5 * (1.0 + value), logits      # the engine's win rate
    if s["kind"] == "callers":          # n threads with one blocking request each, 4 times over
        parts = np.split(s["x"], n)
        got = [g for f in [s["pool"].submit(_caller, pipe, x) for x in parts] for g in f.result()]
        return np.stack([p for p, _ in got]), np.stack([v for _, v in got])
    for k, (x, pol, val) in enumerate(zip(s["in"], s["pol"], s["val"])):
        pipe.forward_batch_device(n, x.data_ptr(), pol.data_ptr(), val.data_ptr(), lane=k)
    return s["pol"], s["val"]


# --- what a pass cannot do without ----------------------------------------------------------

def work(case):
    """3x3 convolutions in Winograd F(4x4,3x3) form (36 products for 16 outputs, 25 tiles a
    board), the 1x1 heads and, where they run in the pass, the fully connected ones; every
    3x3 filter read once a forward in the storage type, planes in, results out."""
    e = 2 if case["precision"] == "fp16" else 4
    F, layers = case["filters"], 2 * case["blocks"]
    n, forwards = case["n"], case["lanes"] * _rounds(case["kind"])
    boards = n * forwards
    macs = 36 * 25 * F * (lz.INPUT_CHANNELS + layers * F) + 361 * 3 * F
    filters = 9 * F * (lz.INPUT_CHANNELS + layers * F) * e + 3 * F * e
    per_board = 4 * (lz.INPUT_SIZE + lz.POL_SIZE + lz.VAL_SIZE)
    if case["kind"] in ("average", "host"):
        macs += 722 * 362 + 361 * 256 + 256
        filters += 4 * (722 * 362 + 361 * 256 + 256)
        per_board = 4 * (lz.INPUT_SIZE + 2 * 362 + 1)
    return {"bytes": filters * forwards + per_board * boards, "flops": 2 * macs * boards}


def tolerance(case):
    """The repository's own parity bars: fp16 storage of every activation and filter through up
    to 81 layers (raw planes within 2e-2), fp32 sums through as many (1e-5 a layer chain, twice
    that between two implementations)."""
    return {"rel": 2e-2} if case["precision"] == "fp16" else {"rel": 2e-5}
