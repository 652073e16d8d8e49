"""Shared helpers of the parity tests: build engine + oracle from the same seeded weights."""
import os
import sys

import torch

from flint_amd.synth import ModelArgs, synth_weights


def log(*a):
    print(*a, flush=True)
    sys.stdout.flush()


# pytest's capture manager (set by conftest.py): record() lines go straight to the terminal while
# a test runs, so a long full-size test (minutes of CPU oracle work) shows its progress as it goes
CAPTURE = None


def say(line):
    """log() past pytest's output capture: the per-step / per-layer lines of the full-size tests,
    which spend minutes on the CPU oracle, reach the terminal as they are made."""
    if CAPTURE is not None:
        with CAPTURE.global_and_fixture_disabled():
            log(line)
    else:
        log(line)


def record(line):
    """say() a parity figure and, when FLINT_AMD_PARITY_OUT names a file, append it there (the
    parity summaries kept beside the profiles)."""
    say(line)
    path = os.environ.get("FLINT_AMD_PARITY_OUT")
    if path:
        os.makedirs(os.path.dirname(os.path.abspath(path)), exist_ok=True)
        with open(path, "a") as f:
            f.write(line + "\n")


def ulp_stats(e, r):
    """Distance of bf16 values e from r (same shape, any float dtype) in bf16 ulps:
    {same: fraction bit-identical, in1: fraction within one ulp of the larger magnitude of the pair,
     top: max |e - r| in ulps of the largest magnitude in the vector}."""
    e, r = e.float().reshape(-1), r.float().reshape(-1)
    d = (e - r).abs()
    own = bf16_ulp(torch.maximum(e.abs(), r.abs()))
    top = bf16_ulp(torch.maximum(e.abs().max(), r.abs().max()))
    return {"same": float((d == 0).float().mean()), "in1": float((d <= own).float().mean()),
            "top": float((d / top).max())}


def gemm_bound(x, dq):
    """(fp64 x . dq^T, the largest distance of bf16 of an fp32 sum of its exact products from it). The sum may
    go in any order of steps of 32 products: at most 32 roundings within a step, one per step of the
    accumulator and 16 where parts meet, each of 2^-23 of the magnitudes that it adds; then half a bf16 ulp."""
    xd, dd = x.double(), dq.double()
    ref = xd @ dd.T
    return ref, (x.shape[1] / 32 + 48) * 2.0 ** -23 * (xd.abs() @ dd.abs().T) + ref.abs() * 2.0 ** -8


def make_pair(name, seed=0, n_layer=None, device="cuda", weight_device="cpu", **over):
    """(args, sd, engine, oracle) for config `name` with identical bf16 master weights."""
    from flint_amd.model import Transformer
    from oracle.model import OracleModel
    cfg = dict(**__import__("flint_amd.synth", fromlist=["CONFIGS"]).CONFIGS[name])
    if n_layer is not None:
        cfg["n_layer"] = n_layer
    cfg.update(over)
    args = ModelArgs(**cfg)
    sd = synth_weights(args, seed, device=weight_device)
    eng = Transformer.from_weights(args, sd, device)
    orc = OracleModel(args, {k: v.cpu() for k, v in sd.items()})
    return args, sd, eng, orc


def fill_kv_random(eng, orc, npos, seed=1):
    """Fill cache slots [0, npos) of both engine and oracle with the same bf16 N(0,1) values."""
    g = torch.Generator().manual_seed(seed)
    shape = eng.k_cache.shape
    k = torch.randn(shape[0], shape[1], npos, shape[3], generator=g).to(torch.bfloat16)
    v = torch.randn(shape[0], shape[1], npos, shape[3], generator=g).to(torch.bfloat16)
    eng.k_cache[:, :, :npos] = k.to(eng.k_cache.device)
    eng.v_cache[:, :, :npos] = v.to(eng.v_cache.device)
    orc.k_cache[:, :, :npos] = k
    orc.v_cache[:, :, :npos] = v


def top2_margin(logits):
    v = torch.topk(logits.float(), 2).values
    return float(v[0] - v[1])


def bf16_ulp(v):
    """ulp of a bf16 value of magnitude |v| (elementwise, v fp32 tensor)."""
    a = v.abs().clamp(min=2.0 ** -126)
    return torch.pow(2.0, torch.floor(torch.log2(a)) - 7)


# fp32 summation-order noise floor of the reference semantics, per test configuration. The
# reference fixes every bf16 rounding point but not the fp32 summation order inside a linear, and
# an order difference flips single bf16 roundings that later layers spread. Each entry is
# (max|dlogit| of a row, mean|dlogit| of a row, mean|dlogit| over all rows): the largest of each
# between torch's F.linear order and other valid implementations of the CPU oracle itself
# (per-128-group partial sums in order, reversed 4-way split-K, 32-element chunks, exp2-based
# softmax / SiLU), over single decode steps at several positions with random N(0, 1) KV and the 24
# rows of one batched causal chain. A row's mean is heavy-tailed (one flipped rounding in the final
# hidden state moves many logits); the mean over many rows is what separates a valid order from a
# misplaced rounding point. tests/test_oracle_floor.py re-measures them (the 40-layer one opted
# in) and checks that a planted rounding-point mistake exceeds the bars built from them. The HIP
# kernels' own arithmetic flips a few more (v_dot2_f32_bf16 is not correctly rounded in about 2e-5
# of cases, by up to 8 ulp, measured on the GPU; exp2 and rcp are the hardware's), so no bar is
# below one layer of the 3B model's: one bf16 ulp of the top logits, and that layer's mean bars.
ORDER_FLOOR = {
    "tiny": (0.015625, 2.68e-3, 1.17e-3),
    "small": (0.04736328125, 9.85e-3, 6.89e-3),    # 4 layers: down to 90.7% of logits within 2e-2
    "wide": (0.0625, 1.11e-2, 5.78e-3),
    "flint-3b-l1": (0.046875, 5.60e-3, 1.61e-3),   # >= 99.4% of a row within 2e-2
    "flint-3b": (0.3671875, 6.31e-2, 5.08e-2),     # 40 layers: only 21-39% of logits within 2e-2
}

ULP_TOP = 2.0 ** -5            # one bf16 ulp at |logit| in [4, 8), the range of the top logits
MEAN_MIN = 2.0 * ORDER_FLOOR["flint-3b-l1"][1]   # smallest per-row mean bar: one 3B layer's
AGG_MIN = 2.0 * ORDER_FLOOR["flint-3b-l1"][2]    # smallest all-rows mean bar: one 3B layer's
NORTH_STAR_TOL = 2e-2


def logit_bar(name):
    """Bar on max|dlogit| for configuration `name`: twice the oracle's own order floor, and at
    least one bf16 ulp of the top logits."""
    return max(2.0 * ORDER_FLOOR[name][0], ULP_TOP)


def mean_bar(name):
    """Bar on one row's mean|dlogit| for configuration `name`: twice the oracle's own floor."""
    return max(2.0 * ORDER_FLOOR[name][1], MEAN_MIN)


def agg_bar(name):
    """Bar on mean|dlogit| over all rows of a check (several steps or verify rows) for
    configuration `name`: twice the oracle's own all-rows floor."""
    return max(2.0 * ORDER_FLOOR[name][2], AGG_MIN)


def near_tie(ref_logits, bar):
    """True when the reference's top-2 logits are within `bar`, so the argmax is not determined by
    the reference semantics themselves (another valid fp32 order can flip it)."""
    v = torch.topk(ref_logits.float(), 2).values
    return float(v[0] - v[1]) <= bar


def logit_stats(eng, ref):
    """{max, mean, within (fraction of logits within 2e-2), same (fraction bit-identical)}."""
    d = (eng.float() - ref.float()).abs()
    return {"max": float(d.max()), "mean": float(d.mean()),
            "within": float((d <= NORTH_STAR_TOL).float().mean()), "same": float((d == 0).float().mean())}


def compare_logits(eng, ref, name):
    """(ok, max|d|, fraction of logits within 2e-2, fraction bit-identical) against configuration
    `name`'s bars: ok = max|d| <= logit_bar(name) and mean|d| <= mean_bar(name)."""
    st = logit_stats(eng, ref)
    ok = st["max"] <= logit_bar(name) and st["mean"] <= mean_bar(name)
    return ok, st["max"], st["within"], st["same"]


def oracle_pair(orc, run):
    """The oracle's result in a second valid implementation (per-group summation order and
    exp2-based softmax / SiLU; run first: a forward writes its cache rows, which the default run
    then overwrites with its own) and in its default implementation: (alt, ref)."""
    orc.set_order("g128+exp2")
    try:
        alt = run()
    finally:
        orc.set_order("torch")
    return alt, run()


def row_bars(name, alt_st):
    """(max bar, row-mean bar) for one row: twice the larger of the configuration's recorded floor
    and this row's own floor (the oracle's second implementation against its default on the same
    input); the floor depends on the input, the recorded one is its minimum."""
    return (max(logit_bar(name), 2.0 * alt_st["max"]), max(mean_bar(name), 2.0 * alt_st["mean"]))


def check_rows(eng, ref, alt, name, label):
    """Parity of logit rows eng [M, V] against the oracle's ref [M, V], with alt [M, V] the
    oracle's second implementation on the same input: every row within row_bars, the mean
    |dlogit| over the rows (when M >= 8) within twice the larger of agg_bar's floor and the
    oracle's own mean over the rows, and the argmax equal except at the oracle's near-ties.
    Returns the number of near-tie argmax flips."""
    ties, means, alt_means = 0, [], []
    for m in range(ref.shape[0]):
        st, fl = logit_stats(eng[m], ref[m]), logit_stats(alt[m], ref[m])
        bar, mbar = row_bars(name, fl)
        means.append(st["mean"])
        alt_means.append(fl["mean"])
        am_e, am_o = int(torch.argmax(eng[m])), int(torch.argmax(ref[m]))
        log(f"{label} row {m}: max|d|={st['max']:.3e} mean {st['mean']:.2e} ({st['within']:.1%} within "
            f"2e-2) | oracle 2nd impl max|d|={fl['max']:.3e} mean {fl['mean']:.2e} | argmax {am_e}/{am_o}")
        assert st["max"] <= bar and st["mean"] <= mbar, (label, m, st, bar, mbar)
        if am_e != am_o:
            assert near_tie(ref[m], bar), (label, m)
            ties += 1
    agg, alt_agg = sum(means) / len(means), sum(alt_means) / len(alt_means)
    abar = max(agg_bar(name), 2.0 * alt_agg)
    log(f"{label}: mean|d| over the rows {agg:.3e}, oracle 2nd impl {alt_agg:.3e} (bar {abar:.2e})")
    if len(means) >= 8:
        assert agg <= abar, (label, agg, abar)
    return ties
