"""Timed cases of the framework: what a user has it do, through the calls they make.

Each case is a dict of plain values.  `kind` names the path; the sizes are
those of the repository's workloads (the 10,000-neuron plain block, the large
block, the region share, the 16-member judge block, the 256-member EnKF, the
window surrogates) or, for drawn cases, spread around them over the range each
path is used in.

listed()            the cases
draw(rng)           one more case of the same ranges
prepare(case, seed) inputs and handles a program holds before the call
run(state)          one pass through the public entry points
work(case)          bytes and operations a pass cannot do without
exact(case, seed)   the outputs in 64 bits, where plain torch gives them
"""
from __future__ import annotations

import math

import numpy as np
import torch

DT = 0.1            # ms per step
BOLD_PAR = dict(epsilon=200, tao_s=0.8, tao_f=0.4, tao_0=1, alpha=0.2, E_0=0.8, V_0=0.02)


def listed():
    return [
        # models/block.py's own loop: one call per step, statistics back every
        # step, then the membrane potentials; the smallest calls of the simulator
        dict(name="dropin_run_10k", kind="dropin_run", n=10_000, in_degree=100, steps=10),
        # the same network through the batched form, untuned, as a program
        # gets it that only needs the statistics afterwards
        dict(name="dropin_steps_10k", kind="dropin_steps", n=10_000, in_degree=100, steps=20),
        # the plain block tuned for its size: a batch of steps in one launch
        dict(name="plain_batch_10k", kind="plain_batch", n=10_000, in_degree=100, delay=1, steps=500),
        # the large block with its BOLD integrator, in its tuned launch shape:
        # long rows, delays 1..10, a bucket of neurons per compute unit
        dict(name="large_block", kind="large", n=5_000_000, in_degree=1000, delay=10, steps=20),
        # one GPU's share of a whole-brain model: 90 uneven regions, a
        # connectome, delays 1..40, external drive, one BOLD voxel per region
        dict(name="region_share", kind="regions", members=1, regions=90, n=10_000_000, k_intra=400, k_inter=100,
             delay=40, steps=20),
        # the judge of a data-assimilation window: copies of 16 whole-brain
        # members, small enough that each step is bound by latency
        dict(name="judge_block", kind="regions", members=16, regions=90, n=10_000, k_intra=80, k_inter=20, delay=40,
             steps=50),
        # the analysis that ends a window, at the ensemble of the whole-brain DA
        dict(name="enkf_256", kind="enkf", members=256, voxels=90, states=10),
        # one training step of the window surrogate: a mini-batch of region
        # rows (18 features, 6 targets), forward, backward and Adam
        dict(name="mlp_train_2048", kind="mlp_train", n_in=18, n_out=6, hidden=512, layers=3, batch=2048),
        # a window's forecast: every region of every member through the surrogate
        dict(name="mlp_predict_23040", kind="mlp_predict", n_in=18, n_out=6, hidden=512, layers=3, rows=23_040),
        # one training step of the recurrent surrogate over a sequence of windows
        dict(name="gru_train_32x64", kind="gru_train", n_in=18, n_out=6, hidden=256, batch=64, steps=32),
        # the surrogate's matrix product at the size it is quoted on
        dict(name="gemm_8192", kind="gemm", m=8192, n=8192, k=8192, act=0, bias=0, half=0),
        # the drop-in BOLD model, one step over every voxel of the ensemble
        dict(name="bold_23040", kind="bold", n=23_040, double=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin_run", "dropin_steps", "plain_batch", "large", "regions", "regions", "enkf", "enkf",
                       "mlp_train", "mlp_predict", "gru_train", "gemm", "bold"])
    if kind == "dropin_run":
        return dict(kind=kind, n=_log(rng, 500, 10_000), in_degree=rng.randint(10, 100), steps=10)
    if kind == "dropin_steps":
        return dict(kind=kind, n=_log(rng, 500, 10_000), in_degree=rng.randint(10, 100), steps=rng.randint(5, 20))
    if kind == "plain_batch":
        return dict(kind=kind, n=_log(rng, 1000, 20_000), in_degree=rng.randint(20, 100),
                    delay=rng.choice([1, 1, 3, 10]), steps=rng.randint(50, 500))
    if kind == "large":
        return dict(kind=kind, n=_log(rng, 150_000, 5_000_000), in_degree=rng.randint(100, 1000),
                    delay=rng.choice([1, 5, 10, 20]), steps=20)
    if kind == "regions":
        if rng.random() < 0.3:
            return dict(kind=kind, members=1, regions=rng.randint(20, 120), n=_log(rng, 300_000, 10_000_000),
                        k_intra=rng.randint(60, 400), k_inter=rng.randint(10, 100), delay=rng.choice([10, 20, 40]),
                        steps=20)
        return dict(kind=kind, members=_log(rng, 4, 256), regions=90, n=rng.randint(6_000, 12_000),
                    k_intra=rng.randint(40, 80), k_inter=rng.randint(5, 20), delay=rng.choice([10, 20, 40]),
                    steps=10 * rng.randint(1, 5))
    if kind == "enkf":
        return dict(kind=kind, members=_log(rng, 8, 256), voxels=_log(rng, 10, 200), states=rng.randint(7, 15))
    if kind == "mlp_train":
        if rng.random() < 0.5:  # a member per row: every voxel's features in, every voxel's targets out
            v = rng.randint(10, 90)
            return dict(kind=kind, n_in=8 * v, n_out=6 * v, hidden=512, layers=3, batch=rng.randint(16, 256))
        return dict(kind=kind, n_in=18, n_out=6, hidden=rng.choice([128, 256, 512]), layers=rng.randint(1, 3),
                    batch=_log(rng, 64, 2048))
    if kind == "mlp_predict":
        return dict(kind=kind, n_in=18, n_out=6, hidden=rng.choice([256, 512]), layers=rng.randint(2, 3),
                    rows=_log(rng, 90, 23_040))
    if kind == "gru_train":
        return dict(kind=kind, n_in=rng.randint(8, 200), n_out=rng.randint(4, 150), hidden=rng.choice([64, 128, 256]),
                    batch=rng.randint(8, 64), steps=rng.randint(4, 32))
    if kind == "gemm":
        return dict(kind=kind, m=32 * _log(rng, 2, 192), n=32 * _log(rng, 2, 192), k=16 * _log(rng, 4, 384),
                    act=rng.randint(0, 1), bias=rng.randint(0, 1), half=rng.randint(0, 1))
    return dict(kind="bold", n=_log(rng, 90, 23_040), double=rng.randint(0, 1))


# --------------------------------------------------------------- simulator
def _dropin_inputs(case, seed):
    """The plain block's parameters (g_ui ~ U[0.001, 0.05], 80% excitatory)
    and a random table of in_degree synapses per neuron, weights U[0, 1],
    shared by the receptors of a pair."""
    from digital_twin_brain_amd import networks

    n, k = case["n"], case["in_degree"]
    props, n_exc = networks.plain_props(n, seed=seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    # distinct synapses: one presynaptic neuron per slot, drawn from its own k-th of the network
    slot = torch.arange(k, device="cuda")
    lo = slot * n // k
    width = (slot + 1) * n // k - lo
    u = torch.rand((n, k), generator=g, device="cuda", dtype=torch.float64)
    pre = (lo + (u * width).long()).reshape(-1)
    post = torch.arange(n, device="cuda").repeat_interleave(k)
    w = torch.rand(n * k, generator=g, device="cuda")
    return props, n_exc, pre.cpu(), post.cpu(), w.cpu()


DROPIN_WARM = 22    # steps before the first pass: past the initial refractory hold (T_ref = 20 steps)
DROPIN_NOISE = 1e-3  # 10 Hz at 0.1 ms


def _prepare_dropin(case, seed):
    from digital_twin_brain_amd.block import block

    props, n_exc, pre, post, w = _dropin_inputs(case, seed)
    n = case["n"]
    ch = torch.where(pre >= n_exc, 2, 0)
    idx = torch.cat([torch.stack([ch, post, pre]), torch.stack([ch + 1, post, pre])], dim=1)
    W = torch.sparse_coo_tensor(idx, torch.cat([w, w]), (4, n, n))
    b = block(torch.from_numpy(props), W, delta_t=DT, seed=seed)
    if case["kind"] == "dropin_run":
        for _ in range(DROPIN_WARM):
            b.run(noise_rate=DROPIN_NOISE)
    else:
        b.run_steps(DROPIN_WARM, noise_rate=DROPIN_NOISE)
    return dict(case=case, block=b)


def _run_dropin(s):
    b, case = s["block"], s["case"]
    if case["kind"] == "dropin_steps":
        freq, vmean = b.run_steps(case["steps"], noise_rate=DROPIN_NOISE)
        return dict(freq=freq, vmean=vmean, V=b.V_i)
    freq, vmean = [], []
    for _ in range(case["steps"]):
        f, v = b.run(noise_rate=DROPIN_NOISE)
        freq.append(f)
        vmean.append(v)
    return dict(freq=torch.stack(freq), vmean=torch.stack(vmean), V=b.V_i)


def _philox_word0(i, step, seed):
    """Word 0 of Philox4x32-10 with counter (i, 0, step, "NOIS") and key seed
    (Salmon et al., SC'11), i an int64 array."""
    m = np.uint64(0xFFFFFFFF)
    c0, c1 = i.astype(np.uint64), np.zeros(i.shape, np.uint64)
    c2, c3 = np.full(i.shape, step, np.uint64), np.full(i.shape, 0x4E4F4953, np.uint64)
    k0, k1 = seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c0, np.uint64(0xCD9E8D57) * c2
        c0, c1, c2, c3 = ((p1 >> np.uint64(32)) ^ c1 ^ np.uint64(k0), p1 & m,
                          (p0 >> np.uint64(32)) ^ c3 ^ np.uint64(k1), p0 & m)
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c0


def _exact_dropin(case, seed):
    """models/block.py:68-150 in float64 on the same inputs and noise."""
    props, n_exc, pre, post, w = _dropin_inputs(case, seed)
    n, steps = case["n"], case["steps"]
    p = torch.from_numpy(props).double()
    S = int(p[:, 3].max()) + 1
    sub = p[:, 3].long()
    size = torch.bincount(sub, minlength=S).double()
    w = w.double()
    inh = (pre >= n_exc).long()
    decay = torch.exp(-DT / p[:, 18:22])
    V = (p[:, 8] + p[:, 9]) / 2
    J = torch.zeros(n, 4, dtype=torch.float64)
    t, t_last = 0.0, torch.zeros(n, dtype=torch.float64)
    ids = np.arange(n, dtype=np.int64)
    freq, vmean = [], []
    rate = float(np.float32(DROPIN_NOISE))
    for k in range(1, DROPIN_WARM + steps + 1):
        t += DT
        isyn = (p[:, 10:14] * (p[:, 14:18] - V[:, None]) * J).sum(1)
        vn = V + DT / p[:, 4] * (-p[:, 6] * (V - p[:, 7]) + isyn + p[:, 2])
        vi = torch.where(t >= t_last + p[:, 5], vn, p[:, 9])
        act = vi >= p[:, 8]
        V = torch.minimum(vi, p[:, 8])
        t_last[act] = t
        u = (_philox_word0(ids, k, seed) >> np.uint64(8)).astype(np.float64) / 16777216.0
        spike = (torch.from_numpy(u) < rate) | act
        hit = spike[pre]
        arr = torch.zeros(n * 2, dtype=torch.float64).index_add_(0, post[hit] * 2 + inh[hit], w[hit]).reshape(n, 2)
        J = J * decay + arr.repeat_interleave(2, dim=1)
        if k > DROPIN_WARM:
            freq.append(torch.bincount(sub[act], minlength=S).double())
            vmean.append(torch.zeros(S, dtype=torch.float64).index_add_(0, sub, V) / size)
    return dict(freq=torch.stack(freq), vmean=torch.stack(vmean), V=V)


def _native_outputs(nb, steps):
    """Device buffers that a program hands to NativeBlock.run once and reuses."""
    out = dict(events=torch.zeros(steps, dtype=torch.int64, device="cuda"),
               spikes=torch.zeros(steps, dtype=torch.int32, device="cuda"),
               freqs=torch.zeros((steps, nb.S), dtype=torch.int32, device="cuda"))
    V = torch.zeros(nb.n, dtype=torch.float32, device="cuda")
    return out, V


def _run_native(s):
    nb = s["nb"]
    nb.run(s["case"]["steps"], noise_mode=1, graph=True, **s["out"])
    nb.get("V", out=s["V"])
    return dict(s["out"], V=s["V"])


def _prepare_plain(case, seed):
    from digital_twin_brain_amd import networks
    from digital_twin_brain_amd.engine import NativeBlock

    props, n_exc = networks.plain_props(case["n"], seed=seed)
    nb = NativeBlock.fixed_indegree(props, n_exc, case["in_degree"], max_delay=case["delay"], conn_seed=seed,
                                    noise_seed=seed + 1)
    nb.set_launch(deliver_mode=2)  # what the tuner picks for blocks of this size
    out, V = _native_outputs(nb, case["steps"])
    return dict(case=case, nb=nb, out=out, V=V)


def _prepare_large(case, seed):
    from digital_twin_brain_amd import networks
    from digital_twin_brain_amd.engine import NativeBlock

    n = case["n"]
    props, n_exc = networks.large_props(n, seed=seed)
    if case["in_degree"] < 1000:  # the same drive from fewer inputs
        props[:, 10:14] *= np.float32(1000.0 / case["in_degree"])
    nb = NativeBlock.fixed_indegree(_scattered(props, seed), n_exc, case["in_degree"], max_delay=case["delay"],
                                    conn_seed=seed, noise_seed=seed + 1)
    # the shape that the tuner keeps for the large block
    nb.set_launch(deliver_mode=1, deliver_grid=1024, stage_segs=256, stage_ept=16, stage_variant=2)
    return _settle(case, nb, props)


def _scattered(props, seed):
    """The parameters that create a block with membrane potentials scattered
    between reset and threshold, and hold them there: V starts at (V_th +
    V_reset) / 2, and without I_ext and refractoriness it hardly moves.  (All
    neurons at one potential would fire their first spikes together.)"""
    p = props.copy()
    v0 = np.random.default_rng(seed).uniform(-65.0, -50.0, size=len(p)).astype(np.float32)
    p[:, 9] = 2.0 * v0 - p[:, 8]
    p[:, 5] = 0.0
    p[:, 2] = 0.0
    return p


def _settle(case, nb, props, nvox_of_pop=None):
    """From scattered potentials to the asynchronous state that the network
    settles in: the refractory hold passes, 40 Hz of noise spikes alone build
    up the inhibition, then the network is connected (connected from silence
    it would first fire a volley of most of its neurons)."""
    nb.run(25, noise_rate=0.0, isolated=True)
    nb.replace_props(props)
    nb.run(600, noise_rate=0.004, isolated=True)
    nb.run(205, noise_mode=1)
    if nvox_of_pop is None:
        nb.attach_bold(steps_per_sample=10, delta_t=1e-3)
    else:
        nb.attach_bold(steps_per_sample=10, delta_t=1e-3, voxel_of_pop=nvox_of_pop)
    out, V = _native_outputs(nb, case["steps"])
    out["bold"] = torch.zeros((case["steps"] // 10, nb.nvox), dtype=torch.float64, device="cuda")
    return dict(case=case, nb=nb, out=out, V=V)


def _prepare_regions(case, seed):
    from digital_twin_brain_amd import networks
    from digital_twin_brain_amd.engine import NativeBlock

    R, E, D = case["regions"], case["members"], case["delay"]
    sizes = networks.region_sizes(R, case["n"], min_size=40, seed=seed)
    cdf = networks.source_cdf(networks.connectome(R, seed=seed + 1))
    ki, kx = case["k_intra"], case["k_inter"]
    parts, spec = [], None
    for m in range(E):
        p, regs = networks.region_props(sizes, ki + kx, seed=seed + 2 + m, dt=DT)
        p[:, 3] += 2 * R * m
        parts.append(p)
        spec = [(a, b, ki, kx) for a, b in regs]
    props = np.concatenate(parts)
    kw = dict(max_delay=D, conn_seed=seed, noise_seed=seed + 1, stats_exclude_blocked=True)
    if E == 1:
        nb = NativeBlock.regions(_scattered(props, seed), spec, cdf, **kw)
    else:
        nb = NativeBlock.region_replicas(_scattered(props, seed), spec, E, cdf, **kw)
    # external Poisson drive: 20% of all input events at 8 Hz
    nb.set_external(0.25 * (ki + kx) * 8.0 * DT * 1e-3, 0.5)
    nb.set_launch(deliver_mode=1, deliver_grid=1024, stage_segs=256 if nb.n > 1_000_000 else 128, stage_ept=16,
                  stage_variant=2)
    return _settle(case, nb, props, nvox_of_pop=(np.arange(nb.S) // 2).astype(np.int32))


# -------------------------------------------------------- data assimilation
def _enkf_inputs(case, seed):
    """A window's hidden state [hp logits, act, s, q, v, f_in, bold]: logits
    spread over a few units, hemodynamics near their resting values."""
    E, V, S = case["members"], case["voxels"], case["states"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)

    w = 0.1 * normal(E, V, S) + 1.0
    w[:, :, : S - 6] = 3.0 * normal(E, V, S - 6)
    w[:, :, S - 1] = 0.01 * normal(E, V) + 0.02
    y = 0.02 + 0.01 * normal(1, V)
    return w, y, normal(E, V)


SIGMA, RHO = 1e-6, 0.8


def _run_enkf(s):
    from digital_twin_brain_amd.enkf import diffusion_enkf

    return diffusion_enkf(s["w"], SIGMA, s["y"], RHO, xi=s["xi"])


def _exact_enkf(case, seed):
    """data_assimilation/DataAssimilation.py:40-60."""
    w, y, xi = _enkf_inputs(case, seed)
    E, V, S = w.shape
    wd = w - w.mean(0, keepdim=True)
    c = (wd[:, :, -1] ** 2).sum(0) / (E - 1) + SIGMA
    gain = wd[:, :, -1] / c / (E - 1)
    innov = y + math.sqrt(SIGMA) * xi - w[:, :, -1]
    local = (gain[:, :, None] * wd).sum(0)
    A = innov @ gain.T / V
    return w + RHO * innov[:, :, None] * local + (1 - RHO) * (A @ wd.reshape(E, V * S)).reshape(E, V, S)


# --------------------------------------------------------------- surrogates
def _table(rows, n_in, n_out, seed):
    """Standardised-looking features and targets that depend on them."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = 0.5 + 2.0 * torch.randn((rows, n_in), generator=g, device="cuda")
    M = torch.randn((n_in, n_out), generator=g, device="cuda") / math.sqrt(n_in)
    Y = 0.1 * torch.tanh(X @ M) + 0.02 * torch.randn((rows, n_out), generator=g, device="cuda")
    return X, Y


def _mlp(case, seed, rows):
    from digital_twin_brain_amd.surrogate import MLPSurrogate

    X, Y = _table(rows, case["n_in"], case["n_out"], seed)
    m = MLPSurrogate(case["n_in"], case["n_out"], hidden=(case["hidden"],) * case["layers"],
                     max_batch=min(rows, 2048), seed=seed)
    m.set_normalization(X.cpu(), Y.cpu())
    return m, X, Y


def _prepare_mlp(case, seed):
    train = case["kind"] == "mlp_train"
    m, X, Y = _mlp(case, seed, case["batch"] if train else case["rows"])
    return dict(case=case, m=m, X=X, Y=Y)


def _run_mlp(s):
    m = s["m"]
    if s["case"]["kind"] == "mlp_predict":
        return m.predict(s["X"])
    loss = m.gradients(s["X"], s["Y"])
    m.step()
    return dict(loss=loss.sum(), dW=list(m.dW), db=list(m.db))


def _exact_mlp(case, seed):
    train = case["kind"] == "mlp_train"
    rows = case["batch"] if train else case["rows"]
    X, Y = (t.double() for t in _table(rows, case["n_in"], case["n_out"], seed))
    pad = lambda n: (n + 31) // 32 * 32  # noqa: E731
    sizes = [pad(case["n_in"])] + [pad(case["hidden"])] * case["layers"] + [pad(case["n_out"])]
    g = torch.Generator().manual_seed(seed)
    Ws, bs = [], []
    for l, (i, o) in enumerate(zip(sizes[:-1], sizes[1:])):  # He initialisation, in the order the surrogate draws it
        w = torch.randn((o, i), generator=g) * np.sqrt(2.0 / i)
        if l == 0:
            w[:, case["n_in"]:] = 0.0
        Ws.append(w.double().cuda().requires_grad_(True))
        bs.append(torch.zeros(o, dtype=torch.float64, device="cuda", requires_grad=True))
    xs, ys = X.std(0).clamp_min(1e-12), Y.std(0).clamp_min(1e-12)
    H = torch.zeros((rows, sizes[0]), dtype=torch.float64, device="cuda")
    H[:, : case["n_in"]] = (X - X.mean(0)) / xs
    for l, (W, b) in enumerate(zip(Ws, bs)):
        H = H @ W.T + b
        if l < len(Ws) - 1:
            H = torch.relu(H)
    out = H[:, : case["n_out"]]
    if not train:
        return (out * ys + Y.mean(0)).detach()
    d = out - (Y - Y.mean(0)) / ys
    (d.square().sum() / (2 * rows)).backward()
    return dict(loss=d.detach().square().sum(), dW=[W.grad for W in Ws], db=[b.grad for b in bs])


def _gru_inputs(case, seed):
    T, B = case["steps"], case["batch"]
    X, Y = _table(T * B, case["n_in"], case["n_out"], seed)
    return X.reshape(T, B, -1), Y.reshape(T, B, -1)


def _prepare_gru(case, seed):
    from digital_twin_brain_amd.surrogate import GRUSurrogate

    X, Y = _gru_inputs(case, seed)
    m = GRUSurrogate(case["n_in"], case["n_out"], hidden=case["hidden"], max_batch=case["batch"],
                     max_steps=case["steps"], seed=seed)
    m.set_normalization(X.cpu(), Y.cpu())
    return dict(m=m, X=X, Y=Y)


def _run_gru(s):
    m = s["m"]
    loss = m.gradients(s["X"], s["Y"])
    m.step()
    return dict(loss=loss.sum(), grad=dict(m.grad))


def _exact_gru(case, seed):
    X, Y = (t.double() for t in _gru_inputs(case, seed))
    T, B = X.shape[:2]
    pad = lambda n: (n + 31) // 32 * 32  # noqa: E731
    I, H, O = pad(case["n_in"]), pad(case["hidden"]), pad(case["n_out"])
    g = torch.Generator().manual_seed(seed)
    s = 1.0 / np.sqrt(H)
    w_ih = (torch.rand((3 * H, I), generator=g) * 2 - 1) * s
    w_ih[:, case["n_in"]:] = 0.0
    p = dict(W_ih=w_ih, b_ih=(torch.rand(3 * H, generator=g) * 2 - 1) * s,
             W_hh=(torch.rand((3 * H, H), generator=g) * 2 - 1) * s, b_hh=(torch.rand(3 * H, generator=g) * 2 - 1) * s,
             W_o=torch.randn((O, H), generator=g) * s, b_o=torch.zeros(O))
    p = {k: v.float().double().cuda().requires_grad_(True) for k, v in p.items()}
    Xf, Yf = X.reshape(T * B, -1), Y.reshape(T * B, -1)
    xs, ys = Xf.std(0).clamp_min(1e-12), Yf.std(0).clamp_min(1e-12)
    Xn = torch.zeros((T, B, I), dtype=torch.float64, device="cuda")
    Xn[:, :, : case["n_in"]] = (X - Xf.mean(0)) / xs
    Tn = (Y - Yf.mean(0)) / ys
    h = torch.zeros((B, H), dtype=torch.float64, device="cuda")
    loss = 0.0
    for t in range(T):
        gi = Xn[t] @ p["W_ih"].T + p["b_ih"]
        gh = h @ p["W_hh"].T + p["b_hh"]
        r = torch.sigmoid(gi[:, :H] + gh[:, :H])
        z = torch.sigmoid(gi[:, H:2 * H] + gh[:, H:2 * H])
        n = torch.tanh(gi[:, 2 * H:] + r * gh[:, 2 * H:])
        h = (1 - z) * n + z * h
        y = h @ p["W_o"].T + p["b_o"]
        loss = loss + (y[:, : case["n_out"]] - Tn[t]).square().sum()
    (loss / (2 * T * B)).backward()
    return dict(loss=loss.detach(), grad={k: v.grad for k, v in p.items()})


def _gemm_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = torch.randn((case["m"], case["k"]), generator=g, device="cuda").to(torch.bfloat16)
    B = torch.randn((case["n"], case["k"]), generator=g, device="cuda").to(torch.bfloat16)
    return A, B, torch.randn(case["n"], generator=g, device="cuda")


def _prepare_gemm(case, seed):
    A, B, b = _gemm_inputs(case, seed)
    C = torch.empty((case["m"], case["n"]), device="cuda")
    return dict(case=case, A=A, B=B, b=b if case["bias"] else None, C=C,
                Cb=torch.empty_like(C, dtype=torch.bfloat16) if case["half"] else None)


def _run_gemm(s):
    from digital_twin_brain_amd import _native as nat

    c, A, B, C, Cb = s["case"], s["A"], s["B"], s["C"], s["Cb"]
    nat.check(nat.lib().dtb_mlp_gemm_bf16_nt(c["m"], c["n"], c["k"], nat.ptr(A), c["k"], nat.ptr(B), c["k"],
                                             nat.ptr(s["b"]), c["act"], nat.ptr(C), c["n"], nat.ptr(Cb), c["n"],
                                             torch.cuda.current_stream().cuda_stream))
    return [C] if Cb is None else [C, Cb]


def _exact_gemm(case, seed):
    A, B, b = _gemm_inputs(case, seed)
    C = A.double() @ B.double().T
    if case["bias"]:
        C += b.double()
    if case["act"]:
        C.clamp_min_(0.0)
    return [C, C] if case["half"] else [C]


# --------------------------------------------------------------------- BOLD
def _bold_inputs(case, seed):
    """A state some seconds into a run and one millisecond's input per voxel."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.float64 if case["double"] else torch.float32
    n = case["n"]
    u = 0.001 * torch.rand(n, generator=g, device="cuda", dtype=dt)
    st = [0.1 * torch.rand(n, generator=g, device="cuda", dtype=dt) + c for c in (0.0, 0.8, 1.0, 1.0)]
    return u, st


def _prepare_bold(case, seed):
    from digital_twin_brain_amd.bold import BOLD

    u, (s, q, v, f) = _bold_inputs(case, seed)
    return dict(u=u, m=BOLD(**BOLD_PAR, delta_t=1e-3, init_s=s, init_q=q, init_v=v, init_f_in=f))


def _run_bold(s):
    m = s["m"]
    out = m.run(s["u"])
    return [out, m.s, m.q, m.v, m.f_in]


def _exact_bold(case, seed):
    """models/bold_model_pytorch.py:69-77."""
    u, (s, q, v, f) = _bold_inputs(case, seed)
    u, s, q, v, f = (x.double() for x in (u, s, q, v, f))
    P, dt = BOLD_PAR, 1e-3
    ds = P["epsilon"] * u - s / P["tao_s"] - (f - 1) / P["tao_f"]
    qp = torch.where(f > 0, 1 - (1 - P["E_0"]) ** (1 / f), torch.ones_like(f))
    qn = q + (f * qp / P["E_0"] - q * v ** (1 / P["alpha"] - 1)) / P["tao_0"] * dt
    vn = v + (f - v ** (1 / P["alpha"])) / P["tao_0"] * dt
    fn = (f + s * dt).clamp_min(0.0)
    sn = s + ds * dt
    out = P["V_0"] * (7 * P["E_0"] * (1 - qn) + 2 * (1 - qn / vn) + (2 * P["E_0"] - 0.2) * (1 - vn))
    return [out, sn, qn, vn, fn]


# -------------------------------------------------------------------- table
_KINDS = {
    "dropin_run": (_prepare_dropin, _run_dropin, _exact_dropin),
    "dropin_steps": (_prepare_dropin, _run_dropin, _exact_dropin),
    "plain_batch": (_prepare_plain, _run_native, None),
    "large": (_prepare_large, _run_native, None),
    "regions": (_prepare_regions, _run_native, None),
    "enkf": (lambda c, s: dict(zip(("w", "y", "xi"), _enkf_inputs(c, s))), _run_enkf, _exact_enkf),
    "mlp_train": (_prepare_mlp, _run_mlp, _exact_mlp),
    "mlp_predict": (_prepare_mlp, _run_mlp, _exact_mlp),
    "gru_train": (_prepare_gru, _run_gru, _exact_gru),
    "gemm": (_prepare_gemm, _run_gemm, _exact_gemm),
    "bold": (_prepare_bold, _run_bold, _exact_bold),
}


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, int(seed) % (1 << 30))
    s["run"] = _KINDS[case["kind"]][1]
    return s


def run(state):
    return state["run"](state)


def exact(case, seed):
    f = _KINDS[case["kind"]][2]
    return f(case, int(seed) % (1 << 30)) if f else None


def work(case):
    k = case["kind"]
    if k in ("dropin_run", "dropin_steps", "plain_batch", "large", "regions"):
        n = case["n"] * case.get("members", 1)
        deg = case.get("in_degree") or case["k_intra"] + case["k_inter"]
        # delivered spikes per neuron and step: the strongly coupled plain
        # block at about 450 Hz, the others at about 20 Hz
        rate = 0.045 if k in ("dropin_run", "dropin_steps", "plain_batch") else 0.002
        # per neuron: V, J, refractory end, conductances and noise rate read,
        # V, J and flags written; per event: the target and its weight
        per_step = n * 65.0 + rate * n * deg * 8.0
        return dict(bytes=per_step * case["steps"] + 4.0 * n, flops=case["steps"] * (60.0 * n + rate * n * deg))
    if k == "enkf":
        E, V, S = case["members"], case["voxels"], case["states"]
        return dict(bytes=8.0 * (2 * E * V * S + E * V + V), flops=2.0 * E * E * V * (S + 1) + 8.0 * E * V * S)
    if k in ("mlp_train", "mlp_predict"):
        dims = [case["n_in"]] + [case["hidden"]] * case["layers"] + [case["n_out"]]
        p = sum(a * b + b for a, b in zip(dims[:-1], dims[1:]))
        rows = case["batch"] if k == "mlp_train" else case["rows"]
        io = 4.0 * rows * (case["n_in"] + case["n_out"])
        if k == "mlp_predict":
            return dict(bytes=io + 2.0 * p, flops=2.0 * rows * p)
        return dict(bytes=io + 28.0 * p, flops=6.0 * rows * p)  # weights, two moments in and out, gradients out
    if k == "gru_train":
        rows, h = case["steps"] * case["batch"], case["hidden"]
        p = 3 * h * (case["n_in"] + h + 2) + case["n_out"] * (h + 1)
        return dict(bytes=4.0 * rows * (case["n_in"] + case["n_out"]) + 28.0 * p, flops=6.0 * rows * p)
    if k == "gemm":
        m, n, kk = case["m"], case["n"], case["k"]
        return dict(bytes=2.0 * (m + n) * kk + (4.0 + 2.0 * case["half"]) * m * n, flops=2.0 * m * n * kk)
    return dict(bytes=(8.0 if case["double"] else 4.0) * 10 * case["n"], flops=100.0 * case["n"])
