"""The work a user of this framework has it do, as cases with inputs, one pass and its cost.

Simulation (the main path): single runs through capi.run from the few
thousand mutations of a test run to the two million of the large benchmark
run, two and three populations with a split, growth, a bottleneck and
migration, and batches through capi.batch_run / surrogate.simulate.
Spectra: the sample, joint and population spectra of host rows.
Surrogate: predictions for a handful of inputs and for hundreds of
thousands, and training (forward, backward and Adam).

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call
    run(state)          one pass through the public entry points
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   the outputs in 64 bits, where they are computed numbers
"""
import ctypes as C
import math

import numpy as np
import torch

MU = 1e-9


def _use_device():
    """torch first on the device, then the library: both then share torch's HIP runtime"""
    torch.zeros(1, device="cuda")
    from parallelpopgen_amd import capi, scenarios, surrogate
    return capi, scenarios, surrogate


# ---------------------------------------------------------------- cases

def listed():
    return [
        # a test-sized run: 8.4e3 live mutations; what a user tries first,
        # and what fitting programs call in a loop (latency and launches)
        dict(name="run_small", kind="run", N=10000, L=2e7, G=1000, gamma=0.0, h=0.5, F=0.0, growth=1.0, interval=35,
             sample_every=0, n=100),
        # the headline run: 2.0e6 live mutations under purifying selection
        dict(name="run_large", kind="run", N=100000, L=5e8, G=5000, gamma=-10.0, h=0.5, F=0.0, growth=1.0,
             interval=35, sample_every=0, n=1000),
        # two populations with a split and exponential growth, the shape of
        # the usual out-of-Africa fit (examples/dadi)
        dict(name="run_split", kind="split", N=10000, L=2e8, G=1001, gamma=-4.0, interval=30, n=1001),
        # three populations: growth, bottleneck, inbreeding, migration,
        # selection that changes over time, preserved mutations
        dict(name="run_three_populations", kind="three", N=20000, L=2e8, G=2000, interval=35, preserve_every=100, n=50),
        # training data for the surrogate: one chunk of parameter draws
        dict(name="batch_draws", kind="draws", sims=8192),
        # a parameter sweep with uneven sizes and lengths, one batch
        dict(name="batch_sweep", kind="sweep", sims=64, n=50),
        # spectrum of a time sample a program already holds on the host
        dict(name="sfs_row", kind="sfs", M=200000, Nc=20000, n=100),
        # joint spectrum of two populations' rows (two-population fits)
        dict(name="joint_sfs", kind="joint", M=100000, Nc=20000, na=40, nb=40),
        # whole-population histogram of a large sample
        dict(name="population_histogram", kind="hist", M=2000000, Nc=200000),
        # a handful of surrogate evaluations: one step of an optimiser
        dict(name="predict_few", kind="predict", n=16, on_device=False, ensemble=4),
        # surrogate evaluations over a grid, inputs and outputs on the GPU
        dict(name="predict_bulk", kind="predict", n=262144, on_device=True, ensemble=4),
        # training: one epoch of Adam over a small set (forward, backward, update)
        dict(name="train_epoch", kind="train", n=32768, batch=512, ensemble=4),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "split", "three", "draws", "sweep", "sfs", "joint", "hist", "predict",
                       "predict", "train"])
    if kind == "run":
        # N, selection, dominance and inbreeding as scenarios.parameter_sweep
        # draws them, 1e3 to 2e6 mutations, growth in a third of the runs
        N = int(_log(rng, 1e3, 1e5))
        live = _log(rng, 1e3, 2e6)
        L = live / (2 * MU * 2 * N * (math.log(2 * N) + 0.5772))
        G = int(min(_log(rng, 100, 5000), 5e9 / live))
        return dict(kind=kind, N=N, L=float(int(L)), G=G, gamma=rng.choice([0.0, rng.uniform(-50, 10)]),
                    h=rng.choice([0.0, 0.3, 0.5, 1.0]), F=rng.choice([0.0, rng.uniform(0, 0.2), 1.0]),
                    growth=rng.choice([1.0, 1.0, _log(rng, 1, 10)]), interval=rng.choice([15, 25, 30, 35]),
                    sample_every=rng.choice([0, 0, max(1, G // 3)]), n=int(_log(rng, 10, 500)))
    if kind == "split":
        return dict(kind=kind, N=int(_log(rng, 2e3, 1e4)), L=float(int(_log(rng, 2e7, 5e8))), G=rng.randint(300, 1001),
                    gamma=rng.uniform(-10, 4), interval=rng.choice([15, 30, 35]), n=int(_log(rng, 10, 1001)))
    if kind == "three":
        return dict(kind=kind, N=int(_log(rng, 2e3, 2e4)), L=float(int(_log(rng, 2e7, 2e8))), G=rng.randint(200, 1500),
                    interval=35, preserve_every=rng.choice([0, 100]), n=rng.randint(10, 100))
    if kind == "draws":
        return dict(kind=kind, sims=int(_log(rng, 64, 8192)))
    if kind == "sweep":
        return dict(kind=kind, sims=rng.randint(4, 48), n=rng.randint(10, 100))
    if kind == "sfs":
        return dict(kind=kind, M=int(_log(rng, 1e3, 2e6)), Nc=int(_log(rng, 4e3, 4e5)), n=int(_log(rng, 10, 1000)))
    if kind == "joint":
        return dict(kind=kind, M=int(_log(rng, 1e3, 2e5)), Nc=int(_log(rng, 4e3, 1e5)), na=rng.randint(5, 50),
                    nb=rng.randint(5, 50))
    if kind == "hist":
        return dict(kind=kind, M=int(_log(rng, 1e3, 2e6)), Nc=int(_log(rng, 2e3, 4e5)))
    if kind == "predict":
        return dict(kind=kind, n=int(_log(rng, 1, 262144)), on_device=rng.choice([False, True]),
                    ensemble=rng.choice([2, 4, 4]))
    return dict(kind="train", n=int(_log(rng, 4096, 32768)), batch=64 * rng.randint(2, 16),
                ensemble=rng.choice([2, 4, 4]))


# ---------------------------------------------------------------- inputs

def _rng(seed):
    return np.random.default_rng(int(seed) & 0x7FFFFFFF)


def _seed1(seed):
    return 1 + (int(seed) & 0x3FFFFFFF)


def _grow(N, growth, G):
    """population size of every generation: exponential growth by a factor over the run"""
    g = np.arange(G + 1)
    return np.floor(N * np.exp(math.log(growth) * g / max(G, 1)) + 0.5).astype(np.int64)


def _single(capi, scenarios, c, seed):
    s = scenarios.selection_from_gamma(c["gamma"], c["N"], c["F"])
    d = scenarios.constant(N=c["N"], L=c["L"], G=c["G"], mu=MU, F=c["F"], h=c["h"], s=s, seed1=_seed1(seed),
                           compact_interval=c["interval"], sample_every=c["sample_every"])
    if c["growth"] != 1.0:
        d.params["N"][:, 0] = _grow(c["N"], c["growth"], c["G"])
    return d


def _split(capi, scenarios, c, seed):
    """one population that doubles at generation 1; a second one founded from
    it at a tenth of the run, growing 100-fold; symmetric migration afterwards"""
    G, N, P = c["G"], c["N"], 2
    t0 = max(2, G // 10)
    g = np.arange(G + 1)
    params = np.zeros((G + 1, P), capi.POP_GEN_DTYPE)
    params["N"][:, 0] = np.where(g == 0, N, 2 * N)
    size = 0.05 * N * np.exp(math.log(100.0) / max(1, G - t0) * np.maximum(g - t0, 0))
    params["N"][:, 1] = np.where(g < t0, 0, np.floor(size + 0.5).astype(np.int64))
    params["h"] = 0.5
    params["mu"] = MU
    params["sel_intercept"] = scenarios.selection_from_gamma(c["gamma"], N, 0.0)
    m = 1.0 / (2.0 * N)
    mig = np.zeros((G + 1, P, P), np.float32)
    mig[:t0 + 1, 0, 0] = 1.0
    mig[t0, 0, 1] = 1.0
    mig[t0 + 1:] = scenarios.migration_constant_equal(m, P)
    return capi.SimDesc(P, c["L"], _seed1(seed), scenarios.SEED2_DEFAULT, G, params, mig,
                        compact_interval=c["interval"])


def _row(rng, M, Nc):
    """frequencies of segregating mutations, counts distributed as 1/x"""
    j = np.floor(np.exp(rng.uniform(0.0, math.log(Nc), M))).astype(np.int64)
    return (np.clip(j, 1, Nc - 1).astype(np.float32) / np.float32(Nc)).astype(np.float32)


def _two_rows(rng, M, Nc):
    """rows of two diverged populations: the second drifts around the first, and
    a third of the mutations are private to one of the two"""
    a = _row(rng, M, Nc)
    x = a.astype(np.float64)
    b = np.clip(np.floor(Nc * (x + rng.normal(0, 1, M) * np.sqrt(0.1 * x * (1 - x))) + 0.5), 0, Nc)
    b = (b.astype(np.float32) / np.float32(Nc)).astype(np.float32)
    u = rng.uniform(0, 1, M)
    b[u < 1 / 6] = 0.0
    a[u > 5 / 6] = 0.0
    return a, b


INS = (64, 512, 512, 512, 512)
OUTS = (512, 512, 512, 512, 128)


def _weights(rng, ensemble):
    """parameters of an ensemble, [member][W_l (out x in), b_l ...]: scale
    sqrt(2 / inputs), small biases, the padding (inputs past 6, outputs past
    100) zero"""
    members = []
    for _ in range(ensemble):
        flat = []
        for l, (i, o) in enumerate(zip(INS, OUTS)):
            ni, no = (6 if l == 0 else i), (100 if l == 4 else o)
            W = np.zeros((o, i), np.float32)
            W[:no, :ni] = rng.standard_normal((no, ni), np.float32) * np.float32(math.sqrt((2.0 if l < 4 else 0.5) / ni))
            b = np.zeros(o, np.float32)
            b[:no] = rng.standard_normal(no, np.float32) * np.float32(0.05)
            if l == 4:
                b[:99] += -np.log(np.arange(1, 100)).astype(np.float32)   # the neutral spectrum's slope
            flat += [W.ravel(), b]
        members.append(np.concatenate(flat))
    return np.stack(members)


def _inputs(surrogate, rng, n):
    return surrogate.features(surrogate.draw(n, rng))


def prepare(case, seed):
    c, kind = case, case["kind"]
    capi, scenarios, surrogate = _use_device()
    rng = _rng(seed)
    s = dict(kind=kind, capi=capi, surrogate=surrogate, case=c)
    if kind == "run":
        s["desc"] = _single(capi, scenarios, c, seed)
        s["sfs"] = [(0, min(c["n"], 100)), (0, c["n"])]
    elif kind == "split":
        s["desc"] = _split(capi, scenarios, c, seed)
        s["sfs"] = [(1, min(c["n"], int(s["desc"].params["N"][-1, 1])))]
    elif kind == "three":
        s["desc"] = scenarios.three_population(seed1=_seed1(seed), G=c["G"], L=c["L"], N0=c["N"],
                                               compact_interval=c["interval"], preserve_every=c["preserve_every"])
        s["sfs"] = [(p, c["n"]) for p in range(3)]
    elif kind == "draws":
        s["p"] = surrogate.draw(c["sims"], rng)
        s["seeds"] = rng.integers(1, 2 ** 31 - 1, c["sims"])
    elif kind == "sweep":
        s["sims"] = scenarios.parameter_sweep(c["sims"], seed=int(seed) & 0x7FFFFFFF, seed_base=_seed1(seed), mu=MU)
    elif kind in ("sfs", "hist"):
        s["row"] = _row(rng, c["M"], c["Nc"])
        s["L"] = float(10 * c["M"])
    elif kind == "joint":
        s["a"], s["b"] = _two_rows(rng, c["M"], c["Nc"])
        s["L"] = float(10 * c["M"])
    elif kind == "predict":
        s["held"] = _Held(surrogate, c["ensemble"])
        s["net"] = s["held"].net
        s["net"].set_params(_weights(rng, c["ensemble"]))
        x = _inputs(surrogate, rng, c["n"])
        if c["on_device"]:
            A = capi.DeviceArray
            s["x"] = A.from_host(x)
            s["out"] = [A((c["n"], surrogate.NBINS)), A(c["n"]), A(c["n"])]
        else:
            s["x"] = x
    else:
        n = c["n"]
        s["net"] = surrogate.Network(ensemble=c["ensemble"])   # Adam's state is its own: never reused
        _TRAINED.append(s["net"])
        s["net"].set_params(_weights(rng, c["ensemble"]))
        s["x"] = _inputs(surrogate, rng, n)
        k = np.arange(1, 100)
        y = rng.gamma(5.0, 1.0, (n, 99)) / k ** (1.0 + 0.3 * s["x"][:, :1])
        s["y"] = (y / y.sum(1, keepdims=True)).astype(np.float32)
        s["t"] = (1.0 + 0.5 * s["x"][:, 0] + 0.05 * rng.standard_normal(n)).astype(np.float32)
    if kind in ("run", "split", "three"):
        d = s["desc"]
        cap, samples = _most(c), 1 + int(d.sample[1:-1].sum())
        s["freq"] = [np.zeros(d.P * cap, np.float32) for _ in range(samples)]
        s["num"] = np.zeros(samples, np.int64)
        s["ids"] = np.zeros((cap, 4), np.int32)
        s["live"] = np.zeros(d.G + 1, np.int64)
    return s


# Networks stay in the program: a serving program keeps the ones it loaded (new
# weights go into a network that no state uses any more), a training program
# the ones it trains.
_IDLE = {}
_TRAINED = []


class _Held:
    def __init__(self, surrogate, ensemble):
        self.ensemble = ensemble
        idle = _IDLE.setdefault(ensemble, [])
        self.net = idle.pop() if idle else surrogate.Network(ensemble=ensemble)

    def __del__(self):
        _IDLE[self.ensemble].append(self.net)


def run(s):
    kind, capi, surrogate, c = s["kind"], s["capi"], s["surrogate"], s["case"]
    if kind in ("run", "split", "three"):
        return _simulate(capi, s)
    if kind == "draws":
        return surrogate.simulate(s["p"], s["seeds"])
    if kind == "sweep":
        r = capi.batch_run(s["sims"], sfs_n=c["n"])
        return dict(sfs=r["sfs"], num_mutations=r["num_mutations"], live=r["live_mutation_generations"])
    if kind == "sfs":
        return capi.site_frequency_spectrum(s["row"], c["n"], s["L"])
    if kind == "joint":
        return capi.joint_site_frequency_spectrum(s["a"], s["b"], c["na"], c["nb"], s["L"])
    if kind == "hist":
        return capi.population_frequency_histogram(s["row"], c["Nc"], s["L"])
    if kind == "predict":
        if not c["on_device"]:
            return s["net"].predict(s["x"])
        s["net"].predict_device(s["x"], *s["out"])
        return [_DeviceView(a).tensor() for a in s["out"]]
    losses = s["net"].train(s["x"], s["y"], s["t"], epochs=1, batch=c["batch"], seed=_TRAIN_SEED)
    return dict(weights=s["net"].get_params(), losses=losses)


_TRAIN_SEED = 7


def _simulate(capi, s):
    """gf_run, the final spectra where the state lies, and every sample, ID and
    live count read into the program's own arrays (flat [P][mutations] rows
    from the start of each; the rest stays zero)"""
    lib, d = capi.load(), s["desc"]
    h = C.c_void_p()
    capi.check(lib.gf_run(C.byref(d.desc), C.byref(h)))
    try:
        last, sfs = lib.gf_result_num_samples(h) - 1, []
        for pop, n in s["sfs"]:
            o = np.empty(n, np.float32)
            capi.check(lib.gf_result_site_frequency_spectrum(h, last, pop, n, d.num_sites, _at(o)))
            sfs.append(o)
        m = C.c_int32()
        for k, f in enumerate(s["freq"]):
            capi.check(lib.gf_result_sample_info(h, k, C.byref(m), None, None, None))
            if d.P * m.value > len(f):
                raise RuntimeError("more mutations than the program's arrays hold")
            capi.check(lib.gf_result_sample_freq(h, k, _at(f)))
            s["num"][k] = m.value
        if lib.gf_result_num_ids(h) > len(s["ids"]):
            raise RuntimeError("more mutations than the program's arrays hold")
        capi.check(lib.gf_result_ids(h, _at(s["ids"])))
        capi.check(lib.gf_result_live_counts(h, _at(s["live"])))
    finally:
        lib.gf_result_free(h)
    return dict(sfs=sfs, num=s["num"], freq=s["freq"], ids=s["ids"], live=s["live"])


def _at(a):
    return a.ctypes.data_as(C.c_void_p)


class _DeviceView:
    """a capi.DeviceArray as a torch tensor of the same memory"""

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr="<f4", data=(a.ptr, False), version=2)

    def tensor(self):
        return torch.as_tensor(self, device="cuda")


# ---------------------------------------------------------------- cost

def _live(N, L, gamma=0.0):
    """segregating mutations expected at equilibrium (additive selection)"""
    Nc = 2 * N
    x = np.arange(1, Nc) / Nc
    w = np.ones_like(x) if abs(gamma) < 1e-3 else -np.expm1(-2 * gamma * (1 - x)) / (-np.expm1(-2 * gamma) * (1 - x))
    return float(np.sum(2 * MU * L / x * np.minimum(w, 1e3)))


def _most(c):
    """room for the mutations of any sample of a run: about twice what is expected"""
    N, L = c["N"], c["L"]
    if c["kind"] == "run":
        up = max(c["gamma"], 0.0)
        return int(2 * _live(int(N * max(c["growth"], 1.0)), L, up)) + 4096
    if c["kind"] == "split":
        return int(2 * (_live(2 * N, L, max(c["gamma"], 0.0)) + _live(5 * N, L, max(c["gamma"], 0.0)))) + 4096
    marks = c["G"] // c["preserve_every"] if c["preserve_every"] else 0
    born = MU * L * 24 * N                      # new mutations a generation, all populations
    return int(4 * _live(10 * N, L) + marks * 7 * born) + 4096


def work(case):
    """simulations: 4 B of state read and 4 B written, and 40 operations, per
    mutation, population and generation; spectra: the rows in, the spectrum
    out, one product per mutation and level; networks: 2 operations per weight
    and example (6 when training), weights, inputs and outputs once"""
    c, kind = case, case["kind"]
    if kind == "run":
        mg = _live(c["N"], c["L"], c["gamma"]) * c["G"]
        return dict(bytes=8 * mg, flops=40 * mg)
    if kind == "split":
        mg = _live(c["N"], c["L"], c["gamma"]) * c["G"] * 2
        return dict(bytes=8 * mg, flops=40 * mg)
    if kind == "three":
        # 1.3e10 mutation-generations at N = 2e4, L = 2e8 over 2,000 generations
        mg = 3 * 1.3e10 * (c["N"] / 2e4) * (c["L"] / 2e8) * (c["G"] / 2e3)
        return dict(bytes=8 * mg, flops=40 * mg)
    if kind == "draws":
        mg = 1200.0 * 37 * c["sims"]      # about 1,200 mutations over 37 generations on average
        return dict(bytes=8 * mg, flops=40 * mg)
    if kind == "sweep":
        mg = 9.6e8 * c["sims"]            # 3.92e12 mutation-generations over the 4,096-simulation sweep
        return dict(bytes=8 * mg, flops=40 * mg)
    if kind == "sfs":
        return dict(bytes=4.0 * (c["M"] + c["n"]), flops=3.0 * c["M"] * min(c["n"], 30))
    if kind == "joint":
        return dict(bytes=4.0 * (2 * c["M"] + (c["na"] + 1) * (c["nb"] + 1)),
                    flops=2.0 * c["M"] * min(c["na"], 15) * min(c["nb"], 15))
    if kind == "hist":
        return dict(bytes=4.0 * (c["M"] + c["Nc"]), flops=2.0 * c["M"])
    weights = 6 * 512 + 3 * 512 * 512 + 512 * 100
    E = c["ensemble"]
    if kind == "predict":
        return dict(bytes=4.0 * c["n"] * (6 + 101) + 2.0 * E * weights, flops=2.0 * E * weights * c["n"])
    steps = c["n"] // c["batch"]
    return dict(bytes=28.0 * E * weights * steps + 4.0 * c["n"] * 106, flops=6.0 * E * weights * steps * c["batch"])


# ---------------------------------------------------------------- 64 bits

def _prob(x, n):
    """P(k of n chromosomes | frequency x), [len(x)][n + 1], 64 bits on the GPU"""
    x = torch.as_tensor(x, device="cuda").double()[:, None]
    k = torch.arange(n + 1, device="cuda", dtype=torch.float64)[None, :]
    lc = math.lgamma(n + 1) - torch.lgamma(k + 1) - torch.lgamma(n - k + 1)
    p = torch.exp(lc + torch.xlogy(k, x) + torch.xlogy(n - k, 1 - x))
    return p


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("run", "split", "three", "draws", "sweep", "train"):
        return None   # random draws, or weights after many steps: no such value
    s = prepare(c, seed)
    if kind == "hist":
        j = np.floor(s["row"].astype(np.float64) * c["Nc"] + 0.5).astype(np.int64)
        j[j == c["Nc"]] = 0
        h = np.bincount(j, minlength=c["Nc"]).astype(np.float64)
        h[0] += s["L"] - c["M"]
        return h
    if kind == "sfs":
        n = c["n"]
        out = torch.zeros(n + 1, dtype=torch.float64, device="cuda")
        for a in range(0, c["M"], 1 << 16):
            out += _prob(s["row"][a:a + (1 << 16)], n).sum(0)
        out[0] += out[n] + s["L"] - c["M"]
        return out[:n].cpu().numpy()
    if kind == "joint":
        out = torch.zeros((c["na"] + 1, c["nb"] + 1), dtype=torch.float64, device="cuda")
        for a in range(0, c["M"], 1 << 16):
            out += _prob(s["a"][a:a + (1 << 16)], c["na"]).t().contiguous() @ _prob(s["b"][a:a + (1 << 16)], c["nb"])
        out[0, 0] += s["L"] - c["M"]
        return out.cpu().numpy()
    # predict: the same network in 64 bits throughout
    rng = _rng(seed)
    w = _weights(rng, c["ensemble"])
    x = torch.as_tensor(_inputs(s["surrogate"], rng, c["n"]), device="cuda").double()
    sfs, tot, dis = [], [], []
    for a in range(0, c["n"], 1 << 15):
        p, t = [], []
        for e in range(c["ensemble"]):
            act, o = x[a:a + (1 << 15)], 0
            for l, (i, m) in enumerate(zip(INS, OUTS)):
                W = torch.as_tensor(w[e, o:o + i * m], device="cuda").double().reshape(m, i)
                b = torch.as_tensor(w[e, o + i * m:o + i * m + m], device="cuda").double()
                o += i * m + m
                act = act @ W[:, :act.shape[1]].t().contiguous() + b
                if l < 4:
                    act = torch.nn.functional.gelu(act, approximate="tanh")
            p.append(torch.softmax(act[:, :99], 1))
            t.append(act[:, 99])
        p, t = torch.stack(p), torch.stack(t)
        mean = p.mean(0)
        sd = torch.sqrt(torch.clamp((p * p).mean(0) - mean * mean, min=0))
        sfs.append(mean)
        tot.append(t.mean(0))
        dis.append(torch.where(mean >= 1e-3, sd / mean, torch.zeros_like(mean)).amax(1))
    out = [torch.cat(v) for v in (sfs, tot, dis)]
    return out if c["on_device"] else tuple(v.cpu().numpy() for v in out)
