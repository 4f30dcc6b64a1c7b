"""The work that programs built on this framework have it do, as timed cases.

A user of the framework steps populations and reads them back.  Most cases
are therefore a running simulation (built and settled by `prepare`) of which
one pass advances some steps and reads the agents, as a program does between
two dumps, two events or two points of its output; the models are the ones of
`qhg4_amd/scenarios.py`, at sizes from a few hundred cells to the 163,842-cell
grid.  The others step an ensemble as one batch and take an environment event.

Worlds (grid, altitudes, NPP) are synthetic and fixed per size; the seed makes
the agents, their genomes, the draws of the steps and, for the event, the new
environment.  Agents start spread over the habitable land, so that the settled
population neither grows nor spreads and every pass is alike.
"""
import ctypes
import functools

import numpy as np

from qhg4_amd import abi, scenarios
from qhg4_amd._lib import check, lib
from qhg4_amd.grids import rect_grid
from qhg4_amd.population import GpuBatch, GpuPopulation

WORLD = 42          # seed of the worlds
# settled live agents per grid cell (measured): lattices at the tutorial's
# rates, land/sea worlds; used by work() only
LATTICE_LIVE = 24.0
WORLD_LIVE = 9.0


def listed():
    return [
        # the smallest call: one step of a small lattice in the reference
        # loop's order, the agents looked at after it (an interactive or
        # coupled program)
        dict(name="lattice_20x13_step", kind="loop", model="lattice", width=20, height=13, steps=1),
        # the plain model on its configured 128 x 128 lattice, between two
        # points of a time series
        dict(name="lattice_128x128", kind="run", model="lattice", width=128, height=128, steps=500),
        # the out-of-Africa model on the smallest grid of the ensembles, run
        # step by step with the extinction check of a driver loop
        dict(name="ooa_level4_loop", kind="loop", model="ooa", level=4, steps=100),
        # the headline configuration's grid, between two dumps
        dict(name="ooa_level6", kind="run", model="ooa", level=6, steps=1000),
        # the largest grid of the ensembles, one population
        dict(name="ooa_level7", kind="run", model="ooa", level=7, steps=1000),
        # 2-bit genetics (256 loci) on the headline grid
        dict(name="genetics_level6", kind="run", model="genetics", level=6, loci=256, steps=500),
        # ... and at the scale run's density on the largest of these grids
        dict(name="genetics_level7", kind="run", model="genetics", level=7, loci=256, steps=500),
        # assortative mating by genome distance, with the permutation
        dict(name="hamming_level6", kind="run", model="hamming", level=6, loci=256, steps=300),
        # assortative mating by equal proteins
        dict(name="protein_level5", kind="run", model="protein", level=5, loci=256, steps=60),
        # sea-ways and bridges along the coasts
        dict(name="navigate_level6", kind="run", model="navigate", level=6, steps=600),
        # an ensemble of unequal replicas stepped as one batch
        dict(name="ensemble_24", kind="batch", members=24, steps=300),
        # a climate and vegetation event: new environment arrays in, the
        # capacity and movement-weight tables out
        dict(name="event_level7", kind="event", level=7),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["lattice", "lattice", "ooa", "ooa", "genetics", "hamming", "protein", "navigate", "batch",
                       "event"])
    if kind == "lattice":
        case = dict(kind=rng.choice(["loop", "run"]), model="lattice", width=rng.randint(11, 128),
                    height=rng.randint(11, 128), steps=_log_int(rng, 1, 500))
    elif kind == "ooa":
        case = dict(kind=rng.choice(["loop", "run", "run"]), model="ooa", level=rng.randint(3, 7),
                    steps=_log_int(rng, 5, 1000))
    elif kind == "genetics":
        case = dict(kind="run", model="genetics", level=rng.randint(4, 6), loci=rng.randint(40, 700),
                    steps=_log_int(rng, 10, 400))
    elif kind == "hamming":
        case = dict(kind="run", model="hamming", level=rng.randint(4, 6), loci=rng.randint(100, 1200),
                    steps=_log_int(rng, 10, 300))
    elif kind == "protein":
        case = dict(kind="run", model="protein", level=rng.randint(4, 5), loci=rng.randint(100, 256),
                    steps=_log_int(rng, 5, 60))
    elif kind == "navigate":
        case = dict(kind="run", model="navigate", level=rng.randint(4, 6), steps=_log_int(rng, 10, 600))
    elif kind == "batch":
        case = dict(kind="batch", members=rng.randint(3, 24), steps=_log_int(rng, 10, 300))
    else:
        case = dict(kind="event", level=rng.randint(4, 7))
        case["npp_scale"] = round(rng.uniform(0.5, 1.5), 3)
    return case


# -- inputs ------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _world(level):
    """Grid, environment and habitable cells of a land/sea world."""
    grid, env, land, good = scenarios.c4_world(level, WORLD)
    return grid, env, good


@functools.lru_cache(maxsize=None)
def _coast(level):
    """A world with ports, sea-ways and bridges (no genetics)."""
    sc = scenarios.c2nav(seed=WORLD, level=level, n_agents=1000, patch_cells=max(50, 4000 >> (2 * (6 - level))),
                         genetics=False)
    alt = sc["env"]["altitude"]
    good = np.flatnonzero((alt > 0) & (alt < 1500) & (sc["env"]["base_npp"] > 0.05)).astype(np.int32)
    return sc["grid"], sc["env"], sc["nav"], good, sc["params"]


def _agents(rng, cells, density, life, last_birth):
    n = int(len(cells) * density)
    at = np.sort(cells[rng.integers(0, len(cells), n)])
    age = rng.uniform(0.0, 40.0, n)
    return {
        "id": np.arange(1, n + 1, dtype=np.int64), "cell": at.astype(np.int32),
        "life": np.full(n, life, dtype=np.uint8), "gender": (rng.random(n) < 0.5).astype(np.uint8),
        "birth_time": -age, "age": age, "last_birth": np.full(n, last_birth), "num_babies": np.zeros(n, np.int32),
        "mate_id": np.full(n, -3, dtype=np.int64),
    }


def _genomes(rng, n, loci, changed):
    """One shared random genome with a few random nucleotides of `changed`
    agents in a hundred changed."""
    words = 2 * abi.genome_words(loci)
    g = np.tile(rng.integers(0, 2 ** 63, size=words, dtype=np.int64).astype(np.uint64), (n, 1))
    rows = np.flatnonzero(rng.random(n) < changed / 100.0)
    for _ in range(4):
        pos = rng.integers(0, 2 * loci, len(rows))
        g[rows, pos // 32] ^= rng.integers(1, 4, len(rows)).astype(np.uint64) << (2 * (pos % 32)).astype(np.uint64)
    return np.ascontiguousarray(g.ravel())


def _population(case, seed):
    """The case's model, agents placed, ready to step."""
    model = case["model"]
    rng = np.random.default_rng([seed, 7])
    nav = None
    if model == "lattice":
        grid, env = rect_grid(case["width"], case["height"]), {}
        params = scenarios.c1(seed=seed, width=4, height=4, n_agents=4)["params"]
        params.verh_b0, params.verh_d0, params.verh_theta = 0.8, 0.001, 0.1   # the tutorial's rates
        agents = _agents(rng, np.arange(grid["num_cells"], dtype=np.int32), 10.0, abi.QHG_LIFE_FERTILE, 0.0)
    elif model == "navigate":
        grid, env, nav, good, params = _coast(case["level"])
        params = type(params).from_buffer_copy(params)
        params.seed = seed
        agents = _agents(rng, good, 10.0, abi.QHG_LIFE_ALIVE, -1.0)
    else:
        grid, env, good = _world(case["level"])
        assort = {"hamming": (0.9, 1), "protein": (1.0, 1)}.get(model)
        params = scenarios.ooa_params(seed, genetics=model != "ooa", assort=assort, protein=model == "protein",
                                      genome_size=case.get("loci", 256))
        agents = _agents(rng, good, 10.0, abi.QHG_LIFE_ALIVE, -1.0)
        if model != "ooa":
            if model == "protein":
                params.gen_mutation_rate = 1e-6   # the matching proteins stay common over a long run
            agents["genome"] = _genomes(rng, len(agents["id"]), case["loci"], 20 if model == "protein" else 100)
    pop = GpuPopulation(grid, env, params, agents)
    if nav is not None:
        pop.set_navigation(nav)
    pop.preLoop(0.0)
    return pop


def _settle(case):
    return {"hamming": 400, "protein": 1200}.get(case["model"], 120)


class _State:
    """What a program keeps: the handles, and host arrays with room for the
    agents it reads back; closed with the state."""

    def __init__(self, case):
        self.case, self.pops, self.batch, self.t = case, [], None, 0.0
        self.out, self.parts = None, []

    def make_room(self):
        room = [(32 if p.grid["connectivity"] == 4 else 12) * p.grid["num_cells"] + 512 for p in self.pops]
        words = self.pops[0].gwords
        self.out = {k: np.zeros(sum(room), dtype=dt) for k, (dt, _) in abi.AGENT_FIELDS.items()}
        if words:
            self.out["genome"] = np.zeros(sum(room) * words, dtype=np.uint64)
        at = 0
        for r in room:
            self.parts.append((r, {k: v[at * words:(at + r) * words] if k == "genome" else v[at:at + r]
                                   for k, v in self.out.items()}))
            at += r

    def read(self):
        """Every population's live agents, in id order, into the arrays."""
        alive = np.zeros(len(self.pops), dtype=np.int64)
        for i, (pop, (room, into)) in enumerate(zip(self.pops, self.parts)):
            alive[i] = pop.getNumAgentsEffective()
            if alive[i] > room:
                raise RuntimeError("no room for %d agents" % alive[i])
            check(lib().qhg_gpu_download_agents(pop.h, ctypes.byref(abi.agents_struct(into, int(alive[i])))),
                  "qhg_gpu_download_agents")
        out = dict(self.out, alive=alive)
        if "genome" in out:
            out["genome"] = out["genome"].view(np.int64)   # the words as they are, signed
        return out

    def __del__(self):
        if self.batch is not None:
            self.batch.close()
        for p in self.pops:
            p.close()


def prepare(case, seed):
    s = _State(case)
    if case["kind"] == "batch":
        s.batch = GpuBatch()
        for k in range(case["members"]):
            # replicas of unequal size: levels 3, 4 and 5
            pop = _population(dict(model="ooa", level=3 + k % 3), 1000 * seed + k)
            s.pops.append(pop)
            s.batch.add(pop)
        s.batch.set_graph(True)
        s.batch.run(120)
        s.batch.sync()
    elif case["kind"] == "event":
        s.pops.append(_population(dict(model="ooa", level=case["level"]), seed))
        s.env = _event_env(case, seed)
    else:
        s.pops.append(_population(case, seed))
        s.pops[0].run(_settle(case))
        s.pops[0].sync()
        s.t = float(_settle(case))
    if case["kind"] != "event":
        s.make_room()
    return s


def _event_env(case, seed):
    """A warmer or wetter world: the NPP rescaled and shifted cell by cell."""
    _, env, _ = _world(case["level"])
    rng = np.random.default_rng([seed, 11])
    npp = env["base_npp"] * case.get("npp_scale", 1.1) + rng.normal(0.0, 0.05, len(env["base_npp"]))
    return {"base_npp": np.clip(npp, 0.0, 2.0), "altitude": env["altitude"] + rng.normal(0.0, 20.0, len(npp))}


# -- a pass -------------------------------------------------------------------
def run(s):
    case = s.case
    if case["kind"] == "event":
        pop = s.pops[0]
        pop.env_event(s.env, abi.EVENT_CLIMATE | abi.EVENT_VEG)
        return {"capacity": pop.capacities(), "weights": pop.env_weights()}
    if case["kind"] == "batch":
        s.batch.run(case["steps"])
        s.batch.sync()
        return s.read()
    pop = s.pops[0]
    if case["kind"] == "run":
        pop.run(case["steps"])
    else:
        for _ in range(case["steps"]):
            # PopLooper::doStep: the phases in order, then the extinction check
            pop.initializeStep(s.t)
            pop.doActions(0, s.t)
            pop.finalizeStep()
            s.t += 1.0
            if pop.getNumAgentsEffective() == 0:
                break
    return s.read()


# -- what a pass cannot do without ----------------------------------------------
def _cells(case):
    return case["width"] * case["height"] if case.get("model") == "lattice" else 10 * 4 ** case["level"] + 2


def _step_work(case, live):
    """Per step, in place: an agent's record read and its changed fields
    written (57 bytes), an occupied cell's rows, the births."""
    cells = _cells(case)
    words = 2 * abi.genome_words(case["loci"]) if "loci" in case else 0
    births = 0.055 * live
    return 57.0 * live + 88.0 * min(cells, live / 10) + births * (60 + 24 * words), 80.0 * live


def work(case):
    if case["kind"] == "event":
        # NPP, altitude, longitude, latitude and neighbours in; capacity and weights out
        return {"bytes": _cells(case) * (4 * 8 + 6 * 4 + 8 + 7 * 8.0), "flops": _cells(case) * 60.0}
    if case["kind"] == "batch":
        parts = [work(dict(kind="run", model="ooa", level=3 + k % 3, steps=case["steps"]))
                 for k in range(case["members"])]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    live = _cells(case) * (LATTICE_LIVE if case["model"] == "lattice" else WORLD_LIVE)
    b, f = _step_work(case, live)
    record = 50 + (16 * abi.genome_words(case["loci"]) if "loci" in case else 0)
    return {"bytes": b * case["steps"] + 2.0 * live * record, "flops": f * case["steps"]}


# -- in 64 bits ------------------------------------------------------------------
def exact(case, seed):
    """The event's tables from their definitions.  A stepped population is a
    sequence of draws and discrete outcomes: its times are whole steps and
    initial ages carried along, for which there is no other value than the
    simulation itself."""
    if case["kind"] != "event":
        return None
    grid, env, _ = _world(case["level"])
    new = _event_env(case, seed)
    alt, npp = new["altitude"], new["base_npp"]
    k_max = 75.0
    af = np.where(alt < 1500, 1.0, np.maximum((2500 - alt) / 1000.0, 0.0))
    tn = npp * af
    oceania = (grid["lon"] > 115) & (grid["lon"] < 150) & (grid["lat"] > -12) & (grid["lat"] < 1)
    tn = np.where(oceania & (npp < 0.0), 0.0, tn)
    K = np.where(alt > 0, np.minimum(np.where(tn > 1.5, k_max, tn * k_max / 1.5), k_max), 0.0)
    xs, vs = np.array(scenarios.sigmoid_polyline()).T
    pref = np.interp(alt.astype(np.float32).astype(np.float64), xs, vs)
    nbr = grid["neighbors"]

    def row(v):
        v = np.maximum(v, 0.0)
        return np.concatenate([v[:, None], np.where(nbr >= 0, v[nbr], 0.0)], axis=1)

    return {"capacity": K, "weights": np.cumsum(row(pref) * row(K), axis=1).ravel()}
