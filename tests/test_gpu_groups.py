"""The step's grouping of cells at its edges: cells of around 64, 128 and 256
agents (a wave, half a block, a block, larger than a block), groups of many
small cells (table rows beyond the block's threads), groups that do not fit a
block, a mix of all; against the oracle, bit for bit.  And a look at the agents
inside a step, which must not change what the step commits."""
import numpy as np
import pytest

from qhg4_amd import abi, scenarios
from qhg4_amd.grids import rect_grid
from qhg4_amd.population import GpuBatch, GpuPopulation
from oracle.oracle import Oracle
from tests.helpers import assert_same_state, tut_verhulst

pytestmark = pytest.mark.gpu


def _counts(kind, ncells, rng):
    n = np.zeros(ncells, dtype=np.int64)
    if kind == "edges":
        sizes = [1, 2, 62, 63, 64, 65, 66, 126, 127, 128, 129, 130, 254, 255, 256, 257, 258, 511, 513]
        at = rng.choice(ncells, len(sizes), replace=False)
        n[at] = sizes
    elif kind == "ones":          # the most cells a group can hold
        n[:] = 1
    elif kind == "sixes":         # groups of 28 cells
        n[:] = 6
    elif kind == "fours":         # groups of 36 cells: weight rows past the block's threads, neighbour rows not
        n[:] = 4
    elif kind == "threes":        # groups of 42 cells: both
        n[:] = 3
    elif kind == "hundreds":      # two or three cells per group, some groups past a block
        n[rng.choice(ncells, 40, replace=False)] = rng.integers(90, 125, 40)
    elif kind == "mixed":
        n[:] = rng.choice([0, 0, 1, 2, 5, 30, 70], ncells)
        n[rng.choice(ncells, 6, replace=False)] = [150, 200, 256, 257, 300, 400]
    elif kind == "alone":
        n[7] = 1
    return n


def _scenario(kind, model, seed):
    rng = np.random.default_rng(seed)
    if model == "lattice":
        sc = tut_verhulst(scenarios.c1(seed=seed, width=23, height=19, n_agents=10))
        sc["params"].verh_K = 400.0
    else:
        sc = scenarios.c2(seed=seed, level=3, n_agents=10, patch_cells=5, genetics=model == "genetics")
        sc["params"].npp_k_max = 600.0
    ncells = sc["grid"]["num_cells"]
    n = _counts(kind, ncells, rng)
    cell = np.repeat(np.arange(ncells), n).astype(np.int32)
    m = len(cell)
    age = rng.uniform(0, 40, m)
    sc["agents"] = {
        "id": rng.permutation(np.arange(1, 3 * m + 1, dtype=np.int64))[:m], "cell": cell,
        "life": np.full(m, abi.QHG_LIFE_FERTILE, dtype=np.uint8), "gender": (rng.random(m) < 0.5).astype(np.uint8),
        "birth_time": -age, "age": age, "last_birth": np.full(m, -5.0), "mate_id": np.full(m, -3, dtype=np.int64),
        "num_babies": np.zeros(m, dtype=np.int32)}
    if model == "genetics":
        sc["agents"]["genome"] = scenarios.initial_genomes(rng, m, 256)
    return sc


KINDS = ["edges", "ones", "fours", "threes", "sixes", "hundreds", "mixed", "alone"]


@pytest.mark.parametrize("model", ["lattice", "ooa", "genetics"])
@pytest.mark.parametrize("kind", KINDS)
def test_groups_match_the_oracle(kind, model):
    sc = _scenario(kind, model, 41)
    gpu, ora = GpuPopulation.from_scenario(sc), Oracle(sc)
    gpu.preLoop()
    ora.pre_loop()
    for k in range(8):
        gpu.run(1)
        ora.run(1)
        assert_same_state(gpu.agents(), ora.agents(), "%s %s step %d" % (kind, model, k))
        gs, os_ = gpu.stats(), ora.stats()
        for f in ("num_alive", "births_last", "deaths_last", "moves_last"):
            assert gs[f] == os_[f], (f, gs[f], os_[f])
    gpu.close()


@pytest.mark.parametrize("group_agents", [1.0, 20.0, 64.0, 4096.0])
def test_group_sizes_do_not_change_results(group_agents):
    sc = _scenario("mixed", "ooa", 43)
    pop, bat, ora = GpuPopulation.from_scenario(sc), GpuPopulation.from_scenario(sc), Oracle(sc)
    pop.set_tuning(group_agents, 1)
    ora.pre_loop()
    b = GpuBatch()
    for p in (pop, bat):
        p.preLoop()
    b.add(bat)
    b.set_tuning(group_agents, 1)
    for k in range(3):
        pop.run(3)
        b.run(3)
        ora.run(3)
        assert_same_state(pop.agents(), ora.agents(), "alone %d" % k)
        assert_same_state(bat.agents(), ora.agents(), "batch %d" % k)
    b.close()


@pytest.mark.parametrize("model", ["lattice", "genetics"])
def test_a_look_inside_a_step_changes_nothing(model):
    sc = _scenario("mixed", model, 47)
    gpu, ora = GpuPopulation.from_scenario(sc), Oracle(sc)
    gpu.preLoop()
    ora.pre_loop()
    for k in range(4):
        before = gpu.agents()
        gpu.initializeStep(float(k))
        gpu.doActions(0, float(k))
        for _ in range(2):
            inside = gpu.agents()
            assert np.array_equal(inside["id"], before["id"])
            assert np.array_equal(inside["birth_time"], before["birth_time"])
            alive = inside["life"] != 0
            assert np.array_equal(inside["age"][alive], (k - inside["birth_time"])[alive])
            gave = inside["num_babies"] - before["num_babies"]
            assert set(gave) <= {0, 1} and np.all(inside["gender"][gave == 1] == 0)
            paired = np.flatnonzero(inside["mate_id"] >= 0)
            at = np.searchsorted(inside["id"], inside["mate_id"][paired])
            assert np.array_equal(inside["mate_id"][at], inside["id"][paired])
            assert np.array_equal(inside["cell"][at], inside["cell"][paired])
        gpu.state_digest()
        gpu.finalizeStep()
        ora.step()
        assert_same_state(gpu.agents(), ora.agents(), "%s step %d" % (model, k))
    gpu.close()


@pytest.mark.parametrize("width,height", [(1, 1), (511, 1), (512, 1), (513, 1), (32, 32), (41, 25), (600, 300)])
def test_scan_tiles_match_the_oracle(width, height):
    """Grids of a tile less one cell, a tile, one more, several; agents in
    every 7th cell and in the last one."""
    sc = tut_verhulst(scenarios.c1(seed=9, width=width, height=height, n_agents=10))
    ncells = width * height
    rng = np.random.default_rng(9)
    cell = np.unique(np.concatenate([np.arange(0, ncells, 7), [ncells - 1]])).repeat(5).astype(np.int32)
    m = len(cell)
    age = rng.uniform(0, 40, m)
    sc["agents"] = {
        "id": np.arange(1, m + 1, dtype=np.int64), "cell": cell,
        "life": np.full(m, abi.QHG_LIFE_FERTILE, dtype=np.uint8), "gender": (rng.random(m) < 0.5).astype(np.uint8),
        "birth_time": -age, "age": age, "last_birth": np.zeros(m), "mate_id": np.full(m, -3, dtype=np.int64),
        "num_babies": np.zeros(m, dtype=np.int32)}
    gpu, ora = GpuPopulation.from_scenario(sc), Oracle(sc)
    gpu.preLoop()
    ora.pre_loop()
    for k in range(4):
        gpu.run(3)
        ora.run(3)
        assert_same_state(gpu.agents(), ora.agents(), "step %d" % (3 * k + 3))
        assert np.array_equal(gpu.getNumAgentsArray(), ora.cell_counts())
    gpu.close()


def _protein_genomes(rng, n, genome_size, proteins):
    """Genomes of about that many proteins per agent: Met, a few codons and a
    stop, again and again, with a few nucleotides changed per agent."""
    words = 2 * abi.genome_words(genome_size)
    nuc = rng.integers(0, 4, 32 * words)
    per = (2 * genome_size // 3) // max(1, proteins)
    for strand in range(2):
        at = strand * 16 * words
        for k in range(0, genome_size // 3 - 3, max(3, per)):
            nuc[at + 3 * k:at + 3 * k + 3] = (0, 3, 2)                    # Met
            nuc[at + 3 * (k + 2):at + 3 * (k + 2) + 3] = (3, 0, 0)        # stop
    g = np.tile(nuc, (n, 1))
    for _ in range(3):
        g[np.arange(n), rng.integers(0, 32 * words, n)] = rng.integers(0, 4, n)
    g = g.reshape(n, words, 32).astype(np.uint64) << (2 * np.arange(32)).astype(np.uint64)
    return np.ascontiguousarray(g.sum(axis=2, dtype=np.uint64).ravel())


@pytest.mark.parametrize("kind", ["edges", "ones", "sixes", "hundreds", "mixed", "alone"])
@pytest.mark.parametrize("model", ["hamming", "hamming_noperm", "hamming_long", "protein", "protein_many"])
def test_assortative_groups_match_the_oracle(kind, model):
    """k_assort_pair at the same edges: 16 lanes per cell, tables of several
    cells, cells too large for a block; digests in the block's pool and past it."""
    rng = np.random.default_rng(51)
    prot = model.startswith("protein")
    size = 1100 if model == "hamming_long" else 256
    sc = scenarios.c2(seed=51, level=3, n_agents=10, patch_cells=5, genetics=True, genome_size=size, protein=prot,
                      assort=((1.0, 1) if prot else (0.9, 0 if model == "hamming_noperm" else 1)))
    sc["params"].npp_k_max = 600.0
    n = _counts(kind, sc["grid"]["num_cells"], rng)
    cell = np.repeat(np.arange(len(n)), n).astype(np.int32)
    m = len(cell)
    age = rng.uniform(0, 40, m)
    sc["agents"] = {
        "id": rng.permutation(np.arange(1, 3 * m + 1, dtype=np.int64))[:m], "cell": cell,
        "life": np.full(m, abi.QHG_LIFE_FERTILE, dtype=np.uint8), "gender": (rng.random(m) < 0.5).astype(np.uint8),
        "birth_time": -age, "age": age, "last_birth": np.full(m, -5.0), "mate_id": np.full(m, -3, dtype=np.int64),
        "num_babies": np.zeros(m, dtype=np.int32),
        "genome": (_protein_genomes(rng, m, size, 12 if model == "protein_many" else 4) if prot
                   else scenarios.initial_genomes(rng, m, size))}
    gpu, ora = GpuPopulation.from_scenario(sc), Oracle(sc)
    gpu.preLoop()
    ora.pre_loop()
    paired = 0
    for k in range(5):
        gpu.run(1)
        ora.run(1)
        got = gpu.agents()
        assert_same_state(got, ora.agents(), "%s %s step %d" % (kind, model, k))
        paired += int((got["mate_id"] >= 0).sum())
    assert paired > 0 or kind in ("ones", "alone")
    gpu.close()


@pytest.mark.parametrize("genome_size,crossovers,rate", [
    (4, 1, 0.2), (32, 5, 0.3), (32, 0, 0.0), (33, -1, 0.1), (97, 9, 0.1), (192, 3, 0.05), (500, 1, 0.02), (1024, -1, 1e-3),
    (1025, 32, 1e-3), (2048, 2, 5e-3)])
def test_genome_draws_match_the_oracle(genome_size, crossovers, rate):
    """Genomes of 2 to 128 words (32 births a pass of a wave to one birth in
    two passes, widths that do not divide a wave); draws within a birth's
    lanes' numbers and past them; mutation counts in and past the binomial
    table's first entries; alone and as a batch's members."""
    print("case: genome size %d, crossovers %d, rate %g" % (genome_size, crossovers, rate), flush=True)
    scs = []
    for seed in (61, 62):
        sc = scenarios.c2(seed=seed, level=3, n_agents=2500, patch_cells=60, genetics=True, genome_size=genome_size)
        p = sc["params"]
        p.gen_num_crossover, p.gen_mutation_rate = crossovers, rate
        words = 2 * abi.genome_words(genome_size)
        rng = np.random.default_rng(seed + genome_size)
        sc["agents"]["genome"] = rng.integers(0, 2**63, len(sc["agents"]["id"]) * words, dtype=np.uint64)
        scs.append(sc)
    gpu, oras = GpuPopulation.from_scenario(scs[0]), [Oracle(sc) for sc in scs]
    members = [GpuPopulation.from_scenario(sc) for sc in scs]
    for pop in [gpu] + members:
        pop.preLoop()
    for ora in oras:
        ora.pre_loop()
    batch = GpuBatch()
    for m in members:
        batch.add(m)
    for k in range(3):
        gpu.run(8)
        batch.run(8)
        for ora in oras:
            ora.run(8)
        assert_same_state(gpu.agents(), oras[0].agents(), "alone, step %d" % (8 * k + 8))
        for m, ora in zip(members, oras):
            assert_same_state(m.agents(), ora.agents(), "in a batch, step %d" % (8 * k + 8))
    assert oras[0].agents()["id"].max() > 2700      # (births: ids past the first 2500)
    batch.close()
    for pop in [gpu] + members:
        pop.close()


@pytest.mark.parametrize("changed", [0, 1, 4])
@pytest.mark.parametrize("model", ["hamming", "hamming_noperm", "protein"])
def test_assortative_rounds_match_the_oracle(model, changed):
    """Rounds of cells up to and past 16 females or males (16 lanes' registers
    and the table in LDS): all matches equal (every female in one round, the
    draws past a window of 16), and few to many different values."""
    rng = np.random.default_rng(57)
    prot = model == "protein"
    sc = scenarios.c2(seed=57, level=3, n_agents=10, patch_cells=5, genetics=True, protein=prot,
                      assort=((1.0, 1) if prot else (0.5, 0 if model == "hamming_noperm" else 1)))
    sc["params"].npp_k_max = 600.0
    sizes = [(1, 1), (1, 16), (16, 1), (2, 3), (3, 2), (4, 5), (7, 8), (8, 7), (9, 12), (15, 16), (16, 15), (16, 16),
             (16, 17), (17, 16), (17, 17), (1, 17), (17, 1), (14, 16), (16, 4), (20, 30)] * 3
    cells = rng.choice(sc["grid"]["num_cells"], len(sizes), replace=False)
    cell = np.concatenate([np.full(f + m, c) for (f, m), c in zip(sizes, cells)]).astype(np.int32)
    gender = np.concatenate([rng.permutation([0] * f + [1] * m) for f, m in sizes]).astype(np.uint8)
    n = len(cell)
    if prot:
        genome = _protein_genomes(np.random.default_rng(3), 1, 256, 4).reshape(1, -1)
    else:
        genome = scenarios.initial_genomes(np.random.default_rng(3), 1, 256).reshape(1, -1)
    genome = np.repeat(genome, n, axis=0)
    for _ in range(changed):
        genome[np.arange(n), rng.integers(0, genome.shape[1], n)] ^= np.uint64(1) << rng.integers(0, 64, n).astype(np.uint64)
    age = rng.uniform(0, 40, n)
    sc["agents"] = {
        "id": rng.permutation(np.arange(1, 3 * n + 1, dtype=np.int64))[:n], "cell": cell,
        "life": np.full(n, abi.QHG_LIFE_FERTILE, dtype=np.uint8), "gender": gender, "birth_time": -age, "age": age,
        "last_birth": np.full(n, -5.0), "mate_id": np.full(n, -3, dtype=np.int64),
        "num_babies": np.zeros(n, dtype=np.int32), "genome": np.ascontiguousarray(genome.ravel())}
    gpu, ora = GpuPopulation.from_scenario(sc), Oracle(sc)
    gpu.preLoop()
    ora.pre_loop()
    paired = 0
    for k in range(4):
        gpu.run(1)
        ora.run(1)
        got = gpu.agents()
        assert_same_state(got, ora.agents(), "%s %d step %d" % (model, changed, k))
        paired += int((got["mate_id"] >= 0).sum())
    assert paired > 0
    gpu.close()
