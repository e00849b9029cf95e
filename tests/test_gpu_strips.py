"""The strip kernel on the shapes that the automatic choice gives to the band
kernel: the checks of the other test modules with strips asked for, by one class
threshold set to its automatic value (which leaves every threshold as it is).
Plain and compensated; footprints wider than any staged table and than a region,
shortened table ids (unfolded direct reads), grids that end inside a region,
XCD groups, the captured form, the allocation-free form, and the records that
k_gather_visits writes."""
import pytest

from mi355_gridding import _lib
import test_gpu_batched as batched
import test_gpu_buckets as buckets
import test_gpu_parity as parity
import test_zz_no_alloc as noalloc

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def strips(gpu):
    ctx = gpu[1].context()
    ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 6)
    yield
    ctx.set_option(_lib.OPT_MIN_STAGE_RUN_W33, 0)


@pytest.mark.parametrize("cfg,N,G,P,smax", parity.CASES)
def test_config_shapes(gpu, cfg, N, G, P, smax):
    parity.test_device_grid_against_fp64_oracle(gpu, cfg, N, G, P, smax)


@pytest.mark.parametrize("G,smax", [(1001, 24), (130, 12), (300, 36)])
def test_grid_sizes(gpu, G, smax):
    parity.test_grid_sizes_off_the_region_grid(gpu, G, smax)


@pytest.mark.parametrize("smax,N", [(100, 4000), (160, 3000)])
def test_large_supports(gpu, smax, N):
    parity.test_large_supports_against_fp64_oracle(gpu, smax, N)


def test_shortened_table_ids(gpu):
    parity.test_many_planes_shortened_table_ids_against_fp64_oracle(gpu)


def test_shortened_table_ids_compensated(gpu):
    torch, ops = gpu
    c = parity.small_config(2, 20_000, 512, 4000, 8, seed=5)
    t, tn, ts = parity.oracle.grid_fsel_d(c)
    g, n, s = parity.run_grid(torch, ops, c, mode="comp")
    assert s == ts and abs(n - tn) <= 1e-12 * abs(tn)
    assert parity.errors(g, t)[0] <= 1e-6


def test_item_splits_and_groups(gpu):
    parity.test_deterministic_and_item_split_invariant(gpu)


@pytest.mark.parametrize("compensated", [0, 1])
def test_captured(gpu, compensated):
    batched.test_graph_replays_equal_eager(gpu, compensated)


def test_batched(gpu):
    batched.test_batched_equals_sequential(gpu)


def test_allocation_free(gpu):
    noalloc.test_noalloc_matches_device_entry_point(gpu)


@pytest.mark.parametrize("cfg,N,G,P,smax,seed", [(2, 30_000, 1024, 80, 72, 7),
                                                 (1, 60_000, 2048, 714, 36, 8)])
def test_records(gpu, cfg, N, G, P, smax, seed):
    buckets.test_buckets_bitexact_against_selection(gpu, cfg, N, G, P, smax, seed, (6, 6, 3, 3))
