"""GPU: the plan (stable CSR / CSC build + schedule) is bit-exact with the numpy
oracle (stable argsort), through the C ABI."""
import numpy as np
import pytest
import torch

from oracle import graph_prep as gp
from torchgt_amd import _lib, workloads
from torchgt_amd.plan import GraphPlan, _plan_bytes

pytestmark = pytest.mark.gpu


def _check_plan(ei_np, N, cuda):
    print(f"plan case N={N} E={ei_np.shape[1]}", flush=True)
    ei = torch.from_numpy(np.ascontiguousarray(ei_np)).to(cuda)
    plan = GraphPlan(ei, N)
    for by, ids in (("dst", (_lib.PLAN_ROWPTR_DST, _lib.PLAN_COL_DST, _lib.PLAN_EID_DST, _lib.PLAN_ITEMS_DST)),
                    ("src", (_lib.PLAN_ROWPTR_SRC, _lib.PLAN_COL_SRC, _lib.PLAN_EID_SRC, _lib.PLAN_ITEMS_SRC))):
        rowptr, col, eid = gp.build_csr(ei_np, N, by)
        np.testing.assert_array_equal(plan.export(ids[0]), rowptr)
        np.testing.assert_array_equal(plan.export(ids[2]), eid)
        np.testing.assert_array_equal(plan.export(ids[1]), col)
        # schedule: items tile every row exactly once, in order, segments <= limit
        items = plan.export(ids[3]).reshape(-1, 4)
        seg = plan.info()["segment_len"]
        assert np.all(items[:, 2] <= seg) and np.all(items[:, 2] >= 0)
        order = np.lexsort((items[:, 1], items[:, 0]))
        it = items[order]
        covered = np.zeros(N, dtype=np.int64)
        np.add.at(covered, it[:, 0], it[:, 2])
        np.testing.assert_array_equal(covered, np.diff(rowptr))
        first = np.ones(len(it), dtype=bool)
        first[1:] = it[1:, 0] != it[:-1, 0]
        np.testing.assert_array_equal(it[first, 1], rowptr[it[first, 0]])
        cont = ~first
        np.testing.assert_array_equal(it[cont, 1], it[np.nonzero(cont)[0] - 1, 1] + it[np.nonzero(cont)[0] - 1, 2])
        split = np.diff(rowptr) > seg
        assert np.all((it[:, 3] >= 0) == split[it[:, 0]])
        parts = np.sort(it[it[:, 3] >= 0, 3])
        np.testing.assert_array_equal(parts, np.arange(len(parts)))
    plan.close()
    return True


def test_plan_small_random(cuda):
    rng = np.random.default_rng(0)
    for N, E in ((1, 0), (1, 3), (7, 0), (5, 1), (100, 1000), (300, 5000), (257, 4097), (70000, 200000)):
        ei = rng.integers(0, N, (2, E))
        _check_plan(ei, N, cuda)


def test_plan_hub_and_duplicates(cuda):
    rng = np.random.default_rng(1)
    N = 3000
    ei = rng.integers(0, N, (2, 20000))
    ei[1, :9000] = 17                      # hub destination with 9000 in-edges (split row)
    ei[0, 9000:15000] = 5                  # hub source
    ei[:, 15000:16000] = ei[:, 16000:17000]   # duplicate edges
    _check_plan(ei, N, cuda)


def test_plan_config1_and_config2_graphs(cuda):
    e1, n1 = workloads.barabasi_albert()
    assert (n1, e1.shape[1]) == (4097, 45024)
    _check_plan(e1, n1, cuda)
    e2, n2 = workloads.power_law_graph()
    assert n2 == 64001 and abs(e2.shape[1] - 530000) < 0.02 * 530000
    _check_plan(e2, n2, cuda)


# Tiles of 1024 and of 4096 keys: one that ends inside, at and behind a tile, the largest sort of small tiles (eight per CU, two views) and the
# first of large ones
def test_plan_at_the_edges_of_the_sorts_tiles(cuda):
    rng = np.random.default_rng(3)
    few = 4 * torch.cuda.get_device_properties(cuda).multi_processor_count * 1024
    for N, E in ((40, 1023), (40, 1024), (40, 1025), (300, 2049), (5000, few), (5000, few + 1), (70000, few - 1), (70000, few + 4096)):
        _check_plan(rng.integers(0, N, (2, E)), N, cuda)


def test_plan_three_radix_passes(cuda):
    # N > 65536 needs three 8-bit passes; ids spread over the whole range
    rng = np.random.default_rng(2)
    N = 300000
    ei = rng.integers(0, N, (2, 400000))
    _check_plan(ei, N, cuda)


def test_plan_rejects_out_of_range(cuda):
    ei = torch.tensor([[0, 1, 9], [1, 2, 0]], device=cuda)
    with pytest.raises(_lib.TorchGTHipError) as exc:
        GraphPlan(ei, 5)
    assert exc.value.code == _lib.ERR_INDEX_RANGE
    ei = torch.tensor([[0, -1], [1, 2]], device=cuda)
    with pytest.raises(_lib.TorchGTHipError):
        GraphPlan(ei, 5)


def test_plan_is_reproducible(cuda):
    rng = np.random.default_rng(3)
    ei = torch.from_numpy(rng.integers(0, 5000, (2, 60000))).to(cuda)
    a, b = GraphPlan(ei, 5000), GraphPlan(ei, 5000)
    for which in range(8):
        np.testing.assert_array_equal(a.export(which), b.export(which))


@pytest.mark.parametrize("near,lengths,rows", [(True, [1, 12, 6, 30], 256), (False, [1, 5, 2, 6], 256), (False, [1, 12, 6, 30], 128)])
def test_windows_of_large_graphs(cuda, near, lengths, rows):
    """From 128 K rows on windows have 256 rows where most neighbours are near or rows are short (below ten edges), else 128: the wave items go window by
    window, and inside one by length class."""
    print(f"windows near={near} lengths={lengths}", flush=True)
    n, g = (1 << 17) + 200, torch.Generator(device=cuda).manual_seed(1)
    dst = torch.repeat_interleave(torch.arange(n, device=cuda), torch.tensor(lengths, device=cuda).repeat(n // 4))
    src = (dst + torch.randint(-500, 501, dst.shape, generator=g, device=cuda)).clamp(0, n - 1) if near else torch.randint(0, n, dst.shape, generator=g, device=cuda)
    plan = GraphPlan(torch.stack([src, dst]), n)
    items = plan.export(6).reshape(-1, 4)[plan.info()["block_items_dst"]:, 0]
    for size, in_order in ((rows, True), (rows // 2, False)):
        assert bool((np.diff(items // size) >= 0).all()) == in_order, size
    assert np.array_equal(np.sort(items), np.arange(n))
    plan.close()


@pytest.mark.parametrize("near", [True, False])
@pytest.mark.parametrize("n,length", [(20000, 5), (64000, 9), (64000, 17), (64000, 33), (140000, 5), (140000, 17), (140000, 33)])
def test_bytes_of_a_cached_plan_are_a_bound(cuda, n, length, near):
    """What the plan cache counts for a plan covers what the plan holds, at the row lengths where a wave record is fullest of rows and emptiest of edges;
    with near neighbours the backward has two lists of records."""
    print(f"plan bytes n={n} length={length} near={near}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(1)
    dst = torch.arange(n, device=cuda).repeat_interleave(length)
    src = (dst + torch.randint(-500, 501, dst.shape, generator=g, device=cuda)).clamp(0, n - 1) if near else torch.randint(0, n, dst.shape, generator=g, device=cuda)
    ei = torch.stack([src, dst])
    before = torch.cuda.memory_allocated()
    plan = GraphPlan(ei, n)
    held = torch.cuda.memory_allocated() - before
    assert plan.info()["near_neighbours"] == int(near and (length >= 10 or n >= 128 << 10))
    # (the allocator rounds each of a plan's arrays up to 512 bytes)
    assert 0 < held <= _plan_bytes(plan) + 32 * 512
    plan.close()
