"""Launch shapes and memory of plan descriptions, on the CPU: the built-in choices as
rick_plan_describe() tells them, and the benchmark's record of them."""
import pytest

import bench
from rick_amd import FP32, FP64, GAUSS, GAUSS_HI_PRECISION, KAISERBESSEL, _lib, serve
from rick_amd.imaging import describe


def desc(nx, planes, rows, precision=FP64, support=7, kernel=KAISERBESSEL, **kw):
    d = _lib.PlanDesc(num_w_planes=planes, grid_size_x=nx, grid_size_y=nx, kernel=kernel,
                      w_support=support, dx=1.0 / nx, dw=1.0 / planes, precision=precision,
                      max_points=rows)
    for k, v in kw.items():
        setattr(d, k, v)
    return d


@pytest.mark.parametrize("nx,planes,rows,tile", [
    (256, 4, 50_000, (64, 32)), (512, 16, 100_000, (64, 32)), (512, 17, 100_000, (64, 64)),
    (4096, 32, 7_745_536, (64, 64)), (8192, 64, 2_900_000, (128, 32))])
def test_builtin_tiles(nx, planes, rows, tile):
    assert describe(desc(nx, planes, rows))["tile"] == tile


@pytest.mark.parametrize("kernel,support,planes,rows,tile", [
    (GAUSS_HI_PRECISION, 9, 2, 4095, (64, 64)), (GAUSS_HI_PRECISION, 9, 2, 4096, (64, 32)),
    (GAUSS_HI_PRECISION, 15, 17, 10 ** 6, (64, 64)), (GAUSS_HI_PRECISION, 15, 16, 10 ** 6, (64, 32)),
    (GAUSS_HI_PRECISION, 7, 2, 700, (64, 32)), (KAISERBESSEL, 9, 2, 700, (64, 32))])
def test_builtin_tile_of_a_dear_footprint(kernel, support, planes, rows, tile):
    assert describe(desc(256, planes, rows, support=support, kernel=kernel))["tile"] == tile


def test_named_shapes_stay():
    d = desc(8192, 8, 100_000, tile_u=32, tile_v=64, rows_per_task=777, footprint_unroll=11)
    s = describe(d)
    assert (s["tile"], s["rows_per_task"], s["unroll"]) == ((32, 64), 777, 11)


# Large FP64 tiles filled record by record keep the bucket order where the grid is large
# beside the rows; those by class, smaller ones and FP32 run their long tasks first.
@pytest.mark.parametrize("kernel,support,unroll,tile,by_class,bucket_order", [
    (KAISERBESSEL, 7, 0, (64, 64), True, False), (KAISERBESSEL, 11, 0, (64, 64), True, False),
    (KAISERBESSEL, 5, 0, (64, 64), False, True), (GAUSS, 3, 0, (64, 64), False, True),
    (KAISERBESSEL, 7, 9, (64, 64), False, True), (KAISERBESSEL, 15, 0, (64, 64), False, True),
    (GAUSS_HI_PRECISION, 7, 0, (64, 64), False, True),
    (KAISERBESSEL, 7, 0, (128, 32), False, True), (KAISERBESSEL, 5, 0, (64, 32), False, False),
    (GAUSS_HI_PRECISION, 7, 0, (32, 32), False, False)])
def test_task_order_follows_the_accumulation(kernel, support, unroll, tile, by_class, bucket_order):
    shape = dict(support=support, kernel=kernel, tile_u=tile[0], tile_v=tile[1],
                 footprint_unroll=unroll)
    most = 16 * 8 * 1024 * 1024 // (20 * support * support)      # 20 bytes a footprint cell
    for rows, order in ((most, bucket_order), (most + 1, False)):
        s = describe(desc(1024, 8, 1_000_000, **shape), rows)
        assert (s["by_class"], s["long_tasks_first"]) == (by_class, not order)
        assert describe(desc(1024, 8, 1_000_000, FP32, **shape), rows)["long_tasks_first"]


# A call takes the task length of its own rows, whatever the plan was made for.
@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("support,kernel", [(7, KAISERBESSEL), (5, KAISERBESSEL),
                                            (15, KAISERBESSEL), (7, GAUSS_HI_PRECISION)])
@pytest.mark.parametrize("rows", [1, 50_000, 516_000, 1_500_000])
def test_task_length_follows_the_call(rows, support, kernel, precision):
    own = describe(desc(1024, 8, rows, precision, support, kernel, tile_u=64, tile_v=64))
    big = describe(desc(1024, 8, 8_000_000, precision, support, kernel, tile_u=64, tile_v=64), rows)
    assert big["rows_per_task"] == own["rows_per_task"]
    assert describe(desc(1024, 8, 8_000_000, rows_per_task=3000), rows)["rows_per_task"] == 3000


def test_tasks_are_longer_before_a_plan_is_refused():
    # 8,387,600 tiles of one workgroup each leave slots for 1000 tasks of records.
    few = describe(desc(32, 8, 500_000, support=5, tile_u=32, tile_v=32))
    many = describe(desc(32, 8_387_600, 500_000, support=5, tile_u=32, tile_v=32))
    assert (few["rows_per_task"], many["rows_per_task"]) == (1024, 2048)


@pytest.mark.parametrize("bad", [{"w_support": 8}, {"tile_u": 48, "tile_v": 48},
                                 {"max_points": 2 ** 31}])
def test_what_no_plan_takes_has_no_shape(bad):
    with pytest.raises(_lib.RickError):
        describe(desc(256, 4, 1000, **bad))
    with pytest.raises(_lib.RickError):
        describe(desc(256, 4, 1000), 1001)


def test_benchmark_records_the_shapes_that_run():
    rows = 2_900_000
    plain, named = desc(8192, 64, rows, FP32), desc(8192, 64, rows, FP32, tile_u=64, tile_v=64,
                                                    rows_per_task=1024)
    got = bench.launch_shapes(plain, named, rows)
    assert got["tile"] == [128, 32] and got["image_tile"] == [64, 64]
    assert got["rows_per_task"] == describe(plain)["rows_per_task"] != 4096
    assert got["image_rows_per_task"] == 1024 and got["footprint_unroll"] == 7


@pytest.mark.parametrize("precision", [FP64, FP32])
@pytest.mark.parametrize("grid,planes,rows", [(256, 4, 50_000), (1024, 16, 1_000_000),
                                              (2048, 12, 3_000_000), (300, 4, 20_000)])
def test_service_charges_the_whole_plan(grid, planes, rows, precision):
    class Cfg:
        kernel, support, n_rows = KAISERBESSEL, 7, rows
    Cfg.grid, Cfg.planes = grid, planes
    cell = 16 if precision == FP64 else 8
    held = (planes * cell + 2 * 8) * grid * grid
    held += describe(desc(grid, planes, rows, precision))["device_bytes"]
    assert serve.grid_footprint(Cfg, precision) == held
    Cfg.support = 8         # refused: the job fails by itself, the service goes on
    assert 0 < serve.grid_footprint(Cfg, precision) < held


@pytest.mark.gpu
@pytest.mark.parametrize("nx,planes,rows,precision", [
    (256, 4, 50_000, FP32), (300, 3, 1000, FP64), (1024, 8, 0, FP32), (2048, 2, 100_000, FP64)])
def test_described_bytes_are_the_plans(nx, planes, rows, precision):
    from rick_amd import Plan
    plan = Plan(nx, nx, planes, precision=precision, max_points=rows)
    assert plan.shape()["device_bytes"] == plan.device_bytes
