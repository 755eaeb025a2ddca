"""bench.py's traffic per H x from counter databases: every kernel of an H x counts, and a
run whose H x differ, or whose kernels are not all there, is refused."""
import sqlite3

import pytest

import bench

TILES = "void (anonymous namespace)::k_apply_tiles<float, 512, 8, 4, 4, true>((anonymous namespace)::DevTables)"
NN = "void bsl::(anonymous namespace)::k_nn<float>(bsl::Tab, float const*, float*, int)"
PP = "bsl::(anonymous namespace)::k_pp(bsl::Tab, float const*, float*)"
OTHER = ["bsl::(anonymous namespace)::k_pp(bsl::Tab, double const*, double*)",
         "void bsl::(anonymous namespace)::k_nn<double>(bsl::Tab, double const*, double*, int)",
         "bsl::(anonymous namespace)::k_pp_fill(int, int const*, float*, double*)"]


def _db(path, rows):
    c = sqlite3.connect(path)
    c.execute("create table counters_collection (dispatch_id integer, kernel_name text, value real, duration integer)")
    c.executemany("insert into counters_collection values (?, ?, ?, ?)", [(i,) + r for i, r in enumerate(rows)])
    c.commit()
    c.close()
    return str(path)


D = 100_000_000
PROBE = ("__amd_rocclr_copyBuffer", 4.0 * D / 1024 / 2, 9)  # the counter reads half


def test_three_kernels(tmp_path):
    h = [(NN, 1000.0, 10), (PP, 2000.0, 20), (TILES, 4000.0, 40)]
    db = _db(tmp_path / "f.db", [(n, 5e6, 1) for n in OTHER] + h + h + [PROBE])
    t = bench.traffic_from_dbs(db, db, D)
    assert t["fetch"]["bytes_per_launch"] == pytest.approx(7000 * 1024 * 2)
    assert t["fetch"]["mean_duration_ns"] == 70 and t["kernel"] == TILES and len(t["kernels"]) == 3
    assert t["bytes_per_launch"] == pytest.approx(2 * 7000 * 1024 * 2)


def test_tile_kernel_alone(tmp_path):
    db = _db(tmp_path / "f.db", [(TILES, 4000.0, 40), (TILES, 6000.0, 40), PROBE])
    t = bench.traffic_from_dbs(db, db, D)
    assert t["fetch"]["bytes_per_launch"] == pytest.approx(5000 * 1024 * 2) and t["kernels"] == [TILES]


@pytest.mark.parametrize("rows", [[(NN, 1.0, 1), (TILES, 4.0, 4)], [(NN, 1.0, 1), (PP, 1.0, 1), (TILES, 4.0, 4), (TILES, 4.0, 4)],
                                  [(TILES, 4.0, 4), (TILES.replace("true", "false"), 4.0, 4)], [(NN, 1.0, 1), (PP, 1.0, 1)]])
def test_refused(rows, tmp_path):
    db = _db(tmp_path / "f.db", rows + [PROBE])
    with pytest.raises(RuntimeError):
        bench.traffic_from_dbs(db, db, D)
