"""bench.py's account of a profile: the unit the roofline is read on and its bytes."""
import bench

N = 128 * 64 * 4


def profile(**launched):
    p = {k: (0.0, 0) for k in ("convdiff", "bc", "rhs", "bicg_init", "bicg_A", "bicg_B", "bicg_C",
                               "bicg_check", "sor_half", "project", "mg", "pb")}
    p.update({"convdiff": (0.02, 1), "project": (0.02, 1)}, **launched)
    return p


def test_launched_phases_count_as_one_iteration():
    p = profile(bicg_A=(4.0, 100), bicg_B=(3.0, 100), bicg_C=(3.0, 100))
    r = bench.step_roofline(p, N, "none", 97)
    assert r["bound"] == "hbm" and r["bytes_per_launch"] == 128 * N
    assert r["avg_launch_us"] == 100.0 and r["achieved"] == round(128 * N / 1e-4 / 1e9, 1)
    assert bench.kernel_table(p, N, bench.launch_bytes(p, 97))["bicg_A"]["GBps"] is not None


def test_a_resident_solve_is_read_by_the_iteration():
    p = profile(bicg_A=(3.4, 1))  # 340 iterations of 10 us in one launch
    r = bench.step_roofline(p, N, "none", 340)
    assert r["bound"] == "latency" and "k_bicg_grid" in r["kernel"]
    assert r["avg_launch_us"] == 10.0 and r["bytes_per_launch"] == 16 * N
    assert bench.kernel_table(p, N, bench.launch_bytes(p, 340))["bicg_A"]["GBps"] is None


def test_sor_launches_are_passes_or_half_sweeps():
    passes = profile(sor_half=(5.0, 182))  # 301 sweeps: 151 passes, the last batch exits
    r = bench.step_roofline(passes, N, "none", 301)
    assert r["kernel"] == "sor_pass" and r["bytes_per_launch"] == 24 * N
    halves = profile(sor_half=(5.0, 634))  # 602 half sweeps
    r = bench.step_roofline(halves, N, "none", 301)
    assert r["kernel"] == "sor_half" and r["bytes_per_launch"] == 16 * N
