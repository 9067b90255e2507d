"""Conditions that the host planners guarantee to the kernels, on the CPU.

The batch kernel sums a gradient term in the sweep that applies the gadget's
inverse, with one barrier after both; a gradient item on its own would read
rows that the next item already writes.  A plan that separates the two must be
refused, and so must an MFMA pass over tiles that do not hold the column blocks
of every wave.
"""
import subprocess

from test_emu_kernels import BUILD, CXX, EMU, FLAGS, drive  # noqa: F401


def _check(source, without, tmp_path):
    """Builds and runs tests/emu/<source>, which includes the source of unit `without`."""
    exe = tmp_path / source.split(".")[0]
    objs = [str(BUILD / f"{u}.o") for u in ("kernels_tile_emu", "kernels_stream_emu", "kernels_rtile_emu", "rtile_plan",
                                            "kernels_batch", "kernels_reduce", "kernels_gemm", "engine", "circuit",
                                            "batch", "emu_rt") if u != without]
    subprocess.run([CXX, *FLAGS, str(EMU / source), *objs, "-o", str(exe), "-lpthread",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)


def test_plans_the_kernels_cannot_run_are_refused(drive, tmp_path):  # noqa: F811
    r = _check("plan_checks.cpp", "batch", tmp_path)
    assert r.returncode == 0 and "ACCEPTED" not in r.stdout, r.stdout + r.stderr


def test_register_tile_passes_access_whole_lines(drive, tmp_path):  # noqa: F811
    r = _check("sweep_checks.cpp", "circuit", tmp_path)
    assert r.returncode == 0, r.stdout + r.stderr
