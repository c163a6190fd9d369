"""Which kernels a call launches, on the CPU: the library's host code against a stand-in HIP
runtime that records the launches (tests/hostmock/route_mock.cpp, routes.cpp). No kernel runs."""
from __future__ import annotations

import os
import pathlib
import re
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
SRC = ROOT / "kwinto-cuda_amd" / "csrc"
MOCK = pathlib.Path(__file__).resolve().parent / "hostmock"
HIPCC = "/opt/rocm/bin/hipcc"
UNITS = ["kwgpu_api", "fd1d_wave", "fd1d_lane", "bs", "surrogate"]
LISTED = ["zero_counters", "plan_windows", "list_windows", "fd1d_windowed"]


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    """routes(request, ...): the kernels that each request launches, a list of names each."""
    if not os.path.exists(HIPCC):
        pytest.skip("ROCm compilers not installed")
    d = tmp_path_factory.mktemp("routes")
    host = [HIPCC, "-O1", "-std=c++17", "-fPIC", "--offload-host-only", f"-I{ROOT / 'include'}",
            f"-I{SRC}", f"-I{MOCK}"]
    src = [SRC / f"{u}.hip" for u in UNITS] + [MOCK / "route_mock.cpp", MOCK / "routes.cpp"]
    jobs = [subprocess.Popen(host + ["-c", str(s), "-o", str(d / (s.stem + ".o"))],
                             stderr=subprocess.PIPE, text=True) for s in src]
    for p, s in zip(jobs, src):
        err = p.communicate(timeout=600)[1]
        assert p.returncode == 0, f"{s}: {err}"
    objs = [str(d / (s.stem + ".o")) for s in src]
    # each unit refers to its (absent) device code object by a generated name
    nm = subprocess.run(["nm", "-u", *objs], capture_output=True, text=True, check=True).stdout
    names = sorted(set(re.findall(r"__hip_fatbin_\w+", nm)))
    (d / "fatbins.cpp").write_text("".join(f'extern "C" {{ char {n}[16]; }}\n' for n in names))
    subprocess.run(["g++", *objs, str(d / "fatbins.cpp"), "-o", str(d / "routes")], check=True)

    def run(*requests):
        r = subprocess.run([str(d / "routes")], input="\n".join(requests) + "\n", text=True,
                           capture_output=True, timeout=120)
        assert r.returncode == 0, r.stderr
        return [re.split(r",(?! )", ln) if ln else [] for ln in r.stdout.split("\n")[:-1]]
    return run


def test_capture_takes_no_shared_scratch(routes, tmp_path):
    """A call captured into a graph may be replayed beside any other: it may only launch
    kernels that keep nothing in the context's or the device's scratch (work counters,
    windows' records and lists)."""
    sizes = ["%s %d %d %d" % (c, n, x, t) for c in ("price", "noalloc") for n, x, t in (
        (64, 512, 128), (2048, 1024, 256), (2049, 1024, 256), (2400, 256, 66), (16384, 512, 512),
        (600, 2048, 256), (1500, 1025, 90), (4000, 2048, 257))]
    free, held = routes("capture 0", *sizes), routes("capture 1", *sizes)
    assert any("plan_windows" in k for k in free)
    # tuned to the 16-row variants on persistent grids
    (tmp_path / "tune").write_text("256 0 2 1\n512 0 5 1\n1024 0 8 1\n2048 0 9 1\n")
    tuned = routes(f"tune {tmp_path / 'tune'}", "capture 1", *sizes)
    for call, k in list(zip(sizes, held[1:])) + list(zip(sizes, tuned[2:])):
        assert len(k) == 1 and k[0].split("<")[0] in ("fd1d_wave", "fd1d_lone"), (call, k)
        assert k[0] == "fd1d_lone" or k[0].split(", ")[4] == "false", (call, k)  # persistent


@pytest.mark.parametrize("variant", [-3, -7, -100])
def test_tune_file_with_an_unknown_march(routes, tmp_path, variant):
    """A tune file's march numbers below those that exist are skipped, as variants that do not
    hold their bucket are: no lane kernel runs without its workspace."""
    f = tmp_path / "tune"
    f.write_text("".join(f"{cap} 0 {variant} 0\n" for cap in (128, 256, 512, 1024, 2048)))
    calls = ["price 100 128 90", "price 3000 512 400", "uneven 300 90 100,256,700,2048",
             "noalloc 3000 512 400", "noalloc_uneven 300 90 100,256,700,2048", "host 50 256 90"]
    plain, tuned = routes(*calls), routes(f"tune {f}", *calls)[1:]
    assert plain == tuned
    # the lane layout itself (-1) is still taken from a file, with its workspace
    f.write_text("512 0 -1 0\n")
    for k in routes(f"tune {f}", "price 3000 512 400", "uneven 300 90 100,256,512,2048")[1:]:
        assert any("fd1d_lane" in x for x in k) and "null workspace" not in k


def test_tuned_whole_grid_march_beside_windows(routes, tmp_path):
    """Where a bucket is tuned to the windowed march, its calls that take no windows (short or small
    uniform batches, Greeks, capture) keep the tuned whole-grid variant; so they do after a save
    and a load."""
    f, g = tmp_path / "tune", tmp_path / "saved"
    f.write_text("512 0 7 0\n512 0 -2 0\n256 0 4 1\n256 0 -2 0\n")
    calls = ["price 2400 512 66", "noalloc 2400 512 66", "price 400 512 40", "greeks 40 512 90", "price 3000 512 512"]
    loaded = routes(f"tune {f}", f"save {g}", *calls, "capture 1", "price 3000 512 512")[2:]
    again = routes(f"tune {g}", *calls, "capture 1", "price 3000 512 512")[1:]
    assert loaded == again
    for k in (*loaded[:4], loaded[6]):
        assert any(x.startswith("fd1d_wave<8, 64, 1") for x in k), k
    assert "fd1d_windowed" in loaded[4]


def test_per_option_grids_take_the_windowed_forms(routes):
    """The forms that test_window_forms.py and test_window_again.py are written for."""
    lone, lone_big, listed, big, small = routes(
        "uneven 64 130 512,512", "uneven 64 130 512,1500", "uneven 2400 130 512", "uneven 1400 130 512,2048",
        "uneven 300 90 60,100")
    assert "fd1d_lone" in lone and "plan_windows" not in lone
    assert "fd1d_lone_big" in lone_big and "fd1d_window_again" in lone_big
    assert [k for k in LISTED if k in listed] == LISTED
    assert "fd1d_windowed_big" in big and "fd1d_window_again" in big
    assert not any("window" in k or "lone" in k for k in small)


def test_rule_for_uniform_batches(routes):
    """Which uniform batches take the windowed march, at the lines of the rule."""
    calls = {"price 1024 896 65": True, "price 1024 897 65": False, "price 1025 256 65": False,
             "price 1025 257 65": True, "price 2048 256 99": False, "price 2048 256 100": True,
             "price 2049 512 256": False, "price 2049 512 257": True, "price 512 1100 65": False,
             "price 1024 1025 400": False, "price 1025 1025 65": True, "price 64 512 64": False,
             "price 64 512 65": True, "price 64 128 400": False, "price 64 129 400": True,
             "price 2049 2049 65": False, "greeks 300 512 512": False}
    for call, k in zip(calls, routes(*calls)):
        assert any("lone" in x or "windowed" in x for x in k) == calls[call], (call, k)
