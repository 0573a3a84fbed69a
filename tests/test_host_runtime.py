"""What the host side of the library allocates, copies and launches, seen by a
HIP runtime that runs on the CPU and computes nothing (tests/native/fake_hip.cpp):
libmfc_lbm.so is loaded in a process of its own, behind that runtime."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PREAMBLE = """
import ctypes as C, os, sys
sys.path[:0] = [{root!r}, {here!r}]
fake = C.CDLL({fake!r}, mode=C.RTLD_GLOBAL)
fake.fake_max_lds.restype = fake.fake_allocated.restype = C.c_size_t
fake.fake_set_free.argtypes = [C.c_size_t]
import numpy as np
from helpers import small_params
from multiphase_flow_codes_amd.lbm import Lattice, lib, _dp
def lattice(n=(20, 18, 16), precision="fp64", storage="ab", **kw):
    return Lattice(small_params(n=n, forcing=False, **kw), precision, storage=storage)
def fields(n, seed=0):
    rng = np.random.default_rng(seed)
    return [rng.normal(size=n[::-1]) for _ in range(4)]
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """Runs a piece of code behind the CPU runtime."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    fake = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run([gxx, "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Werror", "-o", fake,
                    os.path.join(HERE, "native", "fake_hip.cpp")], check=True, timeout=300)

    def go(code, **env):
        pre = PREAMBLE.format(root=ROOT, here=HERE, fake=fake)
        r = subprocess.run([sys.executable, "-c", pre + textwrap.dedent(code) + "\nprint('done')"],
                           capture_output=True, text=True, timeout=300, env=dict(os.environ, **env))
        assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr

    return go


def test_fields_come_back(run):
    run("""
        for n in ((4, 4, 4), (17, 16, 8), (64, 64, 32), (75, 71, 73)):
            lat, a = lattice(n), fields(n)
            lat.upload_macro(*a)
            for x, y in zip(lat.download_macro(), a):
                assert np.array_equal(x, y)
    """)


def test_download_of_nothing_succeeds(run):
    """Each target of mfc_download_macro may be null, all of them too."""
    run("""
        lat, a = lattice(), fields((20, 18, 16))
        lat.upload_macro(*a)
        assert lib().mfc_download_macro(lat.h, None, None, None, None) == 0
        uy = np.empty_like(a[2])
        assert lib().mfc_download_macro(lat.h, None, None, _dp(uy), None) == 0
        assert np.array_equal(uy, a[2])
    """)


def test_results_of_another_device(run):
    """Contexts of device 1 read by threads whose current device is 0: what such
    a read allocates and launches is on device 1, and 0 stays current."""
    run("""
        import threading
        a, got = fields((20, 18, 16)), []
        fake.hipSetDevice(1)
        lat = lattice(npart=2, rad=3.0)
        lat.prt_init(2)
        lat.upload_macro(*a)
        lat.prt_set("ypglb", np.array([[5.0, 5.0, 5.0], [14.0, 12.0, 11.0]]))
        lat.beads_links()
        fake.fake_reset()

        def read():
            lat.sync()
            lat.status()
            got.extend(lat.download_macro())
            got.append(lat.prt_get("ypglb"))
            d = C.c_int(-1)
            fake.hipGetDevice(C.byref(d))
            got.append(d.value)

        t = threading.Thread(target=read)
        t.start()
        t.join()
        assert len(got) == 6 and got[5] == 0
        for x, y in zip(got, a):
            assert np.array_equal(x, y)
        assert got[4][1, 0] == 14.0
        assert fake.fake_launches(b"k_copy_out") == 4 and fake.fake_launches(b"k_link_totals") == 1
        assert fake.fake_foreign() == 0
    """)


@pytest.mark.parametrize("alloc,n,copies", [
    ("hipHostMalloc", (64, 60, 62), 1),   # large: the bus reaches pinned memory without the thread's copy
    ("hipHostMalloc", (20, 18, 16), 0),   # small: the windows are faster
    ("hipMalloc", (64, 60, 62), 1),
    ("hipMalloc", (20, 18, 16), 1),       # the thread may not be able to write it
])
def test_targets_the_runtime_knows(run, alloc, n, copies):
    """Results for memory of the runtime's own are left to its copy, those for
    ordinary memory beside them still go through the windows."""
    run(f"""
        n = {n}
        size = n[0] * n[1] * n[2]
        lat, a = lattice(n), fields(n)
        lat.upload_macro(*a)
        p, out = C.c_void_p(), np.empty(n[::-1])
        assert fake.{alloc}(C.byref(p), C.c_size_t(8 * size), 0) == 0
        p = C.cast(p, C.POINTER(C.c_double))
        for target in (None, _dp(out)):
            fake.fake_reset()
            assert lib().mfc_download_macro(lat.h, None, p, None, target) == 0
            assert np.array_equal(np.ctypeslib.as_array(p, (size,)), a[1].ravel())
            assert fake.fake_copies() == {copies}
            assert (fake.fake_launches(b"k_copy_out") > 0) == (target is not None or not {copies})
        assert np.array_equal(out, a[3])
    """)


def test_padding_of_rows_is_bounded(run):
    """Two buffers take at most an eighth more than their 19 values per node,
    rows of up to 64 nodes no more than those; and a lattice that fits the
    memory without padding is made (and read back) however little is left."""
    run("""
        def populations(n, precision):
            before = fake.fake_allocated()
            lat = lattice(n, precision)
            got = fake.fake_allocated() - before
            # forcing tables, phase tables and the rest of a context
            rest = 4 * 8 * 18 * n[1] * n[2] + 16 * sum(n) + 8 * (16384 + 1024) + 4096
            lat.close()
            return got, rest

        for precision, size in (("fp32", 4), ("fp64", 8), ("fp32x", 4)):
            for nx in list(range(4, 40)) + [48, 50, 63, 64, 65, 66, 70, 75, 90, 96, 100, 111, 112, 113, 115, 120,
                                            129, 130, 150, 170, 200, 257, 262, 300, 1000]:
                n = (nx, 24, 20)
                need = 2 * 19 * size * nx * n[1] * n[2]
                got, rest = populations(n, precision)
                assert need <= got <= (need if nx <= 64 else need * 9 // 8) + rest, (precision, nx, got, need)

        n = (150, 24, 20)
        size = 8 * n[0] * n[1] * n[2]
        tight = 2 * 19 * size + 4 * 8 * 18 * n[1] * n[2] + 4 * size + (1 << 19)
        a = fields(n)
        fake.fake_set_free(tight)
        lat = lattice(n)
        lat.upload_macro(*a)
        assert all(np.array_equal(x, y) for x, y in zip(lat.download_macro(), a))
    """)


@pytest.mark.parametrize("mode", ["1", "2"])
@pytest.mark.parametrize("storage", ["ab", "aa"])
def test_overlapped_step_does_not_wait_for_the_contact_list(run, mode, storage):
    """Contact links are listed behind the refill (in its grid in place, by a grid
    beside the near collide with two buffers), not ahead of the bounce-back,
    except the first one after links built on their own; a call's last
    bounce-back takes them from the other buffer where there is one."""
    run(f"""
        lat = lattice((40, 36, 32), "fp32", "{storage}", npart=2, rad=3.0)
        lat.upload_macro(*fields((40, 36, 32)))
        lat.initpop()
        lat.macrovar()
        lat.prt_init(2)
        lat.prt_set("ypglb", np.array([[9.0, 9.0, 9.0], [28.0, 20.0, 21.0]]))
        lat.beads_links()
        fake.fake_launch.restype = C.c_char_p
        ahead = []
        for first, n in ((1, 6), (7, 3), (10, 1)):
            fake.fake_reset()
            lat.step(first, n)
            names = []
            while fake.fake_launch(len(names)):
                names.append(fake.fake_launch(len(names)).decode())
            names = [x for x in names if any(k in x for k in ("k_contacts", "k_tile_mark", "k_bounce_back", "k_fill"))]
            assert sum("k_bounce_back" in x for x in names) == n
            # listed behind the refill, or where the next step's bounce-back starts
            ahead.append(sum("k_tile_mark" in a and "k_contacts" in b for a, b in zip(names, names[1:])))
            behind = sum("k_fill" in a and "k_contacts" in b for a, b in zip(names, names[1:]))
            assert behind == (n - 1 if "{storage}" == "ab" else 0)
        assert ahead == ([1, 1, 0] if "{storage}" == "ab" else [1, 0, 0])
    """, MFC_OVERLAP=mode)


def test_prerelax_answers_an_interrupt(run):
    """A signal handler's exception ends the loop after a batch of iterations, not
    after all of them; counts and stops as one iteration after the other."""
    run("""
        import math, signal
        lat = lattice((8, 8, 8))
        def start():
            lat.upload_macro(*fields((8, 8, 8)))
            lat.initpop()
            fake.fake_reset()
        start()
        # the CPU runtime's residual is 0
        assert lat.prerelax(0.0, 5) == (0, 0.0)
        for m in (-3, -1, 0, 1, 2.5, 125, 126, 127, 128, 129, 254.9, 300):
            start()
            it, err = lat.prerelax(-1.0, m)
            assert (it, err) == (max(math.floor(m) + 1, 0), 0.0), (m, it)
            assert fake.fake_launches(b"k_rho_residual") == it + 1
        def stop(*_):
            raise KeyboardInterrupt
        signal.signal(signal.SIGALRM, stop)
        for limit in (300000, math.inf, math.nan):
            start()
            signal.setitimer(signal.ITIMER_REAL, 0.03)
            try:
                lat.prerelax(-1.0, limit)
                raise AssertionError
            except KeyboardInterrupt:
                pass
            assert fake.fake_launches(b"k_rho_residual") < 290000
    """)


def test_prerelax_calls_replaced_methods(run):
    run("""
        class Counting(Lattice):
            n = 0
            def rhoupdat(self):
                self.n += 1
                return super().rhoupdat() + (1.0 if self.n < 4 else 0.0)
        lat = Counting(small_params(n=(8, 8, 8), forcing=False), "fp64")
        lat.upload_macro(*fields((8, 8, 8)))
        lat.initpop()
        assert lat.prerelax(0.5) == (3, 0.0) and lat.n == 4
        lat = lattice((8, 8, 8))
        lat.upload_macro(*fields((8, 8, 8)))
        lat.initpop()
        seen = []
        step = lat.streaming
        lat.streaming = lambda: (seen.append(1), step())
        assert lat.prerelax(-1.0, 2) == (3, 0.0) and len(seen) == 4
    """)


def test_spectrum_stays_within_its_lds(run):
    """Transform tiles of lines of up to 2048 entries take at most 96 KB of LDS
    along x, and 72 KB along y and z with 8 B more per shell along z."""
    run("""
        def spectrum(n, nek):
            lat = lattice(n, "fp32")
            lat.upload_macro(*fields(n))
            fake.fake_reset()
            ek = np.zeros(nek)
            assert lib().mfc_diag_spectrum(lat.h, nek, _dp(ek)) == 0
            assert fake.fake_launches(b"invalid") == 0
            return fake.fake_max_lds(b"k_fft")

        sizes = [4, 5, 7, 12, 64, 100, 127, 128, 250, 256, 500, 512, 1000, 682, 683, 1023, 1024, 1025, 1536, 2047, 2048]
        for m in sizes:
            for axis in range(3):
                n = [4, 4, 4]
                n[axis] = m
                for nek in (8, 4096):
                    got = spectrum(tuple(n), nek)
                    assert got <= max(96 * 1024, 72 * 1024 + 8 * nek), (n, nek, got)
    """)
