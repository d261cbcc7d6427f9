"""The library's host code on a stand-in for the HIP runtime (host_runtime/fake_hip.cpp), in processes of their own: what one
device, or a machine with enough memory, does not show.  No device needed."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    where = tmp_path_factory.mktemp("runtime")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-Wno-deprecated-declarations",
                    os.path.join(HERE, "host_runtime", "fake_hip.cpp"), "-Wl,-soname,libamdhip64.so.7",
                    "-Wl,--version-script=" + os.path.join(HERE, "host_runtime", "versions.map"), "-o", str(where / "libamdhip64.so.7")], check=True)
    return where


def on(runtime, program):
    head = """
        import ctypes, sys
        import numpy as np
        from meganeura_amd import capi
        capi.load()
        hip = ctypes.CDLL("libamdhip64.so.7")
        assert hasattr(hip, "fake_launches"), "not the stand-in"
        hip.fake_refuse_allocations_of.argtypes = [ctypes.c_size_t]
        hip.fake_launch_log.restype = ctypes.c_char_p
        def current():
            d = ctypes.c_int()
            hip.hipGetDevice(ctypes.byref(d))
            return d.value
    """
    env = dict(os.environ, LD_LIBRARY_PATH=str(runtime), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(head) + textwrap.dedent(program)], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("nbytes", [5, 3 << 20, 20 << 20])  # one piece of the ring, pieces, slots
def test_copies_belong_to_the_contexts_device(runtime, nbytes):
    """A context's first copies made while another device is current: its events are made on its own device, and the other device is
    current again afterwards."""
    on(runtime, f"""
        with capi.Context(1) as ctx:
            b = ctx.buffer({nbytes})
            hip.hipSetDevice(0)
            want = np.random.default_rng(1).integers(0, 256, {nbytes}, dtype=np.uint8)
            for direction in range(2):
                b.upload(want)
                assert current() == 0
                assert np.array_equal(b.download(np.uint8, {nbytes}), want)
                assert current() == 0
            b.free()
    """)


@pytest.mark.parametrize("nth", [0, 1, 2, 9])
@pytest.mark.parametrize("upload", [True, False])
def test_threads_that_cannot_be_made(runtime, nth, upload):
    """Large copies ask for threads; where the host has no memory for the nth of them, those there are do the work."""
    on(runtime, f"""
        with capi.Context(0) as ctx:
            want = np.random.default_rng(2).integers(0, 256, 20 << 20, dtype=np.uint8)
            b = ctx.buffer(want.size)
            if {upload}:
                hip.fake_fail_allocation(ctypes.c_long({nth}))
            b.upload(want)
            if not {upload}:
                hip.fake_fail_allocation(ctypes.c_long({nth}))
            assert np.array_equal(b.download(np.uint8, want.size), want)
            hip.fake_fail_allocation(ctypes.c_long(-1))
            b.free()
    """)


@pytest.mark.parametrize("fmt", [0, 1])
def test_a_context_without_room_for_the_blocked_kernel(runtime, fmt):
    """The blocked kernel's 96 MiB workspace is not to be had: the context exists without it, and the calls that would take the kernel
    run on the ones behind it."""
    on(runtime, f"""
        m, k, n = 77, 4096, 14336
        assert capi.matmul_block_plan({fmt}, m, k, n).taken
        def run(ctx):
            w = ctx.weight_from_packed({fmt}, np.zeros(capi.packed_size({fmt}, k, n), np.uint8), k, n)
            a, c = ctx.buffer(m * k * 4), ctx.buffer(m * n * 4)
            before = hip.fake_launches(b"12block_kernel"), hip.fake_launches(b"tile_")
            ctx.matmul_q(a, w, c, m)
            ctx.sync()
            return hip.fake_launches(b"12block_kernel") - before[0], hip.fake_launches(b"tile_") - before[1]
        with capi.Context(0) as ctx:
            assert run(ctx) == (1, 0)
        hip.fake_refuse_allocations_of(96 << 20)
        with capi.Context(0) as ctx:
            assert run(ctx)[0] == 0 and run(ctx)[1] > 0
            ctx.set_route(capi.ROUTE_BLOCK_MFMA)
            try:
                run(ctx)
                assert False, "a kernel that has no workspace"
            except capi.MgnError as e:
                assert e.status == capi.EINVAL
    """)


def test_the_automatic_plan_is_what_is_launched(runtime):
    """mgn_matmul_q_auto_plan against the launches of the calls themselves: the kernel, its grid and its threads, in every range of rows,
    for both formats and all three kinds of activations."""
    on(runtime, """
        KERNELS = {capi.ROUTE_GEMV_MFMA: "gemv", capi.ROUTE_GEMM_MFMA: "gemm_mfma_kernel", capi.ROUTE_TILE_MFMA: "tile_", capi.ROUTE_BLOCK_MFMA: "12block_kernel"}
        seen = set()
        with capi.Context(0) as ctx:
            a, c = ctx.buffer(520 * 4096 * 4), ctx.buffer(520 * 14336 * 4)
            for fmt in (0, 1):
                for k, n in ((576, 1536), (1024, 3072), (2048, 2048), (4096, 4096), (4096, 14336), (4096, 1000)):
                    w = ctx.weight_from_packed(fmt, np.zeros(capi.packed_size(fmt, k, n), np.uint8), k, n)
                    for m in (1, 4, 5, 16, 17, 33, 40, 64, 96, 127, 128, 200, 512):
                        for act in ("any", "f16", "range"):
                            ctx.set_activation_range(act == "range")
                            hip.fake_launch_log()
                            (ctx.matmul_q_f16a if act == "f16" else ctx.matmul_q)(a, w, c, m)
                            log = [l.split() for l in hip.fake_launch_log().decode().splitlines()]
                            p = capi.matmul_plan(fmt, m, k, n, act == "f16", fp16_range=act == "range", auto=True)
                            where = (fmt, m, k, n, act, p.route, log)
                            main = [l for l in log if KERNELS[p.route] in l[0]]
                            assert main and all(int(l[4]) == p.threads for l in main), where
                            wgs = p.grid[0] * p.grid[1] * p.grid[2]
                            got = sum(int(l[1]) * int(l[2]) * int(l[3]) for l in main)
                            kind = p.route
                            if p.route == capi.ROUTE_TILE_MFMA:
                                kind = "resident" if p.quads_per_wave == 0 else "general"
                                assert ("tile_resident_kernel" in main[0][0]) == (kind == "resident"), where
                            if p.route == capi.ROUTE_BLOCK_MFMA:
                                tiles = p.grid[1] * p.grid[2]
                                assert got == -(-tiles // 8) * 8 * p.grid[0] and p.quads_per_wave == 1, where
                                assert (p.k_parts > 1) == any("add_parts" in l[0] for l in log), where
                                b = capi.matmul_block_plan(fmt, m, k, n, act == "f16")
                                assert b.taken and (b.row_groups, b.col_groups, b.k_parts) == (p.grid[2], p.grid[1], p.grid[0]), where
                            elif kind == "resident" and p.k_parts > 1:
                                assert got == -(-p.grid[1] * p.grid[2] // 8) * 8 * p.grid[0], where
                            elif kind != "general" or p.quads_per_wave == 1:
                                assert got == wgs, where
                            seen.add((kind, fmt, act))
                    w.free()
            resident_q8 = capi.matmul_plan(1, 64, 1024, 3072, auto=True)
            assert resident_q8.quads_per_wave == 0 and capi.matmul_plan(1, 64, 1024, 3072).quads_per_wave > 0
        assert len({s[0] for s in seen}) >= 4, seen
    """)


@pytest.mark.parametrize("fmt,m,k,n,taken", [(0, 77, 14336, 4096, False), (1, 77, 14336, 4096, False), (0, 33, 8192, 7168, False), (1, 33, 8192, 7168, False),
                                             (0, 512, 1024, 8192, True), (1, 512, 2048, 2048, True)])
def test_the_static_entry_takes_the_same_calls_on_a_forced_blocked_route(runtime, fmt, m, k, n, taken):
    """Of the blocked kernel's calls, those that the kernels behind it could run on the library's array: by the automatic choice and by force."""
    on(runtime, f"""
        assert (capi.matmul_plan({fmt}, {m}, {k}, {n}).workspace_bytes <= capi.STATIC_WORKSPACE_BYTES) == {taken}
        assert capi.matmul_block_plan({fmt}, {m}, {k}, {n}).taken
        with capi.Context(0) as ctx:
            w = ctx.weight_from_packed({fmt}, np.zeros(capi.packed_size({fmt}, {k}, {n}), np.uint8), {k}, {n})
            a, c = ctx.buffer({m * k * 4}), ctx.buffer({m * n * 4})
            for route in (capi.ROUTE_AUTO, capi.ROUTE_BLOCK_MFMA):
                ctx.set_route(route)
                before = hip.fake_launches(b"12block_kernel")
                try:
                    ctx.matmul_q_static(a, w, c, {m})
                    assert {taken} and hip.fake_launches(b"12block_kernel") == before + 1, route
                except capi.MgnError as e:
                    assert not {taken} and e.status == capi.EUNSUPPORTED and hip.fake_launches(b"12block_kernel") == before, route
    """)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("m,k,n,groups,launched", [(333, 3072, 1024, 84, 84), (320, 2080, 1024, 80, 80), (16, 14336, 4352, 17, 17), (250, 2080, 800, 64, 64),
                                                   (300, 2080, 800, 76, 80)])
def test_the_grid_of_k_parts(runtime, fmt, m, k, n, groups, launched):
    """Column groups x row groups of a resident launch with K parts: rounded up to a multiple of 8 where the rounds stay the same, as they are
    where they would not."""
    on(runtime, f"""
        with capi.Context(0) as ctx:
            w = ctx.weight_from_packed({fmt}, np.zeros(capi.packed_size({fmt}, {k}, {n}), np.uint8), {k}, {n})
            a, c = ctx.buffer({m * k * 4}), ctx.buffer({m * n * 4})
            ctx.set_route(capi.ROUTE_TILE_MFMA)
            p = capi.matmul_plan({fmt}, {m}, {k}, {n})
            assert p.quads_per_wave == 0 and p.k_parts > 1 and p.grid[1] * p.grid[2] == {groups}, (p.quads_per_wave, p.k_parts, list(p.grid))
            hip.fake_launch_log()
            ctx.matmul_q(a, w, c, {m})
            log = [l.split() for l in hip.fake_launch_log().decode().splitlines()]
            got = [l for l in log if "tile_resident_kernel" in l[0]]
            assert len(got) == 1 and [int(v) for v in got[0][1:4]] == [{launched}, p.k_parts, 1], log
    """)


@pytest.mark.parametrize("fmt,m,k,n,f16", [(1, 96, 8544, 2606, False), (1, 42, 8096, 253, False), (0, 118, 13056, 1600, False), (0, 641, 9280, 4274, True),
                                           (1, 508, 3456, 5248, False)])
def test_the_blocked_kernel_launches_the_workgroups_that_there_are(runtime, fmt, m, k, n, f16):
    """The tiles of all K parts, dealt out evenly over eight XCDs, and no workgroup more than that takes."""
    on(runtime, f"""
        with capi.Context(0) as ctx:
            w = ctx.weight_from_packed({fmt}, np.zeros(capi.packed_size({fmt}, {k}, {n}), np.uint8), {k}, {n})
            a, c = ctx.buffer({m * k * 4}), ctx.buffer({m * n * 4})
            ctx.set_route(capi.ROUTE_BLOCK_MFMA)
            p = capi.matmul_block_plan({fmt}, {m}, {k}, {n}, {f16})
            tiles = p.row_groups * p.col_groups
            assert p.k_parts > 1 and tiles % 8 and p.launches == 1
            hip.fake_launch_log()
            (ctx.matmul_q_f16a if {f16} else ctx.matmul_q)(a, w, c, {m})
            log = [l.split() for l in hip.fake_launch_log().decode().splitlines()]
            got = [l for l in log if "12block_kernel" in l[0]]
            assert len(got) == 1 and [int(v) for v in got[0][1:4]] == [-(-tiles * p.k_parts // 8) * 8, 1, 1], log
    """)
