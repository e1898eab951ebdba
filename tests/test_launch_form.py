"""What the stencil's launches run, chosen on the host by the library's own selection
(lym_launch_form; no GPU): every form visits every site block once per right-hand
side, and the lattices that the GPU tests name for a form and a block order take them.
"""
import ctypes
import itertools
import os
import shutil
import subprocess

import numpy as np
import pytest

from helpers import ROOT

import leonardym_amd as lym

# (dims, parity, form, orders with blocks in them: plain, x-slice fastest, XCD pairs)
FP64_FIELD = [
    # four waves to a workgroup, each order: all workgroups at once, and sweeping
    ((4, 14, 22, 40), -1, lym.FORM_STAGED, (1, 0, 0)),
    ((16, 4, 28, 32), -1, lym.FORM_STAGED, (0, 1, 0)),
    ((8, 8, 28, 32), -1, lym.FORM_STAGED, (0, 0, 1)),
    ((4, 22, 28, 40), -1, lym.FORM_STAGED, (1, 0, 0)),
    ((40, 4, 16, 40), -1, lym.FORM_STAGED, (0, 1, 0)),
    ((8, 16, 26, 32), -1, lym.FORM_STAGED, (0, 0, 1)),
    # ranges that split x-slices
    ((98, 4, 4, 32), -1, lym.FORM_STAGED, (1, 1, 0)),
    ((194, 4, 4, 32), -1, lym.FORM_STAGED, (1, 1, 0)),
    ((98, 4, 8, 32), 1, lym.FORM_STAGED, (1, 1, 0)),
    ((4, 22, 28, 40), 1, lym.FORM_STAGED, (1, 0, 0)),
    ((40, 4, 16, 40), 1, lym.FORM_STAGED, (0, 1, 0)),
    ((8, 16, 26, 32), 1, lym.FORM_STAGED, (0, 0, 1)),
    # one wave to a workgroup
    ((10, 10, 10, 40), -1, lym.FORM_WAVE, (1, 0, 0)),
    ((16, 4, 14, 48), -1, lym.FORM_WAVE, (0, 1, 0)),
    ((8, 4, 32, 40), -1, lym.FORM_WAVE, (0, 0, 1)),
    ((6, 14, 28, 28), 1, lym.FORM_WAVE, (1, 0, 0)),
    ((40, 4, 16, 26), 1, lym.FORM_WAVE, (0, 1, 0)),
    ((8, 8, 22, 48), 1, lym.FORM_WAVE, (0, 0, 1)),
    ((17, 15, 13, 21), 0, lym.FORM_WAVE, (1, 0, 0)),
    ((14, 14, 14, 14), -1, lym.FORM_WAVE, (1, 0, 0)),
    # the benchmark's apply and the largest lattice
    ((16, 16, 16, 32), -1, lym.FORM_STAGED, (0, 0, 1)),
    ((32, 32, 32, 64), -1, lym.FORM_STAGED, (0, 0, 1)),
]


@pytest.mark.parametrize("dims,parity,form,orders", FP64_FIELD, ids=lambda v: str(v).replace(", ", "x"))
def test_fp64_field(dims, parity, form, orders):
    r = lym.launch_form(dims, parity)
    assert (r["form"], tuple(int(b > 0) for b in r["branches"])) == (form, orders), r["branches"]


@pytest.mark.parametrize("dims,parity,prec,nrhs,form", [
    # FP64: 32768 lanes of one field, whichever the parities
    ((16, 16, 16, 16), 0, 0, 1, lym.FORM_HOP), ((16, 16, 16, 8), -1, 0, 1, lym.FORM_HOP),
    ((16, 16, 16, 18), 0, 0, 1, lym.FORM_WAVE), ((16, 16, 16, 10), -1, 0, 1, lym.FORM_WAVE),
    ((16, 16, 16, 24), 0, 0, 1, lym.FORM_WAVE),
    # over several lanes 8192, over two 49152
    ((8, 8, 8, 8), 0, 0, 4, lym.FORM_HOP), ((8, 8, 8, 8), 1, 0, 6, lym.FORM_LANES),
    ((8, 8, 8, 16), 0, 0, 3, lym.FORM_LANES), ((16, 16, 16, 12), 1, 0, 2, lym.FORM_HOP),
    ((12, 12, 12, 24), -1, 0, 2, lym.FORM_LANES), ((16, 16, 16, 14), 0, 0, 2, lym.FORM_LANES),
    ((12, 12, 12, 24), 0, 0, 12, lym.FORM_LANES), ((4, 4, 4, 4), -1, 0, 16, lym.FORM_HOP),
    # low precision: 49152 of one parity, 32768 of both, over the right-hand sides
    ((16, 16, 16, 24), 0, 1, 1, lym.FORM_HOP), ((16, 16, 16, 24), 0, 2, 1, lym.FORM_HOP),
    ((16, 16, 16, 26), 0, 1, 1, lym.FORM_SPLIT), ((16, 16, 16, 26), 0, 2, 1, lym.FORM_SPLIT),
    ((16, 16, 16, 8), -1, 2, 1, lym.FORM_HOP), ((16, 16, 16, 10), -1, 2, 1, lym.FORM_SPLIT),
    ((12, 12, 12, 12), 0, 2, 4, lym.FORM_HOP), ((12, 12, 12, 12), 0, 2, 6, lym.FORM_SITE),
    # two threads per site up to 131072 sites of a parity
    ((16, 16, 32, 32), 0, 1, 1, lym.FORM_SPLIT), ((16, 18, 32, 32), 0, 1, 1, lym.FORM_SITE),
])
def test_limits(dims, parity, prec, nrhs, form):
    assert lym.launch_form(dims, parity, prec, nrhs, single=nrhs == 1)["form"] == form


def test_matrix_cores():
    for nrhs in (2, 4, 8):
        assert lym.launch_form((8, 8, 8, 8), 0, 2, nrhs, matrix_cores=True)["form"] == lym.FORM_MFMA
    for prec, nrhs in ((2, 3), (2, 16), (1, 4)):
        assert lym.launch_form((8, 8, 8, 8), 0, prec, nrhs, matrix_cores=True)["form"] == lym.FORM_SITE


def test_every_block_once():
    seen = set()
    lattices = [(4, 4, 4, 4), (6, 6, 6, 8), (4, 6, 2, 8), (12, 12, 12, 12), (18, 4, 4, 32), (14, 14, 14, 14),
                (16, 16, 16, 32), (10, 12, 14, 22), (98, 4, 4, 32), (24, 24, 24, 32), (5, 7, 3, 6), (17, 15, 13, 21)]
    options = [dict(nrhs=1), dict(nrhs=1, single=True), dict(nrhs=1, lane_ops=True), dict(nrhs=2),
               dict(nrhs=2, matrix_cores=True), dict(nrhs=3), dict(nrhs=4, lane_ops=True), dict(nrhs=6, threads=192),
               dict(nrhs=8, threads=64), dict(nrhs=12), dict(nrhs=16)]
    for dims, parity, prec, kw in itertools.product(lattices, (-1, 0, 1), (0, 1, 2), options):
        odd = any(d % 2 for d in dims)
        if odd and (parity or kw["nrhs"] > 1 or prec):
            continue  # one site class, FP64 launches of one field
        r = lym.launch_form(dims, parity, prec, **kw)
        want = np.zeros_like(r["visits"])
        want[[0, 1] if parity < 0 else [parity]] = 1 if prec else kw["nrhs"]
        assert np.array_equal(r["visits"], want), (dims, parity, prec, kw)
        per_class = int(np.prod(dims)) // (1 if odd else 2)
        assert r["spb"] * r["nbpp"] >= per_class > r["spb"] * (r["nbpp"] - 1)
        assert r["threads"] <= 512 and r["partials"] == 0
        seen.add(r["form"])
    assert seen == set(range(7))


def test_bad_arguments():
    for kw in (dict(prec=3), dict(nrhs=0), dict(nrhs=17), dict(threads=-1), dict(threads=1024), dict(part_max=-1),
               dict(parity=2), dict(dims=(1, 4, 4, 4)), dict(dims=(5, 4, 4, 4), parity=1)):
        with pytest.raises(lym.LymError):
            lym.launch_form(**{"dims": (4, 4, 4, 4), **kw})


@pytest.mark.parametrize("dims,nrhs,form", [
    # the lanes of the matrix-core form reach a link entry at 288 bytes a site of a parity,
    # a spinor component at 32 bytes a (site, right-hand side), and a buffer holds 2^31 - 1
    ((60, 60, 64, 64), 2, lym.FORM_MFMA), ((60, 60, 64, 64), 8, lym.FORM_MFMA),
    ((60, 62, 64, 64), 2, lym.FORM_SITE), ((60, 62, 64, 64), 8, lym.FORM_SITE), ((64, 64, 64, 64), 4, lym.FORM_SITE),
])
def test_matrix_cores_within_a_buffer(dims, nrhs, form):
    for parity in (-1, 0):
        r = lym.launch_form(dims, parity, 2, nrhs, matrix_cores=True)
        assert r["form"] == form and np.all(r["visits"][0] == 1)
    sites = int(np.prod(dims)) // 2
    assert (288 * sites <= 0x7fffffff and 32 * sites * nrhs <= 0x7fffffff) == (form == lym.FORM_MFMA)


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("step", [1, 2])
def test_a_step_without_room_is_not_taken(prec, step):
    """A launch with more workgroups than the partial sums hold runs without the step and
    says so; with room it leaves one per workgroup."""
    for dims in ((4, 4, 4, 4), (12, 12, 12, 24), (16, 16, 16, 32), (24, 24, 24, 32)):
        r = lym.launch_form(dims, -1, prec, single=True, step=step, part_max=1 << 20)
        assert r["partials"] == r["grid"] > 1
        assert lym.launch_form(dims, -1, prec, single=True, step=step, part_max=r["grid"])["partials"] == r["grid"]
        assert lym.launch_form(dims, -1, prec, single=True, step=step, part_max=r["grid"] - 1)["partials"] == 0
    # several right-hand sides, or a kappa each: never
    assert lym.launch_form((8, 8, 8, 8), -1, prec, nrhs=2, step=step, part_max=1 << 20)["partials"] == 0
    if step == 2 or prec == 0:
        assert lym.launch_form((8, 8, 8, 8), -1, prec, lane_ops=True, step=step, part_max=1 << 20)["partials"] == 0


def test_room_of_the_fp64_solvers():
    """The FP64 solvers' partial sums (8192, or one per 256 sites of a lattice) hold those of
    any launch of theirs."""
    r = np.random.default_rng(5)
    dims = [tuple(int(v) for v in r.integers(2, 40, 4)) for _ in range(150)]
    dims += [(64, 64, 64, 64), (32, 32, 32, 64), (2, 2, 2, 2), (3, 3, 3, 3), (48, 48, 48, 96)]
    for d in dims:
        odd = any(x % 2 for x in d)
        vh = int(np.prod(d)) // (1 if odd else 2)
        for parity in (0,) if odd else (-1, 0, 1):
            q = lym.launch_form(d, parity, step=2, part_max=max(8192, 2 * ((vh + 255) // 256)))
            assert q["partials"] == q["grid"], (d, parity)


@pytest.mark.parametrize("width", [64, 128, 512])
def test_other_workgroup_sizes(width, tmp_path):
    """LYM_DSLASH_THREADS is a build option: with another value every form still visits
    every block once per right-hand side (the selection alone, built with it)."""
    stub, so = tmp_path / "fail.cpp", tmp_path / "plan.so"
    stub.write_text("namespace lym_internal { int fail(int code, const char*, ...) { return code; } }\n")
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.check_call([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-fPIC", "-shared", "-w",
                           "-DLYM_DSLASH_THREADS=%d" % width,
                           os.path.join(ROOT, "leonardym_amd", "csrc", "plan.cpp"), str(stub), "-o", str(so)])
    call = ctypes.CDLL(str(so)).lym_launch_form
    call.argtypes = lym.SIGNATURES["lym_launch_form"][1]
    for dims, parity, prec, nrhs in itertools.product([(4, 4, 4, 4), (12, 12, 12, 24), (16, 16, 16, 32), (10, 12, 14, 22)],
                                                      (-1, 0, 1), (0, 1, 2), (1, 2, 3, 4, 6, 8, 12, 16)):
        info = lym.LaunchInfo()
        args = (np.array(dims, np.int32).ctypes.data, parity, prec, nrhs, 0, 0, 0, 0, ctypes.byref(info))
        assert call(*args, None, 0) == 0
        visits = np.zeros((2, info.nbpp), np.int32)
        assert call(*args, visits.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), visits.size) == 0
        want = np.zeros_like(visits)
        want[[0, 1] if parity < 0 else [parity]] = 1 if prec else nrhs
        assert np.array_equal(visits, want), (dims, parity, prec, nrhs)
        assert info.spb * info.nbpp >= int(np.prod(dims)) // 2
        if info.form == lym.FORM_LANES:
            assert info.spb == 64  # what k_dslash_lanes covers, a wave
