"""What the C-ABI asks of the HIP runtime, and in which order, without a GPU:
plans that calls on any stream read are complete before they are used or the
call that builds them returns, nothing that a capturing stream forbids is
asked of one, and a failed allocation leaves nothing behind. Each case runs in
a process of its own with tests/cpp/hip_recorder.cpp in front of the runtime:
kernels are recorded, not run."""
import ctypes
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SRC = os.path.join(HERE, "cpp", "hip_recorder.cpp")
LIB = os.path.join(HERE, "cpp", "_build", "libhip_recorder.so")
A, B = 0x10, 0x20  # stream handles: the recorder only tells them apart
PTR = 0x1000       # stands for a caller's device array; no kernel runs
PLANS = ("k_query2_vv_local", "k_query2_vf_local", "k_ring_plan", "k_closed_fans")  # kernels that write plans


class Recorder:
    """A mesh on the recorder's device and its log."""

    def __init__(self, fv, patch_size=64):
        sys.path.insert(0, ROOT)
        sys.modules["torch"] = None  # the wrapper starts torch's own HIP runtime where it finds torch
        import rxmesh_amd as rx
        self.rec = ctypes.CDLL(LIB)
        self.rec.rec_log.restype = ctypes.c_char_p
        self.rec.rec_live_bytes.restype = self.rec.rec_live_count.restype = ctypes.c_size_t
        self.host = rx.Mesh(fv, patch_size=patch_size, host_only=True)  # the build itself runs on the host
        self.mesh = rx.Mesh(None, parts=[self.host])
        self.h, self.lib, self.log = self.mesh._h, rx.lib(), []
        self.events()

    def events(self):
        """(what, kernel or "", stream) since the last call."""
        out = []
        for line in self.rec.rec_log().decode().splitlines():
            what, _, rest = line.partition(" ")
            name, _, stream = rest.rpartition("@")
            out.append((what, name.strip(), int(stream) if stream.isdigit() else rest))
        return out

    def __call__(self, name, *args):
        return getattr(self.lib, name)(self.h, *args)

    def smooth(self, iters, stream):
        return self("rxm_laplacian_smooth", PTR, 2 * PTR, 3 * PTR, 0.5, iters, stream)


def check_plans_waited_for(events):
    """Every plan kernel is followed by a wait for its stream before any kernel
    that does not build plans, and before the end."""
    pending = {}
    for what, name, stream in events:
        if what == "launch" and any(p in name for p in PLANS):
            pending[stream] = name
        elif what == "wait":
            pending.pop(stream, None)
        elif what == "launch" and "k_fill" not in name and "k_reset" not in name:
            assert not pending, "%s launched while %s may still run" % (name, pending)
    assert not pending, "returned while %s may still run" % pending


def sphere():
    sys.path.insert(0, ROOT)
    from rxmesh_amd import meshgen as mg
    return mg.icosphere(3, seed=0)[1]


def case_ring_plan():
    """rxm_vv_plan_build, and the smoothing that builds its own ring plan."""
    r = Recorder(sphere())
    assert r("rxm_vv_plan_build", A) == 0
    e = r.events()
    assert any("k_ring_plan" in n for _, n, _ in e)
    check_plans_waited_for(e)
    assert r.smooth(4, B) == 0
    assert [n for w, n, _ in r.events() if w == "launch" and "k_smoothk" not in n] == []
    r = Recorder(sphere())
    assert r("rxm_set_launch_threads", 8, 4) == 0
    assert r.smooth(4, A) == 0
    e = r.events()
    assert any("k_ring_plan" in n for _, n, _ in e) and any("k_smoothk" in n for _, n, _ in e)
    check_plans_waited_for(e)


def case_face_plan():
    """Each entry point that builds the face plan on its first call."""
    for name, args in (("rxm_vertex_normals", (0, PTR, 2 * PTR)), ("rxm_gaussian_curvature", (PTR, 2 * PTR, 3 * PTR)),
                       ("rxm_symdir3_grad", (PTR, 2 * PTR, 3 * PTR)),
                       ("rxm_symdir3_grad_step", (PTR, 2 * PTR, 0.1, 3 * PTR)),
                       ("rxm_smooth_symdir_steps", (PTR, 2 * PTR, 3 * PTR, 0.5, 0.1, 1))):
        r = Recorder(sphere())
        assert r(name, *args, A) == 0
        e = r.events()
        assert any("k_query2_vf_local" in n for _, n, _ in e)
        check_plans_waited_for(e)
        assert r(name, *args, B) == 0
        assert not any(p in n for _, n, _ in r.events() for p in PLANS)


def first_calls():
    """name -> calls of which each builds plans or work arrays on first use."""
    cg = (PTR,) * 7 + (3, 0.0, 0.0, None, None, None)
    return {
        "plan": [("rxm_vv_plan_build",)],
        "smooth": [("rxm_laplacian_smooth", PTR, 2 * PTR, 3 * PTR, 0.5, 4)],
        "smooth, four steps a launch": [("rxm_set_launch_threads", 8, 4),
                                        ("rxm_laplacian_smooth", PTR, 2 * PTR, 3 * PTR, 0.5, 4)],
        "smooth, two steps a launch": [("rxm_set_launch_threads", 4, 1),
                                       ("rxm_laplacian_smooth", PTR, 2 * PTR, 3 * PTR, 0.5, 5)],
        "normals": [("rxm_vertex_normals", 0, PTR, 2 * PTR)],
        "gradient step": [("rxm_symdir3_grad_step", PTR, 2 * PTR, 0.1, 3 * PTR)],
        "rotations": [("rxm_arap_rotations", PTR, 2 * PTR, 3 * PTR, 4 * PTR)],
        "energy": [("rxm_arap_energy_grad", PTR, PTR, PTR, PTR, 2 * PTR, 3 * PTR)],
        "assembly": [("rxm_cot_csr_assemble", PTR, 0.1, 2 * PTR, 3 * PTR, 4 * PTR, 5 * PTR)],
        "cg": [("rxm_mcf_implicit_cg", *cg[:5], 6 * PTR, *cg[7:])],
        "matrix-free cg": [("rxm_mcf_matfree_cg", PTR, PTR, 2 * PTR, 0.1, 0, 0, 3, 0.0, 0.0, None, None, None)],
        "query": [("rxm_query_vv_vf", PTR, 2 * PTR, 3 * PTR, 4 * PTR)],
    }


def last_call(r, calls, stream):
    for c in calls[:-1]:
        assert r(*c) == 0
    r.events()
    return r(*calls[-1], stream)


def case_failed_allocation():
    """Any one allocation of a first call fails: the call says so (or, where
    the plan is an option, does without), leaves no array of the unfinished
    plan behind and no error for the next call, which builds it whole."""
    for what, calls in first_calls().items():
        r = Recorder(sphere())
        assert last_call(r, calls, A) == 0, what
        whole, n = r.rec.rec_live_bytes(), 0
        while True:
            n += 1
            r = Recorder(sphere())
            before = r.rec.rec_live_bytes()
            r.rec.rec_fail_malloc(n)
            rc = last_call(r, calls, A)
            r.rec.rec_fail_malloc(0)
            if rc == 0 and r.rec.rec_live_bytes() == whole:
                break  # fewer than n allocations: none failed
            assert rc in (0, 7), (what, n, rc)
            check_plans_waited_for(r.events())
            kept = r.rec.rec_live_bytes() - before
            assert last_call(r, calls, A) == 0, (what, n, "the call after a failed allocation")
            assert r.rec.rec_live_bytes() == whole, (what, n, kept, r.rec.rec_live_bytes(), whole)
        assert n > 1, what


def case_failed_wait():
    """A plan whose build could not be waited for is not published: the call
    fails, and the next one builds the plan anew."""
    for name, kernel, args in (("rxm_arap_rotations", "k_query2_vv_local", (PTR, 2 * PTR, 3 * PTR, 4 * PTR)),
                               ("rxm_vertex_normals", "k_query2_vf_local", (0, PTR, 2 * PTR))):
        r = Recorder(sphere())
        before = r.rec.rec_live_count()
        r.rec.rec_fail_wait(1)
        assert r(name, *args, A) == 5
        assert r.rec.rec_live_count() == before
        r.rec.rec_fail_wait(0)
        r.rec.hipGetLastError()  # a caller that goes on after such an error has read it
        r.events()
        assert r(name, *args, A) == 0
        assert any(kernel in n for _, n, _ in r.events())


def case_capture():
    """Once a smoothing has built the VV plan, rxm_vv_plan_build and smoothing
    ask nothing of a capturing stream that it forbids; the multi-step plan is
    made by the first call outside."""
    r = Recorder(sphere())
    assert r.smooth(1, A) == 0
    r.events()
    r.rec.rec_capturing(1)
    assert r("rxm_vv_plan_build", A) == 0
    assert r.smooth(4, A) == 0
    e = r.events()
    assert not [x for x in e if x[0] == "illegal"], e
    assert sum("k_smooth_local" in n for _, n, _ in e) == 4
    r.rec.rec_capturing(0)
    assert r("rxm_vv_plan_build", A) == 0
    check_plans_waited_for(r.events())
    r.rec.rec_capturing(1)
    assert r.smooth(4, A) == 0
    e = r.events()
    assert [w for w, _, _ in e] == ["launch"] and "k_smoothk" in e[0][1], e


def case_automatic_smoothing():
    """Tuning the gradient step loop leaves the steps per launch of the
    smoothing alone, and knobs 0 and 8 have a value that means the automatic
    choice."""
    r = Recorder(sphere(), patch_size=1024)
    from rxmesh_amd import autotune
    assert r("rxm_vv_plan_build", A) == 0

    def kernels():
        r.events()
        assert r.smooth(4, A) == 0
        return [n for _, n, _ in r.events()]
    default = kernels()
    assert len(default) == 1 and "k_smoothkILj1024" in default[0]
    autotune.apply(r.mesh, {"smooth_threads": 256, "grad_threads": 256, "grad_queue": 0})
    tuned = kernels()
    assert len(tuned) == 1 and "k_smoothkILj256" in tuned[0], tuned
    for cfg in autotune.smooth_configs():
        autotune.apply(r.mesh, cfg)
        assert (kernels() == default) == (cfg["smooth_steps"] == -1), cfg
    assert r("rxm_set_launch_threads", 8, 0) == 0 and len(kernels()) == 4
    assert r("rxm_set_launch_threads", 0, 0) == 0 and r("rxm_set_launch_threads", 8, -1) == 0
    assert kernels() == default
    for knob, value in ((0, -1), (0, 1), (0, 1024), (8, -2), (8, 7)):
        assert r("rxm_set_launch_threads", knob, value) == 1


def case_one_plan_for_every_steps():
    """Walking the steps per launch upwards (as the tuner does) makes one plan
    that holds them all, beside the automatic one where that was made."""
    for planned in (0, 1):
        r = Recorder(sphere())
        if planned:
            assert r("rxm_vv_plan_build", A) == 0
        assert r.smooth(1, A) == 0
        sizes = []
        r.events()
        for steps in (2, 3, 4, 5, 6, 1, 6):
            assert r("rxm_set_launch_threads", 8, steps) == 0
            assert r.smooth(12, A) == 0
            sizes.append(r.rec.rec_live_bytes())
        assert sum("k_ring_plan" in n for _, n, _ in r.events()) == 2  # its two passes
        assert sizes[-1] == sizes[4] and (planned or len(set(sizes)) == 1)


def case_names():
    return [n[5:] for n in globals() if n.startswith("case_") and n != "case_names"]


@pytest.mark.parametrize("case", case_names())
def test_host_calls(case):
    if not os.path.exists(LIB) or os.path.getmtime(LIB) < os.path.getmtime(SRC):
        os.makedirs(os.path.dirname(LIB), exist_ok=True)
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", SRC, "-o", LIB + ".tmp"])
        os.replace(LIB + ".tmp", LIB)
    q = subprocess.run([sys.executable, os.path.abspath(__file__), case], env=dict(os.environ, LD_PRELOAD=LIB),
                       capture_output=True, text=True, timeout=120)
    assert q.returncode == 0, q.stdout + q.stderr


if __name__ == "__main__":
    globals()["case_" + sys.argv[1]]()
