"""The further state sets a context takes by itself: given back by
hg_set_fused(0) and by a batch in the separate form, and taken back when other
contexts need their memory, between steps and while another thread steps, with
the state bit for bit as in a context that never had them."""
import ctypes as C
import threading

import numpy as np
import pytest

import bench
from hormone_amd import driver as D
from hormone_amd import native
from hormone_amd import problems as P
from hormone_amd.batch import Batch
from hormone_amd.grid import cartesian_grid
from hormone_amd.native import Hydro

pytestmark = pytest.mark.gpu

N = (256, 128, 128)
FIELD = 8 * N[0] * N[1] * N[2]
SETS = 19 * FIELD          # U 9 and W 5 of the second set, W 5 of the third
MARGIN = 256 << 20         # the runtime's own: queues, scratch


def free():
    """Bytes free on the device (the HIP runtime the library itself runs on)."""
    hip, a, b = native.lib(), C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


@pytest.fixture(scope="module")
def flow():
    prm = P.Params(n=N, mag_on=True, rktype=3, bc=(0,) * 12, courant=0.3, t_end=1e30,
                   dt_out=1e30, is_test=False)
    g = cartesian_grid(N, prm.lo, prm.hi)
    r = np.random.default_rng(3)

    def noise(a):
        return a * r.uniform(-1.0, 1.0, g.shape)
    st = P.State(d=1.0 + noise(0.2), p=1.0 + noise(0.2), v=[noise(0.3) for _ in range(3)],
                 b=[noise(0.3) for _ in range(3)], phi=np.zeros(g.shape))
    return prm, g, st


def create(flow):
    prm, g, st = flow
    return Hydro(**D.desc_fields(prm, g))


def load(eng, flow):
    D.load_initial_state(eng, *flow)
    return eng


def form(eng, n, fused):
    """Whether the context is in this form, by the bytes of its RK launch."""
    cells, dim = n[0] * n[1] * n[2], sum(m > 1 for m in n)
    want = bench.kernel_bytes(fused, eng.ufnmax(), 10, dim, True, 3, fused and cells > 1 << 19)[1]
    return eng.profile_read(native.PROF_RK)[2] == pytest.approx(want * cells)


def run(eng, t, tn, steps):
    return eng.run_loop(t, tn, 1e30, 1e30, 1e30, 2, 2, 1 << 40, 1 << 40, steps, 0.5)[:2]


def fields(eng, flow):
    return D.fetch(eng, flow[1], D.SNAP_FIELDS_MAG + (D.F_EINT,) +
                   tuple(D.F_U + q for q in range(9)))


def same(a, b):
    for f in b:
        assert np.array_equal(a[f].view(np.uint64), b[f].view(np.uint64)), f


@pytest.fixture(scope="module")
def separate(hiplib, flow):
    """Memory of a context without further sets, and its state after 3 and 5 steps."""
    # what the process keeps: code, and the queues' scratch memory for both forms
    engs = [load(create(flow), flow) for _ in range(5)]
    for eng in engs:
        run(eng, 0.0, 0, 1)
        eng.set_fused(0)
        run(eng, 0.0, 0, 1)
    for eng in engs:
        eng.close()
    f0 = free()
    eng = create(flow)
    eng.set_fused(0)
    need = f0 - free()
    load(eng, flow)
    t, tn = run(eng, 0.0, 0, 3)
    three = fields(eng, flow)
    end = run(eng, t, tn, 2)
    five = fields(eng, flow)
    eng.close()
    return need, three, five, (t, tn), end


@pytest.mark.parametrize("fused", [None, 2, 1])
def test_gpu_set_fused_off_gives_the_sets_back(hiplib, flow, separate, fused):
    print(f"case sets given back fused={fused}", flush=True)
    need, three, five, mid, end = separate
    eng = create(flow)
    if fused:
        eng.set_fused(fused)
    load(eng, flow)
    assert run(eng, 0.0, 0, 3) == mid
    f0 = free()
    eng.set_fused(0)
    assert free() - f0 >= 0.9 * SETS
    same(fields(eng, flow), three)
    assert run(eng, *mid, 2) == end
    same(fields(eng, flow), five)
    f0 = free()
    eng.set_fused(2)  # and takes them again
    assert f0 - free() >= 0.9 * SETS
    same(fields(eng, flow), five)
    eng.close()


@pytest.mark.parametrize("when", ["before", "after"])
def test_gpu_separate_batch_gives_the_sets_back(hiplib, flow, separate, when):
    need = separate[0]
    print(f"case sets of a separate batch, chosen {when} adding", flush=True)
    out = []
    for own in (True, False):
        f0 = free()
        eng = create(flow)
        if not own:
            eng.set_fused(0)
        load(eng, flow)
        run(eng, 0.0, 0, 3)  # the state is in a further set now
        b = Batch()
        if when == "before":
            b.set_fused(False)
        b.add(eng, t_end=1e30, t_out=1e30, dt_out=1e30)
        b.set_fused(False)
        b.step(3)
        assert f0 - free() <= need + 0.1 * SETS
        b.remove(eng)
        b.close()
        assert form(eng, N, own * 2)  # and takes its own form again
        out.append(fields(eng, flow))
        eng.close()
    same(out[0], out[1])


@pytest.mark.parametrize("n,fused", [((256, 256, 1), 2), ((1024, 1, 1), 2), (N, 0)])
def test_gpu_sets_of_small_boxes_fit_where_large_ones_do_not(hiplib, flow, separate, n, fused):
    """With 4 GiB left: the form a box starts with, by the bytes of its launches."""
    hip, fill = native.lib(), C.c_void_p()
    assert hip.hipMalloc(C.byref(fill), C.c_size_t(free() - (4 << 30))) == 0
    try:
        print(f"case form of {n} with 4 GiB left", flush=True)
        prm = P.Params(n=n, mag_on=True, bc=(0,) * 12, is_test=False)
        eng = Hydro(**D.desc_fields(prm, cartesian_grid(n, prm.lo, prm.hi)))
        assert form(eng, n, fused)
        eng.close()
    finally:
        assert hip.hipFree(fill) == 0


def test_gpu_sets_are_taken_back_before_memory_is_full(hiplib, flow, separate):
    """An allocation that fits, but leaves the runtime next to nothing."""
    need, three, five, mid, end = separate
    hip, fill = native.lib(), C.c_void_p()
    engs = [load(create(flow), flow)]
    try:
        assert run(engs[0], 0.0, 0, 3) == mid
        assert hip.hipMalloc(C.byref(fill), C.c_size_t(free() - need - (64 << 20))) == 0
        print("case a context that leaves 64 MiB", flush=True)
        engs.append(load(create(flow), flow))
        assert free() >= 0.9 * SETS
        assert run(engs[1], 0.0, 0, 3) == mid
        for eng in engs:
            same(fields(eng, flow), three)
            assert run(eng, *mid, 2) == end
            same(fields(eng, flow), five)
    finally:
        for eng in engs:
            eng.close()
        assert hip.hipFree(fill) == 0


@pytest.mark.parametrize("busy", [False, True], ids=["idle", "stepping"])
def test_gpu_contexts_that_fit_without_the_sets_fit(hiplib, flow, separate, busy):
    """Two contexts with further sets, then memory for three more once one of
    them has lost its own."""
    need, three, five, mid, end = separate
    hip, fill = native.lib(), C.c_void_p()
    f0 = free()
    engs, after = [load(create(flow), flow) for _ in range(2)], {}
    assert f0 - free() >= 2 * (need + 0.9 * SETS)
    try:
        for eng in engs:
            assert run(eng, 0.0, 0, 3) == mid
        room = 3 * need + MARGIN - SETS
        assert hip.hipMalloc(C.byref(fill), C.c_size_t(free() - room)) == 0
        first = engs[0]

        def stepping():
            t, tn = mid
            for _ in range(60):
                t, tn = run(first, t, tn, 1)
            after["end"], after["fields"] = (t, tn), fields(first, flow)
        th = threading.Thread(target=stepping)
        if busy:
            th.start()
        for q in range(3):
            print(f"case context {q + 3} of {need >> 20} MiB, busy={busy}", flush=True)
            engs.append(load(create(flow), flow))
            assert run(engs[-1], 0.0, 0, 3) == mid
        if busy:
            th.join()
        for eng in engs[busy:]:
            same(fields(eng, flow), three)
            assert run(eng, *mid, 2) == end
            same(fields(eng, flow), five)
    finally:
        for eng in engs:
            eng.close()
        assert hip.hipFree(fill) == 0
    if busy:
        eng = create(flow)
        eng.set_fused(0)
        load(eng, flow)
        assert run(eng, 0.0, 0, mid[1] + 60) == after["end"]
        same(after["fields"], fields(eng, flow))
        eng.close()
