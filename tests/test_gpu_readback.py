"""What a viewer reads each frame (mesh, normals, wind map), with the staging the
context keeps: it serves calls of every size and order, and no call allocates
once the largest has run."""
import numpy as np
import pytest

from simplewinderosion_amd import Batch, World, capi

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


def _free():
    return torch.cuda.mem_get_info()[0]


def _views(w):
    return dict(normals=w.normals(), windmap=w.windmap(), mesh=w.mesh())


@pytest.mark.parametrize("nx,ny", [(1, 1), (3, 5), (113, 145), (512, 512)])
def test_views_in_any_order(nx, ny):
    print("case views", nx, ny, flush=True)
    rng = np.random.default_rng(nx)
    w = World(nx, ny)
    w.upload(rng.random((nx, ny)).astype(np.float32))
    w.upload_fields(momentum=rng.standard_normal((3, nx, ny)).astype(np.float32))
    first = _views(w)  # growing: 3, 4, 12 floats a cell
    mesh = first["mesh"]
    assert np.array_equal(mesh[..., 0], np.broadcast_to(np.arange(nx)[:, None], (nx, ny)))
    assert np.array_equal(mesh[..., 3:6], np.moveaxis(first["normals"], 0, -1))
    assert np.all(first["windmap"][..., 3] == 1.0)
    for _ in range(2):  # 12, 3, 4: what the larger left behind is not read
        again = dict(mesh=w.mesh(), normals=w.normals(), windmap=w.windmap())
        for k in first:
            assert np.array_equal(first[k], again[k]), k
    w.close()


def test_a_frame_keeps_its_staging():
    """A context holds the staging from the first frame to its end: the device
    memory that is free does not change between frames, and all of it is back
    after the context."""
    print("case views staging", flush=True)
    w = World(1024, 1024)
    w.upload(np.random.default_rng(1).random((1024, 1024)).astype(np.float32))
    w.windmap()
    before = _free()
    w.mesh()
    held = _free()
    assert before - held >= (12 - 4) * 4 << 20  # the mesh's staging stays
    for _ in range(3):
        _views(w)
        assert _free() == held
    w.close()
    assert _free() > held


def test_batch_views_of_several_sizes():
    print("case views batch", flush=True)
    sizes = [(40, 30), (7, 5), (128, 130)]
    b = Batch(sizes, periodic=True)
    hs = [np.random.default_rng(k).random(s).astype(np.float32) for k, s in enumerate(sizes)]
    for k, h in enumerate(hs):
        b.upload(k, h)
    for k in (1, 2, 0, 1):
        nx, ny = sizes[k]
        n = 3 * nx * ny
        got, want = np.empty(n, np.float32), np.empty(n, np.float32)
        fp = lambda a: a.ctypes.data_as(capi._FP)
        assert b.lib.swe_normals_terrain(b.ctx, k, fp(got)) == 0
        w = World(nx, ny, periodic=True)
        w.upload(hs[k])
        assert w.lib.swe_normals(w.ctx, fp(want)) == 0
        assert np.array_equal(got, want), k
        w.close()
    b.close()


def test_threads_read_one_context():
    """The staging is held by one call at a time: views read by several threads
    at once, growing it in between, are those read alone."""
    import threading

    print("case views threads", flush=True)
    w = World(96, 160)
    w.upload(np.random.default_rng(3).random((96, 160)).astype(np.float32))
    bad = []

    def read(names, want):
        for i in range(40):
            for nm in names:
                if not np.array_equal(getattr(w, nm)(), want[nm]):
                    bad.append((nm, i))

    ref = World(96, 160)
    ref.upload(np.random.default_rng(3).random((96, 160)).astype(np.float32))
    want = _views(ref)
    orders = (("windmap", "normals", "mesh"), ("normals", "mesh", "windmap"), ("mesh", "windmap", "normals"))
    ts = [threading.Thread(target=read, args=(o, want)) for o in orders]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad[:4]
    ref.close()
    w.close()
