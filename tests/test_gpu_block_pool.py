"""GPU test of the reuse of device memory: buffers of very different lives
(solves, renewed operators, vectors destroyed while others live) give the same
results again and again, a vector's memory handed out anew starts at zero and
is not written by work queued before, also when the old owner's last work was
still running, and torch work on a vector's memory on another stream is
finished before that memory serves another vector; what is kept is bounded and
goes back to the device on request while other objects live."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_renewed_problems_repeat_bit_for_bit():
    print("case renewed problems", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    rng = np.random.default_rng(3)
    thetas = [rng.normal(size=16 ** 3) * 0.5 for _ in range(3)]
    first = {}
    d = U.DomainDiscretization(0, 4)
    b = U.Vector(d.num_dofs())
    for k in range(9):
        d.set_theta(thetas[k % 3])
        A = U.SparseMatrix()                    # the last one's memory is free again
        d.assemble_linear(A, b)
        S = U.CG(U.GeometricMultiGrid(d, precision="f32" if k % 2 else "f64"), reduction=1e-10)
        S.init(A)
        x = U.Vector(d.num_dofs())
        assert S.apply(x, b)
        got = (x.numpy(), A.download_csr()[2])
        key = (k % 3, k % 2)
        if key in first:
            assert all(np.array_equal(p, q) for p, q in zip(got, first[key]))
        first[key] = got


def test_new_vectors_are_zero_while_old_work_runs():
    print("case new vectors after queued work", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    n = 1 << 22
    keep = U.Vector(n)                          # the pool is not emptied
    for k in range(20):
        a = U.Vector(n)
        for _ in range(8):
            U.lib().ugx_vec_scale_add2_f64(n, a.device_ptr(), 1.0, a.device_ptr(), 1.0, keep.device_ptr(), None)
        a.set(float(k + 1))
        del a                                   # released behind the queued work
        v = U.Vector(n)
        assert not v.numpy().any()
        keep.set(float(k))


def test_work_on_another_stream_ends_before_reuse():
    print("case torch stream", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    import torch

    class Memory:
        def __init__(self, v):
            self.__cuda_array_interface__ = {"shape": (v.size(),), "typestr": "<f8", "data": (v.device_ptr(), False),
                                             "version": 2}
    n = 1 << 22
    keep = U.Vector(n)
    s = torch.cuda.Stream()
    for k in range(10):
        v = U.Vector(n)
        U.synchronize()
        with torch.cuda.stream(s):
            t = torch.as_tensor(Memory(v), device="cuda")
            for _ in range(30):
                t.add_(1.0)
        del t, v
        w = U.Vector(n)                         # the same size: most likely the same memory
        assert not w.numpy().any()
    assert keep.size() == n


def test_kept_memory_goes_back_on_request():
    print("case trim memory", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    import torch
    keep = U.Vector(1000)
    keep.set(2.0)
    n = 1 << 27                                 # 1 GiB
    U.trim_memory()
    v = U.Vector(n)
    U.synchronize()
    used = torch.cuda.mem_get_info()[0]
    del v
    assert torch.cuda.mem_get_info()[0] <= used + (n << 2)      # kept
    assert U.trim_memory() >= 8 * n
    # up to the chunks of a few MB that the runtime takes for itself in between
    assert torch.cuda.mem_get_info()[0] >= used + 8 * n - (32 << 20)
    assert U.trim_memory() == 0
    assert np.all(keep.numpy() == 2.0)
    w = U.Vector(n)                             # allocated anew, zero
    assert not w.numpy().any()


def test_the_number_of_kept_blocks_is_bounded():
    print("case block count", flush=True)
    sys.stdout.flush()
    import ugcore_amd as U
    keep = U.Vector(64)
    U.trim_memory()
    for _ in range(2):
        vs = [U.Vector(64) for _ in range(1500)]
        assert not any(v.numpy().any() for v in vs[::100])
        for k, v in enumerate(vs):
            v.set(float(k))
        del vs, v
    assert 0 < U.trim_memory() <= 512 * 512
    assert not keep.numpy().any()
