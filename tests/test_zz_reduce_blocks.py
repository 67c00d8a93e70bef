"""The divergence check's reduction where its rule changes: as many blocks as
there are partial slots, each with its own, and one tile more, where blocks share
the slots by atomics.  Exact maxima, so equal to the host's bit for bit; every
second call's field is smaller, so a slot the call before left filled would
show."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,shapes", [
    (np.float64, ((128, 128, 64), (128, 128, 65), (192, 192, 60), (128, 128, 64))),
    (np.float32, ((128, 128, 128), (128, 128, 129), (192, 192, 100), (128, 128, 128))),
])
def test_shared_and_own_slots(gpu_lib, dtype, shapes):
    import torch
    f = gpu_lib.melt_divgck_noalloc
    f.restype = C.c_int
    rng = np.random.default_rng(3)
    box = 2.0
    for n1, n2, n3 in shapes:
        u = [rng.standard_normal((n3, n2, n1), dtype=np.float32).astype(dtype) for _ in range(3)]
        h = (n1 / box, n2 / box, n3 / box)
        q = torch.full((1,), -1.0, dtype=torch.float64, device="cuda")
        print(f"# divgck_noalloc {n1}x{n2}x{n3} {np.dtype(dtype).name}", flush=True)
        for scale in (1.0, 0.5, 0.25):
            x, y, z = ((a * dtype(scale)).astype(dtype) for a in u)
            dev = [torch.from_numpy(a).cuda() for a in (x, y, z)]
            rc = f(*(C.c_void_p(t.data_ptr()) for t in dev), n1, n2, n3, C.c_double(box), C.c_double(box), C.c_double(box),
                   x.itemsize, C.c_void_p(torch.cuda.current_stream().cuda_stream), C.c_void_p(q.data_ptr()))
            assert rc == 0
            x, y, z = (a.astype(np.float64) for a in (x, y, z))
            want = np.abs((np.roll(x, -1, 2) - x) * h[0] + (np.roll(y, -1, 1) - y) * h[1] + (np.roll(z, -1, 0) - z) * h[2]).max()
            assert q.item() == want, (n1, n2, n3, scale)
