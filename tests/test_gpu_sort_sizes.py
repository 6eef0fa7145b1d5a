"""The launcher layer's cell sort where its kernels change: one block up to 8,192 pairs, two kernels
a digit to 1,048,576 (256 tiles of 4,096), four beyond; one to four digits of the cell count, one
digit copied back by the bounds kernel. Hashes, indices and cell bounds are numpy's stable sort's,
exactly. The time of a large sort grows with its size: 16 million pairs against 4 million (4 times
the pairs) take at most 6 times as long, which allows half as much again for the caches and is far
from the square's 16."""
import numpy as np
import pytest

from test_gpu_launchers import call, dev, host, ptr

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def check(n, ncell, keys):
    index = np.random.default_rng(n).permutation(n).astype(np.uint32)
    d = [dev(a) for a in (keys, index, np.zeros(ncell, np.uint32), np.zeros(ncell, np.uint32), np.zeros(n, np.uint32))]
    call("xdem_reserve_workspace", n)
    call("xdem_cu_reorderDataAndFindCellStart", *(ptr(t) for t in d), n, ncell)
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    sk = keys[order]
    first = np.nonzero(np.r_[True, sk[1:] != sk[:-1]])[0]
    cs, ce = np.full(ncell, 0xFFFFFFFF, np.uint32), np.zeros(ncell, np.uint32)
    cs[sk[first]] = first
    ce[sk[first]] = np.r_[first[1:], n]
    for t, want in zip(d, (sk, index[order], cs, ce, index[order])):
        assert np.array_equal(host(t, np.uint32), want)


@pytest.mark.parametrize("ncell", [1, 200, 256, 257, 1 << 15, (1 << 24) + 1])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 40001, (1 << 20) + 1])
def test_sort_at_the_edges_of_its_kernels(n, ncell):
    print(f"[sort sizes] n={n} ncell={ncell}", flush=True)
    rng = np.random.default_rng(n + ncell)
    keys = np.where(rng.random(n) < 0.5, rng.integers(0, min(64, ncell), n), rng.integers(0, ncell, n)).astype(np.uint32)
    check(n, ncell, keys)


@pytest.mark.parametrize("n,ncell,spread", [(1 << 20, 128**3, "all"), (5000011, 128**3, "all"), (5000011, 1 << 16, "last"),
                                            (4 * 131072 * 8 + 4097, 1 << 24, "ramp")])
def test_large_sort(n, ncell, spread):
    """Keys over all cells, in the last cell only, and falling with the index."""
    print(f"[sort sizes] large n={n} ncell={ncell} {spread}", flush=True)
    if spread == "all":
        keys = np.random.default_rng(n).integers(0, ncell, n)
    else:
        keys = np.full(n, ncell - 1) if spread == "last" else (ncell - 1) - np.arange(n) % ncell
    check(n, ncell, keys.astype(np.uint32))


def test_time_grows_with_the_size():
    ncell, ms = 1 << 24, {}
    call("xdem_reserve_workspace", 16000000)
    for n in (4000000, 16000000):
        key0 = torch.randint(0, ncell, (n,), device="cuda", dtype=torch.int32)
        key, idx, out = key0.clone(), torch.arange(n, device="cuda", dtype=torch.int32), torch.empty_like(key0)
        cs, ce = (torch.empty(ncell, device="cuda", dtype=torch.int32) for _ in range(2))
        for _ in range(6):
            key.copy_(key0)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            call("xdem_cu_reorderDataAndFindCellStart", *(ptr(t) for t in (key, idx, cs, ce, out)), n, ncell)
            b.record()
            torch.cuda.synchronize()
            ms.setdefault(n, []).append(a.elapsed_time(b))
    print(f"[sort sizes] ms {ms}", flush=True)
    assert min(ms[16000000]) <= 6.0 * min(ms[4000000])
