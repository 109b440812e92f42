"""Host threads that share a stream: the launches of one call, which hand data to each other through the stream's workspace, are
not mixed with another thread's."""

import sys
import threading
from _ctypes import FUNCFLAG_PYTHONAPI

import pytest
import torch

from flash_model_architectures_amd import _native, ops
from flash_model_architectures_amd.functional.routing import route_tokens


def test_native_calls_hold_the_interpreter_lock():
    lib = _native.load()
    for name in _native.PROTOTYPES:
        assert getattr(lib, name)._flags_ & FUNCFLAG_PYTHONAPI, name


def _split_gemm(dtype, sizes, n, k, seed):
    """A grouped product whose last tiles are cut along the reduction; small integers, exact in any order."""

    g = torch.Generator("cuda").manual_seed(seed)
    ends = torch.tensor(sizes).cumsum(0).tolist()
    offsets = torch.tensor([0] + ends, dtype=torch.int32, device="cuda")
    a = torch.randint(-2, 3, (ends[-1], k), generator=g, device="cuda").to(dtype)
    w = torch.randint(-1, 2, (len(sizes), n, k), generator=g, device="cuda").to(dtype)
    index = torch.arange(ends[-1], dtype=torch.int32, device="cuda")
    want = torch.cat([(a[e - s : e].double() @ w[i].double().T) for i, (s, e) in enumerate(zip(sizes, ends))]).to(dtype)

    def run():
        out = torch.full_like(want, float("nan"))
        ops.scatter2scatter(a, w.permute(0, 2, 1), index, index, out, 1, True, True, offsets)
        return out

    return run, want


def _sort(seed):
    """A counting sort of several launches."""

    ids = torch.randint(0, 300, (50000,), generator=torch.Generator("cuda").manual_seed(seed), device="cuda")
    return (lambda: route_tokens(ids, 300).sorted_scattered_idxs), torch.sort(ids, stable=True).indices.int()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp32", "bf16", "sort"])
def test_two_threads_on_one_stream(kind):
    if kind == "fp32":  # 3 and 8 parts
        work = [_split_gemm(torch.float32, [1024, 1, 2050, 1100], 2040, k, k) for k in (2004, 4100)]
    elif kind == "bf16":  # 2 and 4 parts
        work = [_split_gemm(torch.bfloat16, [200, 70, 130, 40, 10], 136, k, k) for k in (4160, 8320)]
    else:
        work = [_sort(seed) for seed in (0, 1)]
    results, errors = [[], []], []
    start = threading.Barrier(2)

    def loop(i):
        try:
            start.wait(60)
            for _ in range(30):
                results[i].append(work[i][0]())
        except BaseException as e:  # noqa: BLE001 (handed to the main thread)
            errors.append(e)

    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=loop, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not errors
    for got, (_, want) in zip(results, work):
        assert len(got) == 30 and all(torch.equal(y, want) for y in got)
