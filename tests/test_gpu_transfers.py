"""Host transfers of fields: dense rows (one copy), padded rows and views (through the dense block on the
device), several pieces of the block, every element size, and several threads at once."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import parallelstencil as ps

pytestmark = pytest.mark.gpu
ps.init_parallel_stencil(ps.AMDGPU, ps.Float64, 3, module=__name__)
NP = {ps.Float64: np.float64, ps.Float32: np.float32, ps.BFloat16: np.uint16, ps.Bool: np.bool_, ps.Int32: np.int32}


def _host(shape, et, seed):
    return np.asfortranarray(np.random.default_rng(seed).integers(0, 2 if et == ps.Bool else 60000, size=shape).astype(NP[et]))


@pytest.mark.parametrize("shape,et", [((1,), ps.Float64), ((1000,), ps.Float32), ((1, 7), ps.Float64), ((32, 5), ps.Float64), ((33, 5, 4), ps.Float64),
                                      ((64, 64), ps.Float32), ((65, 1, 9), ps.Float32), ((127, 9, 3), ps.BFloat16), ((300, 11), ps.Bool),
                                      ((5, 70000), ps.Int32), ((301, 200, 101), ps.Float64), ((0, 4), ps.Float64)])
def test_round_trip(shape, et):
    h = _host(shape, et, 1)
    A = ps.zeros(*shape, eltype=et).copy_from(h)
    assert np.array_equal(A.to_host(), h)


@pytest.mark.parametrize("lo,hi", [((1, 1, 1), (33, 20, 9)), ((2, 3, 4), (31, 20, 9)), ((5, 7, 2), (5, 7, 8)), ((1, 4, 3), (33, 4, 3)), ((2, 1, 1), (2, 20, 9))])
def test_views_touch_only_their_box(lo, hi):
    h = _host((33, 20, 9), ps.Float64, 2)
    A = ps.zeros(33, 20, 9, eltype=ps.Float64).copy_from(h)
    box = tuple(slice(a - 1, b) for a, b in zip(lo, hi))
    v = A.view(lo, hi)
    assert np.array_equal(v.to_host(), h[box])
    new = _host(v.shape, ps.Float64, 3)
    v.copy_from(new)
    h[box] = new
    assert np.array_equal(A.to_host(), h)


def test_threads_transfer_at_once():
    hs = [_host((100 + i, 50, 40), ps.Float64, i) for i in range(6)]
    fields = [ps.zeros(*h.shape, eltype=ps.Float64) for h in hs]

    def work(i):
        st = ps.get_stream(1 + i % 3)
        for _ in range(4):
            fields[i].copy_from(hs[i], st)
            if not np.array_equal(fields[i].to_host(st), hs[i]):
                return False
        return True

    with ThreadPoolExecutor(6) as pool:  # result() raises what a worker raised
        assert [f.result() for f in [pool.submit(work, i) for i in range(6)]] == [True] * 6


@pytest.mark.parametrize("shape,et", [((1,), ps.Float64), ((1001,), ps.Float32), ((33, 3), ps.Float64), ((1025, 70, 1), ps.Float32), ((130, 9, 7), ps.BFloat16),
                                      ((65, 1, 9), ps.Bool), ((2, 70000), ps.Float64), ((1, 9, 7001), ps.Float32), ((7, 3, 9000), ps.Float64),
                                      ((17, 5, 4099), ps.BFloat16), ((5, 3), ps.Bool), ((1030, 2), ps.Float64), ((3, 70000, 2), ps.Int32)])
def test_device_copies(shape, et):
    h = _host(shape, et, 4)
    A, B = ps.zeros(*shape, eltype=et).copy_from(h), ps.zeros(*shape, eltype=et)
    B.copy_(A)
    assert np.array_equal(B.to_host(), h)


@pytest.mark.parametrize("lo,hi", [((2, 1, 1), (33, 20, 9)), ((5, 3, 2), (30, 19, 8)), ((3, 4, 5), (3, 20, 5)), ((1, 1, 1), (1, 20, 9)),
                                   ((32, 1, 1), (33, 20, 9)), ((2, 5, 2), (9, 5, 8)), ((4, 2, 3), (4, 2, 3))])
def test_device_copies_of_views(lo, hi):
    # rows that start off a 16-byte boundary, and elements beside the view that must stay
    ha, hb = _host((33, 20, 9), ps.Float64, 5), _host((40, 21, 9), ps.Float64, 6)
    A, B = ps.zeros(33, 20, 9, eltype=ps.Float64).copy_from(ha), ps.zeros(40, 21, 9, eltype=ps.Float64).copy_from(hb)
    box = tuple(slice(a - 1, b) for a, b in zip(lo, hi))
    B.view(lo, hi).copy_(A.view(lo, hi))
    hb[box] = ha[box]
    assert np.array_equal(B.to_host(), hb) and np.array_equal(A.to_host(), ha)
