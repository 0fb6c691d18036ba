"""The eight-wave kernel of small batches: every form it is dispatched in against the K-split decode kernel (identical bits)
and the oracle."""
import numpy as np
import pytest

import tritium_amd as T
from helpers import f32_to_bf16_bits, same_bits, scales, ternary
from oracle_lib import FMT_TQ2_0

pytestmark = pytest.mark.gpu


def make(backend, rng, n, k, planes):
    ws = [ternary(rng, n, k, p0) for p0 in (0.4, 0.7, 0.85)[:planes]]
    scs = [scales(rng, n) for _ in ws]
    packed = [T.pack_rows(w, n, k) for w in ws]
    return packed, scs, backend.linear(packed, scs, n, k)


def forced(backend, run):
    backend.set_decode_kernel(1)
    try:
        run()
    finally:
        backend.set_decode_kernel(0)


# rows around the edges of the 32-row tiles, K blocks around the eight waves (1, 8, 9, 17 of them, a ragged last one), an
# odd and an even number of column tiles, a ragged last one
@pytest.mark.parametrize("m,n,k,planes", [(3, 17, 200, 1), (16, 40, 2048, 1), (31, 64, 2304, 1), (32, 33, 4352, 1), (33, 130, 2050, 1), (64, 48, 300, 1),
                                          (3, 33, 1500, 2), (32, 16, 2304, 2), (64, 50, 4100, 2), (9, 17, 700, 3), (32, 200, 2560, 3)])
def test_int8_contract(backend, oracle, m, n, k, planes):
    print("case waves a8", m, n, k, planes, flush=True)
    rng = np.random.default_rng(m * 7 + n + k + planes)
    packed, scs, layer = make(backend, rng, n, k, planes)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[m - 1, k // 2] = np.nan
    res = rng.standard_normal((m, n)).astype(np.float32)
    dact, dres, o, o2 = backend.to_device(act, "f32"), backend.to_device(res, "f32"), backend.empty(m * n, "f32"), backend.empty(m * n, "f32")
    backend.linear_a8(layer, dact, m, o)
    assert backend.last_kernel() == "waves", backend.last_kernel()
    got, want = o.to_host().reshape(m, n), oracle.cpu_linear_a8_planes(packed, FMT_TQ2_0, scs, act, m, n, k).reshape(m, n)
    assert same_bits(got[:-1], want[:-1]) and np.array_equal(got[-1], want[-1], equal_nan=True)  # (a NaN's own bits are the host's choice)
    forced(backend, lambda: backend.linear_a8(layer, dact, m, o2))
    assert same_bits(got, o2.to_host())
    backend.linear_a8_residual(layer, dact, m, dres, o)
    assert backend.last_kernel() == "waves", backend.last_kernel()
    forced(backend, lambda: backend.linear_a8_residual(layer, dact, m, dres, o2))
    assert same_bits(o.to_host(), o2.to_host())
    for a in (dact, dres, o, o2):
        a.free()
    layer.free()


@pytest.mark.parametrize("m,n,k,planes,dtype", [(2, 17, 2304, 1, "f32"), (8, 33, 700, 1, "bf16"), (9, 64, 2050, 1, "f32"), (16, 130, 4352, 2, "bf16"),
                                                (3, 40, 300, 2, "f32"), (8, 48, 2560, 3, "bf16")])
def test_float_contract(backend, m, n, k, planes, dtype):
    print("case waves float", m, n, k, planes, dtype, flush=True)
    rng = np.random.default_rng(m * 11 + n + k + planes)
    _, _, layer = make(backend, rng, n, k, planes)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[0, k // 3] = np.inf
    dact, o, o2 = backend.to_device(f32_to_bf16_bits(act) if dtype == "bf16" else act, dtype), backend.empty(m * n, dtype), backend.empty(m * n, dtype)
    backend.linear_float(layer, dact, m, o)
    assert backend.last_kernel() == "waves", backend.last_kernel()
    forced(backend, lambda: backend.linear_float(layer, dact, m, o2))
    assert o.to_host().tobytes() == o2.to_host().tobytes()
    for a in (dact, o, o2):
        a.free()
    layer.free()


@pytest.mark.parametrize("mode,planes,ms", [(1, 1, (5, 5, 5)), (1, 2, (33, 40, 3)), (0, 1, (4, 8, 16)), (0, 3, (2, 3, 8))])
def test_groups(backend, mode, planes, ms):
    """Members of different widths and token counts in one launch, one of them a single tile; behind an RMSNorm under the int8
    contract."""
    rng = np.random.default_rng(77 + planes + mode)
    k = 1300
    shapes = [(70, k), (16, k), (161, 2304)]
    layers = [make(backend, rng, n, kk, planes)[2] for n, kk in shapes]
    acts = [backend.to_device(rng.standard_normal((m, kk)).astype(np.float32), "f32") for m, (_, kk) in zip(ms, shapes)]
    norms = [(backend.to_device(rng.uniform(0.5, 1.5, kk).astype(np.float32), "f32"), 1e-5, False) for _, kk in shapes]
    outs = []
    for force in (0, 1):
        backend.set_decode_kernel(force)
        try:
            o = [backend.empty(m * n, "f32") for m, (n, _) in zip(ms, shapes)]
            g = backend.group(list(zip(layers, acts, ms, o)), mode, "f32", "f32", **({"norms": norms} if mode == 1 else {}))
            for _ in range(2):
                g.launch()
                assert backend.last_kernel() == ("ksplit_decode" if force else "waves"), backend.last_kernel()
            outs.append([x.to_host() for x in o])
            g.destroy()
            for x in o:
                x.free()
        finally:
            backend.set_decode_kernel(0)
    for a, b in zip(*outs):
        assert same_bits(a, b)
    for a in acts + [n[0] for n in norms]:
        a.free()
    for layer in layers:
        layer.free()
