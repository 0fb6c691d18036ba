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


# both sides of the lines of the dispatch rule: the kernel that the eight waves replace, short and long rows, within a round of
# workgroups and beyond one
@pytest.mark.parametrize("m,n,k,planes,kernel", [
    (18, 17024, 256, 1, "gemm64"), (32, 16400, 256, 1, "gemm64"), (18, 16384, 256, 1, "waves"), (24, 16900, 2560, 1, "waves"),   # prefill kernel
    (40, 16400, 512, 1, "gemm64"), (48, 16384, 300, 1, "waves"),
    (4, 16400, 300, 1, "waves"), (12, 16400, 300, 1, "ksplit_decode"), (12, 16400, 2200, 1, "waves"),                             # K-split kernel
    (3, 8208, 8192, 1, "ksplit_decode"), (4, 8208, 8192, 1, "waves"),
    (4, 10560, 2816, 3, "flow"), (8, 1280, 2048, 3, "waves"), (8, 1280, 1792, 3, "flow"), (4, 2560, 1024, 2, "flow"),             # flow kernel
    (24, 16384, 512, 3, "flow"), (24, 16384, 768, 3, "waves")])
def test_both_sides_of_the_dispatch_rule(backend, m, n, k, planes, kernel):
    print("case waves rule", m, n, k, planes, kernel, flush=True)
    rng = np.random.default_rng(m + n + k + planes)
    packed = [T.pack_rows(rng.integers(-1, 2, (n, k), dtype=np.int8), n, k) for _ in range(planes)]
    layer = backend.linear(packed, [scales(rng, n) for _ in packed], n, k)
    dact = backend.to_device(f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32)), "bf16")
    o, o2 = backend.empty(m * n, "bf16"), backend.empty(m * n, "bf16")
    backend.linear_a8(layer, dact, m, o)
    assert backend.last_kernel() == kernel, backend.last_kernel()
    forced(backend, lambda: backend.linear_a8(layer, dact, m, o2))
    assert o.to_host().tobytes() == o2.to_host().tobytes()
    for a in (dact, o, o2):
        a.free()
    layer.free()


@pytest.mark.parametrize("m,shapes,planes,kernel", [
    (16, [(6912, 6912)] * 6, 1, "waves"),               # rows within LDS, several workgroups of the K-split kernel per CU
    (16, [(130, 10496), (70, 2304)], 2, "waves"),       # one member's rows beyond LDS
    (16, [(48, 10496)] * 3, 3, "waves"),
    (8, [(8448, 512)] * 2, 2, "flow"), (40, [(8448, 512)] * 2, 1, "gemm64")])
def test_both_sides_of_the_dispatch_rule_in_groups(backend, m, shapes, planes, kernel):
    print("case waves rule group", m, shapes, planes, kernel, flush=True)
    rng = np.random.default_rng(m + len(shapes) + planes)
    made, acts, members = {}, {}, []
    for n, k in shapes:
        if (n, k) not in made:
            packed = [T.pack_rows(rng.integers(-1, 2, (n, k), dtype=np.int8), n, k) for _ in range(planes)]
            made[(n, k)] = backend.linear(packed, [scales(rng, n) for _ in packed], n, k)
        if k not in acts:
            acts[k] = backend.to_device(rng.standard_normal((m, k)).astype(np.float32), "f32")
    results = []
    for force in (0, 1):
        outs = [backend.empty(m * n, "f32") for n, _ in shapes]
        backend.set_decode_kernel(force)
        try:
            g = backend.group([(made[s], acts[s[1]], m, o) for s, o in zip(shapes, outs)], 1, "f32", "f32")
        finally:
            backend.set_decode_kernel(0)
        g.launch()
        assert backend.last_kernel() == ("ksplit_decode" if force else kernel), backend.last_kernel()
        results.append([o.to_host() for o in outs])
        g.destroy()
        for o in outs:
            o.free()
    for a, b in zip(*results):
        assert same_bits(a, b)
    for x in list(acts.values()) + list(made.values()):
        x.free()


def test_sparse_planes_leave_only_the_flow_kernel_its_calls(backend):
    """Planes with a zero-chunk map: the flow kernel, which skips their chunks, keeps what it was chosen for; the K-split and the
    prefill kernel do not read the map, and their calls go to the eight waves as any other's."""
    rng = np.random.default_rng(3)
    backend.set_zero_skip(2)
    try:
        for m, n, k, planes, kernel in ((16, 640, 2560, 1, "waves"), (32, 640, 2560, 1, "waves"), (8, 5120, 2560, 2, "flow")):
            packed = []
            for _ in range(planes):
                w = rng.integers(-1, 2, (n, k), dtype=np.int8)
                w[16:48] = 0  # whole chunks of zeros
                packed.append(T.pack_rows(w, n, k))
            layer = backend.linear(packed, [scales(rng, n) for _ in packed], n, k)
            dact, o, o2 = backend.to_device(rng.standard_normal((m, k)).astype(np.float32), "f32"), backend.empty(m * n, "f32"), backend.empty(m * n, "f32")
            backend.linear_a8(layer, dact, m, o)
            assert backend.last_kernel() == kernel, (m, n, k, backend.last_kernel())
            forced(backend, lambda: backend.linear_a8(layer, dact, m, o2))
            assert same_bits(o.to_host(), o2.to_host())
            for a in (dact, o, o2):
                a.free()
            layer.free()
    finally:
        backend.set_zero_skip(0)
