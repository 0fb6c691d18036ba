"""Block-scale additive planes (SALT) through the device-resident C ABI.

The host definition (dequantize the row, planes in order; then one f32 accumulator over k:
crates/tritium-format/src/salt.rs:720-738, crates/tritium-nn/src/layers/packed_salt.rs:585-628) is the
oracle. The reference-order kernel must reproduce it bit for bit; the matrix-core form is held to the
bound the reference sets for its own GPU kernel, 1e-4 (crates/tritium-cuda/kernels/tq2_0_add.cu:651-655)."""
import ctypes as C

import numpy as np
import pytest

import tritium_amd as T
from helpers import accepts, bf16_bits_to_f32, f32_to_bf16_bits, rel_err, same_bits, ternary
from test_oracle_salt import f16_bits

pytestmark = pytest.mark.gpu

SALT_REL = 1e-4  # tq2_0_add.cu:651-655


def make_planes(backend, oracle, rng, n, k, t_planes):
    nb = (k + 255) // 256
    packed, bufs = [], []
    for p in range(t_planes):
        trits = ternary(rng, n, k, (0.4, 0.7, 0.85, 0.85)[p])
        sc = f16_bits(rng.uniform(0.02, 1.0, (n, nb)) * (0.5 ** p))
        packed.append(oracle.pack_matrix_scaled(trits, sc, n, k))
        bufs.append(backend.upload_weights_scaled(packed[-1], T.GemmShape(0, n, k)))
    return packed, bufs


@pytest.mark.parametrize("m,n,k,t_planes", [(1, 48, 256, 1), (3, 33, 700, 2), (5, 130, 1000, 3), (17, 20, 300, 4)])
def test_reference_order_kernel_is_bit_exact(backend, oracle, m, n, k, t_planes):
    print("case salt-seq", m, n, k, t_planes, flush=True)
    rng = np.random.default_rng(m * 13 + n + k)
    packed, bufs = make_planes(backend, oracle, rng, n, k, t_planes)
    act = rng.standard_normal((m, k)).astype(np.float32)
    rc, want = oracle.salt_mpgemm(packed, n, k, act, m)
    dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, "f32")
    backend.linear_salt(bufs, dact, m, dout, seq=True)
    assert rc == 0 and same_bits(dout.to_host(), want)
    for a in [dact, dout] + bufs:
        a.free()


@pytest.mark.parametrize("t_planes", [1, 2, 3, 4])
@pytest.mark.parametrize("m,n,k", [(1, 48, 256), (2, 130, 700), (4, 64, 2048), (5, 33, 1000), (8, 257, 2560), (16, 96, 2048)])
def test_matrix_core_form_within_the_reference_bound(backend, oracle, m, n, k, t_planes):
    print("case salt-flow", m, n, k, t_planes, flush=True)
    rng = np.random.default_rng(m * 17 + n + k + t_planes)
    packed, bufs = make_planes(backend, oracle, rng, n, k, t_planes)
    bits = f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32) * 2)
    act = bf16_bits_to_f32(bits).reshape(m, k)
    rc, want = oracle.salt_mpgemm(packed, n, k, act, m)
    for dtype, dev in (("bf16", bits), ("f32", act)):
        dact, dout = backend.to_device(dev, dtype), backend.empty(m * n, "f32")
        backend.linear_salt(bufs, dact, m, dout)
        got = dout.to_host().reshape(m, n)
        assert rc == 0 and accepts(got, want, rel=SALT_REL, floor=1.0).all()
        assert rel_err(got, want) < 2e-5  # what it actually achieves: the f32 fold's own rounding
        dact.free()
        dout.free()
    for b in bufs:
        b.free()


def test_tokens_with_nan_or_inf_take_the_host_order(backend, oracle):
    rng = np.random.default_rng(40)
    m, n, k = 4, 40, 600
    packed, bufs = make_planes(backend, oracle, rng, n, k, 2)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[1, 7] = np.nan
    act[2, 300] = np.inf
    rc, want = oracle.salt_mpgemm(packed, n, k, act, m)
    dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, "f32")
    backend.linear_salt(bufs, dact, m, dout)
    got = dout.to_host().reshape(m, n)
    assert same_bits(got[1], want[1]) and same_bits(got[2], want[2])
    assert accepts(got[[0, 3]], want[[0, 3]], rel=SALT_REL, floor=1.0).all()
    for a in [dact, dout] + bufs:
        a.free()


@pytest.mark.parametrize("m,n,k", [(40, 72, 768), (9, 40, 5000)])
def test_passes_where_the_workspace_cannot_grow(oracle, m, n, k):
    """A context whose workspace has the size of a few tokens, under stream capture: the call may not allocate there and runs in
    passes of as many tokens as the flow form takes (16, 16, 8; 7, 2). The bits of the call in one launch, on every replay."""
    print("case salt-passes", m, n, k, flush=True)
    backend = T.Mi355xBackend(0)
    hip = C.CDLL("libamdhip64.so.7")
    stream = C.c_void_p(backend.stream_handle())
    rng = np.random.default_rng(m + n + k)
    packed, bufs = make_planes(backend, oracle, rng, n, k, 2)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[m - 1, 3] = np.nan
    few = min(16, 163840 // ((k + 255) // 256 * 1040))
    dact, dout, dfew = backend.to_device(act, "f32"), backend.empty(m * n, "f32"), backend.empty(16 * n, "f32")
    for count in (few, m % few):
        backend.linear_salt(bufs, dact, count, dfew)
    graph, gexec, nodes = C.c_void_p(), C.c_void_p(), C.c_size_t(0)
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    try:
        backend.linear_salt(bufs, dact, m, dout)
    finally:
        rc = hip.hipStreamEndCapture(stream, C.byref(graph))
    assert rc == 0 and hip.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0
    assert nodes.value == 2 * ((m + few - 1) // few)  # a digit split and a flow launch per pass
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0
    got = []
    for _ in range(3):
        dout.copy_from(np.zeros(m * n, np.float32))
        backend.linear_salt(bufs, dact, few, dfew)
        assert hip.hipGraphLaunch(gexec, stream) == 0
        backend.sync()
        got.append(dout.to_host())
    assert hip.hipGraphExecDestroy(gexec) == 0 and hip.hipGraphDestroy(graph) == 0
    backend.linear_salt(bufs, dact, m, dout)  # eager: the workspace grows, one launch
    want = dout.to_host()
    assert all(same_bits(x, want) for x in got)
    rc, host = oracle.salt_mpgemm(packed, n, k, act, m)
    assert accepts(want.reshape(m, n)[:-1], host[:-1], rel=SALT_REL, floor=1.0).all() and np.isnan(want.reshape(m, n)[-1]).any()
    for a in [dact, dout, dfew] + bufs:
        a.free()
    backend.close()


def test_more_than_16_tokens_run_in_slices(backend, oracle):
    """40 tokens are one launch: three slices of 16 operand tokens (64 rows), the last one of 8 tokens."""
    rng = np.random.default_rng(41)
    m, n, k = 40, 72, 768
    packed, bufs = make_planes(backend, oracle, rng, n, k, 2)
    act = rng.standard_normal((m, k)).astype(np.float32)
    rc, want = oracle.salt_mpgemm(packed, n, k, act, m)
    for dtype in ("f32", "bf16"):
        dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, dtype)
        backend.linear_salt(bufs, dact, m, dout)
        got = dout.to_host().reshape(m, n)
        if dtype == "bf16":
            got = bf16_bits_to_f32(got).reshape(m, n)
            assert accepts(got, want, rel=4e-3, floor=1.0).all()  # bf16 output: 8 bits
        else:
            assert accepts(got, want, rel=SALT_REL, floor=1.0).all() and rel_err(got, want) < 2e-5
        dact.free()
        dout.free()
    for b in bufs:
        b.free()


def test_rows_too_long_for_lds_fall_back(backend, oracle):
    """K = 10240 needs 164 KiB for the rows of 16 tokens: the launch takes the reference-order kernel."""
    rng = np.random.default_rng(43)
    m, n, k = 2, 20, 10240
    packed, bufs = make_planes(backend, oracle, rng, n, k, 1)
    act = rng.standard_normal((m, k)).astype(np.float32)
    rc, want = oracle.salt_mpgemm(packed, n, k, act, m)
    dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, "f32")
    backend.linear_salt(bufs, dact, m, dout)
    got = dout.to_host().reshape(m, n)
    assert accepts(got, want, rel=SALT_REL, floor=1.0).all()
    for a in [dact, dout] + bufs:
        a.free()


def test_scaled_upload_still_serves_the_plain_contract(backend, oracle):
    """mpgemm ignores block scales (crates/tritium-cpu/src/lib.rs:302-345), also on a buffer that kept them;
    and a buffer without them is refused by the block-scale entry point."""
    rng = np.random.default_rng(42)
    m, n, k = 2, 20, 512
    packed, bufs = make_planes(backend, oracle, rng, n, k, 1)
    act = rng.standard_normal((m, k)).astype(np.float32)
    sc = rng.uniform(0.01, 0.1, n).astype(np.float32)
    out = np.zeros((m, n), np.float32)
    backend.mpgemm(T.MpGemm(act, bufs[0], sc, T.GemmShape(m, n, k), T.TernaryFormat.Tq2_0, out))
    from oracle_lib import FMT_TQ2_0
    rc, want = oracle.cpu_mpgemm(packed[0], FMT_TQ2_0, act, sc, m, n, k)
    assert rc == 0 and same_bits(out, want)
    plain = backend.upload_weights(packed[0], T.GemmShape(0, n, k), T.TernaryFormat.Tq2_0)
    dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, "f32")
    with pytest.raises(T.InvalidInput):
        backend.linear_salt([plain], dact, m, dout)
    for a in [dact, dout, plain] + bufs:
        a.free()


def test_every_f16_block_scale_reaches_the_kernels_exactly(backend, oracle):
    """One row per f16 bit pattern, one non-zero trit against an activation of 1: the output is the
    block scale itself, so the device's f16 -> f32 conversion is checked over all 65,536 patterns
    (subnormals, zeros, infinities, NaNs) through both kernels."""
    n, k = 65536, 256
    trits = np.zeros((n, k), np.int8)
    trits[:, 0] = 1
    bits = np.arange(n, dtype=np.uint16).reshape(n, 1)
    packed = oracle.pack_matrix_scaled(trits, bits, n, k)
    buf = backend.upload_weights_scaled(packed, T.GemmShape(0, n, k))
    act = np.zeros((1, k), np.float32)
    act[0, 0] = 1.0
    rc, want = oracle.salt_mpgemm([packed], n, k, act, 1)
    want = want.reshape(-1)
    scale = bits.reshape(-1).view(np.float16).astype(np.float32)
    finite = np.isfinite(scale)
    scale[0x8000] = 0.0  # 0.0 + (-0.0) * 1 is +0.0: the one pattern whose row is not the scale's own bits
    assert rc == 0 and (want[finite].view(np.uint32) == scale[finite].view(np.uint32)).all()
    assert np.isnan(want[~finite]).all()  # an infinite scale times a zero trit is NaN, on the host too
    dact, dout = backend.to_device(act, "f32"), backend.empty(n, "f32")
    backend.linear_salt([buf], dact, 1, dout, seq=True)
    got = dout.to_host()
    assert np.isnan(got[~finite]).all() and (got[finite].view(np.uint32) == want[finite].view(np.uint32)).all()
    # the matrix-core form multiplies the block's integer sum by the scale once: the same values for
    # every finite scale (an infinite or NaN scale gives Inf or NaN there, the host NaN)
    backend.linear_salt([buf], dact, 1, dout)
    got = dout.to_host()
    assert (got[finite].view(np.uint32) == want[finite].view(np.uint32)).all()
    assert (~np.isfinite(got[~finite])).all()
    for a in (dact, dout, buf):
        a.free()


@pytest.mark.parametrize("m,n,k,t_planes,dtype", [(17, 130, 256, 1, "f32"), (33, 33, 700, 2, "f32"), (64, 257, 2560, 3, "bf16"), (65, 15, 1000, 4, "f32"),
                                                  (130, 96, 2048, 2, "bf16"), (1027, 40, 300, 1, "f32"),
                                                  (512, 4100, 300, 1, "f32"),  # the 64-column waves
                                                  (9, 70, 5000, 2, "f32")])    # seven such tokens fit the flow form (of K = 2560 fifteen)
def test_many_tokens_have_the_bits_of_sixteen_at_a_time(backend, oracle, m, n, k, t_planes, dtype):
    """The many-token form adds the same exact block values in the same order as the flow form: identical bits, rows past the
    last row tile, columns past the last pair, a token holding NaN and a second pass of tokens included."""
    print("case salt-many", m, n, k, t_planes, dtype, flush=True)
    rng = np.random.default_rng(m * 19 + n + k + t_planes)
    packed, bufs = make_planes(backend, oracle, rng, n, k, t_planes)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[m // 2, k // 3] = np.nan
    host = f32_to_bf16_bits(act) if dtype == "bf16" else act
    dout = backend.empty(m * n, dtype)
    many = backend.to_device(host, dtype)
    backend.linear_salt(bufs, many, m, dout)
    got = dout.to_host().reshape(m, n)
    want = np.empty_like(got)
    rows = np.asarray(host).reshape(m, k)
    step = min(16, 163840 // ((k + 255) // 256 * 1040))  # tokens that the flow form holds in LDS
    for m0 in range(0, m, step):
        part = rows[m0:m0 + step]
        dact, dpart = backend.to_device(part, dtype), backend.empty(len(part) * n, dtype)
        backend.linear_salt(bufs, dact, len(part), dpart)
        want[m0:m0 + step] = dpart.to_host().reshape(-1, n)
        dact.free()
        dpart.free()
    assert same_bits(got, want) if dtype == "f32" else (got == want).all()
    for a in [many, dout] + bufs:
        a.free()


@pytest.mark.parametrize("m,n,k,t_planes", [(17, 300, 2560, 1), (16, 200, 5000, 2), (9, 130, 8192, 3), (1030, 40, 2600, 1)])
def test_long_rows_are_no_less_exact_than_the_host_order(backend, m, n, k, t_planes):
    """Calls whose rows do not fit the flow form stand in for the host's order, f32 sums over k: their error against float64
    may not be larger, in any token and in the outputs that miss a token's largest element either (its weights there are
    zero, so the values are small next to the element that sets the token's grid)."""
    print("case salt-exactness", m, n, k, t_planes, flush=True)
    rng = np.random.default_rng(m + n + k + t_planes)
    nb = (k + 255) // 256
    w64, bufs = np.zeros((n, k)), []
    for p in range(t_planes):
        trits = ternary(rng, n, k, (0.4, 0.7, 0.85)[p])
        trits[: n // 2, 5] = 0
        bits = f16_bits(rng.uniform(0.02, 1.0, (n, nb)) * (0.5 ** p))
        packed = T.pack_rows(trits, n, k).reshape(n, nb, 66).copy()
        packed[:, :, 64:] = bits.reshape(n, nb, 1).view(np.uint8)
        bufs.append(backend.upload_weights_scaled(packed.reshape(-1), T.GemmShape(0, n, k)))
        w64 += trits * np.repeat(bits.view(np.float16).astype(np.float64), 256, 1)[:, :k]
    dout = backend.empty(m * n, "f32")
    for name in ("normal", "log-normal", "outlier 2^6", "outlier 2^11", "outlier 2^13", "outlier 2^16", "outlier 2^20"):
        act = rng.standard_normal((m, k))
        if name == "log-normal":
            act = np.sign(act) * np.exp(2 * rng.standard_normal((m, k)))
        elif name != "normal":
            act[:, 5] *= 2.0 ** int(name[10:])
        act = act.astype(np.float32)
        want = act.astype(np.float64) @ w64.T
        dact = backend.to_device(act, "f32")
        errors = []
        for seq in (False, True):
            backend.linear_salt(bufs, dact, m, dout, seq=seq)
            d = dout.to_host().reshape(m, n) - want
            miss = slice(0, n // 2)
            errors.append((np.linalg.norm(d) / np.linalg.norm(want), np.linalg.norm(d[:, miss]) / np.linalg.norm(want[:, miss])))
        assert errors[0][0] <= errors[1][0] and errors[0][1] <= errors[1][1], (name, errors)
        dact.free()
    for a in [dout] + bufs:
        a.free()


@pytest.mark.parametrize("m,n,k,t_planes,dtype", [(21, 70, 2501, 1, "f32"), (9, 33, 5003, 2, "bf16"), (130, 40, 2307, 4, "f32"), (17, 600, 2560, 3, "bf16"),
                                                  (1024, 1030, 2560, 1, "f32")])  # (the 64-column waves)
def test_flagged_tokens_of_the_many_token_form_have_the_bits_of_the_host_order(backend, m, n, k, t_planes, dtype):
    """Tokens with one element 2^40 times the others, beside ordinary ones, up to all of a launch: the reference-order kernel's bits."""
    print("case salt-flagged", m, n, k, t_planes, dtype, flush=True)
    rng = np.random.default_rng(m + n + k + t_planes)
    nb = (k + 255) // 256
    bufs = []
    for p in range(t_planes):
        packed = T.pack_rows(ternary(rng, n, k, (0.4, 0.7, 0.85, 0.85)[p]), n, k).reshape(n, nb, 66).copy()
        packed[:, :, 64:] = f16_bits(rng.uniform(0.02, 1.0, (n, nb)) * (0.5 ** p)).reshape(n, nb, 1).view(np.uint8)
        bufs.append(backend.upload_weights_scaled(packed.reshape(-1), T.GemmShape(0, n, k)))
    dout = backend.empty(m * n, "f32")
    plain = rng.standard_normal((m, k)).astype(np.float32)
    for tokens in ([m // 2], [0, 5, m - 1], list(range(m))):
        act = plain.copy()
        act[tokens, k - 1] = np.float32(2.0 ** 40)
        dact = backend.to_device(f32_to_bf16_bits(act) if dtype == "bf16" else act, dtype)
        results = []
        for seq in (False, True):
            backend.linear_salt(bufs, dact, m, dout, seq=seq)
            results.append(dout.to_host().reshape(m, n))
        assert same_bits(results[0][tokens], results[1][tokens])
        assert accepts(results[0], results[1], rel=SALT_REL, floor=1.0).all()
        dact.free()
    for a in [dout] + bufs:
        a.free()


def test_flagged_tokens_cost_no_more_than_the_host_order(backend):
    """A call of long rows whose tokens are all flagged is not slower than the reference-order kernel, which such calls took
    before the many-token form (measured: 0.45 of it; one dot after the other in a lane it was 7.6 times)."""
    import time
    rng = np.random.default_rng(9)
    m, n, k = 16, 2560, 2560
    packed = T.pack_rows(ternary(rng, n, k), n, k).reshape(n, 10, 66).copy()
    packed[:, :, 64:] = f16_bits(rng.uniform(0.02, 1.0, (n, 10))).reshape(n, 10, 1).view(np.uint8)
    buf = backend.upload_weights_scaled(packed.reshape(-1), T.GemmShape(0, n, k))
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[:, 7] = np.nan
    dact, dout = backend.to_device(act, "f32"), backend.empty(m * n, "f32")
    best = {}
    for seq in (False, True):
        for _ in range(4):
            backend.sync()
            t0 = time.perf_counter()
            for _ in range(3):
                backend.linear_salt([buf], dact, m, dout, seq=seq)
            backend.sync()
            best[seq] = min(best.get(seq, 1e9), time.perf_counter() - t0)
    print("salt flagged / host order", {s: round(v * 1e6 / 3, 1) for s, v in best.items()}, "us", flush=True)
    assert best[False] <= 1.2 * best[True], best
    for a in (dact, dout, buf):
        a.free()
