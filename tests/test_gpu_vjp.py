"""TernaryBackend::mpgemm_projected_vjp through the C ABI: the reference's own cases
(crates/tritium-cpu/src/lib.rs:496-700, crates/tritium-cuda/src/cuda/tests.rs:724-800), bit for bit
against the CPU oracle's scalar path (the reference's bar between backends is 1e-4 relative)."""
import numpy as np
import pytest

import tritium_amd as T
from helpers import same_bits, ternary
from oracle_lib import FMT_TQ1_0, FMT_TQ2_0

pytestmark = pytest.mark.gpu


def _vjp(backend, packed, fmt, act, scales, gy, m, n, k, bias=True):
    buf = backend.upload_weights(packed, T.GemmShape(m, n, k), T.TernaryFormat(fmt))
    ga = np.full((m, k), np.nan, np.float32)
    gw = np.full((n, k), np.nan, np.float32)
    gb = np.full(n, np.nan, np.float32) if bias else None
    backend.mpgemm_projected_vjp(T.MpGemmProjectedVjp(
        act=np.asarray(act, np.float32), weights=buf, scales=np.asarray(scales, np.float32),
        grad_output=np.asarray(gy, np.float32), shape=T.GemmShape(m, n, k), format=T.TernaryFormat(fmt),
        grad_act=ga, grad_projected_weight=gw, grad_bias=gb))
    return ga, gw, gb


def test_reference_known_answer(backend, oracle):
    """crates/tritium-cpu/src/lib.rs:500-533."""
    packed = oracle.pack_matrix(np.array([[1, 0, -1], [-1, 1, 1]], np.int8), 2, 3, FMT_TQ2_0)
    ga, gw, gb = _vjp(backend, packed, FMT_TQ2_0, [1.0, 2.0, 3.0, -1.0, 4.0, 0.5], [2.0, 0.5], [3.0, -2.0, 4.0, 1.0], 2, 2, 3)
    assert ga.reshape(-1).tolist() == [7.0, -1.0, -7.0, 7.5, 0.5, -7.5]
    assert gw.reshape(-1).tolist() == [-1.0, 22.0, 11.0, -3.0, 0.0, -5.5]
    assert gb.tolist() == [7.0, -1.0]


@pytest.mark.parametrize("fmt", [FMT_TQ2_0, FMT_TQ1_0])
@pytest.mark.parametrize("m,n,k", [(2, 3, 5), (7, 4, 257), (1, 33, 64), (2, 3, 257), (17, 35, 576), (33, 130, 1100),
                                   (70, 16, 256), (16, 64, 1024)])
def test_bits_of_the_cpu_scalar_path(backend, oracle, fmt, m, n, k):
    """The first three shapes are the reference's device test (tests.rs:734), the fourth its
    packed-decode test (lib.rs:536), (17, 35, 576) its training shape (tests.rs:818-820); the rest
    cross every tile edge of the kernels (16 tokens, 16 / 64 rows, 64 / 256 / 1024 columns)."""
    print("case vjp", fmt, m, n, k, flush=True)
    rng = np.random.default_rng(m * 1000 + n * 10 + k)
    w = ternary(rng, n, k)
    packed = oracle.pack_matrix(w, n, k, fmt)
    act = rng.uniform(-2, 2, (m, k)).astype(np.float32)
    sc = rng.uniform(0.05, 1.5, n).astype(np.float32)
    sc[0] = -sc[0]
    gy = rng.uniform(-1, 1, (m, n)).astype(np.float32)
    rc, ga_w, gw_w, gb_w = oracle.cpu_projected_vjp(packed, fmt, act, sc, gy, m, n, k)
    assert rc == 0
    ga, gw, gb = _vjp(backend, packed, fmt, act, sc, gy, m, n, k)
    assert same_bits(ga, ga_w) and same_bits(gw, gw_w) and same_bits(gb, gb_w)
    ga, gw, gb = _vjp(backend, packed, fmt, act, sc, gy, m, n, k, bias=False)
    assert same_bits(ga, ga_w) and same_bits(gw, gw_w) and gb is None


@pytest.mark.parametrize("m,n,k", [(9, 40, 2), (5, 3, 9), (6, 515, 1030), (3, 1100, 1001), (5, 3301, 2560), (290, 70, 3900), (1030, 67, 3300)])
def test_every_tile_of_the_gradient_kernels(backend, oracle, m, n, k):
    """One shape per tile size that the launch picks (rows of weights x columns per lane: 1 x 1, 4 x 1, 8 x 2, 8 x 4; token
    tiles per wave of grad_act: 1, 2, 4), each with ragged edges. Sums and products in the CPU's order: bits."""
    print("case vjp tiles", m, n, k, flush=True)
    rng = np.random.default_rng(m + n + k)
    packed = oracle.pack_matrix(ternary(rng, n, k), n, k, FMT_TQ2_0)
    act = rng.standard_normal((m, k)).astype(np.float32)
    sc = rng.uniform(0.05, 1.5, n).astype(np.float32)
    gy = (rng.standard_normal((m, n)) * 10.0 ** rng.integers(-6, 3, (m, n))).astype(np.float32)
    gy[0, :] *= np.float32(1e-38)  # products that are denormal
    rc, ga_w, gw_w, gb_w = oracle.cpu_projected_vjp(packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    ga, gw, gb = _vjp(backend, packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    assert rc == 0 and same_bits(ga, ga_w) and same_bits(gw, gw_w) and same_bits(gb, gb_w)


def test_product_that_overflows_under_a_zero_trit(backend, oracle):
    """upstream * scale beyond the largest float: the CPU multiplies the scale with the trit first, so a zero trit still
    contributes 0 and only the columns with a non-zero trit become infinite."""
    rng = np.random.default_rng(21)
    m, n, k = 37, 100, 700
    packed = oracle.pack_matrix(ternary(rng, n, k), n, k, FMT_TQ2_0)
    act = rng.standard_normal((m, k)).astype(np.float32)
    sc = rng.uniform(0.05, 1.5, n).astype(np.float32)
    sc[50] = np.float32(1e30)
    gy = rng.standard_normal((m, n)).astype(np.float32)
    gy[17, 50] = np.float32(-1e20)
    rc, ga_w, gw_w, gb_w = oracle.cpu_projected_vjp(packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    ga, gw, gb = _vjp(backend, packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    assert rc == 0 and np.isinf(ga_w[17]).any() and np.isfinite(ga_w[17]).any()
    assert same_bits(ga, ga_w) and same_bits(gw, gw_w) and same_bits(gb, gb_w)


def test_non_finite_values_follow_the_host(backend, oracle):
    """Inf upstream times a zero trit is NaN on the host (upstream * (0 * scale)); so it is here."""
    rng = np.random.default_rng(12)
    m, n, k = 3, 20, 300
    w = ternary(rng, n, k)
    packed = oracle.pack_matrix(w, n, k, FMT_TQ2_0)
    act = rng.standard_normal((m, k)).astype(np.float32)
    act[1, 7] = np.nan
    sc = rng.uniform(0.1, 1, n).astype(np.float32)
    sc[3] = np.inf
    gy = rng.standard_normal((m, n)).astype(np.float32)
    gy[0, 5] = np.inf
    gy[2, 9] = -np.inf
    rc, ga_w, gw_w, gb_w = oracle.cpu_projected_vjp(packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    ga, gw, gb = _vjp(backend, packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    for got, want in ((ga, ga_w), (gw, gw_w), (gb, gb_w)):
        nan = np.isnan(want)
        assert (np.isnan(got) == nan).all() and same_bits(got[~nan], want[~nan])


@pytest.mark.parametrize("m,n,k", [(37, 100, 700), (290, 70, 3900), (1030, 67, 3300)])
def test_sums_that_leave_the_finite_range(backend, oracle, m, n, k):
    """Every token-tile size of grad_act (1, 2 and 4 tiles of 16 per wave): infinities and NaN upstream, sums that overflow on
    the way and meet the other infinity, products of finite factors that overflow under zero and non-zero trits, all beside
    tokens that stay finite."""
    print("case vjp range", m, n, k, flush=True)
    rng = np.random.default_rng(m + 7 * n + k)
    packed = oracle.pack_matrix(ternary(rng, n, k), n, k, FMT_TQ2_0)
    act = rng.standard_normal((m, k)).astype(np.float32)
    sc = rng.uniform(0.05, 1.5, n).astype(np.float32)
    sc[50], sc[3], sc[4], sc[61] = np.float32(1e30), 1.0, 1.0, 1.0
    base = rng.standard_normal((m, n)).astype(np.float32)
    base[:, 50] *= np.float32(1e-25)  # (so that only the planted products overflow)
    big = np.float32(2.5e38)
    for rows in ((), (1, 2), (1, 2, m - 1), tuple(range(m))):
        gy = base.copy()
        for i, row in enumerate(rows):
            if i % 3 == 0:
                gy[row, 5], gy[row, 40] = np.inf, (np.nan if row % 2 else 1.0)
            elif i % 3 == 1:
                gy[row, [3, 4, 61]] = big, big, -big
            else:
                gy[row, 50] = np.float32(-1e20)
        rc, ga_w, gw_w, gb_w = oracle.cpu_projected_vjp(packed, FMT_TQ2_0, act, sc, gy, m, n, k)
        assert rc == 0 and np.isfinite(ga_w).all() == (not rows)
        ga, gw, gb = _vjp(backend, packed, FMT_TQ2_0, act, sc, gy, m, n, k)
        for got, want in ((ga, ga_w), (gw, gw_w), (gb, gb_w)):
            nan = np.isnan(want)
            assert (np.isnan(got) == nan).all() and same_bits(got[~nan], want[~nan]), len(rows)


def test_non_finite_upstream_costs_no_more_than_the_unfused_sums(backend, oracle):
    """A step of loss scaling that overflows is an ordinary step. Multiply and add per term on the vector ALU took ten times
    the matrix form at this size, whatever the values: no call may take longer than that, whichever tokens hold an
    infinity, a NaN or an overflowing product (measured: 1.1, 1.2 and 3.6 times the finite call)."""
    import time
    rng = np.random.default_rng(5)
    m, n, k = 512, 2560, 2560
    packed = T.pack_rows(ternary(rng, n, k), n, k)
    buf = backend.upload_weights(packed, T.GemmShape(0, n, k), T.TernaryFormat.Tq2_0)
    sc = rng.uniform(0.05, 1.5, n).astype(np.float32)
    sc[50] = np.float32(1e30)
    gy = rng.standard_normal((m, n)).astype(np.float32)
    gy[:, 50] *= np.float32(1e-25)
    one, nan, over = gy.copy(), gy.copy(), gy.copy()
    one[m // 2, 7] = np.inf
    nan[:, 7] = np.nan
    over[:, 50] = np.float32(1e20)
    dact, dsc, ga = backend.to_device(np.ones((m, k), np.float32), "f32"), backend.to_device(sc, "f32"), backend.empty(m * k, "f32")
    times = {}
    for name, up in (("finite", gy), ("one", one), ("nan", nan), ("over", over)):
        dup = backend.to_device(up, "f32")
        best = 1e9
        for _ in range(4):
            backend.sync()
            t0 = time.perf_counter()
            for _ in range(5):
                backend.projected_vjp(buf, dsc, dact, dup, m, ga, None, None)
            backend.sync()
            best = min(best, time.perf_counter() - t0)
        times[name] = best
        dup.free()
    print("vjp times", {key: round(v * 2e5, 1) for key, v in times.items()}, "us", flush=True)
    assert max(times.values()) <= 10 * times["finite"], times
    for a in (dact, dsc, ga, buf):
        a.free()


def test_device_resident_form_equals_the_host_form(backend, oracle):
    rng = np.random.default_rng(13)
    m, n, k = 40, 100, 700
    packed = oracle.pack_matrix(ternary(rng, n, k), n, k, FMT_TQ2_0)
    act = rng.standard_normal((m, k)).astype(np.float32)
    sc = rng.uniform(0.1, 1, n).astype(np.float32)
    gy = rng.standard_normal((m, n)).astype(np.float32)
    ga_w, gw_w, gb_w = _vjp(backend, packed, FMT_TQ2_0, act, sc, gy, m, n, k)
    buf = backend.upload_weights(packed, T.GemmShape(0, n, k), T.TernaryFormat(FMT_TQ2_0))
    d = [backend.to_device(x, "f32") for x in (sc, act, gy)]
    o = [backend.empty(c, "f32") for c in (m * k, n * k, n)]
    backend.projected_vjp(buf, d[0], d[1], d[2], m, o[0], o[1], o[2])
    backend.sync()
    assert same_bits(o[0].to_host(), ga_w) and same_bits(o[1].to_host(), gw_w) and same_bits(o[2].to_host(), gb_w)
    for a in d + o:
        a.free()


def test_reserved_code_is_refused_before_any_write(backend, oracle):
    """lib.rs:600-638."""
    for corrupt in (0, 1):
        packed = oracle.pack_matrix(np.ones((1, 1), np.int8), 1, 1, FMT_TQ2_0).copy()
        packed[corrupt] |= 3
        buf = backend.upload_weights(packed, T.GemmShape(1, 1, 1), T.TernaryFormat.Tq2_0)
        ga, gw, gb = np.array([41.0], np.float32), np.array([42.0], np.float32), np.array([43.0], np.float32)
        with pytest.raises(T.Backend, match="unpack row 0: decoded value 2 outside ternary range"):
            backend.mpgemm_projected_vjp(T.MpGemmProjectedVjp(
                act=np.ones(1, np.float32), weights=buf, scales=np.ones(1, np.float32), grad_output=np.ones(1, np.float32),
                shape=T.GemmShape(1, 1, 1), format=T.TernaryFormat.Tq2_0, grad_act=ga, grad_projected_weight=gw, grad_bias=gb))
        assert (ga[0], gw[0], gb[0]) == (41.0, 42.0, 43.0)


def test_zero_dimensions(backend, oracle):
    """lib.rs:640-666 (k = 0: the bias is still summed); m = 0 and n = 0 zero-fill (kernel.rs:122-129)."""
    buf = backend.upload_weights(np.zeros(0, np.uint8), T.GemmShape(2, 3, 0), T.TernaryFormat.Tq2_0)
    gb = np.full(3, np.nan, np.float32)
    backend.mpgemm_projected_vjp(T.MpGemmProjectedVjp(
        act=np.zeros(0, np.float32), weights=buf, scales=np.array([1, 2, 3], np.float32),
        grad_output=np.array([1, 2, 3, 1, 2, 4], np.float32), shape=T.GemmShape(2, 3, 0), format=T.TernaryFormat.Tq2_0,
        grad_act=np.zeros(0, np.float32), grad_projected_weight=np.zeros(0, np.float32), grad_bias=gb))
    assert gb.tolist() == [2.0, 4.0, 7.0]
    n, k = 5, 40
    rng = np.random.default_rng(2)
    packed = oracle.pack_matrix(ternary(rng, n, k), n, k, FMT_TQ2_0)
    buf = backend.upload_weights(packed, T.GemmShape(0, n, k), T.TernaryFormat.Tq2_0)
    gw, gb = np.full((n, k), np.nan, np.float32), np.full(n, np.nan, np.float32)
    backend.mpgemm_projected_vjp(T.MpGemmProjectedVjp(
        act=np.zeros(0, np.float32), weights=buf, scales=np.ones(n, np.float32), grad_output=np.zeros(0, np.float32),
        shape=T.GemmShape(0, n, k), format=T.TernaryFormat.Tq2_0, grad_act=np.zeros(0, np.float32),
        grad_projected_weight=gw, grad_bias=gb))
    assert not gw.any() and not gb.any()


def test_length_and_identity_errors(backend, oracle):
    """lib.rs:668-700 and the order of kernel.rs:102-120; identity first (lib.rs:363)."""
    packed = oracle.pack_matrix(np.ones((1, 1), np.int8), 1, 1, FMT_TQ2_0)
    buf = backend.upload_weights(packed, T.GemmShape(1, 1, 1), T.TernaryFormat.Tq2_0)
    one = lambda: np.ones(1, np.float32)  # noqa: E731

    def call(**kw):
        args = dict(act=one(), weights=buf, scales=one(), grad_output=one(), shape=T.GemmShape(1, 1, 1),
                    format=T.TernaryFormat.Tq2_0, grad_act=one(), grad_projected_weight=one(), grad_bias=None)
        args.update(kw)
        backend.mpgemm_projected_vjp(T.MpGemmProjectedVjp(**args))

    with pytest.raises(T.ShapeMismatch) as e:
        call(grad_act=np.zeros(0, np.float32))
    assert (e.value.expected, e.value.got) == (1, 0)
    with pytest.raises(T.ShapeMismatch) as e:
        call(act=np.zeros(3, np.float32), grad_output=np.zeros(2, np.float32))  # act is checked first
    assert (e.value.expected, e.value.got) == (1, 3)
    with pytest.raises(T.ShapeMismatch) as e:
        call(grad_bias=np.zeros(2, np.float32))
    assert (e.value.expected, e.value.got) == (1, 2)
    with pytest.raises(T.InvalidInput):
        call(shape=T.GemmShape(1, 2, 1), act=np.zeros(7, np.float32))  # identity before lengths
    call()
