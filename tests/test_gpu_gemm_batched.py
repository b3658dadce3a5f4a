"""GPU parity of the batched W8A16 projection (af_w8a16_gemm_batched) and the
paged serving step's fused QKV projection + RoPE + paged append
(af_paged_qkv_rope_append).

Batched projection: every token row within half an fp16 ulp plus the fp32
summation bound of the float64 oracle (the reference's per-token GEMV,
qkv_gemm.cu:32-110), the same bar as af_w8a16_gemv. Fused kernel: bit for bit
the batched projection followed by af_paged_rope_append, whole pool compared.
"""
import numpy as np
import pytest

import atomflow_amd
import oracle
from atomflow_amd import device as dev
from atomflow_amd import kv
from inputs import HD, KV_DIM, NKV, NQ, QKV, THETA, fp16_ulp, gemv_abs_terms, gemv_case

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[case] {msg}", flush=True)


def up(a):
    return dev.DeviceBuffer.from_array(a)


def batched_gpu(w, xs, s, group=128, x_stride=None):
    n, k = w.shape
    m = xs.shape[0]
    stride = x_stride or k
    xb = np.zeros((max(m, 1), stride), np.float16)
    xb[:m, :k] = xs
    y = dev.DeviceBuffer(max(m, 1) * n * 2)
    kv.launch_w8a16_gemm_batched(up(xb), stride, m, up(w), up(s), y, n, n, k, group)
    return y.download(np.float16, (max(m, 1), n))[:m]


@pytest.mark.parametrize("n,k,m,group", [(QKV, 3072, 32, 128), (QKV, 3072, 1, 128),
                                         (3072, 3072, 7, 128), (8192, 3072, 45, 128),
                                         (3072, 8192, 16, 128), (100, 1024, 33, 128),
                                         (512, 1024, 20, 32), (256, 768, 5, 96), (272, 640, 3, 64)])
def test_gemm_batched_parity(gpu, n, k, m, group):
    """Group sizes 32 and 96 take the 32-k chunk path (8 weight bytes per MFMA),
    the others the 64-k path with the activations staged through LDS."""
    say(f"batched gemm n={n} k={k} m={m} group={group}")
    w, _, s = gemv_case(n, k, 0xA70F30 + n + k, group=group)
    xs = np.random.default_rng(m + n).standard_normal((m, k)).astype(np.float16)
    got = batched_gpu(w, xs, s, group, x_stride=k + (8 if m % 2 else 0)).astype(np.float64)
    assert np.all(np.isfinite(got))
    for i in range(m):
        y64 = oracle.w8a16_gemv_f64(w, xs[i], s, group)
        bound = k * 2.0 ** -24 * gemv_abs_terms(w, xs[i], s, group)
        err = np.abs(got[i] - y64)
        assert np.all(err <= 0.5 * fp16_ulp(y64) + bound), f"token {i}: max err {err.max():.3e}"


def test_gemm_batched_rejects_bad_shapes(gpu):
    say("batched gemm argument checks")
    w, x, s = gemv_case(64, 1024, 5)
    lib = atomflow_amd.lib()
    y = dev.DeviceBuffer(64 * 2)
    dx, dw, ds = up(x), up(w), up(s)
    call = lib.af_w8a16_gemm_batched
    assert call(dx.ptr, 1024, 1, dw.ptr, ds.ptr, y.ptr, 64, 64, 1000, 128,
                None) == atomflow_amd.AF_ERR_UNSUPPORTED
    assert call(dx.ptr, 1000, 1, dw.ptr, ds.ptr, y.ptr, 64, 64, 1024, 128,
                None) == atomflow_amd.AF_ERR_INVALID_ARG
    assert call(dx.ptr, 1024, 1, dw.ptr, ds.ptr, y.ptr, 32, 64, 1024, 128,
                None) == atomflow_amd.AF_ERR_INVALID_ARG
    assert call(dx.ptr, 1024, 0, dw.ptr, ds.ptr, y.ptr, 64, 64, 1024, 128, None) == 0


@pytest.mark.parametrize("fp8,group,m,bad", [(False, 128, 19, 5), (True, 128, 19, 5),
                                              (False, 32, 19, 5), (False, 128, 1, None),
                                              (True, 128, 1, None), (True, 128, 1, "pos"),
                                              (False, 128, 1, "slot")])
def test_paged_qkv_rope_append_equals_unfused(gpu, fp8, group, m, bad):
    """m = 1 takes the single-token GEMV form; it must still equal the batched
    projection (itself the GEMV at m = 1) followed by the paged append."""
    say(f"paged qkv rope append, fp8 {fp8}, group {group}, m {m}, out of range {bad}")
    k_in, bs, total, max_pos = 3072, 16, 96, 700
    w, _, s = gemv_case(QKV, k_in, 0xA70F31, group=group)
    xs = np.random.default_rng(3).standard_normal((m, k_in)).astype(np.float16)
    r = np.random.default_rng(4)
    slots = r.permutation(total * bs)[:m].astype(np.int64)
    positions = r.integers(0, max_pos, m).astype(np.int32)
    # an out-of-range token: its projection stays unrotated, nothing is appended
    bad_row = None
    if bad == "pos" or isinstance(bad, int):
        bad_row = bad if isinstance(bad, int) else 0
        positions[bad_row] = max_pos
    elif bad == "slot":
        bad_row = 0
        slots[0] = total * bs
    esz = 1 if fp8 else 2
    pool_bytes = 2 * 2 * total * bs * KV_DIM * esz  # two layers
    init = r.integers(0, 256, pool_bytes, dtype=np.uint8)
    scales = up(np.full((2, 2, NKV), 0.04, np.float32)) if fp8 else None
    dtype = atomflow_amd.AF_KV_FP8_E4M3 if fp8 else atomflow_amd.AF_KV_FP16
    pools = []
    for _ in range(2):
        buf = up(init)
        pools.append((buf, kv.make_pool(buf, dtype, bs, 2, NKV, HD, total, scales)))
    c, sn = oracle.rope_table(max_pos, HD, THETA)
    d_c, d_s = up(c), up(sn)
    dx, dw, ds = up(xs), up(w), up(s)
    d_slots, d_pos = up(slots), up(positions)
    # fused
    q1 = dev.DeviceBuffer(m * QKV * 2)
    st = up(np.zeros(1, np.int32))
    kv.launch_paged_qkv_rope_append(dx, k_in, m, dw, ds, k_in, q1, pools[0][1], 1, d_slots,
                                    d_pos, d_c, d_s, max_pos, NQ, d_status=st, group_size=group)
    # unfused: batched projection, then the paged append
    q2 = dev.DeviceBuffer(m * QKV * 2)
    kv.launch_w8a16_gemm_batched(dx, k_in, m, dw, ds, q2, QKV, QKV, k_in, group)
    kv.launch_paged_rope_append(q2, m, pools[1][1], 1, d_slots, d_pos, d_c, d_s, max_pos, NQ)
    assert np.array_equal(q1.download(np.uint16, (m, QKV)), q2.download(np.uint16, (m, QKV)))
    p1 = pools[0][0].download(np.uint8, (pool_bytes,))
    p2 = pools[1][0].download(np.uint8, (pool_bytes,))
    assert np.array_equal(p1, p2)
    plain = batched_gpu(w, xs, s, group)
    if m == 1:  # the batched projection of one token is the GEMV, bit for bit
        y = dev.DeviceBuffer(QKV * 2)
        kv.launch_w8a16_gemv(dx, dw, ds, y, QKV, k_in, group)
        assert np.array_equal(plain[0].view(np.uint16), y.download(np.uint16, (QKV,)))
    status = st.download(np.int32, (1,))[0]
    if bad_row is None:
        assert status == 0
        assert not np.array_equal(p1, init)  # something was appended
        # the appended row matches the oracle's append of the rotated projection
        if m == 1:
            host = init.reshape(2, 2, total * bs, KV_DIM * esz).copy()
            rq = oracle.rope_append(plain[0], np.zeros((1, KV_DIM), np.float16),
                                    np.zeros((1, KV_DIM), np.float16), c[positions[0]:],
                                    sn[positions[0]:], 0, NQ, NKV, HD)
            assert np.array_equal(q1.download(np.uint16, (QKV,)), rq.view(np.uint16))
            kr, vr = rq[NQ * HD:NQ * HD + KV_DIM], rq[NQ * HD + KV_DIM:]
            if fp8:
                hk = host[1, 0].reshape(-1, KV_DIM)
                hv = host[1, 1].reshape(-1, KV_DIM)
                oracle.paged_write_fp8(kr, vr, hk, hv, int(slots[0]), KV_DIM, HD,
                                       np.full(NKV, 0.04, np.float32),
                                       np.full(NKV, 0.04, np.float32))
            else:
                host[1, 0, slots[0]] = kr.view(np.uint8)
                host[1, 1, slots[0]] = vr.view(np.uint8)
            assert np.array_equal(p1, host.reshape(-1))
    else:
        assert status == atomflow_amd.AF_ERR_OUT_OF_RANGE
        assert np.array_equal(q1.download(np.uint16, (m, QKV))[bad_row],
                              plain[bad_row].view(np.uint16))
        if m == 1:
            assert np.array_equal(p1, init)  # nothing appended


def test_paged_qkv_rope_append_graph_replays(gpu):
    """Captured in a hipGraph and replayed three times (device positions advanced
    between replays by the eager side): every replay equals the eager launch."""
    say("paged qkv rope append under graph replay")
    k_in, m, bs, total, max_pos = 3072, 8, 16, 64, 256
    w, _, s = gemv_case(QKV, k_in, 0xA70F32, group=128)
    xs = np.random.default_rng(6).standard_normal((m, k_in)).astype(np.float16)
    slots = np.arange(m, dtype=np.int64) * 5
    c, sn = oracle.rope_table(max_pos, HD, THETA)
    d_c, d_s = up(c), up(sn)
    dx, dw, ds = up(xs), up(w), up(s)
    pool_bytes = 2 * total * bs * KV_DIM * 2
    bufs = [dev.DeviceBuffer(pool_bytes) for _ in range(2)]
    for b in bufs:
        b.fill_u32(0, None)
    dev.synchronize()
    pools = [kv.make_pool(b, atomflow_amd.AF_KV_FP16, bs, 1, NKV, HD, total) for b in bufs]
    outs = [dev.DeviceBuffer(m * QKV * 2) for _ in range(2)]
    d_slots = up(slots)
    d_pos = [up(np.zeros(m, np.int32)) for _ in range(2)]
    stream = dev.Stream()
    run = lambda i: kv.launch_paged_qkv_rope_append(dx, k_in, m, dw, ds, k_in, outs[i], pools[i],
                                                    0, d_slots, d_pos[i], d_c, d_s, max_pos, NQ,
                                                    stream=stream)
    graph = dev.Graph.capture(stream, lambda: run(1))
    for step in range(3):
        pos = (np.arange(m) * 7 + 11 * step).astype(np.int32)
        for dp in d_pos:
            dp.upload(pos)
        run(0)
        graph.launch(stream)
        stream.sync()
        assert np.array_equal(outs[0].download(np.uint16, (m, QKV)),
                              outs[1].download(np.uint16, (m, QKV))), f"replay {step}"
        assert np.array_equal(bufs[0].download(np.uint8, (pool_bytes,)),
                              bufs[1].download(np.uint8, (pool_bytes,))), f"replay {step}"
    graph.destroy()


def deq(w, s, group):
    """float64 weights of E4M3 codes and fp16 group scales."""
    n, k = w.shape
    table = oracle.e4m3_decode_table().astype(np.float64)
    return (table[w].reshape(n, k // group, group) * s.astype(np.float64)[:, :, None]).reshape(n, k)


@pytest.mark.parametrize("n,k,m,group,y_off", [
    (4100, 64, 2, 64, 0), (4100, 640, 33, 128, 1), (4100, 640, 2, 128, 0), (1000, 640, 520, 128, 1),
    (1000, 1024, 520, 128, 0), (4100, 3072, 2, 128, 0), (8200, 1536, 65, 512, 0),
    (8200, 3072, 65, 128, 0), (4100, 128, 2100, 128, 0), (3072, 3072, 2100, 128, 0), (4100, 640, 1000, 128, 1)])
def test_gemm_tiled_parity(gpu, n, k, m, group, y_off):
    """One case or more for each tile of the tiled kernel, with partial token and
    column tiles, fewer groups than K parts, parts of unequal length, output rows
    that are not 16-byte aligned, and a zero and a very small group scale. Every
    output within half an fp16 ulp plus the fp32 summation bound; bytes around the
    outputs are untouched."""
    say(f"tiled gemm n={n} k={k} m={m} group={group} y offset {y_off}")
    w, _, s = gemv_case(n, k, 0xA70F40 + n + k, group=group)
    s = s.copy()
    s[1, 0] = 0.0
    s[2, -1] = np.float16(6e-8)
    x = np.random.default_rng(m + n).standard_normal((m, k)).astype(np.float16)
    stride = n + (5 if y_off else 8)
    y = dev.DeviceBuffer((m * stride + y_off + 1) // 2 * 4)
    y.fill_u32(0x7a7a7a7a)
    kv.launch_w8a16_gemm_batched(up(x), k, m, up(w), up(s), y.ptr + 2 * y_off, stride, n, k, group)
    raw = y.download(np.uint16)
    assert np.all(raw[:y_off] == 0x7a7a)
    rows = np.lib.stride_tricks.as_strided(raw[y_off:], (m, n), (2 * stride, 2)).copy()
    pad = np.lib.stride_tricks.as_strided(raw[y_off + n:], (m, stride - n), (2 * stride, 2))
    assert np.all(pad == 0x7a7a)
    got = rows.view(np.float16).astype(np.float64)
    assert np.all(np.isfinite(got))
    wd = deq(w, s, group)
    want = x.astype(np.float64) @ wd.T
    bound = k * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(wd).T)
    err = np.abs(got - want)
    assert np.all(err <= 0.5 * fp16_ulp(want) + bound), f"max err {err.max():.3e}"


@pytest.mark.parametrize("fp8,m,q_off,nq,k_in", [
    (False, 17, 0, NQ, 3072), (True, 40, 0, NQ, 3072), (True, 65, 0, NQ, 3072),
    (False, 131, 1, NQ, 3072), (True, 300, 1, NQ, 3072), (False, 513, 0, NQ, 3072),
    (True, 1100, 0, NQ, 3072), (False, 1300, 0, NQ, 3072), (True, 1300, 1, NQ, 3072),
    (False, 257, 0, 32, 4096), (False, 9, 1, 8, 1024), (True, 9, 0, 8, 1024), (False, 30, 0, 8, 1024),
    (True, 30, 1, 8, 1024)])
def test_paged_qkv_rope_append_many_tokens(gpu, fp8, m, q_off, nq, k_in):
    """Every fused form, the tiles' (24 heads of k 3072) and the 16-row kernel's two (8 heads):
    bit for bit the batched projection followed by the paged append, whole pool compared,
    with tokens out of range at both ends; q_off: qkv rows that are not 16-byte aligned."""
    bs, total, max_pos = 16, 96, 700
    qkv_dim = (nq + 2 * NKV) * HD
    say(f"paged qkv rope append of {m} tokens, fp8 {fp8}, {nq} query heads, k {k_in}")
    w, _, s = gemv_case(qkv_dim, k_in, 0xA70F33, group=128)
    xs = np.random.default_rng(13).standard_normal((m, k_in)).astype(np.float16)
    r = np.random.default_rng(14)
    slots = r.permutation(total * bs)[:m].astype(np.int64)
    positions = r.integers(0, max_pos, m).astype(np.int32)
    positions[7], slots[m - 1] = max_pos, total * bs
    pool_bytes = 2 * 2 * total * bs * KV_DIM * (1 if fp8 else 2)
    init = r.integers(0, 256, pool_bytes, dtype=np.uint8)
    scales = up(np.full((2, 2, NKV), 0.04, np.float32)) if fp8 else None
    dtype = atomflow_amd.AF_KV_FP8_E4M3 if fp8 else atomflow_amd.AF_KV_FP16
    pools = []
    for _ in range(2):
        buf = up(init)
        pools.append((buf, kv.make_pool(buf, dtype, bs, 2, NKV, HD, total, scales)))
    c, sn = oracle.rope_table(max_pos, HD, THETA)
    d_c, d_s, dx, dw, ds = up(c), up(sn), up(xs), up(w), up(s)
    d_slots, d_pos = up(slots), up(positions)
    q1, q2 = dev.DeviceBuffer(m * qkv_dim * 2 + 16), dev.DeviceBuffer(m * qkv_dim * 2)
    st = up(np.zeros(1, np.int32))
    kv.launch_paged_qkv_rope_append(dx, k_in, m, dw, ds, k_in, q1.ptr + 2 * q_off, pools[0][1], 1,
                                    d_slots, d_pos, d_c, d_s, max_pos, nq, d_status=st)
    kv.launch_w8a16_gemm_batched(dx, k_in, m, dw, ds, q2, qkv_dim, qkv_dim, k_in)
    plain = q2.download(np.uint16, (m, qkv_dim))
    kv.launch_paged_rope_append(q2, m, pools[1][1], 1, d_slots, d_pos, d_c, d_s, max_pos, nq)
    got = q1.download(np.uint16)[q_off:q_off + m * qkv_dim].reshape(m, qkv_dim)
    want = q2.download(np.uint16, (m, qkv_dim))
    want[[7, m - 1]] = plain[[7, m - 1]]
    assert np.array_equal(got, want)
    assert np.array_equal(pools[0][0].download(np.uint8), pools[1][0].download(np.uint8))
    assert st.download(np.int32, (1,))[0] == atomflow_amd.AF_ERR_OUT_OF_RANGE


def odd_values(w, s, x):
    """Zero, subnormal, negative, huge, infinite and NaN group scales, infinite and NaN
    activations in and out of zero-scale groups, and a NaN weight code."""
    w, s, x = w.copy(), s.copy(), x.copy()
    s[0, 0] = s[1, -1] = 0.0
    s[2, :] = 0.0
    s[3, 0] = s[3, -1] = np.inf
    s[4, s.shape[1] // 2] = np.nan
    s[5, 0], s[5, -1] = np.float16(6e-8), 65504.0
    s[6, :] = -s[6, :]
    s[7, -1] = -np.inf
    w[9, 3] = 0x7f
    x[0, 1], x[1, -1], x[-1, 0] = np.inf, -np.inf, np.nan
    x[-2, ::2], x[-2, 1::2] = 65504.0, -65504.0
    return w, s, x


# one or more of every form: the 16-row kernel's two, and each tile; group sizes of one to
# sixteen 64-k steps, from one group to more than eight per part, fewer groups than parts
@pytest.mark.parametrize("n,k,m,group", [
    (4100, 640, 20, 128), (5125, 3072, 5, 128), (3072, 8192, 17, 128), (5125, 3072, 33, 128),
    (4100, 4608, 40, 192), (5125, 3072, 70, 128), (4100, 1536, 70, 512), (5125, 3072, 129, 128),
    (1000, 1024, 517, 128), (8200, 1024, 40, 1024), (4100, 1152, 300, 192), (5125, 3072, 200, 128),
    (5125, 3072, 600, 128), (5125, 3072, 1300, 128), (4100, 320, 1500, 64), (4100, 256, 1500, 64)])
@pytest.mark.parametrize("odd", [False, True])
def test_gemm_bits_do_not_depend_on_the_launch(gpu, n, k, m, group, odd):
    """A token's results have the same bits in a launch of m tokens and all n rows as in
    one of up to 16 tokens and 64 rows, which the 16-row kernel runs."""
    say(f"gemm bits n={n} k={k} m={m} group={group} odd {odd}")
    w, _, s = gemv_case(n, k, 0xA70F50 + n + k, group=group)
    x = np.random.default_rng(m + k).standard_normal((m, k)).astype(np.float16)
    if odd:
        w, s, x = odd_values(w, s, x)
    got = batched_gpu(w, x, s, group)
    rows, toks = min(n, 64), min(m, 16)
    for t in sorted({0, (m - toks) // 2, m - toks}):
        for r in (0, n - rows):
            want = batched_gpu(w[r:r + rows], x[t:t + toks], s[r:r + rows], group)
            part = got[t:t + toks, r:r + rows]
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(part), nan), (t, r)
            assert np.array_equal(np.where(nan, 0, part.view(np.uint16)),
                                  np.where(nan, 0, want.view(np.uint16))), (t, r)
            assert odd or not nan.any()
