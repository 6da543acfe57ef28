"""Launches of chunk_kernel (2 to 32 positions, and one with a norm): the reference's
quantized_tensor_matmul_f32 (src/quantized_matvec.cpp:164-224) and the norm,
bias and SwiGLU around it, at the edges of the kernel's cuts: row groups of
16, rounds of 4 positions, fragments of 8, 16 and 32, K in one workgroup or
in chunks, partial 128-weight units.

Bar: every row of every position within 1e-5 * sum |w x| of the oracle, the
bar of every product here. The kernel's activations are two f16 limbs under a
power of two per position and unit, within 2^-23 of each value that is within
2^28 of the unit's largest, so a value 2^26 below its unit's largest must
count as on the VALU kernels."""
import numpy as np
import pytest

import _blocks as B

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def hip(qmv):
    import importlib
    return importlib.import_module("my-inference-engine_amd.hip_runtime")


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _tensor(qmv, t, rows, cols, seed):
    raw = qmv.synth_tensor(t, rows, cols, seed=seed)
    return raw, qmv.DeviceTensor(qmv.make_view(raw, t, rows, cols))


def _check(oracle, raw, t, rows, cols, x, y, what, scale=1.0):
    for b in range(x.shape[0]):
        ref = oracle.matvec(raw, t, rows, cols, x[b])
        _, absdot = oracle.row_stats(raw, t, rows, cols, x[b])
        assert (np.abs(y[b].astype(np.float64) - ref) <= scale * TOL * absdot).all(), f"{what}: position {b}"


# K: one unit, an odd number, the last that one workgroup takes, chunks; the
# 32-weight formats also with a partial last unit.
KS = {B.Q4_K: [256, 1280, 4352, 8960], B.Q6_K: [256, 1280, 4096, 10240],
      B.Q8_0: [32, 480, 1536, 4864], B.Q5_0: [96, 672, 2080, 5120]}


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("rows,batch", [(1, 2), (15, 4), (16, 5), (17, 8), (65, 9), (130, 16), (47, 17), (1000, 32)])
def test_chunk_edges(qmv, oracle, gpu, hip, t, rows, batch):
    with hip.Stream() as s:
        for cols in KS[t]:
            raw, dt = _tensor(qmv, t, rows, cols, rows + batch)
            x = qmv.synth_normal(batch * cols, seed=batch).reshape(batch, cols)
            dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * (batch * rows + 64))
            dy.fill(0x7F)  # nothing past the outputs is written
            print(f"chunks: {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
            dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
            s.synchronize()
            y = dy.to_array(np.float32, (batch * rows + 64,))
            assert np.all(_bits(y[batch * rows:]) == 0x7F7F7F7F)
            _check(oracle, raw, t, rows, cols, x, y[:batch * rows].reshape(batch, rows), f"K={cols}")
            dt.close()


@pytest.mark.parametrize("t,one", [(B.Q8_0, 1), (B.Q5_0, 17)])
@pytest.mark.parametrize("batch", [2, 8, 24])
def test_chunk_holds_activations(qmv, gpu, hip, t, one, batch):
    """Row r has the weight 1 at column r and zeros, whose products are exact,
    so the outputs are the activations as the limbs hold them: within 2^-23 of
    the value down to 2^-28 of its unit's largest, else within 2^-51 of that."""
    n = 128
    w = np.zeros((n, n // 32, B.BLOCK_BYTES[t]), np.uint8)
    w[:, :, 1] = 0x3C  # f16 1.0
    for r in range(n):
        if t == B.Q8_0:
            w[r, r // 32, 2 + r % 32] = one
        else:  # codes of 16, and one of 17
            w[r, :, 2:6] = 0xFF
            w[r, r // 32, 6 + r % 16] = (one & 15) << (4 * (r % 32 // 16))
    dt = qmv.DeviceTensor(qmv.make_view(np.ascontiguousarray(w.reshape(-1)), t, n, n))
    rng = np.random.default_rng(batch)
    x = (rng.uniform(1, 2, (batch, n)) * rng.choice([-1, 1], (batch, n))).astype(np.float32)
    x[0] *= np.float32(2.0) ** rng.integers(-60, 60, n).astype(np.float32)
    x[1] *= np.float32(2.0) ** rng.integers(-25, 1, n).astype(np.float32)
    x[1, 5] = 2.0 ** -120  # far below the rest
    with hip.Stream() as s:
        dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * batch * n)
        print(f"chunks: activations held {B.NAMES[t]} M={batch}", flush=True)
        dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        s.synchronize()
        y = dy.to_array(np.float32, (batch, n)).astype(np.float64)
    v = x.astype(np.float64)
    largest = np.abs(v).max(1, keepdims=True)
    err = np.abs(y - v)
    assert (err <= np.where(np.abs(v) >= largest * 2.0 ** -28, np.abs(v) * 2.0 ** -23, largest * 2.0 ** -51)).all()
    dt.close()


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("batch", [2, 6, 20])
def test_chunk_small_beside_large(qmv, oracle, gpu, hip, t, batch):
    """The first sub-block's scale is 0, so its products are 0, and its
    activations are 2^26 times the others of the same unit: the others keep
    full precision."""
    rows, cols = 40, 1024
    raw = qmv.synth_tensor(t, rows, cols, seed=9).reshape(rows, -1).copy()
    w = raw.reshape(rows, cols // B.BLOCK_ELEMENTS[t], -1)
    if t == B.Q4_K:  # 6-bit scale and minimum of sub-block 0
        w[:, 0, 4] &= 0xC0
        w[:, 0, 8] &= 0xC0
    elif t == B.Q6_K:
        w[:, 0, 192] = 0
    else:
        w[:, 0, :2] = 0
    raw = np.ascontiguousarray(raw.reshape(-1))
    dt = qmv.DeviceTensor(qmv.make_view(raw, t, rows, cols))
    x = qmv.synth_normal(batch * cols, seed=10).reshape(batch, cols)
    x[:, :16 if t == B.Q6_K else 32] *= np.float32(2.0 ** 26)
    with hip.Stream() as s:
        dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * batch * rows)
        print(f"chunks: {B.NAMES[t]} outliers M={batch}", flush=True)
        dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        s.synchronize()
        _check(oracle, raw, t, rows, cols, x, dy.to_array(np.float32, (batch, rows)), "outliers")
    dt.close()


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("batch,cols", [(1, 1024), (3, 1024), (8, 1024), (12, 1024), (32, 1024), (13, 5120), (6, 8960)])
def test_chunk_norm_group(qmv, oracle, gpu, hip, t, batch, cols):
    """RMSNorm, three tensors of unequal rows and biases in one call, then the
    gate and up pair, against the oracle's norm and products; a NaN in one
    position stays there, and an infinity gives no finite row."""
    rows = [100, 16, 33]
    raws, dts = zip(*[_tensor(qmv, t, r, cols, 40 + i) for i, r in enumerate(rows)])
    rng = np.random.default_rng(batch)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    bias = [rng.standard_normal(r).astype(np.float32) for r in rows]
    normed = np.stack([oracle.rms_norm(x[b], nw, 1e-6)[1] for b in range(batch)])
    with hip.Stream() as s:
        dx, dw, dn = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer.from_array(nw), hip.DeviceBuffer(4 * batch * cols)
        db = [hip.DeviceBuffer.from_array(b) for b in bias]
        ys = [hip.DeviceBuffer(4 * batch * r) for r in rows]

        def call():
            qmv.device_rms_norm_matvec_add_group(list(dts), dx.ptr, dw.ptr, 1e-6, batch, [b.ptr for b in db], [0, 0, 0],
                                                 [y.ptr for y in ys], dn.ptr, s.handle)
            s.synchronize()
            return [y.to_array(np.float32, (batch, r)) for y, r in zip(ys, rows)]

        print(f"chunks: {B.NAMES[t]} norm group K={cols} M={batch}", flush=True)
        first = call()
        for raw, r, y, b in zip(raws, rows, first, bias):
            _check(oracle, raw, t, r, cols, normed, y - b[None, :], f"rows {r}", scale=2.0)
        for bad in (np.nan, np.inf) if batch > 1 else ():
            x2 = x.copy()
            x2[1, cols // 3] = bad
            dx = hip.DeviceBuffer.from_array(x2)
            again = call()
            for a, f in zip(again, first):
                keep = [p for p in range(batch) if p != 1]
                assert np.array_equal(_bits(a[keep]), _bits(f[keep]))
                assert np.isnan(a[1]).all() if np.isnan(bad) else not np.isfinite(a[1]).any()
        dx = hip.DeviceBuffer.from_array(x)
        raw_u, du = _tensor(qmv, t, rows[0], cols, 77)
        gate, up, act = (hip.DeviceBuffer(4 * batch * rows[0]) for _ in range(3))
        dxn = hip.DeviceBuffer.from_array(normed)
        qmv.device_matvec_group([dts[0], du], dxn.ptr, batch, [gate.ptr, up.ptr], s.handle)
        qmv.device_rms_norm_matvec_swiglu(dts[0], du, dx.ptr, dw.ptr, 1e-6, batch, act.ptr, dn.ptr, s.handle)
        s.synchronize()
        g, u, a = (v.to_array(np.float32, (batch, rows[0])).astype(np.float64) for v in (gate, up, act))
        absg, absu = (np.stack([oracle.row_stats(r, t, rows[0], cols, normed[b])[1] for b in range(batch)])
                      for r in (raws[0], raw_u))
        # |d silu| <= 1.1 |d g|; both projections within 2e-5 of their sums
        bound = 2 * TOL * (1.1 * absg * np.abs(u) + absu * np.abs(g / (1 + np.exp(-g))) + 2 * TOL * absg * absu) + 1e-6
        assert (np.abs(a - u * g / (1 + np.exp(-g))) <= bound).all()
        du.close()
    for d in dts:
        d.close()


@pytest.mark.parametrize("t,rows,cols,batch", [(B.Q4_K, 64, 256, 32), (B.Q8_0, 900, 96, 20), (B.Q6_K, 5200, 512, 24)])
def test_chunk_capture_without_a_first_call(qmv, oracle, gpu, hip, t, rows, cols, batch):
    """Launches over one or two K-units need no workspace, so a stream that
    never ran one can capture them; replays match the eager launch's bar."""
    raw, dt = _tensor(qmv, t, rows, cols, 5)
    x = qmv.synth_normal(batch * cols, seed=6).reshape(batch, cols)
    dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * batch * rows)
    with hip.Stream() as s, hip.Graph(s) as g:
        print(f"chunks: capture {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
        g.begin()
        dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        g.end()
        for _ in range(3):
            dy.fill(0)
            g.replay()
            s.synchronize()
            _check(oracle, raw, t, rows, cols, x, dy.to_array(np.float32, (batch, rows)), "replay")
    dt.close()


def test_chunk_output_over_norm_weights(qmv, oracle, gpu, hip):
    """An output that lies over the norm weights is written after they are
    read (the norm then runs as a launch of its own)."""
    t, rows, cols, batch = B.Q4_K, 64, 512, 4
    raw, dt = _tensor(qmv, t, rows, cols, 8)
    x = qmv.synth_normal(batch * cols, seed=6).reshape(batch, cols)
    nw = np.abs(qmv.synth_normal(cols, seed=7)).astype(np.float32) + 0.5
    normed = np.stack([oracle.rms_norm(x[b], nw, 1e-6)[1] for b in range(batch)])
    with hip.Stream() as s:
        dx, dw, dn = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer.from_array(nw), hip.DeviceBuffer(4 * batch * cols)
        print("chunks: output over norm weights", flush=True)
        qmv.device_rms_norm_matvec_add_group([dt], dx.ptr, dw.ptr, 1e-6, batch, [0], [0], [dw.ptr], dn.ptr, s.handle)
        s.synchronize()
        _check(oracle, raw, t, rows, cols, normed, dw.to_array(np.float32, (cols,))[:batch * rows].reshape(batch, rows),
               "over the weights", scale=2.0)
    dt.close()


@pytest.mark.parametrize("t,rows,cols,batch", [(B.Q4_K, 4000, 1024, 170), (B.Q8_0, 3000, 512, 77),
                                               (B.Q8_0, 900, 256, 550)])
def test_host_calls_of_several_launches(qmv, oracle, gpu, hip, t, rows, cols, batch):
    """A host call of more launches than parts in which it is copied out (550
    positions: 18), one of 6 and one of three, whose inputs and outputs are
    copied while launches run:
    the bits of the same positions in calls of one launch each; an input
    inside the output's memory is read before it is overwritten."""
    raw = qmv.synth_tensor(t, rows, cols, seed=21)
    v = qmv.make_view(raw, t, rows, cols)
    x = qmv.synth_normal(batch * cols, seed=22).reshape(batch, cols)
    print(f"chunks: host {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
    y = qmv.matvec(v, x)
    parts = np.concatenate([qmv.matvec(v, x[b:b + 32]).reshape(-1, rows) for b in range(0, batch, 32)])
    assert np.array_equal(_bits(y), _bits(parts))
    shared = np.zeros(batch * rows, dtype=np.float32)
    inp = shared[-batch * cols:]
    inp[:] = x.reshape(-1)
    assert qmv.quantized_tensor_matmul_f32(v, inp, cols, batch, shared, rows) == 1
    assert np.array_equal(_bits(shared), _bits(y.reshape(-1)))
    qmv.release_tensor(v.data)


@pytest.mark.parametrize("t,rows,cols,batch,norm", [(B.Q4_K, 151936, 1024, 25, False), (B.Q6_K, 151936, 1024, 17, False),
                                                    (B.Q8_0, 262144, 640, 17, False), (B.Q8_0, 262144, 640, 9, True)])
def test_chunk_capture_of_short_rows(qmv, oracle, gpu, hip, t, rows, cols, batch, norm):
    """Many short rows, whose fastest launch has a workspace: captured on a
    stream that has none, at positions that leave one over from eights; the
    replays against the oracle at three positions."""
    raw, dt = _tensor(qmv, t, rows, cols, 5)
    x = qmv.synth_normal(batch * cols, seed=6).reshape(batch, cols)
    nw = (1 + 0.1 * qmv.synth_normal(cols, seed=7)).astype(np.float32)
    dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * batch * rows)
    dw, dn = hip.DeviceBuffer.from_array(nw), hip.DeviceBuffer(4 * batch * cols)
    ref_x = np.stack([oracle.rms_norm(v, nw, 1e-6)[1] for v in x]) if norm else x
    with hip.Stream() as s, hip.Graph(s) as g:
        print(f"chunks: capture of short rows {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
        g.begin()
        if norm:
            qmv.device_rms_norm_matvec_add_group([dt], dx.ptr, dw.ptr, 1e-6, batch, [0], [0], [dy.ptr], dn.ptr, s.handle)
        else:
            dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        g.end()
        for _ in range(2):
            dy.fill(0)
            g.replay()
            s.synchronize()
            some = [0, batch // 2, batch - 1]
            _check(oracle, raw, t, rows, cols, ref_x[some], dy.to_array(np.float32, (batch, rows))[some], "replay",
                   scale=2.0 if norm else 1.0)
    dt.close()


@pytest.mark.parametrize("t,rows,cols,warm,batch", [(B.Q8_0, 1000, 1280, 8, 1), (B.Q6_K, 1000, 2560, 4, 1),
                                                    (B.Q5_0, 1000, 1280, 16, 4), (B.Q4_K, 300, 8960, 32, 5)])
def test_chunk_call_then_capture_of_another_kernel(qmv, oracle, gpu, hip, t, rows, cols, warm, batch):
    """A call of chunk_kernel, then the first call of the same tensor on a
    matvec kernel, captured: the stream's workspace holds what it needs."""
    raw, dt = _tensor(qmv, t, rows, cols, 15)
    x = qmv.synth_normal(warm * cols, seed=16).reshape(warm, cols)
    dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * warm * rows)
    with hip.Stream() as s, hip.Graph(s) as g:
        print(f"chunks: capture after {warm}: {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
        dt.matvec(dx.ptr, warm, dy.ptr, s.handle)
        s.synchronize()
        g.begin()
        dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        g.end()
        for _ in range(3):
            dy.fill(0)
            g.replay()
            s.synchronize()
            y = dy.to_array(np.float32, (warm, rows))[:batch]
            _check(oracle, raw, t, rows, cols, x[:batch], y, "replay")
            dt.matvec(dx.ptr, warm, dy.ptr, s.handle)
            s.synchronize()
    dt.close()


def _class(a):
    """+inf, -inf, NaN or finite, as numbers"""
    return np.where(np.isnan(a), 3, np.where(np.isinf(a), np.sign(np.where(np.isinf(a), a, 0)), 0))


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("rows,cols,batch", [(96, 1024, 2), (33, 1024, 4), (96, 512, 7), (70, 1024, 8), (48, 1024, 11),
                                             (96, 5120, 16), (40, 8960, 21), (600, 1024, 32)])
def test_chunk_infinities(qmv, oracle, gpu, hip, t, rows, cols, batch):
    """An infinity gives the rows of its position the infinity of its
    weight's sign (NaN where the weight is 0), as the reference's sum does;
    two may cancel to NaN; a NaN stays NaN; the other positions keep their
    bits, and nothing past the outputs is written."""
    raw, dt = _tensor(qmv, t, rows, cols, 31)
    x = qmv.synth_normal(batch * cols, seed=32).reshape(batch, cols)
    bad = x.copy()
    bad[0, cols // 3] = np.inf
    bad[1, cols - 1] = -np.inf
    if batch > 3:
        bad[2, [0, cols // 2]] = np.inf
        bad[batch - 1, 7] = np.nan
    with hip.Stream() as s:
        print(f"chunks: infinities {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
        ys = []
        for v in (x, bad):
            dx, dy = hip.DeviceBuffer.from_array(v), hip.DeviceBuffer(4 * (batch * rows + 64))
            dy.fill(0x7F)
            dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
            s.synchronize()
            y = dy.to_array(np.float32, (batch * rows + 64,))
            assert np.all(_bits(y[batch * rows:]) == 0x7F7F7F7F)
            ys.append(y[:batch * rows].reshape(batch, rows))
    for b in range(batch):
        if np.isfinite(bad[b]).all():
            assert np.array_equal(_bits(ys[1][b]), _bits(ys[0][b])), b
        else:
            ref = oracle.matvec(raw, t, rows, cols, bad[b])
            assert np.array_equal(_class(ys[1][b]), _class(ref)), b
    dt.close()


@pytest.mark.parametrize("t", [B.Q4_K, B.Q6_K])
@pytest.mark.parametrize("batch", [2, 7, 16, 32])
def test_chunk_subnormal_operands(qmv, oracle, gpu, hip, t, batch):
    """Sub-block scales of 1 (Q6_K: and -1) and codes next to the centre, whose
    matrix operands are f16 subnormals: they count in full. Against 64 bits
    (measured 6e-8 to 8e-8; the bar is the rounding of an fp32 sum, and operands
    taken as zero would be off by more than 0.1)."""
    rows, cols = 64, 1024
    rng = np.random.default_rng(batch)
    raw = qmv.synth_tensor(t, rows, cols, seed=9).reshape(rows, cols // 256, -1).copy()
    if t == B.Q4_K:  # scales 1, minimums 0; codes 7, 8, 9
        raw[:, :, 2:4] = 0
        raw[:, :, 4:16] = 0
        raw[:, :, 4:8] = 1
        raw[:, :, 12:16] = 1
        q = rng.integers(7, 10, (2, rows, cols // 256, 128))
        raw[:, :, 16:] = q[0] | q[1] << 4
    else:  # scales 1 and -1; low nibbles 5 .. 11
        raw[:, :, 192:208] = rng.choice([1, 255], (rows, cols // 256, 16))
        q = rng.integers(5, 12, (2, rows, cols // 256, 128))
        raw[:, :, :128] = q[0] | q[1] << 4
    raw = np.ascontiguousarray(raw.reshape(-1))
    dt = qmv.DeviceTensor(qmv.make_view(raw, t, rows, cols))
    w = oracle.dequantize_rows(raw, t, rows, cols, 0, rows).reshape(rows, cols).astype(np.float64)
    if t == B.Q4_K:  # pairs that cancel: the 8 of every code adds nothing
        x = rng.standard_normal((batch, cols)).astype(np.float32)
        x[:, 1::2] = -x[:, ::2]
    else:
        x = rng.standard_normal((batch, cols)).astype(np.float32)
    ref = x.astype(np.float64) @ w.T
    with hip.Stream() as s:
        dx, dy = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * batch * rows)
        print(f"chunks: subnormal operands {B.NAMES[t]} M={batch}", flush=True)
        dt.matvec(dx.ptr, batch, dy.ptr, s.handle)
        s.synchronize()
        y = dy.to_array(np.float32, (batch, rows)).astype(np.float64)
    err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    print(f"relative error {err:.2g}", flush=True)
    assert err <= 3e-7
    dt.close()


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("rows,units,batch", [(1, 1, 9), (8193, 2, 16), (8200, 3, 17), (12300, 4, 12), (8192, 4, 32), (20011, 1, 31),
                                              (8195, 8, 10)])
def test_chunk_direct(qmv, oracle, gpu, hip, t, rows, units, batch):
    """Launches whose waves take whole rows and store them, at the sizes where
    these begin, one segment and several, with rows that fill no group and a
    partial last unit; three tensors at once with an addend each, one in place and one
    bias; an infinity keeps its sign."""
    cols = units * (256 if t in (B.Q4_K, B.Q6_K) else 128) - (0 if t in (B.Q4_K, B.Q6_K) else 32)
    shape = [rows, 33, 16]
    raws, dts = zip(*[_tensor(qmv, t, r, cols, 60 + i) for i, r in enumerate(shape)])
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[1, cols // 2] = np.inf
    adds = [rng.standard_normal((batch, rows)).astype(np.float32), rng.standard_normal(33).astype(np.float32), None]
    with hip.Stream() as s:
        dx = hip.DeviceBuffer.from_array(x)
        ys = [hip.DeviceBuffer(4 * (batch * r + 64)) for r in shape]
        for y in ys:
            y.fill(0x7F)
        ys[0] = hip.DeviceBuffer.from_array(np.concatenate([adds[0].reshape(-1), np.full(64, 7, np.float32)]))
        bias = hip.DeviceBuffer.from_array(adds[1])
        print(f"chunks: direct {B.NAMES[t]} {rows}x{cols} M={batch}", flush=True)
        qmv.device_matvec_add_group(list(dts), dx.ptr, batch, [ys[0].ptr, bias.ptr, 0], [rows, 0, 0], [y.ptr for y in ys],
                                    s.handle)
        s.synchronize()
        out = [y.to_array(np.float32, (batch * r + 64,)) for y, r in zip(ys, shape)]
    assert (out[0][batch * rows:] == 7).all()
    assert all((_bits(o[batch * r:]) == 0x7F7F7F7F).all() for o, r in zip(out[1:], shape[1:]))
    for raw, r, o, add in zip(raws, shape, out, (adds[0], adds[1][None, :], np.zeros((1, 1), np.float32))):
        y = o[:batch * r].reshape(batch, r)
        some = [0, 2, batch // 2, batch - 1]
        _check(oracle, raw, t, r, cols, x[some], (y - add)[some], f"rows {r}", scale=1.5)
        assert np.array_equal(_class(y[1]), _class(oracle.matvec(raw, t, r, cols, x[1])))
    for d in dts:
        d.close()


@pytest.mark.parametrize("t", B.ALL_TYPES)
@pytest.mark.parametrize("batch,cols", [(3, 512), (20, 1024)])
def test_chunk_norm_weights_that_overflow(qmv, oracle, gpu, hip, t, batch, cols):
    """Inputs times norm weights past fp32's range where the normalised values
    are within it: the reference divides first, and so must the rows."""
    rows = 40
    raw, dt = _tensor(qmv, t, rows, cols, 71)
    x = (qmv.synth_normal(batch * cols, seed=72).reshape(batch, cols) * np.float32(1e15)).astype(np.float32)
    nw = np.full(cols, 1e25, np.float32)
    normed = np.stack([oracle.rms_norm(v, nw, 1e-6)[1] for v in x])
    assert np.isfinite(normed).all()
    with hip.Stream() as s:
        dx, dw, dn = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer.from_array(nw), hip.DeviceBuffer(4 * batch * cols)
        dy = hip.DeviceBuffer(4 * batch * rows)
        print(f"chunks: norm overflow {B.NAMES[t]} K={cols} M={batch}", flush=True)
        qmv.device_rms_norm_matvec_add_group([dt], dx.ptr, dw.ptr, 1e-6, batch, [0], [0], [dy.ptr], dn.ptr, s.handle)
        s.synchronize()
        _check(oracle, raw, t, rows, cols, normed, dy.to_array(np.float32, (batch, rows)), "overflow", scale=2.0)
    dt.close()
