"""GGML-format GEMV with candle's CPU arithmetic (pgd_matrix_gemv_q8act_dev):
each activation row quantized to Q8_K (Q4_K / Q6_K) or Q8_0 (Q8_0 / Q5_0) and
integer block dots, against the oracle's restatement of the same kernels
(oracle.c: q8k_quantize_block, vec_dot_q4k_q8k, vec_dot_q6k_q8k,
vec_dot_q8_0_q8_0, vec_dot_q5_0_q8_0). The integer parts are exact and the
f32 terms are added in GGML's scalar order (eight residue-class sums per
256-block, block after block), so every output is bit-equal to the oracle."""
import numpy as np
import pytest

from checkpoints import GGML_Q5_0, GGML_Q8_0, random_blocks
from oracle import pyoracle as ora

pytestmark = pytest.mark.gpu

def close(y, ref):
    """Bit-equal to the oracle's f32 outputs."""
    return bool(np.array_equal(np.asarray(y, np.float32).view(np.uint32), np.asarray(ref, np.float32).view(np.uint32)))


def oracle_rows(fmt, blocks, n_out, n_in, x):
    out = []
    for row in x:
        if fmt in (1, 2):
            out.append(ora.kq_vec_dot_q8k(fmt, blocks, n_out, n_in, ora.q8k_quantize(row)))
        else:
            out.append(ora.q8_0_vec_dot(fmt, blocks, n_out, n_in, ora.q8_0_quantize_act(row)))
    return np.stack(out).astype(np.float32)


def make(dev, fmt, n_out, n_in, seed):
    from pagoda_amd import Matrix

    rng = np.random.default_rng(seed)
    if fmt in (1, 2):
        w = rng.normal(0, 0.02, (n_out, n_in)).astype(np.float32)
        blk = ora.q4k_quantize(w) if fmt == 1 else ora.q6k_quantize(w)
    else:
        blk = random_blocks(rng, GGML_Q8_0 if fmt == 3 else GGML_Q5_0, n_out, n_in, d_std=2e-3)
    return Matrix.upload_kq(dev, fmt, blk, n_out, n_in), blk


SHAPES = [(4864, 896), (896, 4864), (1152, 896), (151936, 896), (40, 320)]


@pytest.mark.parametrize("fmt", [1, 2, 3, 4])
@pytest.mark.parametrize("shape", SHAPES)
def test_q8act_gemv_matches_oracle(dev, fmt, shape):
    n_out, n_in = shape
    if fmt in (3, 4) and n_out == 151936:
        n_out = 8192  # keeps the random 32-weight blocks small
    m, blk = make(dev, fmt, n_out, n_in, 100 * fmt + n_in % 97)
    rng = np.random.default_rng(n_out + fmt)
    x = rng.normal(0, 1, (9, n_in)).astype(np.float32)
    x[3, :] = 0.0  # an all-zero row: d = 0 blocks
    x[4, 5] = 40.0  # one outlier sets its block's scale
    xd = dev.upload(x)
    ref = oracle_rows(fmt, blk, n_out, n_in, x)
    outs = {}
    for rows in (1, 4, 9):
        yd = dev.alloc(rows * n_out * 4)
        m.gemv_q8act_dev(xd, n_in, rows, yd, n_out)
        outs[rows] = dev.download(yd, (rows, n_out), np.float32)
        dev.free(yd)
        assert close(outs[rows], ref[:rows]), (rows, np.abs(outs[rows] - ref[:rows]).max(),
                                                 int((outs[rows] != ref[:rows]).sum()))
    # a row's result does not depend on how many rows share its launch
    np.testing.assert_array_equal(outs[4][0].view(np.uint32), outs[1][0].view(np.uint32))
    np.testing.assert_array_equal(outs[9][:4].view(np.uint32), outs[4].view(np.uint32))
    # residual form
    res = rng.normal(0, 1, (4, n_out)).astype(np.float32)
    rd = dev.upload(res)
    m.gemv_q8act_dev(xd, n_in, 4, rd, n_out, rd, n_out)
    got = dev.download(rd, (4, n_out), np.float32)
    np.testing.assert_array_equal(got.view(np.uint32), (res + outs[4]).view(np.uint32))
    dev.free(rd)
    dev.free(xd)
    m.free()


@pytest.mark.parametrize("fa,fb", [(1, 2), (2, 1), (3, 4)])
def test_q8act_pair_equals_two_launches(dev, fa, fb):
    """Two matrices over one input in one launch (the attention's stacked
    q|k and v): each output bit-equal to its own launch, at 1, 4 and 9 rows
    (1-, 4- and 16-row launches), with a row stride wider than either."""
    n_in, na, nb = 896, 1024, 128
    if fa == 3:
        na = 1000  # a partly filled last tile
    ma, _ = make(dev, fa, na, n_in, 11 * fa)
    mb, _ = make(dev, fb, nb, n_in, 13 * fb)
    rng = np.random.default_rng(fa * 10 + fb)
    x = rng.normal(0, 1, (9, n_in)).astype(np.float32)
    xd = dev.upload(x)
    ld = na + nb + 16
    for rows in (1, 4, 9):
        ys, ya, yb = dev.alloc(rows * ld * 4), dev.alloc(rows * na * 4), dev.alloc(rows * nb * 4)
        ma.gemv_q8act_pair_dev(ys, mb, ys + na * 4, xd, n_in, rows, ld)
        ma.gemv_q8act_dev(xd, n_in, rows, ya, na)
        mb.gemv_q8act_dev(xd, n_in, rows, yb, nb)
        got = dev.download(ys, (rows, ld), np.float32)
        a = dev.download(ya, (rows, na), np.float32)
        b = dev.download(yb, (rows, nb), np.float32)
        np.testing.assert_array_equal(got[:, :na].view(np.uint32), a.view(np.uint32), err_msg=f"a rows={rows}")
        np.testing.assert_array_equal(got[:, na:na + nb].view(np.uint32), b.view(np.uint32), err_msg=f"b rows={rows}")
        for p in (ys, ya, yb):
            dev.free(p)
    dev.free(xd)
    ma.free()
    mb.free()


def test_q8act_pair_rejects_mixed_activation_types(dev):
    from pagoda_amd import PagodaError

    ma, _ = make(dev, 1, 64, 256, 1)
    mb, _ = make(dev, 3, 64, 256, 2)
    xd = dev.upload(np.ones((1, 256), np.float32))
    yd = dev.alloc(128 * 4)
    with pytest.raises(PagodaError):
        ma.gemv_q8act_pair_dev(yd, mb, yd + 256, xd, 256, 1, 128)
    for p in (xd, yd):
        dev.free(p)
    ma.free()
    mb.free()


def test_q8act_rejects_a8(dev):
    from pagoda_amd import Matrix, PagodaError

    m = Matrix.synth(dev, 0, 64, 256, 1, 1, 0.02)
    xd = dev.upload(np.ones((1, 256), np.float32))
    yd = dev.alloc(64 * 4)
    with pytest.raises(PagodaError):
        m.gemv_q8act_dev(xd, 256, 1, yd, 64)
    dev.free(xd)
    dev.free(yd)


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("n_in", [8960, 18944])
def test_q8act_wide_rows_16(dev, fmt, n_in):
    """Down projections of the larger Qwen2 sizes (intermediate 8960: 1.5B,
    18944: 7B): 16 quantized rows of these widths do not fit the LDS at once,
    so the launch takes fewer rows at a time with the same per-row arithmetic."""
    n_out = 256
    m, blk = make(dev, fmt, n_out, n_in, 7 * fmt + n_in % 89)
    x = np.random.default_rng(n_in).normal(0, 1, (16, n_in)).astype(np.float32)
    xd = dev.upload(x)
    yd = dev.alloc(16 * n_out * 4)
    m.gemv_q8act_dev(xd, n_in, 16, yd, n_out)
    y = dev.download(yd, (16, n_out), np.float32)
    assert close(y, oracle_rows(fmt, blk, n_out, n_in, x))
    y1 = dev.alloc(n_out * 4)
    m.gemv_q8act_dev(xd, n_in, 1, y1, n_out)
    np.testing.assert_array_equal(dev.download(y1, (1, n_out), np.float32)[0].view(np.uint32), y[0].view(np.uint32))
    for p in (xd, yd, y1):
        dev.free(p)
    m.free()


def extreme_blocks(rng, fmt, n_out, n_in):
    """Blocks of random bytes (every scale, min and code) at a moderate d, the
    first rows all at the ends of the integer ranges."""
    nsb = (n_in + 255) // 256
    d = np.frombuffer(np.float16(2e-4).tobytes(), np.uint8)
    if fmt == 1:
        b = rng.integers(0, 256, (n_out, nsb, 144)).astype(np.uint8)
        b[0, :, 4:] = 0xFF  # scales and mins 63, codes 15
        b[:, :, 0:2] = b[:, :, 2:4] = d
    else:
        b = rng.integers(0, 256, (n_out, nsb, 210)).astype(np.uint8)
        b[:2, :, :192] = 0  # codes -32
        b[0, :, 192:208] = 0x80  # scales -128
        b[1, :, 192:208] = 0x8F  # -113: -128 and +15 in the two operands
        b[:, :, 208:] = d
    return b


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("n_out,n_in,rows", [
    (40, 320, 1),       # one row; a K tail; partly filled weight tile
    (40, 320, 4),
    (40, 320, 5),       # five and six rows of the vector-ALU kernel
    (40, 320, 6),
    (40, 320, 7),       # the fewest on the matrix cores
    (4000, 5120, 2),    # 20 blocks over 10 waves, two per wave
    (1000, 5120, 6),
    (9728, 512, 2),     # 608 tiles: the matrix cores from 4 rows on
    (33, 4864, 6),      # 19 blocks over 10 waves, 6 rows
    (33, 18944, 2),     # 74 blocks: the most rows whose terms fit the LDS together
    (33, 18944, 3),     # 74 blocks: rows one launch at a time
    (33040, 256, 1),    # more tiles than workgroups
    (16, 256, 16),      # one subtile, one block, one whole activation tile
    (129, 1280, 17),    # one row into the second activation tile
    (3216, 896, 161),   # two activation tiles per workgroup, the last group's second one missing
    (48, 512, 1027),    # rows past one prepared chunk
])
def test_q8act_kernels_match_oracle(dev, fmt, n_out, n_in, rows):
    """Both K-quant kernels: bit-equal to the oracle at the edges of their tiles
    and at the largest integers (class sums of 2^24), and to their pair form."""
    from pagoda_amd import Matrix

    rng = np.random.default_rng(n_out + rows)
    blk = extreme_blocks(rng, fmt, n_out, n_in)
    m = Matrix.upload_kq(dev, fmt, blk, n_out, n_in)
    x = rng.normal(0, 1, (rows, n_in)).astype(np.float32)
    x[0] = 3.0   # every q is -128
    x[1:2] = 0.0
    x[2:3, ::8] = -100.0  # one residue class carries each block
    xd, yd, y2 = dev.upload(x), dev.alloc(rows * n_out * 4), dev.alloc(rows * 2 * n_out * 4)
    ref = oracle_rows(fmt, blk, n_out, n_in, x)
    m.gemv_q8act_dev(xd, n_in, rows, yd, n_out)
    got = dev.download(yd, (rows, n_out), np.float32)
    assert close(got, ref), (np.abs(got - ref).max(), int((got != ref).sum()))
    res = rng.normal(0, 1, (rows, n_out)).astype(np.float32)
    rd = dev.upload(res)
    m.gemv_q8act_dev(xd, n_in, rows, rd, n_out, rd, n_out)
    assert close(dev.download(rd, (rows, n_out), np.float32), res + ref)
    m.gemv_q8act_pair_dev(y2, m, y2 + n_out * 4, xd, n_in, rows, 2 * n_out)
    pair = dev.download(y2, (rows, 2 * n_out), np.float32)
    assert close(pair[:, :n_out], ref) and close(pair[:, n_out:], ref)
    for p in (xd, yd, y2, rd):
        dev.free(p)
    m.free()


@pytest.mark.parametrize("pair", [False, True])
def test_q8act_calls_from_two_threads(dev, pair):
    """Two host threads issue matrix-core launches on one device handle without
    a lock of their own: each call's product takes its own rows' operands,
    whatever the other thread queues meanwhile (other rows, widths and buffer
    sizes). Every output is bit-equal to the same call on one thread."""
    import threading

    from pagoda_amd import Matrix

    calls, jobs, bad = 150, [], []
    for fmt, n_out, n_in, rows, seed in ((1, 48, 1024, 33, 1), (2, 80, 512, 70, 2)):
        m, _ = make(dev, fmt, n_out, n_in, seed)
        x = np.random.default_rng(seed).normal(0, 1, (rows, n_in)).astype(np.float32)
        out = dev.upload(np.zeros((calls + 1, rows, 2, n_out), np.float32))
        jobs.append((m, dev.upload(x), n_in, rows, n_out, out))

    def issue(job, i):
        m, xd, n_in, rows, n_out, out = job
        y = out + i * rows * 2 * n_out * 4
        if pair:
            m.gemv_q8act_pair_dev(y, m, y + n_out * 4, xd, n_in, rows, 2 * n_out)
        else:
            m.gemv_q8act_dev(xd, n_in, rows, y, 2 * n_out)

    def work(job):
        try:
            for i in range(1, calls + 1):
                issue(job, i)
        except Exception as e:  # reported by the main thread
            bad.append(e)

    for job in jobs:
        issue(job, 0)
        dev.sync()
    threads = [threading.Thread(target=work, args=(job,)) for job in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    for m, xd, n_in, rows, n_out, out in jobs:
        got = dev.download(out, (calls + 1, rows, 2, n_out), np.float32).view(np.uint32)
        wrong = [i for i in range(1, calls + 1) if not np.array_equal(got[i], got[0])]
        assert not wrong, wrong
        dev.free(xd)
        dev.free(out)
        m.free()


def test_device_close_gives_scratch_back():
    """Launch scratch is kept per device handle (here the prepared operands of
    1024 rows of 4096, 9 MB a handle) and freed with it."""
    import ctypes as C

    from pagoda_amd import Device, Matrix

    def used():
        free, total = C.c_size_t(), C.c_size_t()
        # the runtime library the backend has loaded
        assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return total.value - free.value

    def run(n):
        devs = [Device("hip") for _ in range(n)]
        for d in devs:
            m = Matrix.synth(d, 1, 16, 4096, 1, 1)
            xd, yd = d.alloc(1024 * 4096 * 4), d.alloc(1024 * 16 * 4)
            m.gemv_q8act_dev(xd, 4096, 1024, yd, 16)
            d.sync()
            m.free()
            d.free(xd)
            d.free(yd)
        held = used()
        for d in devs:
            d.close()
        return held

    run(1)
    before = used()
    held = run(6)
    assert held - before > 48 << 20, (held, before)
    assert used() - before < 16 << 20, (used(), before)
