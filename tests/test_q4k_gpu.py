"""Parity of the gfx950 Q4_K GEMV and activation quantiser against the CPU
oracle (or_quant_q8 restating quant_kernel, src/kernel/q4k_gemv.cu:9-33;
or_gemv_q4k: the dequantised product in double, the value gemv_kernel
q4k_gemv.cu:35-91 computes in fp32).

Quantisation is bit-exact (IEEE divide and round-to-nearest-even on both
sides).  The GEMV sums in fp32 in its own order: the tolerance is 2e-6 of the
row's sum of |terms| (the reference's own self-test allows 1e-5 of one block,
tests/selftest_q4k.cpp:72-74)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_blocks(rng, rows, cols):
    b = rng.integers(0, 256, (rows, cols // 256, 144), dtype=np.uint8)
    b[..., 0:2] = rng.uniform(2e-4, 4e-3, (rows, cols // 256, 1)).astype(np.float16).view(np.uint8)
    b[..., 2:4] = rng.uniform(1e-4, 2e-3, (rows, cols // 256, 1)).astype(np.float16).view(np.uint8)
    return b


def abs_terms(oracle, w, rows, cols, qs, d):
    """sum over k of |w_rk * x_k| (dequantised), for the tolerance"""
    out = np.empty(rows)
    xq = np.abs(qs[0].astype(np.float64) * np.repeat(d[0].astype(np.float64), 32))
    for r in range(rows):
        y = np.concatenate([oracle.q4k_dequant_block(w[r, b]) for b in range(cols // 256)]).astype(np.float64)
        out[r] = np.abs(y) @ xq
    return out


@pytest.mark.parametrize("rows,cols", [(3, 3584), (1, 18944), (2, 256), (4, 32768)])
def test_quant_bit_exact(rows, cols, nova7, oracle):
    nova = nova7
    print(f"[case] quant rows={rows} cols={cols}", flush=True)
    rng = np.random.default_rng(cols + rows)
    x = (rng.standard_normal((rows, cols)) * rng.uniform(0.01, 20, (rows, 1))).astype(np.float32)
    x[0, 64:96] = 0.0                                          # an all-zero block
    dx = nova.upload(x)
    qs, d, s = nova.alloc(rows * cols), nova.alloc(rows * cols // 8), nova.alloc(rows * cols // 4)
    nova.launch_quant_q8(qs.ptr, d.ptr, s.ptr, dx.ptr, rows, cols, None)
    nova.dev_sync()
    rq, rd, rs = oracle.quant_q8(x)
    assert np.array_equal(qs.numpy((rows, cols), np.int8), rq)
    assert np.array_equal(d.numpy((rows, cols // 32), np.float32), rd)
    assert np.array_equal(s.numpy((rows, cols // 16), np.int32), rs)


@pytest.mark.parametrize("rows,cols", [(1, 32), (1, 96), (5, 160), (7, 1056), (33, 992)])
def test_quant_partial_workgroups(rows, cols, nova7, oracle):
    """Blocks that do not fill a wave or a workgroup (8 lanes per block), rows
    whose blocks straddle waves, and nothing written past the last block."""
    nova = nova7
    print(f"[case] quant partial rows={rows} cols={cols}", flush=True)
    rng = np.random.default_rng(rows * 31 + cols)
    x = (rng.standard_normal((rows, cols)) * rng.uniform(1e-3, 50, (rows, 1))).astype(np.float32)
    x[-1, -32:] = 0.0
    n = rows * cols
    dx = nova.upload(x)
    qs, d, s = (nova.upload(np.full(b + 64, 0x5A, np.uint8)) for b in (n, n // 8, n // 4))
    nova.launch_quant_q8(qs.ptr, d.ptr, s.ptr, dx.ptr, rows, cols, None)
    nova.dev_sync()
    rq, rd, rs = oracle.quant_q8(x)
    for buf, ref in ((qs, rq), (d, rd), (s, rs)):
        got = buf.numpy((ref.nbytes + 64,), np.uint8)
        assert np.array_equal(got[:ref.nbytes], np.ascontiguousarray(ref).view(np.uint8).ravel())
        assert np.all(got[ref.nbytes:] == 0x5A)


@pytest.mark.parametrize("rows,cols", [(37, 256), (20, 1536), (512, 3584), (3584, 3584), (50, 5120), (11, 8192),
                                       (70, 8960), (33, 13824), (130, 18944), (9, 32768), (1000, 2560),
                                       (1, 3584), (3, 18944)])
def test_gemv_matches_oracle(rows, cols, nova7, oracle):
    nova = nova7
    print(f"[case] gemv rows={rows} cols={cols}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols)
    w = random_blocks(rng, rows, cols)
    x = rng.standard_normal((1, cols)).astype(np.float32)
    qs, d, s = oracle.quant_q8(x)
    dw, dq, dd, ds = nova.upload(w), nova.upload(qs), nova.upload(d), nova.upload(s)
    out = nova.upload(np.full(rows, np.nan, np.float32))
    nova.launch_gemv_q4k(dw.ptr, rows, cols, dq.ptr, dd.ptr, ds.ptr, out.ptr, None)
    nova.dev_sync()
    got = out.numpy((rows,), np.float32).astype(np.float64)
    ref = oracle.gemv_q4k(w, rows, cols, qs, d, s)
    check = slice(None) if rows <= 600 else slice(0, rows, max(rows // 300, 1))
    scale = abs_terms(oracle, w[check], len(range(rows)[check]), cols, qs, d)
    err = np.abs(got[check] - ref[check])
    assert np.all(np.isfinite(got))
    assert np.all(err <= 2e-6 * scale), f"max err/scale {np.max(err / scale):.2e}"
    print(f"  max |gpu-oracle| / sum|terms| = {np.max(err / scale):.2e}")


@pytest.mark.parametrize("cols,rows", [(3584, (37, 0, 512)), (3584, (3584,)), (18944, (130, 61)), (256, (5, 1, 2, 9)),
                                       (8960, (33, 70)), (32768, (3, 4))])
def test_gemv_f32_fused(cols, rows, nova7, oracle):
    """launch_gemv_q4k_f32 (quantise inside the launch, up to 4 matrices over one
    activation) equals launch_quant_q8 + launch_gemv_q4k per matrix bit for
    bit, and the oracle within the GEMV tolerance."""
    import ctypes as C
    nova = nova7
    print(f"[case] gemv f32 fused cols={cols} rows={rows}", flush=True)
    rng = np.random.default_rng(cols + sum(rows))
    ws = [random_blocks(rng, r, cols) for r in rows]
    x = (rng.standard_normal((1, cols)) * rng.uniform(0.1, 8.0)).astype(np.float32)
    x[0, 64:96] = 0.0                                      # an all-zero 32-block: d = 0
    dx = nova.upload(x)
    dws = [nova.upload(w) if w.size else nova.alloc(16) for w in ws]
    fused = [nova.upload(np.full(max(r, 1), np.nan, np.float32)) for r in rows]
    sep = [nova.upload(np.full(max(r, 1), np.nan, np.float32)) for r in rows]
    n = len(rows)
    bl = (C.c_void_p * n)(*[d.ptr for d in dws])
    rw = (C.c_int64 * n)(*rows)
    ou = (C.c_void_p * n)(*[o.ptr for o in fused])
    nova.launch_gemv_q4k_f32(bl, rw, ou, n, cols, dx.ptr, None)
    qs, dd, ss = nova.alloc(cols), nova.alloc(cols // 8), nova.alloc(cols // 4)
    nova.launch_quant_q8(qs.ptr, dd.ptr, ss.ptr, dx.ptr, 1, cols, None)
    for m, r in enumerate(rows):
        nova.launch_gemv_q4k(dws[m].ptr, r, cols, qs.ptr, dd.ptr, ss.ptr, sep[m].ptr, None)
    nova.dev_sync()
    oq, od, os_ = oracle.quant_q8(x)
    for m, r in enumerate(rows):
        if r == 0:
            assert np.isnan(fused[m].numpy((1,), np.float32)[0])       # nothing written
            continue
        got = fused[m].numpy((r,), np.float32)
        assert np.array_equal(got.view(np.uint32), sep[m].numpy((r,), np.float32).view(np.uint32)), m
        check = slice(None) if r <= 600 else slice(0, r, max(r // 300, 1))
        ref = oracle.gemv_q4k(ws[m], r, cols, oq, od, os_)
        scale = abs_terms(oracle, ws[m][check], len(range(r)[check]), cols, oq, od)
        err = np.abs(got[check].astype(np.float64) - ref[check])
        assert np.all(err <= 2e-6 * scale), f"matrix {m}: max err/scale {np.max(err / scale):.2e}"


@pytest.mark.parametrize("rows,cols", [(37, 256), (512, 3584), (3584, 3584), (130, 18944), (70, 8960),
                                       (33, 13824), (5, 28672), (1, 1536),
                                       # 32M weights and up (ragged 16-row blocks too)
                                       (2051, 16384), (20001, 2048), (18944, 3584), (3584, 18944)])
def test_gemv4_matches_single_token(rows, cols, nova7, oracle):
    """launch_gemv4_q4k (4 stacked tokens, one weight read): every token's
    output within the GEMV tolerance of the oracle, and of launch_gemv_q4k on
    that token (the same terms summed in another order: both kernels are
    within 2e-6 of the row's sum of |terms| of the exact value)."""
    nova = nova7
    print(f"[case] gemv4 rows={rows} cols={cols}", flush=True)
    rng = np.random.default_rng(rows * 13 + cols)
    w = random_blocks(rng, rows, cols)
    x = (rng.standard_normal((4, cols)) * rng.uniform(0.2, 5.0, (4, 1))).astype(np.float32)
    x[2, :32] = 0.0
    qs, d, s = oracle.quant_q8(x)
    dw, dq, dd, ds = nova.upload(w), nova.upload(qs), nova.upload(d), nova.upload(s)
    out4 = nova.upload(np.full(4 * rows + 64, np.nan, np.float32))      # 64 words past the output: left as they are
    nova.launch_gemv4_q4k(dw.ptr, rows, cols, dq.ptr, dd.ptr, ds.ptr, out4.ptr, None)
    singles = []
    for t in range(4):
        o1 = nova.upload(np.full(rows, np.nan, np.float32))
        nova.launch_gemv_q4k(dw.ptr, rows, cols, dq.ptr + t * cols, dd.ptr + t * (cols // 32) * 4,
                             ds.ptr + t * (cols // 16) * 4, o1.ptr, None)
        singles.append(o1)
    nova.dev_sync()
    whole = out4.numpy((4 * rows + 64,), np.float32)
    assert np.all(np.isnan(whole[4 * rows:])), "written past the output"
    got = whole[:4 * rows].reshape(4, rows)
    # every row up to 600, else ~300 spread rows and the last 17 (a ragged last 16-row block)
    check = np.arange(rows) if rows <= 600 else np.unique(np.r_[np.arange(0, rows, rows // 300), np.arange(rows - 17, rows)])
    for t in range(4):
        one = singles[t].numpy((rows,), np.float32)
        ref = oracle.gemv_q4k(w, rows, cols, qs[t:t + 1], d[t:t + 1], s[t:t + 1])
        scale = abs_terms(oracle, w[check], len(check), cols, qs[t:t + 1], d[t:t + 1])
        err = np.abs(got[t][check].astype(np.float64) - ref[check])
        assert np.all(err <= 2e-6 * scale), f"token {t}: max err/scale {np.max(err / scale):.2e}"
        diff = np.abs(got[t][check].astype(np.float64) - one[check])
        assert np.all(diff <= 4e-6 * scale), f"token {t} vs one-token: {np.max(diff / scale):.2e}"


@pytest.mark.parametrize("rows,cols", [(1, 256), (15, 512), (17, 768), (40, 28672), (9301, 1024), (74003, 256)])
def test_gemv4_edges(rows, cols, nova7, oracle):
    """One super-block per row (one wave per 16-row block), ragged last blocks,
    the widest rows, and more blocks than fit at once (a workgroup walks several,
    its last one ragged)."""
    test_gemv4_matches_single_token(rows, cols, nova7, oracle)


@pytest.mark.parametrize("shift", [4, 8])
@pytest.mark.parametrize("rows,cols", [(37, 256), (130, 3584), (33, 18944)])
def test_gemv4_weights_off_16_bytes(rows, cols, shift, nova7, oracle):
    """Weights that do not start on 16 B take the one-token kernel per token:
    its bits for aligned weights, and nothing written past the output."""
    nova = nova7
    print(f"[case] gemv4 rows={rows} cols={cols} weights + {shift} B", flush=True)
    rng = np.random.default_rng(rows + cols + shift)
    w = np.ascontiguousarray(random_blocks(rng, rows, cols)).view(np.uint8).ravel()
    x = rng.standard_normal((4, cols)).astype(np.float32)
    dq, dd, ds = (nova.upload(a) for a in oracle.quant_q8(x))
    aligned, shifted = nova.upload(w), nova.upload(np.concatenate([np.zeros(shift, np.uint8), w]))
    out4 = nova.upload(np.full(4 * rows + 64, np.nan, np.float32))
    one = nova.upload(np.full(4 * rows, np.nan, np.float32))
    nova.launch_gemv4_q4k(shifted.ptr + shift, rows, cols, dq.ptr, dd.ptr, ds.ptr, out4.ptr, None)
    for t in range(4):
        nova.launch_gemv_q4k(aligned.ptr, rows, cols, dq.ptr + t * cols, dd.ptr + t * (cols // 32) * 4,
                             ds.ptr + t * (cols // 16) * 4, one.ptr + t * rows * 4, None)
    nova.dev_sync()
    got, ref = out4.numpy((4 * rows + 64,), np.float32), one.numpy((4 * rows,), np.float32)
    assert np.array_equal(got[:4 * rows].view(np.uint32), ref.view(np.uint32))
    assert np.all(np.isnan(got[4 * rows:]))


@pytest.mark.parametrize("rows,cols,shift", [(1, 256, 1), (9, 4096, 2), (7, 4352, 1), (520, 8192, 4), (20, 8448, 12),
                                             (9, 12544, 8), (17, 16384, 1), (4, 16640, 4), (13, 24576, 2),
                                             (5, 24832, 8), (1030, 28672, 4), (9301, 1024, 4)])
def test_gemv4_off_16_bytes_edges(rows, cols, shift, nova7, oracle):
    """Rows of whole and broken steps of 16 super-blocks, both sides of each
    change of steps and of waves per row, workgroups that are not full, and more
    rows than are resident at once; weights at any byte."""
    test_gemv4_weights_off_16_bytes(rows, cols, shift, nova7, oracle)


def _gemv_us(nova, rows, cols, calls):
    """us per launch of each (entry point, shift): the shortest of ten replays
    over copies of the weights, `shift` bytes off 16, that the last-level cache
    does not hold."""
    n = rows * (cols // 256) * 144
    copies = max(10, -(-380_000_000 // n))
    rng = np.random.default_rng(rows)
    w = nova.upload(rng.integers(0, 64, copies * n + 16, dtype=np.uint8))
    xq = nova.upload(rng.integers(-127, 128, (4, cols), dtype=np.int8))
    xd = nova.upload(np.ones((4, cols // 32), np.float32))
    xs = nova.upload(np.zeros((4, cols // 16), np.int32))
    out = nova.alloc(4 * rows * 4)
    stream = nova.dev_stream_create()
    start, stop = nova.dev_event_create(), nova.dev_event_create()
    us = []
    for launch, shift in calls:
        nova.dev_graph_begin(stream)
        for c in range(copies):
            launch(w.ptr + c * n + shift, rows, cols, xq.ptr, xd.ptr, xs.ptr, out.ptr, stream)
        graph = nova.dev_graph_end(stream)
        took = []
        for _ in range(10):
            nova.dev_event_record(start, stream)
            nova.dev_graph_launch(graph, stream)
            nova.dev_event_record(stop, stream)
            took.append(nova.dev_event_elapsed_ms(start, stop))
        nova.dev_graph_destroy(graph)
        us.append(min(took) * 1e3 / copies)
    nova.dev_event_destroy(start)
    nova.dev_event_destroy(stop)
    nova.dev_stream_destroy(stream)
    return us


@pytest.mark.parametrize("rows,cols", [(18944, 3584), (3584, 18944)])
def test_gemv4_off_16_bytes_reads_weights_once(rows, cols, nova7):
    """Four tokens over weights off 16 B cost less than 2.5 one-token launches
    over the same weights: 1.3 and 1.5 where the weights are read once, 4 where
    the call is four of them."""
    nova = nova7
    print(f"[case] gemv4 one read rows={rows} cols={cols}", flush=True)
    one, four = _gemv_us(nova, rows, cols, [(nova.launch_gemv_q4k, 4), (nova.launch_gemv4_q4k, 4)])
    print(f"  one token {one:.2f} us, four {four:.2f} us")
    assert four < 2.5 * one


@pytest.mark.parametrize("rows,cols", [(512, 18944), (1024, 20480)])
def test_gemv4_few_long_rows_are_spread(rows, cols, nova7):
    """Weights on 16 B are not slower than the same off 16 B, also where there
    are too few 16-row blocks for the chip: 1.0 times as long, 1.3 and 1.4 with
    the blocks' kernel."""
    nova = nova7
    print(f"[case] gemv4 few long rows rows={rows} cols={cols}", flush=True)
    on, off = _gemv_us(nova, rows, cols, [(nova.launch_gemv4_q4k, 0), (nova.launch_gemv4_q4k, 4)])
    print(f"  on 16 B {on:.2f} us, off {off:.2f} us")
    assert on < 1.2 * off


@pytest.mark.parametrize("rows,cols", [(1, 8448), (1024, 8448), (1025, 8448), (1024, 8192), (7, 12288), (1024, 12544),
                                       (1025, 12544), (5, 16384), (1023, 16640), (1025, 16640), (14, 24576), (9, 24832),
                                       (1024, 28672)])
def test_gemv4_few_long_rows(rows, cols, nova7, oracle):
    """Both sides of the lines between the kernel by rows and the one by 16-row
    blocks (33 super-blocks, 1024 rows on 256 CUs) and of its changes of waves
    per row, against the oracle and the one-token kernel."""
    test_gemv4_matches_single_token(rows, cols, nova7, oracle)


@pytest.mark.parametrize("shift", [1, 2, 6])
@pytest.mark.parametrize("rows,cols", [(37, 256), (50, 5120), (33, 13824), (20, 18944)])
def test_gemv_weights_at_any_byte(rows, cols, shift, nova7, oracle):
    """The one-token entry points over weights at any byte: the bits of the same
    weights on 16 B."""
    import ctypes as C
    nova = nova7
    print(f"[case] gemv rows={rows} cols={cols} weights + {shift} B", flush=True)
    rng = np.random.default_rng(rows + cols + shift)
    w = np.ascontiguousarray(random_blocks(rng, rows, cols)).view(np.uint8).ravel()
    x = rng.standard_normal((1, cols)).astype(np.float32)
    dx = nova.upload(x)
    dq, dd, ds = (nova.upload(a) for a in oracle.quant_q8(x))
    got = []
    for off in (0, shift):
        dw = nova.upload(np.concatenate([np.zeros(off, np.uint8), w]))
        out, out32 = (nova.upload(np.full(rows, np.nan, np.float32)) for _ in range(2))
        nova.launch_gemv_q4k(dw.ptr + off, rows, cols, dq.ptr, dd.ptr, ds.ptr, out.ptr, None)
        nova.launch_gemv_q4k_f32((C.c_void_p * 1)(dw.ptr + off), (C.c_int64 * 1)(rows), (C.c_void_p * 1)(out32.ptr),
                                 1, cols, dx.ptr, None)
        nova.dev_sync()
        got.append([o.numpy((rows,), np.uint32) for o in (out, out32)])
    assert np.isfinite(got[0][0].view(np.float32)).all()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
