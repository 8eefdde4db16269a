"""GPU parity of the quantized prefill projection (Q4_K GEMM on the matrix cores)
against the CPU oracle: prefill = the Q4_K matvec applied per token
(LC/src/cpu/ops/q4k_matvec.rs:31-90, the Metal prefill loop LC/src/metal/prefill.rs:21-110).

Bar: max|gpu - cpu| / max|cpu| <= 1e-3 over the checked token rows (fp16 operands with
f32 accumulation; measured ~1e-4)."""
import numpy as np
import pytest

import larql_hip
import oracle

pytestmark = pytest.mark.gpu

REL_TOL = 1e-3


def rel_err(got, ref):
    return float(np.max(np.abs(got.astype(np.float64) - ref)) / max(np.max(np.abs(ref)), 1e-30))


def check_rows(q4k, x, got, rows, cols, token_rows):
    errs = []
    for t in token_rows:
        ref = oracle.q4k_matvec(q4k, x[t], rows, cols)
        errs.append(rel_err(got[t], ref))
    e = max(errs)
    print(f"  rel_err max over {len(token_rows)} tokens = {e:.3e}", flush=True)
    assert e <= REL_TOL, e


@pytest.mark.parametrize("rows,cols,m", [(300, 512, 37), (1000, 2560, 130), (64, 256, 2), (129, 768, 129),
                                         (300, 512, 700), (72, 256, 1030), (1000, 2560, 513)])
def test_q4k_matmul_small_shapes(hip, rows, cols, m):
    print(f"[prefill] rows={rows} cols={cols} m={m}", flush=True)
    w = oracle.gauss(61, rows * cols, 0.0, 0.02)
    q4k = oracle.quantize_q4_k(w)
    x = oracle.gauss(62, m * cols).reshape(m, cols)
    got = hip.q4k_matmul(q4k, x, rows, cols)
    check_rows(q4k, x, got, rows, cols, range(m))


def test_q4k_matmul_fuzzed_bytes(hip):
    """Random 148-byte blocks (all nibbles and scale codes), bounded f16 d / dmin."""
    rows, cols, m = 200, 1024, 70
    rng = np.random.default_rng(63)
    q4k = rng.integers(0, 256, size=rows * cols // 256 * 148, dtype=np.uint8)
    blocks = q4k.reshape(-1, 148)
    dd = rng.uniform(-0.01, 0.01, size=(blocks.shape[0], 2)).astype(np.float16)
    blocks[:, 0:4] = dd.view(np.uint8).reshape(-1, 4)
    x = oracle.gauss(64, m * cols).reshape(m, cols)
    got = hip.q4k_matmul(q4k, x, rows, cols)
    check_rows(q4k, x, got, rows, cols, range(m))


def test_q4k_prefill_512_tokens_full_shape(hip):
    """The prefill workload: Q4_K W [10240 x 2560] from N(0, 0.02), X [512 x 2560] N(0,1),
    through the device path (matvec_dev with m = 512); every token row is checked against
    the oracle (its matvecs spread over the host's threads)."""
    torch = pytest.importorskip("torch")
    rows, cols, m = 10240, 2560, 512
    w = oracle.gauss(71, rows * cols, 0.0, 0.02)
    q4k = oracle.quantize_q4_k(w)
    x = oracle.gauss(72, m * cols).reshape(m, cols)
    h = hip.register_weight(larql_hip.Q4_K, q4k, rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        got = dy.cpu().numpy().reshape(m, rows)
        assert np.all(np.isfinite(got))
        import os
        from concurrent.futures import ThreadPoolExecutor

        with ThreadPoolExecutor(max(1, min(16, len(os.sched_getaffinity(0))))) as pool:
            errs = list(pool.map(lambda t: rel_err(got[t], oracle.q4k_matvec(q4k, x[t], rows, cols)), range(m)))
        e = max(errs)
        print(f"  rel_err max over all {m} tokens = {e:.3e}", flush=True)
        assert e <= REL_TOL, e
    finally:
        hip.release_weight(h)


def test_q4k_matmul_m1_equals_matvec(hip):
    rows, cols = 512, 1024
    q4k = oracle.quantize_q4_k(oracle.gauss(81, rows * cols, 0.0, 0.02))
    x = oracle.gauss(82, cols)
    a = hip.q4k_matmul(q4k, x[None, :], rows, cols)[0]
    b = hip.q4k_matvec(q4k, x, rows, cols)
    np.testing.assert_array_equal(a, b)


# (4096, 14336, 64): the Llama-3-8B down projection; (300, 512, 37): a ragged tile; (70, 1024,
# 9, scaled): token rows scaled by 1e6 .. 1e-30, far outside fp16 (the GEMM's operand pairs
# are fp16: each row must be brought into range by its own power of two), and a zero row
# the others: the edges of 16-token tiles and of one to three tiles per workgroup, of 16-row
# tiles and 256-row workgroups, and K split over 1 .. 16 workgroups
@pytest.mark.parametrize("rows,cols,m,scaled", [(4096, 14336, 64, False), (300, 512, 37, False), (70, 1024, 9, True),
                                                (300, 256, 16, False), (70, 512, 17, False), (257, 1024, 48, False),
                                                (64, 256, 49, False), (1, 4096, 33, False), (272, 2304, 97, False),
                                                (520, 4352, 2, False)])
def test_q6k_gemm_rows_match_matvec_oracle(hip, rows, cols, m, scaled):
    """The Q6_K f32-accuracy GEMM of the prompt pass (matvec_dev with m > 1 on a Q6_K handle)
    at the Llama-3-8B down-projection shape: every token row against the oracle's Q6_K
    matvec (LC/src/cpu/ops/q6k_matvec.rs), within 1e-3 (fp16 operand pairs: measured ~1e-6)."""
    import os
    from concurrent.futures import ThreadPoolExecutor

    torch = pytest.importorskip("torch")
    print(f"[q6k gemm] rows={rows} cols={cols} m={m} scaled={scaled}", flush=True)
    q6k = oracle.quantize_q6_k(oracle.gauss(91, rows * cols, 0.0, 0.02))
    x = oracle.gauss(92, m * cols).reshape(m, cols)
    if scaled:
        f = np.array([1e6, 1e3, 3e4, 1.0, 1e-3, 1e-8, 1e-20, 1e-30, 0.0], np.float32)
        x = (x * f[:, None]).astype(np.float32)
    h = hip.register_weight(larql_hip.Q6_K, q6k, rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        got = dy.cpu().numpy().reshape(m, rows)
        with ThreadPoolExecutor(max(1, min(16, len(os.sched_getaffinity(0))))) as pool:
            refs = list(pool.map(lambda t: oracle.q6k_matvec(q6k, x[t], rows, cols), range(m)))
        errs = [rel_err(got[t], refs[t]) if np.any(refs[t]) else float(np.max(np.abs(got[t]))) for t in range(m)]
        e = max(errs)
        print(f"  rel_err max over all {m} tokens = {e:.3e}", flush=True)
        assert e <= REL_TOL, e
    finally:
        hip.release_weight(h)
        hip.forget_host(q6k)


def _q4k_values(b, rows, cols):
    """d, dmin, scales, mins and codes of 148-byte blocks -> f64 weights."""
    b = b.reshape(-1, 148)
    d, dmin = (b[:, i:i + 2].copy().view(np.float16).astype(np.float64) for i in (0, 2))
    sc = (b[:, 4:12] & 63).astype(np.float64)
    mn = np.concatenate([b[:, 16:20] & 15, b[:, 16:20] >> 4], 1).astype(np.float64)
    q = np.stack([b[:, 20:] & 15, b[:, 20:] >> 4], -1).reshape(-1, 8, 32).astype(np.float64)
    return (q * (d * sc)[..., None] - (dmin * mn)[..., None]).reshape(rows, cols)


# 2 .. 64 tokens, odd row counts, one super-block, K split over up to 16 workgroups, rows of more
# than 16384 (packed by the separate kernels); the larger shapes are those the small-batch route takes
@pytest.mark.parametrize("rows,cols,m", [(300, 4096, 2), (4096, 4096, 16), (1000, 2560, 17), (257, 14336, 33),
                                         (4096, 8192, 48), (130, 4352, 64), (64, 17408, 5), (14336, 4096, 6)])
def test_q4k_small_batch_rows(hip, rows, cols, m):
    """Small batches of Q4_K (matvec_dev, the f32-accuracy GEMM): every output against the f64
    product of the dequantized weights.  One token scaled by 1e6 and one by 1e-20 (each row has its
    own power of two), and super-blocks with a minimum scale of 300, past the range of the usual
    fp16 minimum operand.  The weight rows with such a block and the others are compared apart, each
    with the rms of its own outputs: 4e-6 (an error of 2.3e-7 of the norm, normal over up to 14336
    outputs, and f32 sums; for the former, whose outputs are the few large minima, 1e-5)."""
    torch = pytest.importorskip("torch")
    print(f"[q4k small] rows={rows} cols={cols} m={m}", flush=True)
    b = oracle.quantize_q4_k(oracle.gauss(95, rows * cols, 0.0, 0.02)).reshape(-1, 148).copy()
    b[5::97, 2:4] = np.array([300.0], np.float16).view(np.uint8)
    large = np.zeros(rows, bool)
    large[np.arange(5, rows * (cols // 256), 97) // (cols // 256)] = True
    x = oracle.gauss(96, m * cols).reshape(m, cols).copy()
    x[0] *= np.float32(1e6)
    x[m - 1] *= np.float32(1e-20)
    h = hip.register_weight(larql_hip.Q4_K, b.reshape(-1), rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        got = dy.cpu().numpy().reshape(m, rows).astype(np.float64)
        ref = x.astype(np.float64) @ _q4k_values(b, rows, cols).T
        assert not np.all(large)
        for which, bar in ((~large, 4e-6), (large, 1e-5)):
            e = np.max(np.abs(got - ref)[:, which], 1) / np.sqrt(np.mean(ref[:, which] ** 2, 1))
            print(f"  {which.sum()} weight rows: {np.max(e):.2e}", flush=True)
            assert np.max(e) <= bar
    finally:
        hip.release_weight(h)


def test_q4k_small_batch_infinite_elements(hip):
    """A token with one infinite element: every output is that infinity times the sign of its weight
    (as the f32 sum gives it), the other tokens' outputs are unaffected; a NaN makes its token NaN."""
    torch = pytest.importorskip("torch")
    rows, cols, m = 4096, 4096, 4
    b = oracle.quantize_q4_k(oracle.gauss(97, rows * cols, 0.0, 0.02))
    W = _q4k_values(b, rows, cols)
    x = oracle.gauss(98, m * cols).reshape(m, cols).copy()
    x[1, 77] = np.inf
    x[2, 1000] = np.nan
    h = hip.register_weight(larql_hip.Q4_K, b, rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        got = dy.cpu().numpy().reshape(m, rows)
        clear = np.abs(W[:, 77]) > 1e-6   # (a weight at the rounding of zero may have either sign)
        assert clear.mean() > 0.99
        np.testing.assert_array_equal(got[1][clear], np.sign(W[clear, 77]) * np.inf)
        assert np.all(np.isnan(got[2]))
        for t in (0, 3):
            ref = x[t].astype(np.float64) @ W.T
            assert np.max(np.abs(got[t] - ref)) <= 1e-5 * np.max(np.abs(ref))
    finally:
        hip.release_weight(h)


@pytest.mark.parametrize("cols,m", [(4096, 4), (14336, 17), (2048, 40)])
def test_q4k_f32_gemm_keeps_f32_accuracy(hip, cols, m):
    """Ordinary tokens and weights through the f32-accuracy GEMM: 4e-7 of the output's norm (the pair's
    2^-22, and f32 sums: a few 2^-24 of terms about three times the weights, whose codes and minima
    are multiplied apart).  Operands below fp16's normal range cost the matrix cores' sums 1.9e-6 at
    4096."""
    torch = pytest.importorskip("torch")
    rows = 512
    b = oracle.quantize_q4_k(oracle.gauss(103, rows * cols, 0.0, 0.02))
    x = oracle.gauss(104, m * cols).reshape(m, cols)
    h = hip.register_weight(larql_hip.Q4_K, b, rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        ref = x.astype(np.float64) @ _q4k_values(b, rows, cols).T
        e = np.linalg.norm(dy.cpu().numpy().reshape(m, rows) - ref) / np.linalg.norm(ref)
        print(f"[f32 gemm] cols={cols} m={m}: {e:.2e}", flush=True)
        assert e <= 4e-7
    finally:
        hip.release_weight(h)


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
@pytest.mark.parametrize("col", [518, 519])
def test_f32_gemm_rows_with_an_outlier(hip, fmt, col):
    """A token whose largest element (1e6, ordinary ones ~1) meets only zero weights: the elements are
    held to 2^-24 in units that put the largest in [2^14, 2^15), here 2^-19, at even and odd
    positions alike, so the error grows over the same token's without it by 2^-19 / sqrt(12) =
    5.5e-7 of the output's norm; twice that."""
    torch = pytest.importorskip("torch")
    rows, cols, m = 256, 4096, 4
    w = oracle.gauss(101, rows * cols, 0.0, 0.02)
    sb, e = divmod(col, 256)
    if fmt == "q4_k":
        b = oracle.quantize_q4_k(w).reshape(rows, cols // 256, 148).copy()
        b[:, :, 2:4] = 0                                    # no minima (their sums have a step of their own)
        b[:, sb, 20 + e // 2] &= 0x0F if e % 2 else 0xF0    # code 0
        W = _q4k_values(b, rows, cols)
    else:
        b = oracle.quantize_q6_k(w).reshape(rows, cols // 256, 210).copy()
        b[:, sb, e // 2] &= 0x0F if e % 2 else 0xF0         # code 32: nibble 0, high bits 2
        b[:, sb, 128 + e // 4] = (b[:, sb, 128 + e // 4] & (0xFF ^ (3 << (2 * (e % 4))))) | (2 << (2 * (e % 4)))
        p = b.reshape(-1, 210)
        q = np.stack([p[:, :128] & 15, p[:, :128] >> 4], -1).reshape(-1, 256).astype(np.float64)
        q += 16.0 * np.stack([(p[:, 128:192] >> (2 * i)) & 3 for i in range(4)], -1).reshape(-1, 256) - 32.0
        d = p[:, 208:210].copy().view(np.float16).astype(np.float64)
        W = (q.reshape(-1, 16, 16) * (p[:, 192:208].copy().view(np.int8) * d)[..., None]).reshape(rows, cols)
    assert np.all(W[:, col] == 0)
    x = oracle.gauss(102, m * cols).reshape(m, cols).copy()
    h = hip.register_weight(larql_hip.Q4_K if fmt == "q4_k" else larql_hip.Q6_K, b.reshape(-1), rows, cols)

    def error():
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        ref = x.astype(np.float64) @ W.T
        return np.linalg.norm(dy.cpu().numpy().reshape(m, rows) - ref) / np.linalg.norm(ref)

    try:
        x[:, col] = 1.0
        plain = error()
        x[:, col] = 1e6
        outlier = error()
        print(f"[outlier] {fmt} col={col}: {plain:.2e} -> {outlier:.2e}", flush=True)
        assert outlier <= plain + 1.1e-6
    finally:
        hip.release_weight(h)


@pytest.mark.parametrize("rows,cols,m", [(4096, 4096, 4), (257, 14336, 5), (130, 4352, 3)])
def test_q4k_small_batch_nonfinite_sums(hip, rows, cols, m):
    """Tokens whose packed operands overflow, rows of any width: several infinities of either sign (each
    output their products' sum: an infinity, or NaN where they disagree or meet a zero weight), a token
    of infinities only, one whose largest element is next to f32's limit (finite outputs), beside
    ordinary ones."""
    torch = pytest.importorskip("torch")
    b = oracle.quantize_q4_k(oracle.gauss(105, rows * cols, 0.0, 0.02))
    W = _q4k_values(b, rows, cols)
    x = oracle.gauss(106, m * cols).reshape(m, cols).copy()
    x[0, [3, 700]] = np.inf
    x[1, [9, 256]], x[1, 1029] = -np.inf, np.inf
    x[2, 77] = np.float32(3.4025e38)
    if m > 3:
        x[3] = np.inf
    h = hip.register_weight(larql_hip.Q4_K, b, rows, cols)
    try:
        dx = torch.from_numpy(x).cuda()
        dy = torch.empty(m * rows, device="cuda", dtype=torch.float32)
        hip.matvec_dev(h, dx, dy, m=m)
        hip.synchronize()
        got = dy.cpu().numpy().reshape(m, rows)
        for t in range(m):
            inf = np.flatnonzero(np.isinf(x[t]))
            if inf.size:
                clear = np.all(np.abs(W[:, inf]) > 1e-6, 1) if inf.size < 9 else np.ones(rows, bool)
                with np.errstate(invalid="ignore"):
                    want = np.sum(np.sign(np.float32(W[:, inf])) * x[t, inf], 1)
                np.testing.assert_array_equal(got[t][clear], want[clear].astype(np.float32))
            else:   # (the plain sum's order: 2^-24 per term, random signs)
                ref = x[t].astype(np.float64) @ W.T
                assert np.max(np.abs(got[t] - ref)) <= 1e-5 * np.max(np.abs(ref)), t
    finally:
        hip.release_weight(h)


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_q4k_small_batch_with_one_nonfinite_token_is_no_slow_path(hip, value):
    """One infinite or NaN token among six costs its share of a pass over the weights' scales, not a
    serial sum per output (30 times the call): less than three times the ordinary call."""
    torch = pytest.importorskip("torch")
    rows, cols, m = 14336, 4096, 6
    h = hip.register_weight(larql_hip.Q4_K, oracle.quantize_q4_k(oracle.gauss(107, rows * cols, 0.0, 0.02)), rows, cols)
    stream = torch.cuda.Stream()
    out = torch.empty(m * rows, device="cuda", dtype=torch.float32)

    def us(x):
        dx = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        best = np.inf
        for _ in range(5):
            a, b = torch.cuda.Event(True), torch.cuda.Event(True)
            a.record(stream)
            for _ in range(10):
                hip.matvec_dev(h, dx, out, m=m, stream=stream)
            b.record(stream)
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best

    try:
        x = oracle.gauss(108, m * cols).reshape(m, cols).copy()
        plain = us(x)
        x[2, 1500] = value
        other = us(x)
        print(f"[nonfinite token] {value}: {plain:.1f} -> {other:.1f} us", flush=True)
        assert other <= 3 * plain
    finally:
        hip.release_weight(h)


@pytest.mark.parametrize("m", [6, 700])
def test_q4k_batches_above_2gib_are_refused(hip, m):
    """Q4_K weights whose nibbles fill 2 GiB: both GEMMs of several rows say so, whatever the batch."""
    torch = pytest.importorskip("torch")
    rows, cols = 1048577, 4096
    raw = torch.zeros(rows * (cols // 256) * 148, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    h = hip.register_weight_device(larql_hip.Q4_K, raw, raw.numel(), rows, cols)
    del raw
    try:
        x = torch.ones(m, cols, device="cuda")
        out = torch.empty(m, rows, device="cuda")
        torch.cuda.synchronize()
        with pytest.raises(larql_hip.LarqlHipError, match="2 GiB"):
            hip.matvec_dev(h, x, out, m=m)
    finally:
        hip.synchronize()
        hip.release_weight(h)
        torch.cuda.empty_cache()


def test_q4k_batch_workspace_grows_only_with_the_batch(hip):
    """A context whose largest batch of a Q4_K weight has run allocates nothing for smaller ones, though
    their K splits differ, so they record into a HIP graph; three replays with eager work between
    them give the eager results."""
    torch = pytest.importorskip("torch")
    rows, cols, sizes = 14336, 4096, (2, 16, 33, 48, 64, 96)
    be = larql_hip.HipBackend(0, strict=True)
    h = be.register_weight(larql_hip.Q4_K, oracle.quantize_q4_k(oracle.gauss(109, rows * cols, 0.0, 0.02)), rows, cols)
    try:
        x = torch.from_numpy(oracle.gauss(110, 512 * cols).reshape(512, cols)).cuda()
        out, ref = (torch.empty(512, rows, device="cuda") for _ in range(2))
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        be.matvec_dev(h, x, out, m=512, stream=side)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for m in sizes:
            be.matvec_dev(h, x, ref, m=m, stream=side)
            torch.cuda.synchronize()
            assert torch.cuda.mem_get_info()[0] == free, m
        for m in sizes:
            print(f"[q4k graph] m={m}", flush=True)
            be.matvec_dev(h, x, ref, m=m, stream=side)
            torch.cuda.synchronize()
            want = ref[:m].clone()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                be.matvec_dev(h, x, out, m=m, stream=side)
            for _ in range(3):
                out.fill_(7.0)
                be.matvec_dev(h, x, ref, m=64, stream=side)
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(out[:m], want)
            del graph
    finally:
        be.synchronize()
        be.close()
