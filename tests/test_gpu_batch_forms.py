"""The batched forms that read the weights once for many vectors: Q8_0 / Q4_0 / Q5_0 on the matrix cores
(k_gemv_int), and the fp32-activation kernels (k_gemv_float, k_gemv_float_many): unquantised weights, and block
formats at alignments and row pitches the integer kernels do not take.  Batches are bit-identical to single
vectors, and within the GEMV bar of the fp64 oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import qorvix_amd as qvx
from conftest import max_rel
from test_gpu_kernels import dev, f32bits, random_weight

pytestmark = pytest.mark.gpu

GEMV_TOL = 1e-3
# fp32 activations and exact weight values: a lane's sum is one chain of FMAs over its chunks, K / 64 of them, and
# 6 tree adds follow, so an output's error is at most (K / 64 + 6) 2^-24 sum |w x|; sum |w x| <= 0.4 sqrt(K) max |ref|
# for these inputs, so 178 * 6e-8 * 42 = 4.5e-4 of max |ref| at K = 11008.  Such a bound assumes that every rounding
# errs the same way; they are held to a fifth of it.
FP32_TOL = 9e-5


def _run(torch, w, t, X, rows, cols, bias=None):
    n = X.shape[0]
    out = torch.full((n, rows), float("nan"), dtype=torch.float32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    rc = qvx.qmatmul_n_bias(out.data_ptr(), w.data_ptr(), t, X.data_ptr(), bias.data_ptr() if bias is not None else 0,
                            n, rows, cols, st)
    assert rc == qvx.OK, qvx.strerror(rc)
    return out


def _singles(torch, w, t, X, rows, cols, which):
    return torch.cat([_run(torch, w, t, X[i:i + 1].contiguous(), rows, cols) for i in which])


def _check(torch, t, rows, cols, n, seed, bias=False, zero_vec=False, tol=GEMV_TOL, offset=0):
    rng = np.random.default_rng(seed)
    w_np = random_weight(t, rows, cols, rng)
    X_np = rng.standard_normal((n, cols)).astype(np.float32)
    if zero_vec:
        X_np[1] = 0.0
    w, X = dev(torch, np.concatenate([np.zeros(offset, np.uint8), w_np]))[offset:], dev(torch, X_np)
    got = _run(torch, w, t, X, rows, cols)
    which = sorted({0, min(1, n - 1), n // 2, max(n - 2, 0), n - 1})
    one = _singles(torch, w, t, X, rows, cols, which)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(f32bits(got[which].cpu().numpy()), f32bits(one.cpu().numpy()))
    ref = oracle.matmul_f64(w_np, t, X_np[which], len(which), rows, cols)
    assert max_rel(got[which].cpu().numpy(), ref) <= tol
    if bias:
        b = dev(torch, rng.standard_normal(rows).astype(np.float32))
        gb = _run(torch, w, t, X, rows, cols, b)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(f32bits(gb.cpu().numpy()), f32bits((got + b).cpu().numpy()))


# Slots of 64 elements: a short row's padded tree (4 of 8, 12 of 16, 20 of 32, 40 of 64); exactly one 64-slot block;
# four slots past it; several blocks with a partial last one.  (A row of 1, 6 or 65 slots is no multiple of 16 bytes: those
# cases run on the fp32-activation kernels.)  Rows: one, ragged, whole tiles.  Vectors: the fewest (9, or 5 or 7 on large
# weights), one tile, one past it, several workgroups; few waves take the K parts, many do not.
INT_CASES = [(3, 256, 9), (33, 768, 20), (31, 4352, 18), (8200, 4096, 8), (5000, 14336, 6), (5000, 14336, 8),
             (1, 64, 9), (4, 512, 12), (36, 2560, 16), (4200, 4096, 5), (8200, 4096, 7), (1, 64, 17), (33, 384, 20), (40, 1280, 33), (64, 4096, 17), (70, 4096, 65), (31, 4160, 18),
             (100, 11008, 24), (1030, 4096, 70), (2080, 1024, 130), (1100, 4096, 260)]


@pytest.mark.parametrize("t", [qvx.Q8_0, qvx.Q4_0, qvx.Q5_0])
@pytest.mark.parametrize("rows,cols,n", INT_CASES)
def test_int_batches_match_single_vectors(cuda, t, rows, cols, n):
    _check(cuda, t, rows, cols, n, seed=rows + cols + n, bias=True, zero_vec=True)


def test_int_batch_in_parts(cuda):
    """A batch whose converted activations pass the workspace's bound runs in parts of 992 vectors (32768 columns), the
    last one ragged: bit-identical to single vectors around the parts' edge, eagerly with a bias and in a plan."""
    from qorvix_amd import decode
    rng = np.random.default_rng(9)
    t, rows, cols, n = qvx.Q4_0, 33, 32768, 1003
    w = dev(cuda, random_weight(t, rows, cols, rng))
    X = cuda.randn(n, cols, device="cuda", generator=cuda.Generator(device="cuda").manual_seed(1))
    bias = dev(cuda, rng.standard_normal(rows).astype(np.float32))
    which = [0, 15, 16, 990, 991, 992, 993, 1001, 1002]
    one = _singles(cuda, w, t, X, rows, cols, which)
    got = _run(cuda, w, t, X, rows, cols, bias)
    np.testing.assert_array_equal(f32bits(got[which].cpu().numpy()), f32bits((one + bias).cpu().numpy()))
    out = cuda.empty((n, rows), dtype=cuda.float32, device="cuda")
    plan = decode.Plan()
    plan.add(out, decode.DevWeight(w, t, rows, cols), X, n)
    plan.instantiate()
    for _ in range(3):
        out.fill_(float("nan"))
        plan.launch(cuda.cuda.current_stream().cuda_stream)
        cuda.cuda.synchronize()
        np.testing.assert_array_equal(f32bits(out[which].cpu().numpy()), f32bits(one.cpu().numpy()))
    plan.close()


def test_int_batch_keeps_non_finite_vectors_apart(cuda):
    """A non-finite activation makes its own vector's outputs NaN and leaves the tile's other vectors as they
    are."""
    rng = np.random.default_rng(3)
    t, rows, cols, n = qvx.Q8_0, 50, 512, 19
    w_np = random_weight(t, rows, cols, rng)
    X_np = rng.standard_normal((n, cols)).astype(np.float32)
    w = dev(cuda, w_np)
    clean = _run(cuda, w, t, dev(cuda, X_np), rows, cols).cpu().numpy()
    X_np[3, 7], X_np[16, 500] = np.inf, np.nan
    got = _run(cuda, w, t, dev(cuda, X_np), rows, cols).cpu().numpy()
    assert np.isnan(got[[3, 16]]).all()
    keep = [i for i in range(n) if i not in (3, 16)]
    np.testing.assert_array_equal(f32bits(got[keep]), f32bits(clean[keep]))


# Slots a row: 4 of 8, 12 of 16, one whole block of 64, two blocks and 44 of 64.
@pytest.mark.parametrize("t", [qvx.Q8_0, qvx.Q4_0, qvx.Q5_0])
@pytest.mark.parametrize("cols", [256, 768, 4096, 11008])
def test_int_batch_non_finite_scales(cuda, t, cols):
    """Infinite and NaN block scales, also in a row's last slot (whose sum the padding lanes mirror), give a
    batch what they give single vectors, and leave other rows as they are."""
    rng = np.random.default_rng(cols)
    rows, n = 37, 19
    nb = qvx.row_bytes(t, cols) // (cols // 32)  # a block starts with its fp16 scale
    w_np = random_weight(t, rows, cols, rng).reshape(rows, cols // 32, nb)
    X = dev(cuda, rng.standard_normal((n, cols)).astype(np.float32))
    clean = _run(cuda, dev(cuda, w_np.reshape(-1)), t, X, rows, cols).cpu().numpy()
    bad = {3: (-1, np.inf), 8: (-2, -np.inf), 9: (-1, np.nan), 21: (0, np.inf), 36: (-1, -np.inf)}
    for r, (block, scale) in bad.items():
        w_np[r, block, :2] = np.array([scale], np.float16).view(np.uint8)
    w = dev(cuda, w_np.reshape(-1))
    got = _run(cuda, w, t, X, rows, cols).cpu().numpy()
    one = _singles(cuda, w, t, X, rows, cols, range(n)).cpu().numpy()
    np.testing.assert_array_equal(got, one)  # NaN at the same places
    assert not np.isfinite(got[:, list(bad)]).any()
    keep = [r for r in range(rows) if r not in bad]
    np.testing.assert_array_equal(f32bits(got[:, keep]), f32bits(clean[:, keep]))


# Chunks of 16 bytes: less than a segment of 64, a partial one, one segment (fp16), one chunk past it, more than a
# stage of two segments; rows and vectors around the tiles of 32 x 8.
FLOAT_CASES = [(1, 8, 9), (33, 40, 9), (17, 384, 20), (48, 512, 33), (65, 520, 64), (40, 1536, 31), (1040, 384, 1030)]


@pytest.mark.parametrize("t", [qvx.F16, qvx.BF16, qvx.F32])
@pytest.mark.parametrize("rows,cols,n", FLOAT_CASES)
def test_float_batches_match_single_vectors(cuda, t, rows, cols, n):
    _check(cuda, t, rows, cols, n, seed=rows + cols + n, bias=True, zero_vec=True)


# Block formats on the fp32-activation kernels: the types no integer kernel computes, row pitches that are
# not multiples of 16 bytes (Q6_K rows of an odd number of super-blocks lie at 2-byte offsets), and weights
# whose first byte is unaligned.  K: less than a segment of 512, a partial last one, many.
LOOSE_CASES = [(qvx.Q6_K, 1, 256, 0), (qvx.Q6_K, 37, 768, 0), (qvx.Q6_K, 300, 5632, 0), (qvx.Q6_K, 70, 11008, 0),
               (qvx.Q6_K, 33, 2048, 2), (qvx.Q8_0, 45, 96, 0), (qvx.Q8_0, 130, 4128, 0), (qvx.Q4_0, 45, 192, 0),
               (qvx.Q5_0, 77, 832, 0), (qvx.Q4_1, 50, 1056, 0), (qvx.Q5_1, 50, 544, 0), (qvx.Q8_1, 50, 4096, 0),
               (qvx.Q4_K, 40, 1280, 1), (qvx.Q5_K, 40, 1280, 4), (qvx.F16, 40, 520, 2), (qvx.BF16, 40, 520, 2),
               (qvx.F32, 40, 520, 4)]


@pytest.mark.parametrize("t,rows,cols,offset", LOOSE_CASES)
@pytest.mark.parametrize("n", [1, 3, 9, 70])
def test_loose_blocks(cuda, t, rows, cols, offset, n):
    _check(cuda, t, rows, cols, n, seed=rows + cols + n, bias=True, tol=FP32_TOL, offset=offset)


# The formats whose values are a code (less an offset) times a scale: the block's bytes up to its codes, and the
# whole block as bytes that make every value positive under a positive scale.
POSITIVE = {qvx.Q8_0: (2, 5), qvx.Q8_1: (4, 5), qvx.Q4_0: (2, 0xFF), qvx.Q5_0: (2, 0xFF)}


@pytest.mark.parametrize("t", [*POSITIVE, qvx.Q6_K])
@pytest.mark.parametrize("n", [1, 3, 9])
def test_loose_blocks_infinite_scales(cuda, t, n):
    """An infinite scale over codes of one sign makes the outputs infinite, not NaN, on the fp32-activation
    kernels: each value is its code times the scale, as the block formats define it."""
    rng = np.random.default_rng(n)
    rows, cols, offset = 40, 768, 2
    w_np = random_weight(t, rows, cols, rng)
    if t == qvx.Q6_K:
        b = w_np.reshape(rows, 3, 210)
        for r, sc in ((2, 1), (3, 0xFF)):  # scales +1 and -1
            b[r, 1, :192], b[r, 1, 192:208] = 0xFF, sc
            b[r, 1, 208:] = np.array([np.inf], np.float16).view(np.uint8)
    else:
        at, code = POSITIVE[t]
        b = w_np.reshape(rows, cols // 32, -1)
        for r, d in ((2, np.inf), (3, -np.inf)):
            b[r, 5, at:] = code
            b[r, 5, :2] = np.array([d], np.float16).view(np.uint8)
    X_np = (np.abs(rng.standard_normal((n, cols))) + 0.1).astype(np.float32)
    w = dev(cuda, np.concatenate([np.zeros(offset, np.uint8), w_np]))[offset:]
    got = _run(cuda, w, t, dev(cuda, X_np), rows, cols).cpu().numpy()
    assert (got[:, 2] == np.inf).all() and (got[:, 3] == -np.inf).all()
    assert np.isfinite(np.delete(got, [2, 3], axis=1)).all()


@pytest.mark.parametrize("t", [qvx.Q4_1, qvx.F16])
@pytest.mark.parametrize("n", [1, 2, 3, 7])
def test_loose_rows_past_the_staging_budget(cuda, t, n):
    """Rows of more than 32768 elements read their activations from global memory, up to four vectors a launch."""
    _check(cuda, t, 5, 33024, n, seed=5, tol=3e-4, bias=True)


# Around the tiled form's lines (9 vectors; 5 on 8192 rows), and 3 and 5 to 8 vectors a launch on short rows.
@pytest.mark.parametrize("t", [qvx.F16, qvx.Q4_1])
@pytest.mark.parametrize("rows,cols,n", [(8191, 64, 5), (8192, 64, 5), (8193, 1056, 8), (700, 1024, 8), (65, 1024, 3),
                                         (65, 1056, 3), (1, 64, 7), (4097, 256, 6), (513, 5888, 4)])
def test_float_batch_lines(cuda, t, rows, cols, n):
    _check(cuda, t, rows, cols, n, seed=rows + n, bias=True, tol=FP32_TOL)


def test_unaligned_row_pitch_rmsnorm(cuda):
    """A fused norm on rows no kernel folds it into: the bits of the standalone norm followed by the product."""
    t, rows, cols = qvx.Q6_K, 40, 1536
    rng = np.random.default_rng(cols)
    w = dev(cuda, random_weight(t, rows, cols, rng))
    X = dev(cuda, rng.standard_normal((3, cols)).astype(np.float32))
    nw = dev(cuda, (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32))
    got = qvx.qmatmul_rmsnorm_t(w, t, X, nw, 1e-5, rows, cols)
    want = qvx.qmatmul_t(w, t, qvx.rmsnorm_t(X, nw, 1e-5), rows, cols)
    cuda.cuda.synchronize()
    np.testing.assert_array_equal(f32bits(got.cpu().numpy()), f32bits(want.cpu().numpy()))


@pytest.mark.parametrize("t,n", [(qvx.Q4_0, 21), (qvx.Q4_K, 9), (qvx.Q4_K, 21)])
def test_batch_in_plan_and_capture(cuda, t, n):
    """A plan's batch (its workspace made at instantiation) and a captured call (no temporary, but for the last
    case) give the eager call's bits on every replay."""
    from qorvix_amd import decode
    rng = np.random.default_rng(11)
    rows, cols = 96, 1024
    w = decode.DevWeight(dev(cuda, random_weight(t, rows, cols, rng)), t, rows, cols)
    X = dev(cuda, rng.standard_normal((n, cols)).astype(np.float32))
    want = f32bits(qvx.qmatmul_t(w.data, t, X, rows, cols).cpu().numpy())
    out = cuda.empty((n, rows), dtype=cuda.float32, device="cuda")
    plan = decode.Plan()
    plan.add(out, w, X, n)
    plan.instantiate()
    cap = cuda.empty((n, rows), dtype=cuda.float32, device="cuda")
    graph = cuda.cuda.CUDAGraph()
    with cuda.cuda.graph(graph):
        qvx.qmatmul_t(w.data, t, X, rows, cols, out=cap)
    for _ in range(3):
        out.zero_(), cap.zero_()
        plan.launch(cuda.cuda.current_stream().cuda_stream)
        graph.replay()
        cuda.cuda.synchronize()
        np.testing.assert_array_equal(f32bits(out.cpu().numpy()), want)
        np.testing.assert_array_equal(f32bits(cap.cpu().numpy()), want)


# Grouped one-vector products of one type: rows per lane group 1, 2, 3-4 and more (chunks), members smaller than
# a workgroup's groups, short rows (several groups a wave), rows of several waves with two conversion tasks.
GROUP_CASES = [(qvx.Q8_0, 4096, [4096, 4096, 4096]), (qvx.Q8_0, 512, [40, 7, 300]), (qvx.Q8_0, 4096, [11008, 11008]),
               (qvx.Q4_0, 11008, [1000, 33, 1, 64]), (qvx.Q4_0, 1024, [20000, 17]), (qvx.Q5_0, 4096, [1024, 1024]),
               (qvx.Q5_K, 2048, [515, 2048]), (qvx.Q6_K, 4096, [1024, 4096]), (qvx.Q6_K, 14336, [100, 300])]


@pytest.mark.parametrize("t,cols,rows", GROUP_CASES)
def test_same_type_group_matches_members(cuda, t, cols, rows):
    rng = np.random.default_rng(cols + sum(rows))
    ws = [dev(cuda, random_weight(t, r, cols, rng)) for r in rows]
    x = dev(cuda, rng.standard_normal((1, cols)).astype(np.float32))
    outs = [cuda.full((r,), float("nan"), dtype=cuda.float32, device="cuda") for r in rows]
    st = cuda.cuda.current_stream().cuda_stream
    assert qvx.qmatmul_group([o.data_ptr() for o in outs], [w.data_ptr() for w in ws], [t] * len(rows), rows,
                             x.data_ptr(), cols, st) == qvx.OK
    for o, w, r in zip(outs, ws, rows):
        np.testing.assert_array_equal(f32bits(o.cpu().numpy()), f32bits(_run(cuda, w, t, x, r, cols)[0].cpu().numpy()))


@pytest.mark.parametrize("t", [qvx.Q8_0, qvx.Q4_K])
def test_plan_groups_only_independent_calls(cuda, t):
    """A plan whose consecutive calls share x (grouped when instantiated), then write what the next reads, or
    write one output twice: the replay gives the calls' results in order, every time."""
    from qorvix_amd import decode
    rng = np.random.default_rng(t)
    n = 512
    w = [decode.DevWeight(dev(cuda, random_weight(t, n, n, rng, scale=1e-3)), t, n, n) for _ in range(4)]
    x0 = dev(cuda, rng.standard_normal((1, n)).astype(np.float32))
    x = x0.clone()
    a, b, c = (cuda.zeros((1, n), dtype=cuda.float32, device="cuda") for _ in range(3))
    steps = [(a, 0, x), (b, 1, x), (c, 2, x), (x, 3, x), (a, 1, x), (a, 2, x), (b, 0, a)]
    plan = decode.Plan()
    for out, i, src in steps:
        plan.add(out, w[i], src, 1)
    assert len(plan) == len(steps)
    plan.instantiate()
    st = cuda.cuda.current_stream().cuda_stream
    want = {k: v.clone() for k, v in zip("xabc", (x0, a, b, c))}
    name = {id(x): "x", id(a): "a", id(b): "b", id(c): "c"}
    for out, i, src in steps:
        want[name[id(out)]] = _run(cuda, w[i].data, t, want[name[id(src)]].clone(), n, n)
    for run in (plan.launch, plan.launch, plan.run_eager):
        x.copy_(x0)
        run(st)
        cuda.cuda.synchronize()
        for k, v in zip("xabc", (x, a, b, c)):
            np.testing.assert_array_equal(f32bits(v.cpu().numpy()), f32bits(want[k].cpu().numpy()))
    plan.close()


# Q4_K batches on converted activations (k_gemv_q4b): fewer super-blocks than K ranges, ragged rows, several
# launches with a short last one, one vector tile a launch (rows past 22528), many tiles a workgroup.
Q4B_CASES = [(1, 256, 9), (33, 512, 17), (4096, 2048, 8), (1000, 2304, 64), (300, 10240, 5), (40, 24576, 20),
             (70000, 256, 12), (515, 14336, 33), (9000, 4096, 32)]


@pytest.mark.parametrize("rows,cols,n", Q4B_CASES)
def test_q4k_batches_match_single_vectors(cuda, rows, cols, n):
    _check(cuda, qvx.Q4_K, rows, cols, n, seed=rows + cols + n, bias=True, zero_vec=True)


# Q4_K batches of few long rows, their K ranges split over workgroups (k_gemv_q4s): one row, ragged rows, one and
# two items a wave, 8 and 16 vectors a launch, two launches, ranges of unequal length.
Q4S_CASES = [(1, 8192, 5), (33, 8448, 8), (1000, 8192, 16), (70, 11264, 9), (515, 14336, 7), (64, 24576, 17),
             (40, 20480, 23), (3000, 24576, 12), (2047, 32768, 16)]


@pytest.mark.parametrize("rows,cols,n", Q4S_CASES)
def test_q4k_batches_of_few_long_rows_match_single_vectors(cuda, rows, cols, n):
    _check(cuda, qvx.Q4_K, rows, cols, n, seed=rows + cols + n, bias=True, zero_vec=True)


@pytest.mark.parametrize("rows,cols,n", [(64, 512, 6), (320, 4096, 16), (96, 1024, 40), (9216, 1024, 9)])
def test_q4k_batches_norm_and_swiglu_match_single_vectors(cuda, rows, cols, n):
    rng = np.random.default_rng(rows + n)
    w = dev(cuda, random_weight(qvx.Q4_K, rows, cols, rng))
    X = dev(cuda, rng.standard_normal((n, cols)).astype(np.float32))
    nw = dev(cuda, (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32))
    for call in (lambda x: qvx.qmatmul_rmsnorm_t(w, qvx.Q4_K, x, nw, 1e-5, rows, cols),
                 lambda x: qvx.qmatmul_swiglu_t(w, qvx.Q4_K, x, rows // 2, cols),
                 lambda x: qvx.qmatmul_swiglu_t(w, qvx.Q4_K, x, rows // 2, cols, norm_w=nw, eps=1e-5)):
        one = cuda.cat([call(X[i:i + 1].contiguous()) for i in (0, n - 1)])
        np.testing.assert_array_equal(f32bits(call(X)[[0, n - 1]].cpu().numpy()), f32bits(one.cpu().numpy()))


def test_plan_batches_share_only_unchanged_activations(cuda):
    """Consecutive batches on the same activations share their conversion inside a plan, unless the call
    between them writes the activations, uses others, or is of another form."""
    from qorvix_amd import decode
    rng = np.random.default_rng(21)
    n, d = 9, 512
    w = [decode.DevWeight(dev(cuda, random_weight(qvx.Q4_K, d, d, rng, scale=1e-3)), qvx.Q4_K, d, d) for _ in range(3)]
    v = decode.DevWeight(dev(cuda, random_weight(qvx.Q6_K, 64, d, rng, scale=1e-3)), qvx.Q6_K, 64, d)
    x0 = dev(cuda, rng.standard_normal((n, d)).astype(np.float32))
    x, u = x0.clone(), dev(cuda, rng.standard_normal((n, d)).astype(np.float32))
    outs = [cuda.zeros((n, d), dtype=cuda.float32, device="cuda") for _ in range(5)]
    ov = cuda.zeros((n, 64), dtype=cuda.float32, device="cuda")
    steps = [(outs[0], w[0], x), (outs[1], w[1], x), (x, w[2], x), (outs[2], w[0], x), (ov, v, x), (outs[3], w[1], x),
             (outs[4], w[0], u)]
    plan = decode.Plan()
    for o, ww, src in steps:
        plan.add(o, ww, src, n)
    plan.instantiate()
    st = cuda.cuda.current_stream().cuda_stream
    xa = qvx.qmatmul_t(w[2].data, qvx.Q4_K, x0, d, d)
    want = [qvx.qmatmul_t(ww.data, ww.type, src, ww.rows, d)
            for ww, src in ((w[0], x0), (w[1], x0), (w[0], xa), (w[1], xa), (w[0], u), (v, xa))]
    for run in (plan.launch, plan.launch, plan.run_eager):
        x.copy_(x0)
        run(st)
        cuda.cuda.synchronize()
        for o, e in zip(outs + [ov, x], want + [xa]):
            np.testing.assert_array_equal(f32bits(o.cpu().numpy()), f32bits(e.cpu().numpy()))
    plan.close()


@pytest.mark.parametrize("n", [1, 9])
def test_plan_shares_norms_only_as_recorded(cuda, n):
    """Consecutive calls on one x with a norm folded in share their conversion (batches) or a launch (one vector),
    unless the norm weight or eps differs, or a call before writes the norm weight."""
    from qorvix_amd import decode
    rng = np.random.default_rng(n)
    d = 512
    w = [decode.DevWeight(dev(cuda, random_weight(qvx.Q4_K, d, d, rng, scale=1e-3)), qvx.Q4_K, d, d) for _ in range(3)]
    x = dev(cuda, rng.standard_normal((n, d)).astype(np.float32))
    na0, nb = (dev(cuda, (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)) for _ in range(2))
    buf = cuda.empty(n * d, dtype=cuda.float32, device="cuda")  # an output whose first row is a norm weight
    na = buf[:d]
    outs = [cuda.zeros((n, d), dtype=cuda.float32, device="cuda") for _ in range(6)]
    steps = [(outs[0], w[0], na, 1e-5), (outs[1], w[1], na, 1e-5), (outs[2], w[0], nb, 1e-5), (outs[3], w[0], nb, 1e-1),
             (buf.view(n, d), w[2], nb, 1e-1), (outs[4], w[1], na, 1e-5), (outs[5], w[0], na, 1e-5)]
    plan = decode.Plan()
    for o, ww, nw, eps in steps:
        plan.add_rmsnorm(o, ww, x, nw, eps, n)
    plan.instantiate()
    call = lambda ww, nw, eps: qvx.qmatmul_rmsnorm_t(ww.data, ww.type, x, nw, eps, d, d)  # noqa: E731
    written = call(w[2], nb, 1e-1)
    want = [call(w[0], na0, 1e-5), call(w[1], na0, 1e-5), call(w[0], nb, 1e-5), call(w[0], nb, 1e-1),
            call(w[1], written[0].contiguous(), 1e-5), call(w[0], written[0].contiguous(), 1e-5)]
    st = cuda.cuda.current_stream().cuda_stream
    for run in (plan.launch, plan.launch, plan.run_eager):
        na.copy_(na0)
        run(st)
        cuda.cuda.synchronize()
        for o, e in zip(outs, want):
            np.testing.assert_array_equal(f32bits(o.cpu().numpy()), f32bits(e.cpu().numpy()))
    plan.close()


# K splits of the prefill GEMM whose partial tiles a launch of their own sums (k_split_sum): a last split shorter than
# the others, subtiles and rows past M, columns past N.  splits: as planned for 256 CUs (0: Q6_K, not exposed; 14, 8
# and 4 by the same rule).
@pytest.mark.parametrize("t,M,rows,cols,splits", [(qvx.Q4_K, 17, 2048, 1024, 4), (qvx.Q4_K, 257, 4096, 14336, 5),
                                                  (qvx.Q4_K, 65, 3300, 3328, 7), (qvx.Q4_K, 201, 1001, 4096, 8),
                                                  (qvx.Q4_K, 1, 256, 2304, 5), (qvx.Q4_K, 128, 6144, 1024, 2),
                                                  (qvx.Q4_K, 130, 3000, 1024, 2), (qvx.Q6_K, 17, 4096, 14336, 0),
                                                  (qvx.Q6_K, 130, 1001, 4096, 0), (qvx.Q6_K, 97, 300, 2048, 0)])
@pytest.mark.parametrize("variant", [qvx.GEMM_BF16, qvx.GEMM_F16])
def test_gemm_k_split_sum(cuda, t, M, rows, cols, splits, variant):
    if splits:
        plan = qvx.qgemm_plan_q4k(M, rows, cols, 256)
        assert plan[0]["splits"] == splits and (splits > 2 or plan[0]["tiles"] <= 32)
    rng = np.random.default_rng(M + rows)
    w = dev(cuda, random_weight(t, rows, cols, rng, scale=1e-3))
    X = dev(cuda, (0.5 * rng.standard_normal((M, cols))).astype(np.float16))
    out = cuda.full((M + 1, rows), 7.0, dtype=cuda.float32, device="cuda")
    qvx.qgemm_t(w, t, X, rows, cols, variant, out=out[:M])
    got = out.cpu().numpy()
    assert (got[M] == 7.0).all()
    Wd = oracle.dequantize(t, w.cpu().numpy(), rows * cols).reshape(rows, cols).astype(np.float64)
    ref = X.cpu().numpy().astype(np.float64) @ Wd.T
    # each product's operands rounded to 8 or 11 bits, and fp32 sums of `cols` products
    eps = 2.0 ** (-8 if variant == qvx.GEMM_BF16 else -11)
    bound = (2 * eps + cols * 2.0 ** -24) * (np.abs(X.cpu().numpy().astype(np.float64)) @ np.abs(Wd).T)
    assert (np.abs(got[:M] - ref) <= bound).all()


# The int8 prefill GEMM's two parts (integer products on the int8 matrix cores, minimums on the fp32 one), against
# the quantised operands in fp64: one token, remainders of the 32-token subtiles, 128-token and 256-row tiles, K splits
# with and without a short last one.
@pytest.mark.parametrize("M,rows,cols", [(1, 1, 256), (33, 257, 768), (97, 300, 1280), (129, 255, 4096), (512, 513, 1024)])
def test_gemm_i8_minimums(cuda, M, rows, cols):
    rng = np.random.default_rng(M + rows)
    w = random_weight(qvx.Q4_K, rows, cols, rng, scale=1e-3)
    X = (0.5 * rng.standard_normal((M, cols)) + 0.25).astype(np.float16)  # a mean: the minimums weigh in
    out = cuda.full((M + 1, rows), 7.0, dtype=cuda.float32, device="cuda")
    qvx.qgemm_t(dev(cuda, w), qvx.Q4_K, dev(cuda, X), rows, cols, qvx.GEMM_I8, out=out[:M])
    got = out.cpu().numpy()
    assert (got[M] == 7.0).all()
    q, s, _ = oracle.quantize_q8_act(X.astype(np.float32))
    Xq = q.astype(np.float64) * np.repeat(s.astype(np.float64), 32, axis=1)
    zero = w.reshape(-1, 144).copy()
    zero[:, 16:] = 0  # codes 0: the values are -dmin * m
    Wd = oracle.dequantize(qvx.Q4_K, w, rows * cols).reshape(rows, cols).astype(np.float64)
    Wm = oracle.dequantize(qvx.Q4_K, zero.reshape(-1), rows * cols).reshape(rows, cols).astype(np.float64)
    # two fp32 terms a 32-element block, each rounded at most 4 times before it is added
    bound = (cols / 16 + 8) * 2.0 ** -24 * (np.abs(Xq) @ (np.abs(Wd - Wm) + np.abs(Wm)).T)
    assert (np.abs(got[:M] - Xq @ Wd.T) <= bound + 1e-30).all()
