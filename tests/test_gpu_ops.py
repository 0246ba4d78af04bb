"""GPU parity of the op surface (Batch ops behind the C ABI) against the CPU
oracle, mirroring the reference's own GPU op tests
(crates/metal-backend/tests/affine.rs, operations.rs).  Integer outputs
(expert ids, dispatch permutation) must be bit-exact; float outputs use the
reference tests' element tolerance |a-b| < tol*(1+|b|)."""
import numpy as np
import pytest

import oracle
from helpers import close, zipf_bias
from hip_backend import BF16, F16, F32, Gpu, ShapeError, Tensor, synth

pytestmark = pytest.mark.gpu


def _pattern_tensor(dims, bits, group, st):
    n = int(np.prod(dims))
    packed, s, b = oracle.affine_pattern(n, bits, group, st)
    return Tensor.affine(dims, packed, s, b, bits, group, st)


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("st", [F32, F16, BF16])
def test_affine_gemv_and_prefill_all_layouts(gpu, bits, group, st):
    # crates/metal-backend/tests/affine.rs:53-89
    print(f"[case] affine matmul bits={bits} group={group} st={st}", flush=True)
    t = _pattern_tensor([256, 19], bits, group, st)
    w = gpu.weight_tensor(t)
    for count in [1, 3, 4, 17]:
        x = (np.sin(np.arange(256 * count, dtype=np.float32) * np.float32(0.27)) * np.float32(0.1))
        x = x.astype(np.float32)
        xb = gpu.upload(x)
        y = gpu.zeros(19 * count)
        with gpu.batch() as b:
            b.matmul(w, xb, y, count)
        close(gpu.read(y), oracle.matmul(t, x, count))


@pytest.mark.parametrize("kind", [("dense", F32), ("dense", BF16), ("dense", F16), (4, 64, BF16),
                                  (8, 128, F16), (2, 32, F32)])
@pytest.mark.parametrize("tokens", [4, 17, 64, 4096])
def test_matmul_tiled_f32_tokens(gpu, kind, tokens):
    """Batch::matmul at 4 tokens or more runs the tiled F32 product (the
    reference's affine_mm / gemm_simd switch, matrix.rs:77-123) on the F32
    matrix cores: every token's row against orc_matmul (affine.rs:46-51
    tolerance), at the dense projection shape h 2048 -> 512 (the shared
    expert's gate), for every dtype; below 4 tokens the GEMV runs."""
    from helpers import make_tensor
    print(f"[case] tiled matmul kind={kind} tokens={tokens}", flush=True)
    t = make_tensor([2048, 512], kind, seed=tokens + len(kind))
    w = gpu.weight_tensor(t)
    x = synth.normal(7000 + tokens, tokens * 2048).reshape(tokens, 2048)
    xb, y = gpu.upload(x), gpu.zeros(tokens * 512)
    gpu.profile_reset()
    gpu.profile(True)
    with gpu.batch() as b:
        b.matmul(w, xb, y, tokens)
    prof = gpu.profile_read()
    gpu.profile(False)
    assert "matmul_f32" in prof, sorted(prof)
    rows = range(tokens) if tokens <= 64 else list(range(0, tokens, 97)) + [tokens - 1]
    rows = np.array(list(rows))
    got = gpu.read(y).reshape(tokens, 512)
    if tokens <= 64:
        ref = oracle.matmul(t, x, tokens).reshape(tokens, 512)
        close(got, ref)
    else:
        close(got[rows], oracle.matmul(t, x[rows], len(rows)).reshape(len(rows), 512))
    for b_ in (xb, y):
        gpu.release(b_)


def test_matmul_unaligned_input_uses_gemv(gpu):
    """An input view that is not 16-byte aligned keeps the per-token GEMV
    (the tiled product loads 16-byte vectors), with the same results."""
    t = _pattern_tensor([256, 40], 4, 64, BF16)
    w = gpu.weight_tensor(t)
    T = 8
    x = synth.normal(7100, T * 256 + 1)
    xb = gpu.upload(x)
    y = gpu.zeros(T * 40)
    gpu.profile_reset()
    gpu.profile(True)
    with gpu.batch() as b:
        b.matmul(w, xb.view(1, T * 256), y, T)
    prof = gpu.profile_read()
    gpu.profile(False)
    assert "matmul_f32" not in prof
    close(gpu.read(y), oracle.matmul(t, x[1:], T))


def test_affine_experts_use_gpu_selected_ids(gpu):
    # crates/metal-backend/tests/affine.rs:91-113
    t = _pattern_tensor([64, 3, 4], 4, 32, F16)
    values = oracle.decode(t)
    w = gpu.weight_tensor(t)
    logits = gpu.upload(np.array([1, 4, 3, 2], np.float32))
    ids = gpu.zeros(2)
    probs = gpu.zeros(2)
    x = np.arange(64, dtype=np.float32) * np.float32(0.01)
    xb = gpu.upload(x)
    out = gpu.zeros(6)
    with gpu.batch() as b:
        b.route(logits, ids, probs, True)
        b.expert_matmul(w, xb, ids, out, False)
    assert gpu.read_u32(ids).tolist() == [1, 2]
    expected = np.concatenate([oracle.matvec(values[e * 3 * 64:(e + 1) * 3 * 64], x) for e in [1, 2]])
    close(gpu.read(out), expected)
    e4, e3 = np.exp(4.0), np.exp(3.0)
    np.testing.assert_allclose(gpu.read(probs), [e4 / (e4 + e3), e3 / (e4 + e3)], rtol=1e-6)


def test_expert_matmul_per_expert_input_and_out_of_range_id(gpu):
    t = _pattern_tensor([64, 5, 6], 8, 64, BF16)
    w = gpu.weight_tensor(t)
    ids = np.array([5, 0, 9], np.uint32)  # 9 >= E: zeros (affine.metal:91)
    x = synth.normal(5, 3 * 64)
    out = gpu.zeros(15)
    xb, ib = gpu.upload(x), gpu.upload_u32(ids)
    with gpu.batch() as b:
        b.expert_matmul(w, xb, ib, out, True)
    ref = oracle.expert_matmul(t, x, ids, True)
    close(gpu.read(out), ref)
    assert (gpu.read(out)[10:] == 0).all()


def test_expert_matmul_single_row_weight_honours_ids(gpu):
    """A one-row, one-expert weight ([64, 1, 1]) under expert_matmul with a
    GPU id: id 0 gives the product, id 5 (>= E) gives 0 (affine.metal:91,
    matrix.metal:52-55) -- the one-row fast path applies only without ids."""
    t = _pattern_tensor([64, 1, 1], 4, 32, BF16)
    w = gpu.weight_tensor(t)
    x = synth.normal(8, 64)
    xb = gpu.upload(x)
    for e in (0, 5):
        ib, out = gpu.upload_u32(np.array([e], np.uint32)), gpu.zeros(1)
        with gpu.batch() as b:
            b.expert_matmul(w, xb, ib, out, False)
        ref = oracle.expert_matmul(t, x, np.array([e], np.uint32), False)
        close(gpu.read(out), ref)
        if e == 5:
            assert gpu.read(out)[0] == 0.0
        else:
            assert ref[0] != 0.0


def test_actual_gpu_ops(gpu):
    # crates/metal-backend/tests/operations.rs:8-28
    data = np.sin(np.arange(65 * 7, dtype=np.float32) * np.float32(0.13)).astype(np.float32)
    x = (np.arange(65, dtype=np.float32) / np.float32(65)).astype(np.float32)
    w = gpu.weight_f32(data, [65, 7])
    nw = gpu.weight_f32(np.ones(65, np.float32), [65])
    xb = gpu.upload(x)
    y = gpu.zeros(7)
    norm = gpu.zeros(65)
    with gpu.batch() as b:
        b.matmul(w, xb, y, 1)
        b.norm(xb, nw, norm, 1, 65, 1e-5)
    close(gpu.read(y), oracle.matvec(data, x), 2e-4)
    close(gpu.read(norm), oracle.rms_norm(x, np.ones(65, np.float32), 1e-5), 2e-4)


@pytest.mark.parametrize("dtype", [F32, F16, BF16])
def test_dense_matmul_dtypes(gpu, dtype):
    v = synth.normal(11, 96 * 33, 0.0, 0.5)
    if dtype == F32:
        t = Tensor.dense([96, 33], v)
    elif dtype == F16:
        t = Tensor.dense([96, 33], v.astype(np.float16).view(np.uint16), F16)
    else:
        t = Tensor.dense([96, 33], synth.f32_to_bf16_bits(v), BF16)
    x = synth.normal(12, 96 * 5)
    y = gpu.zeros(33 * 5)
    wt, xb = gpu.weight_tensor(t), gpu.upload(x)
    with gpu.batch() as b:
        b.matmul(wt, xb, y, 5)
    close(gpu.read(y), oracle.matmul(t, x, 5), 2e-4)


def test_rejects_aliases_and_foreign_buffers(gpu):
    # crates/metal-backend/tests/operations.rs:101-111
    other = Gpu()
    w = gpu.weight_f32(np.ones(64, np.float32), [8, 8])
    x = gpu.upload(np.ones(8, np.float32))
    foreign = other.upload(np.ones(8, np.float32))
    with gpu.batch() as b:
        with pytest.raises(ShapeError):
            b.matmul(w, x, x, 1)
        with pytest.raises(ShapeError):
            b.add(x, foreign, x)
        # exact in-place add is allowed (commands.rs:35,52)
        b.add(x, x, x)
    assert (gpu.read(x) == 2).all()
    other.close()


def test_shape_checks_mirror_the_reference(gpu):
    w = gpu.weight_f32(np.ones(64, np.float32), [8, 8])
    x = gpu.zeros(8)
    y = gpu.zeros(9)
    ids = gpu.zeros(3)
    z2, z3, z2b, z2c, z8 = gpu.zeros(2), gpu.zeros(3), gpu.zeros(2), gpu.zeros(2), gpu.zeros(8)
    with gpu.batch() as b:
        with pytest.raises(ShapeError):
            b.matmul(w, x, y, 1)            # matrix.rs:64-75
        with pytest.raises(ShapeError):
            b.route(x, ids, z2, True)       # sampling.rs:28
        with pytest.raises(ShapeError):
            b.mix(x, z3, z2b)               # elementwise.rs:93
        with pytest.raises(ShapeError):
            b.gate_scalar(x, z2c, z8)       # elementwise.rs:80
    with pytest.raises(ShapeError):         # memory access while a batch is open
        with gpu.batch() as b:
            gpu.zeros(4)
    from hip_backend.api import Batch
    with pytest.raises(ShapeError):   # ops need an open batch (the Batch borrow)
        Batch(gpu, begin=False).add(x, x, x)


# ----------------------------------------------------------------- routing --
def _route_case(gpu, logits, k, normalize):
    T, E = logits.shape
    lb = gpu.upload(logits)
    ids = gpu.zeros(T * k)
    w = gpu.zeros(T * k)
    with gpu.batch() as b:
        b.route_tokens(lb, ids, w, T, normalize)
    got_ids = gpu.read_u32(ids).reshape(T, k)
    got_w = gpu.read(w).reshape(T, k)
    ref_ids, ref_w = oracle.route_tokens(logits, k, normalize)
    assert np.array_equal(got_ids, ref_ids)
    both_nan = np.isnan(got_w) & np.isnan(ref_w)
    assert (np.isnan(got_w) == np.isnan(ref_w)).all()
    np.testing.assert_allclose(got_w[~both_nan], ref_w[~both_nan], rtol=2e-6, atol=1e-9)


@pytest.mark.parametrize("normalize", [True, False])
def test_route_bit_exact_random(gpu, normalize):
    logits = synth.normal(21, 257 * 512, 0.0, 1.0).reshape(257, 512)
    _route_case(gpu, logits, 10, normalize)


def test_route_bit_exact_heavy_ties(gpu):
    # logits drawn from 5 values -> many exact ties; order must be lowest index first
    rng = np.random.default_rng(22)
    vals = np.array([-1.0, 0.0, 0.5, 0.5 + 2 ** -20, 2.0], np.float32)
    logits = vals[rng.integers(0, 5, (300, 128))]
    _route_case(gpu, logits, 8, True)
    _route_case(gpu, logits[:, :64], 64, False)  # K = E


def test_route_nonfinite(gpu):
    logits = np.array([[1.0, np.nan, 3.0, -np.inf],
                       [-np.inf, -np.inf, -np.inf, 2.0],
                       [-0.0, 0.0, -1.0, -0.0]], np.float32)
    _route_case(gpu, logits, 3, True)


# ---------------------------------------------------------------- dispatch --
# (4096, 8, 128) runs the single-pass kernel with per-chunk count tables;
# (8192, 8, 512) the same kernel without them (16 chunks x 512 experts of
# tables exceed its 64 KiB of LDS); (4096, 10, 512) and (5600, 10, 512) the
# tables at 10 and 14 chunks over 512 experts (the Qwen3-Next prefill's
# dispatch), the latter filling the 64 KiB
@pytest.mark.parametrize("T,K,E", [(4096, 8, 128), (8192, 8, 512), (4096, 10, 512), (5600, 10, 512),
                                   (64, 10, 512), (1, 10, 512), (777, 3, 40)])
def test_dispatch_bit_exact(gpu, T, K, E):
    logits = synth.normal(23 + T, T * E).reshape(T, E) + zipf_bias(T, E, 5)
    ids, _ = oracle.route_tokens(logits, K, True)
    counts, offsets, perm, pos = (gpu.zeros(E), gpu.zeros(E + 1), gpu.zeros(T * K), gpu.zeros(T * K))
    ib = gpu.upload_u32(ids.ravel())
    with gpu.batch() as b:
        b.dispatch(ib, T, K, E, counts, offsets, perm, pos)
    rc, ro, rp, rpos = oracle.dispatch(ids, E)
    assert np.array_equal(gpu.read_u32(counts), rc)
    assert np.array_equal(gpu.read_u32(offsets), ro)
    assert np.array_equal(gpu.read_u32(perm), rp)
    assert np.array_equal(gpu.read_u32(pos), rpos)


# ------------------------------------------------------------- elementwise --
def test_elementwise_ops(gpu):
    a = synth.normal(31, 1000) * 4
    bb = synth.normal(32, 1000)
    ab, bbuf = gpu.upload(a), gpu.upload(bb)
    y1, y2, y3 = gpu.zeros(1000), gpu.zeros(1000), gpu.zeros(1000)
    g = gpu.upload(np.array([0.3], np.float32))
    xk = synth.normal(33, 4 * 250)
    wk = np.array([0.5, -0.25, 1.5, 0.0], np.float32)
    ym = gpu.zeros(250)
    xkb, wkb = gpu.upload(xk), gpu.upload(wk)
    with gpu.batch() as b:
        b.swiglu(ab, bbuf, y1)
        b.add(ab, bbuf, y2)
        b.gate_scalar(ab, g, y3)
        b.mix(xkb, wkb, ym)
        b.swiglu(ab, bbuf, ab)  # exact in-place (commands.rs:35)
    close(gpu.read(y1), oracle.swiglu(a, bb), 1e-5)
    close(gpu.read(y2), oracle.add(a, bb), 1e-6)
    close(gpu.read(y3), oracle.gate_scalar(a, 0.3), 1e-5)
    close(gpu.read(ym), oracle.mix(xk, wk), 1e-5)
    close(gpu.read(ab), oracle.swiglu(a, bb), 1e-5)


def test_allocation_error_carries_bytes(gpu):
    """Error::Allocation(usize) carries the requested size
    (crates/metal-backend/src/lib.rs:12-13, apple/memory.rs:9-26): zero-sized
    and over-limit requests report their byte counts; a later shape error
    clears it."""
    from hip_backend import AllocationError, ShapeError
    with pytest.raises(AllocationError) as e:
        gpu.zeros(1 << 33)  # more than u32::MAX elements (memory.rs:10)
    assert e.value.bytes == 4 << 33
    with pytest.raises(AllocationError) as e:
        gpu.zeros(0)
    assert e.value.bytes == 0
    with pytest.raises(AllocationError) as e:
        gpu.zeros(1 << 33)
    b = gpu.zeros(4)
    with pytest.raises(ShapeError):
        b.view(2, 8)
    with pytest.raises(ShapeError):
        with gpu.batch() as bt:
            bt.add(b, b.view(0, 2), b)
    from hip_backend.api import _lib
    assert _lib.moe_last_error_bytes(gpu._h) == 0
    gpu.release(b)


def test_zero_fills_end_before_the_call_returns(gpu):
    """A zero fill that queues behind a large one is over before a product
    writes the buffer: the fills run on the null stream, which the gpu's own
    streams do not wait for."""
    w = synth.normal(61, 64 * 256)
    x = synth.normal(62, 64)
    wt, xb = gpu.weight_tensor(Tensor.dense([64, 256], w)), gpu.upload(x)
    for clear in (False, True):
        big = gpu.zeros(1 << 28)
        y = gpu.zeros(256)
        if clear:
            gpu.clear(big)
            gpu.clear(y)
        with gpu.batch() as b:
            b.matmul(wt, xb, y, 1)
        close(gpu.read(y), w.reshape(256, 64) @ x)
        gpu.release(big)
        gpu.release(y)
    gpu.release(xb)


def test_zeros_wait_for_no_other_stream(gpu):
    """moe_zeros returns while a host's own work on the null stream still runs
    (about 0.1 s of fills of 8 GB, queued through the HIP runtime in use)."""
    import ctypes
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipMemsetD32Async.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, ctypes.c_void_p]
    hip.hipStreamQuery.argtypes = hip.hipStreamSynchronize.argtypes = [ctypes.c_void_p]
    big = gpu.zeros(1 << 31)
    for _ in range(50):
        assert hip.hipMemsetD32Async(big.ptr, 1, 1 << 31, None) == 0
    small = gpu.zeros(1000)
    busy = hip.hipStreamQuery(None)
    assert hip.hipStreamSynchronize(None) == 0
    assert busy == 600  # hipErrorNotReady
    assert not gpu.read(small).any()
    for b_ in (big, small):
        gpu.release(b_)


@pytest.mark.parametrize("n,heads,pad", [(1, 2, 0), (64, 5, 3), (128, 16, 0), (255, 2, 1), (260, 3, 4), (1023, 1, 0),
                                         (2047, 2, 0), (2048, 3, 0), (2052, 2, 0), (5000, 2, 8)])
@pytest.mark.parametrize("dtype", [F32, F16, BF16])
def test_norm_rows(gpu, n, heads, pad, dtype):
    """Batch::norm at the edges of its block: rows shorter than a wave, of
    whole and ragged groups of four, rows past the values a block holds, padded
    strides, and an input that is not 16-byte aligned.  F32 sums of n products:
    n * 2^-24 is far below the 2e-4 the op's fixture uses."""
    print(f"[case] norm n={n} heads={heads} pad={pad} dtype={dtype}", flush=True)
    stride = n + pad
    x = synth.normal(900 + n, 1 + (heads - 1) * stride + n)
    w = synth.normal(901 + n, n, 1.0, 0.1)
    if dtype == F32:
        t, wf = Tensor.dense([n], w), w
    elif dtype == BF16:
        bits = synth.f32_to_bf16_bits(w)
        t, wf = Tensor.dense([n], bits, BF16), synth.bf16_bits_to_f32(bits)
    else:
        h = w.astype(np.float16)
        t, wf = Tensor.dense([n], h.view(np.uint16), F16), h.astype(np.float32)
    wt, buf = gpu.weight_tensor(t), gpu.upload(x)
    for first in (0, 1):  # aligned, and one element off
        y = gpu.zeros(heads * n)
        with gpu.batch() as b:
            b.norm(buf.view(first, len(x) - 1), wt, y, heads, stride, 1e-5)
        got = gpu.read(y).reshape(heads, n)
        for i in range(heads):
            row = x[first + i * stride:first + i * stride + n]
            close(got[i], oracle.rms_norm(row, wf, 1e-5), 2e-4)
        gpu.release(y)
    gpu.release(buf)


def test_norm_longest_rows(gpu):
    """One row whose length lies within a block's stride of 2^32 (17 GB): the
    walk over it ends, and its first and last values are normalised."""
    from hip_backend.api import MoeRegionC, MoeWeightC, Weight
    n = (1 << 32) - 512
    print(f"[case] norm n={n}", flush=True)
    x, y, wb = gpu.zeros(n), gpu.zeros(n), gpu.zeros(n // 2)
    w = MoeWeightC()
    w.data = MoeRegionC()
    w.data.ptr, w.data.bytes = wb.ptr, 2 * n
    w.dtype, w.ndims, w.dims[0] = BF16, 1, n
    first, last = np.array([3.0, -1.0], np.float32), np.array([2.0, 4.0], np.float32)
    for b_, at, v in ((x, 0, first), (x, n - 2, last)):
        gpu.write(b_.view(at, 2), v)
    one = synth.f32_to_bf16_bits(np.array([1.0, 0.5], np.float32)).view(np.float32)
    for at in (0, n // 2 - 1):
        gpu.write(wb.view(at, 1), one)
    with gpu.batch() as b:
        b.norm(x, Weight(w, [w.data], [n], 0), y, 1, n, 1e-5)
    scale = np.array([1.0, 0.5]) / np.sqrt((9.0 + 1 + 4 + 16) / n + 1e-5)
    np.testing.assert_allclose(gpu.read(y.view(0, 2)), first * scale, rtol=1e-6)
    np.testing.assert_allclose(gpu.read(y.view(n - 2, 2)), last * scale, rtol=1e-6)
    assert not gpu.read(y.view(2, 4096)).any() and not gpu.read(y.view(n - 4098, 4096)).any()
    for b_ in (x, y, wb):
        gpu.release(b_)


@pytest.mark.parametrize("bits,group,st", [(2, 32, F32), (2, 64, BF16), (2, 128, F16), (4, 32, BF16), (4, 64, F16),
                                           (4, 128, F32), (8, 32, F16), (8, 64, F32), (8, 128, BF16)])
@pytest.mark.parametrize("n_in,out,tokens", [(128, 1, 4), (256, 17, 15), (384, 130, 16), (512, 64, 17), (640, 255, 33),
                                             (1152, 1040, 500)])
def test_matmul_split_products(gpu, bits, group, st, n_in, out, tokens):
    """Batch::matmul of affine weights from 4 tokens on (split f16 products) at
    the edges of its tiles: one to nine units of 128 values, output rows and
    tokens around 16, both tile counts per wave, over rows of unlike magnitude
    (2^-30 .. 2^30 from row to row, one of zeros).  The bound per output is that of the method:
    2^-22 of each product (the split of x) and F32 additions of one sum per
    group, under 2^-20 * sum |w x| together."""
    print(f"[case] split {bits}/{group}/{st} [{n_in},{out}] tokens={tokens}", flush=True)
    q = synth.quantize_affine(synth.normal(31 * n_in + bits, n_in * out, 0.0, 0.5), bits, group, st)
    t = Tensor.affine([n_in, out], *q, bits, group, st)
    x = synth.normal(32 * n_in + tokens, tokens * n_in).reshape(tokens, n_in)
    x = (x * np.exp2(np.linspace(-30, 30, tokens))[:, None]).astype(np.float32)
    x[tokens // 2] = 0.0
    w = gpu.weight_tensor(t)
    xb, y = gpu.upload(x), gpu.zeros(tokens * out)
    with gpu.batch() as b:
        b.matmul(w, xb, y, tokens)
    got = gpu.read(y).reshape(tokens, out).astype(np.float64)
    wd = np.asarray(oracle.decode(t), np.float64).reshape(out, n_in)
    ref, mag = x.astype(np.float64) @ wd.T, np.abs(x.astype(np.float64)) @ np.abs(wd).T
    assert np.all(np.abs(got - ref) <= 2.0 ** -20 * mag)
    for b_ in (xb, y):
        gpu.release(b_)


@pytest.mark.parametrize("bits,n_in", [(2, 2048), (4, 2048), (8, 2048), (8, 4096)])
def test_matmul_split_sum_of_groups(gpu, bits, n_in):
    """The split products' running sum over groups of 32 rounds once per group:
    within what an F32 sum of n_in / 32 terms of random sign rounds to (2^-24 /
    sqrt(3) of it times sqrt(n / 2))."""
    out, tokens = 300, 9
    print(f"[case] split groups {bits}/32 [{n_in},{out}]", flush=True)
    q = synth.quantize_affine(synth.normal(51 + bits, n_in * out, 0.0, 0.02), bits, 32, BF16)
    t = Tensor.affine([n_in, out], *q, bits, 32, BF16)
    x = synth.normal(52 + n_in, tokens * n_in).reshape(tokens, n_in)
    w, xb, y = gpu.weight_tensor(t), gpu.upload(x), gpu.zeros(tokens * out)
    with gpu.batch() as b:
        b.matmul(w, xb, y, tokens)
    # the weights as they are, code * scale + bias unrounded
    codes = (q[0].reshape(-1, 1) >> np.arange(0, 32, bits, dtype=np.uint32)) & ((1 << bits) - 1)
    s, c = (synth.bf16_bits_to_f32(v).astype(np.float64)[:, None] for v in q[1:])
    wd = (codes.reshape(-1, 32) * s + c).reshape(out, n_in)
    ref = x.astype(np.float64) @ wd.T
    err = np.linalg.norm(gpu.read(y).reshape(tokens, out) - ref) / np.linalg.norm(ref)
    assert err <= 2.0 ** -24 / np.sqrt(3) * np.sqrt(n_in / 32 / 2), err
    for b_ in (xb, y):
        gpu.release(b_)


@pytest.mark.parametrize("n_in,out,tokens", [(256, 40, 5), (1152, 130, 40)])
def test_matmul_split_wide_units(gpu, n_in, out, tokens):
    """Magnitudes of 2^-40 .. 2^0 and one of 2^30 inside every 128 values, the
    largest at weights of exactly 0 (code 8 under scale s and bias -8 s), where
    an F32 product would not see them.  The split is off by at most 2^-22 of a
    value or 2^-39 of the largest of its 128, and the sums of the rest by F32's."""
    print(f"[case] split wide units [{n_in},{out}] tokens={tokens}", flush=True)
    rng = np.random.default_rng(n_in)
    codes = rng.integers(0, 16, (out, n_in)).astype(np.uint32)
    cols = np.arange(77, n_in, 128)
    codes[:, cols] = 8
    words = (codes.reshape(out, n_in // 8, 8) << (4 * np.arange(8, dtype=np.uint32))).sum(2, dtype=np.uint32)
    n = out * n_in // 64
    s = synth.f32_to_bf16_bits(np.full(n, 2.0 ** -7, np.float32))
    b = synth.f32_to_bf16_bits(np.full(n, -(2.0 ** -4), np.float32))
    t = Tensor.affine([n_in, out], words.ravel(), s, b, 4, 64, BF16)
    x = synth.normal(53 + n_in, tokens * n_in).reshape(tokens, n_in)
    x = (x * np.exp2(rng.integers(-40, 1, x.shape))).astype(np.float32)
    x[:, cols] = np.float32(2.0 ** 30)
    w, xb, y = gpu.weight_tensor(t), gpu.upload(x), gpu.zeros(tokens * out)
    with gpu.batch() as bt:
        bt.matmul(w, xb, y, tokens)
    got = gpu.read(y).reshape(tokens, out).astype(np.float64)
    wd = ((codes.astype(np.float64) - 8) * 2.0 ** -7)
    x64 = x.astype(np.float64)
    split = np.maximum(2.0 ** -22 * np.abs(x64), 2.0 ** -39 * 2.0 ** 30)
    bound = split @ np.abs(wd).T + 2.0 ** -20 * (np.abs(x64) @ np.abs(wd).T)
    assert np.all(np.abs(got - x64 @ wd.T) <= bound)
    for b_ in (xb, y):
        gpu.release(b_)


def test_matmul_split_nonfinite_rows(gpu):
    """A NaN or an infinity in a token's row reaches every output of that token
    and of no other."""
    t = Tensor.affine([256, 40], *synth.quantize_affine(synth.normal(5, 256 * 40), 4, 64, BF16), 4, 64, BF16)
    x = synth.normal(6, 6 * 256).reshape(6, 256)
    x[1, 200], x[3, 7], x[4, 8] = np.nan, np.inf, -np.inf
    w, xb, y = gpu.weight_tensor(t), gpu.upload(x), gpu.zeros(6 * 40)
    with gpu.batch() as b:
        b.matmul(w, xb, y, 6)
    got = gpu.read(y).reshape(6, 40)
    for i in (1, 3, 4):
        assert not np.isfinite(got[i]).any()
    for i in (0, 2, 5):
        assert np.isfinite(got[i]).all()
    for b_ in (xb, y):
        gpu.release(b_)


@pytest.mark.parametrize("bits,group,st", [(2, 32, F32), (4, 64, BF16), (8, 128, F16)])
@pytest.mark.parametrize("tokens", [4, 19])
def test_matmul_split_infinities_and_overflow(gpu, bits, group, st, tokens):
    """Tiled products of rows the split has no finite value for: every output
    is the one its decoded weights give (oracle.matmul) -- an infinity of the
    products' sign, NaN where two meet or a weight is 0 -- and finite inputs of
    about 2^121 give finite results."""
    print(f"[case] split infinities {bits}/{group}/{st} tokens={tokens}", flush=True)
    n_in, out = 384, 70
    q = synth.quantize_affine(synth.normal(41 + bits, n_in * out, 0.0, 2.0 ** -8), bits, group, st)
    t = Tensor.affine([n_in, out], *q, bits, group, st)
    x = synth.normal(42 + tokens, tokens * n_in).reshape(tokens, n_in)
    x[0, 130] = np.inf
    x[1, 383] = -np.inf
    x[2, 5], x[2, 300] = np.inf, -np.inf
    x[tokens - 1] *= np.float32(2.0 ** 121)
    w, xb, y = gpu.weight_tensor(t), gpu.upload(x), gpu.zeros(tokens * out)
    with gpu.batch() as b:
        b.matmul(w, xb, y, tokens)
    got = gpu.read(y).reshape(tokens, out)
    ref = np.asarray(oracle.matmul(t, x, tokens)).reshape(tokens, out)
    assert np.array_equal(got[:3], ref[:3], equal_nan=True)
    assert np.isposinf(got[:2]).any() and np.isneginf(got[:2]).any()
    # F32 sums of 384 products each: under 2^-20 of sum |w x|
    wd = np.abs(np.asarray(oracle.decode(t), np.float64)).reshape(out, n_in)
    mag = np.abs(x[3:].astype(np.float64)) @ wd.T
    assert np.isfinite(ref[3:]).all() and np.isfinite(got[3:]).all()
    assert np.all(np.abs(got[3:].astype(np.float64) - ref[3:]) <= 2.0 ** -20 * mag)
    for b_ in (xb, y):
        gpu.release(b_)


def test_matmul_split_long_runs(gpu):
    """More token rows than one launch's grid holds (65535 entries of 16): the
    rows on both sides of the boundary and the last ones."""
    n_in, out, tokens = 128, 3, 65535 * 16 + 21
    t = Tensor.affine([n_in, out], *synth.quantize_affine(synth.normal(8, n_in * out), 4, 64, BF16), 4, 64, BF16)
    base = synth.normal(9, 997 * n_in).reshape(997, n_in)
    x = np.resize(base, (tokens, n_in))
    w, xb, y = gpu.weight_tensor(t), gpu.upload(x), gpu.zeros(tokens * out)
    with gpu.batch() as b:
        b.matmul(w, xb, y, tokens)
    got = gpu.read(y).reshape(tokens, out)
    ref = oracle.matmul(t, base, 997).reshape(997, out)
    close(got, np.resize(ref, (tokens, out)))
    for b_ in (xb, y):
        gpu.release(b_)
