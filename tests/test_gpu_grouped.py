"""GPU parity: grouped GEMM through the C ABI (`group_gemm_fn`) against the CPU oracle.
The reference's own check is `torch.allclose(ref, out, atol=1e-2, rtol=0)` on rand() inputs of
sizes 1024, 512, 256, 128 (python/tutorials/08-grouped-gemm.py:190-214)."""
import numpy as np
import pytest
import torch

import triton_amd
from oracle import formats, gemm
from util import bits_equal, from_np, to_np, set_knob

pytestmark = pytest.mark.gpu


def _run(gpu, ga, gb, dtype, **kw):
    ta = [from_np(a, dtype, gpu) for a in ga]
    tb = [from_np(b, dtype, gpu) for b in gb]
    return [to_np(c) for c in triton_amd.group_gemm_fn(ta, tb, **kw)]


def _run_device_tables(gpu, ta, tb, dtype, nprog=0):
    """The same through mi355_grouped_gemm, whose five tables live on the device."""
    from triton_amd import _lib

    tc = [torch.full((a.shape[0], b.shape[1]), 7.0, dtype=a.dtype, device=gpu) for a, b in zip(ta, tb)]
    pointers = [torch.tensor([t.data_ptr() for t in g], device=gpu, dtype=torch.int64) for g in (ta, tb, tc)]
    sizes = torch.tensor([v for a, b in zip(ta, tb) for v in (a.shape[0], b.shape[1], a.shape[1])], dtype=torch.int32, device=gpu)
    lds = torch.tensor([v for a, b, c in zip(ta, tb, tc) for v in (a.stride(0), b.stride(0), c.stride(0))], dtype=torch.int32, device=gpu)
    assert _lib.load().mi355_grouped_gemm(*(t.data_ptr() for t in pointers), sizes.data_ptr(), lds.data_ptr(), len(ta),
                                          _lib.F16 if dtype == "fp16" else _lib.BF16, nprog, torch.cuda.current_stream().cuda_stream) == 0
    return tc


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_reference_example_sizes(gpu, dtype):
    # 08:190-205: square problems 1024, 512, 256, 128 of uniform [0, 1) values
    rng = np.random.default_rng(0)
    ga = [formats.round_to(rng.random((d, d)).astype(np.float32), dtype) for d in (1024, 512, 256, 128)]
    gb = [formats.round_to(rng.random((d, d)).astype(np.float32), dtype) for d in (1024, 512, 256, 128)]
    outs = _run(gpu, ga, gb, dtype)
    for a, b, c in zip(ga, gb, outs):
        ref = gemm.matmul_closed_form(a, b, out_dtype=dtype)
        # results reach 2^8: one unit in the last place is 0.25 (fp16) / 2 (bf16), so the reference's
        # absolute 1e-2 only holds where both sides round the same way; the bar here is rtol 1e-2
        assert np.allclose(c, ref, rtol=1e-2, atol=1e-2)
        assert np.mean(c == ref) > 0.98


@pytest.mark.parametrize("big_min", [None, 1])
@pytest.mark.parametrize("nprog", [0, 1, 7, 100])
def test_ragged_problems_are_bit_exact_on_integers(gpu, nprog, big_min, monkeypatch):
    # partial tiles, a single row, K tails (K % 32 != 0), and problems without 16-byte rows: tables in host memory (ring and
    # any-stride kernels, whatever MI355_GROUPED_BIG_MIN says of a group that is not whole 256x256 tiles) and on the device, there
    # with the tile size that is picked for this group (128x128: fewer 256x256 tiles than CUs) and with the 256x256 form (=1)
    if big_min is not None:
        set_knob(monkeypatch, "MI355_GROUPED_BIG_MIN", str(big_min))
    rng = np.random.default_rng(nprog)
    shapes = [(256, 128, 64), (130, 72, 40), (1, 304, 8), (128, 128, 128), (100, 70, 50), (37, 19, 7), (300, 264, 520)]
    ga = [rng.integers(-2, 3, size=(m, k)).astype(np.float32) for m, n, k in shapes]
    gb = [rng.integers(-2, 3, size=(k, n)).astype(np.float32) for m, n, k in shapes]
    ref = gemm.grouped_matmul(ga, gb, num_programs=max(nprog, 1), out_dtype="fp32")
    for dtype in ("fp16", "bf16"):
        outs = _run(gpu, ga, gb, dtype, num_programs=nprog)
        for c, r in zip(outs, ref):
            assert bits_equal(c, r)   # integer results below 2^11 are exact in fp16 and bf16
        ta, tb = ([from_np(x, dtype, gpu) for x in g] for g in (ga, gb))
        for c, r in zip(_run_device_tables(gpu, ta, tb, dtype, nprog), ref):
            assert bits_equal(to_np(c), r)


def test_strided_rows_and_empty_group(gpu):
    rng = np.random.default_rng(9)
    big_a = torch.from_numpy(rng.integers(-2, 3, size=(96, 200)).astype(np.float32)).to(gpu).half()
    big_b = torch.from_numpy(rng.integers(-2, 3, size=(64, 400)).astype(np.float32)).to(gpu).half()
    a, b = big_a[:, :64], big_b[:, 8:136]          # lda = 200, ldb = 400 elements
    (c,) = triton_amd.group_gemm_fn([a], [b])
    assert torch.equal(c.float(), a.float() @ b.float())
    assert triton_amd.group_gemm_fn([], []) == []
    with pytest.raises(AssertionError):
        triton_amd.group_gemm_fn([a], [b, b])


@pytest.mark.parametrize("chunk", [4, 1, 3])
@pytest.mark.parametrize("nprog", [0, 7, 100])
def test_groups_of_whole_256_tiles(gpu, nprog, chunk, monkeypatch):
    # every problem whole 256x256 tiles and K % 128 == 0: the four-wave 16x16-MFMA kernel takes the group, behind either
    # kind of table (thresholds lowered so that 20 tiles and K = 128 are enough); exact sums of small integers, rounded
    # once; K from one pair of stages up to several, M != N, problems of one tile between larger ones
    set_knob(monkeypatch, "MI355_GROUPED_BIG_MIN", "1")
    set_knob(monkeypatch, "MI355_GROUPED_WAVE128_MIN_K", "128")
    # a program's tiles: chunks of up to 4 / 1 / 3 consecutive tiles (7 programs, 20 tiles: chunks of 3, runs that
    # cross from one problem into the next and runs of several tiles inside one problem)
    set_knob(monkeypatch, "MI355_GROUPED_CHUNK", str(chunk))
    rng = np.random.default_rng(40 + nprog)
    shapes = [(256, 256, 128), (512, 256, 256), (256, 256, 1024), (256, 768, 384), (1024, 512, 128), (256, 256, 256), (512, 512, 640)]
    ga = [rng.integers(-2, 3, size=(m, k)).astype(np.float32) for m, n, k in shapes]
    gb = [rng.integers(-2, 3, size=(k, n)).astype(np.float32) for m, n, k in shapes]
    ref = [a @ b for a, b in zip(ga, gb)]
    for dtype in ("fp16", "bf16"):
        outs = _run(gpu, ga, gb, dtype, num_programs=nprog)
        for c, r in zip(outs, ref):
            assert bits_equal(c, formats.round_to(r, dtype))   # (K = 1024 reaches beyond bf16's exact integers)
        ta, tb = ([from_np(x, dtype, gpu) for x in g] for g in (ga, gb))
        for c, r in zip(_run_device_tables(gpu, ta, tb, dtype, nprog), ref):
            assert bits_equal(to_np(c), formats.round_to(r, dtype))
    # the same group without that kernel: the ring kernels behind a host table, the eight-wave ones behind the device's
    set_knob(monkeypatch, "MI355_GROUPED_WAVE128_MIN_K", "0")
    for c, r in zip(_run(gpu, ga, gb, "fp16", num_programs=nprog), ref):
        assert bits_equal(c, r)
    ta, tb = ([from_np(x, "fp16", gpu) for x in g] for g in (ga, gb))
    for c, r in zip(_run_device_tables(gpu, ta, tb, "fp16", nprog), ref):
        assert bits_equal(to_np(c), r)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
def test_whole_tile_groups_at_the_default_thresholds_against_closed_form(gpu, dtype):
    # 256 tiles of 256x256 with K = 2048 select the four-wave kernel without any knob: N(0,1) operands, padded
    # rows of A and C-sized B pitch of 512-byte multiples in the second problem.  A B pitch that is no such
    # multiple (third case) sends the group to the ring kernels (tables on the device: the eight-wave ones).
    rng = np.random.default_rng(5)
    mk = lambda shape: formats.round_to(rng.standard_normal(shape).astype(np.float32), dtype)
    a = [mk((2048, 2048)) for _ in range(4)]
    b = [mk((2048, 2048)) for _ in range(4)]
    ref = [gemm.matmul_closed_form(x, y, out_dtype=dtype) for x, y in zip(a, b)]
    ta = [from_np(x, dtype, gpu) for x in a]
    tb = [from_np(y, dtype, gpu) for y in b]
    ta[1] = from_np(np.pad(a[1], ((0, 0), (0, 64))), dtype, gpu)[:, :2048]
    for pad in (0, 256, 8):
        if pad:
            tb[1] = from_np(np.pad(b[1], ((0, 0), (pad, 0))), dtype, gpu)[:, pad:]
        for outs in (triton_amd.group_gemm_fn(ta, tb), _run_device_tables(gpu, ta, tb, dtype)):
            for c, r in zip(outs, ref):
                assert np.allclose(to_np(c), r, rtol=1e-2, atol=1e-2), pad
                assert np.mean(to_np(c) == r) > 0.98


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("nprog", [0, 5])
def test_host_tables_and_device_tables_agree_bit_for_bit(gpu, nprog, dtype):
    # more problems than one table holds (64), tiles of 64 and of 128 rows next to each other, K shorter than the ring and
    # with a tail, problems without 16-byte rows in between; the device-table entry on the same matrices (its 128x128 form)
    rng = np.random.default_rng(70 + nprog)
    shapes = [(17 + 31 * (i % 9), 8 * (1 + i % 7), 8 * (1 + i % 23)) for i in range(66)] + [(256, 512, 1024), (512, 256, 704), (33, 19, 7), (1, 64, 8)]
    ga = [from_np(rng.integers(-1, 2, size=(m, k)).astype(np.float32), dtype, gpu) for m, n, k in shapes]
    gb = [from_np(rng.integers(-1, 2, size=(k, n)).astype(np.float32), dtype, gpu) for m, n, k in shapes]
    outs = triton_amd.group_gemm_fn(ga, gb, num_programs=nprog)
    for a, b, c in zip(ga, gb, outs):
        assert torch.equal(c.float(), (a.float() @ b.float()).to(c.dtype).float()), (a.shape, b.shape)
    assert all(torch.equal(c, d) for c, d in zip(outs, _run_device_tables(gpu, ga, gb, dtype, nprog)))


@pytest.mark.parametrize("extension", [True, False])
def test_row_strides_beyond_32_bits_are_refused(gpu, extension, monkeypatch):
    from triton_amd import _lib

    if not extension:
        monkeypatch.setattr(_lib, "ext", lambda: None)
    row = torch.zeros(8, device=gpu, dtype=torch.float16).as_strided((1, 8), ((1 << 32) + 8, 1))
    with pytest.raises(RuntimeError):
        triton_amd.group_gemm_fn([row], [torch.zeros(8, 8, device=gpu, dtype=torch.float16)])


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("extension", [True, False])
def test_rows_of_a_and_b_may_overlap(gpu, extension, dtype, monkeypatch):
    # one row repeated (row stride 0) and windows shifted by less than a row, in A and in B, next to an ordinary problem;
    # exact sums of small integers
    from triton_amd import _lib

    if not extension:
        monkeypatch.setattr(_lib, "ext", lambda: None)
    rng = np.random.default_rng(3)
    ints = lambda *shape: from_np(rng.integers(-2, 3, size=shape).astype(np.float32), dtype, gpu)   # noqa: E731
    a = [ints(1, 64).expand(96, 64), ints(96, 64), ints(1024).as_strided((96, 64), (8, 1)), ints(72, 64), ints(96, 64), ints(1, 8).expand(1, 8)]
    b = [ints(64, 80), ints(1, 80).expand(64, 80), ints(64, 80), ints(1024).as_strided((64, 80), (8, 1)), ints(64, 80), ints(1, 72).expand(8, 72)]
    for x, y, c in zip(a, b, triton_amd.group_gemm_fn(a, b)):
        assert torch.equal(c.float(), x.float() @ y.float())


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("every", [1, 2, 40])
def test_problems_without_16_byte_rows_share_a_launch(gpu, dtype, every):
    # 70 problems (a table holds 64), all of them, every other one and two (one in each table) without 16-byte rows: odd sizes, a
    # base that is not aligned, one row, one column, K = 1, several tiles; exact sums of small integers
    rng = np.random.default_rng(every)
    odd = [(37, 19, 7), (1, 1, 1), (130, 65, 33), (1, 200, 250), (200, 1, 70), (64, 64, 65), (65, 130, 8)]
    ga, gb = [], []
    for i in range(70):
        m, n, k = odd[(i // every) % len(odd)] if i % every == 0 else (16 + 8 * (i % 9), 8 * (1 + i % 7), 64)
        x, y = (from_np(rng.integers(-2, 3, size=s).astype(np.float32), dtype, gpu) for s in ((m, k), (k * n + 1,)))
        ga.append(x)
        gb.append((y[1:] if i % every == 0 else y[:-1]).view(k, n))
    for x, y, c in zip(ga, gb, triton_amd.group_gemm_fn(ga, gb)):
        assert torch.equal(c.float(), (x.float() @ y.float()).to(c.dtype).float()), (x.shape, y.shape)


def test_matrices_of_other_libraries(gpu):
    # whatever has data_ptr(), dtype, shape, stride(i) and device, next to a tensor of torch's and alone
    class Foreign:
        def __init__(self, t):
            self.t, self.dtype, self.shape, self.device = t, t.dtype, tuple(t.shape), t.device

        def data_ptr(self):
            return self.t.data_ptr()

        def stride(self, i):
            return self.t.stride(i)

    rng = np.random.default_rng(8)
    a, b = ([from_np(rng.integers(-2, 3, size=(64, 64)).astype(np.float32), "fp16", gpu) for _ in range(2)] for _ in range(2))
    want = [x.float() @ y.float() for x, y in zip(a, b)]
    for ga, gb in (([Foreign(a[0]), a[1]], [b[0], b[1]]), ([Foreign(x) for x in a], [Foreign(y) for y in b])):
        assert all(torch.equal(c.float(), w) for c, w in zip(triton_amd.group_gemm_fn(ga, gb), want))


def test_groups_checked_in_native_code_are_the_python_function_s(gpu, monkeypatch):
    # lists and tuples of plain tensors go past the Python function's checks: the same bits as through them, and everything else -
    # modes, subclasses, refusals - is still the Python function's
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    from triton_amd import _lib
    g = torch.Generator(device=gpu).manual_seed(5)
    shapes = [(33, 64, 40), (1, 8, 1), (256, 128, 512), (0, 16, 8), (5, 7, 0)]
    a = [torch.randn(m, k, device=gpu, generator=g).half() for m, n, k in shapes]
    b = [torch.randn(k, n, device=gpu, generator=g).half() for m, n, k in shapes]
    ext = _lib.ext()
    want = ext.group_gemm(a, b, 0)
    for got in (triton_amd.group_gemm_fn(a, b), triton_amd.group_gemm_fn(tuple(a), tuple(b)), ext.group_gemm_plain(a, b, 0)):
        assert isinstance(got, list) and all(torch.equal(x, y) and x.dtype == y.dtype and not x.requires_grad for x, y in zip(got, want))
    with torch.inference_mode():
        assert all(x.is_inference() for x in triton_amd.group_gemm_fn(a, b))

    class Sub(torch.Tensor):
        pass

    refused = [([a[0].as_subclass(Sub)], [b[0]]), ([a[0]], [b[0].bfloat16()]), ([a[0]], [b[1]]), ([a[0].t()], [b[0].t()]), ([a[0].cpu()], [b[0]]),
               ([a[0].float()], [b[0].float()]), ([a[0][0]], [b[0]]), ([None], [b[0]]), (a[:2], b[:1]), ([], []), (iter(a), iter(b))]
    assert all(ext.group_gemm_plain(*r, 0) is None for r in refused)

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Dispatch.seen += 1
            return func(*args, **(kwargs or {}))

    for mode in (Functions(), Dispatch()):
        with mode:
            assert ext.group_gemm_plain(a, b, 0) is None
    with Dispatch():
        triton_amd.matmul(a[0], b[0])
    assert Dispatch.seen > 0


@pytest.mark.parametrize("run", [None, 0, 1, 16])
@pytest.mark.parametrize("shape", [0, 2, 4, 5])
def test_every_form_of_a_group_in_every_order_is_bit_exact_on_integers(gpu, monkeypatch, shape, run):
    # tiles of either size, in two stages, of both sizes in one launch; eighths for the XCDs, runs of one and of sixteen tiles, the form's own choice; one
    # tile and more than CUs, partial tiles, several tiles a program.  Whole numbers up to 4096: exact in fp32, rounded once
    set_knob(monkeypatch, "MI355_GROUPED_SHAPE", shape)
    if run is not None:
        set_knob(monkeypatch, "MI355_GROUPED_RUN", run)
    for sizes in ([(1, 8, 8)], [(1800, 1800, 136), (40, 72, 1032), (300, 1104, 520), (65, 640, 64), (1, 8, 2048), (129, 136, 8)]):
        g = torch.Generator(device=gpu).manual_seed(shape)
        a = [torch.randint(-1, 2, (m, k), device=gpu, generator=g).half() for m, n, k in sizes]
        b = [torch.randint(-1, 2, (k, n), device=gpu, generator=g).half() for m, n, k in sizes]
        for nprog in (0, 1, 100):
            for x, y, c in zip(a, b, triton_amd.group_gemm_fn(a, b, num_programs=nprog)):
                assert torch.equal(c, (x.float() @ y.float()).half()), (x.shape, y.shape, nprog)


@pytest.mark.parametrize("nprog", [0, 7])
@pytest.mark.parametrize("sizes", [
    [(m, 256, 3072) for m in (1, 130, 65, 300)],                          # 64x64 tiles
    [(m, 1024, 1280) for m in (18, 1615, 32, 112, 371, 524)],             # 128x128 tiles
    [(m, 2304, 256) for m in (314, 305, 626, 369, 35, 1464, 1, 1154)],    # of those, two workgroups on a CU
    [(728, 1320, 1120), (1128, 1064, 192), (360, 136, 128), (112, 592, 1192), (1, 8, 8), (1900, 1608, 552)]])
def test_every_shape_of_tiles_is_bit_exact_on_integers(gpu, sizes, nprog):
    # several tiles a program, K steps fewer than stages, partial tiles.  Whole numbers up to 4096: exact in fp32, rounded once
    g = torch.Generator(device=gpu).manual_seed(len(sizes))
    a = [torch.randint(-1, 2, (m, k), device=gpu, generator=g).bfloat16() for m, n, k in sizes]
    b = [torch.randint(-1, 2, (k, n), device=gpu, generator=g).bfloat16() for m, n, k in sizes]
    for x, y, c in zip(a, b, triton_amd.group_gemm_fn(a, b, num_programs=nprog)):
        assert torch.equal(c, (x.float() @ y.float()).bfloat16()), (x.shape, y.shape)
