"""Parity of the HIP kernels (through the C ABI) with the CPU oracle.  Needs an MI355X.

Bars: amax, scales and fp8 bytes bit-exact (NaN codes may differ in the sign
bit); GEMM within a stated tolerance of the emulated fp32 product.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

from tests.helpers import CODE_DT, F8, TORCH_DT, fp8_bytes, np_for_c, same_bytes_mod_nan_sign

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def nat():
    if not torch.cuda.is_available():
        pytest.fail("these tests need a GPU (run with -m gpu on an MI355X box)")
    from float8_experimental_amd import _native

    _native.lib()
    return _native


def _oracles():
    from oracle import c_oracle as co
    from oracle import torch_oracle as to

    return co, to


def heavy(shape, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    t = torch.distributions.StudentT(3.0).sample(shape)
    mask = torch.rand(shape, generator=g) < 0.001
    return torch.where(mask, t * 1000, t).to(dtype)


# ------------------------------------------------------------------ K1 amax


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1,), (7,), (4, 8), (33, 47), (257, 1031), (1024, 4096), (3, 5, 64)])
def test_amax_scale_matches_oracle(nat, dt, shape):
    co, to = _oracles()
    torch.manual_seed(hash((dt, shape)) % 1000)
    x = heavy(shape, TORCH_DT[dt], 1)
    xd = x.to(DEV)
    for fmt, (code, tdt) in F8.items():
        amax, scale = nat.amax_scale(xd, tdt)
        want_a = to.tensor_to_amax(x).float()
        want_s = to.tensor_to_scale(x, tdt)
        assert amax.cpu().view(torch.int32).item() == want_a.view(torch.int32).item()
        assert scale.cpu().view(torch.int32).item() == want_s.view(torch.int32).item(), (dt, fmt, shape)
        # fp32 math (delayed-scaling buffers)
        _, s32 = nat.amax_scale(xd, tdt, math_dtype=torch.float32)
        want = to.amax_to_scale(want_a, tdt, TORCH_DT[dt])
        assert s32.cpu().view(torch.int32).item() == want.view(torch.int32).item()


def test_amax_strided_rows_and_unaligned_views(nat):
    co, to = _oracles()
    torch.manual_seed(3)
    base = torch.randn(64, 300).to(torch.bfloat16)
    based = base.to(DEV)
    for view in (lambda t: t[:, 3:259], lambda t: t[5:40, 1:2], lambda t: t[:, ::2], lambda t: t.t()):
        x, xd = view(base), view(based)
        amax, scale = nat.amax_scale(xd, torch.float8_e4m3fn)
        assert amax.item() == to.tensor_to_amax(x).float().item()
        assert scale.item() == to.tensor_to_scale(x, torch.float8_e4m3fn).item()


def test_amax_specials(nat):
    co, to = _oracles()
    for dt in (torch.bfloat16, torch.float16, torch.float32):
        z = torch.zeros(1000, dtype=dt, device=DEV)
        for f8 in (torch.float8_e4m3fn, torch.float8_e5m2):
            a, s = nat.amax_scale(z, f8)
            assert a.item() == 0.0
            assert s.item() == to.tensor_to_scale(torch.zeros(4, dtype=dt), f8).item()
        z[77] = float("nan")
        a, s = nat.amax_scale(z, torch.float8_e4m3fn)
        assert torch.isnan(a).item() and torch.isnan(s).item()
        z[77] = float("-inf")
        a, s = nat.amax_scale(z, torch.float8_e4m3fn)
        assert a.item() == float("inf") and s.item() == 0.0
    # the workspace is left clean: a later call on other data is unaffected
    a, _ = nat.amax_scale(torch.full((10,), 0.5, dtype=torch.bfloat16, device=DEV), torch.float8_e4m3fn)
    assert a.item() == 0.5


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
def test_amax_of_many_tensors_in_one_pass_matches_oracle(nat, dt):
    """f8mi_amax_scale_multi: sizes around the tile (32 KB) and vector (16 B) boundaries, an empty tensor,
    a NaN and an inf, against the oracle and against the one-tensor entry point, bit for bit."""
    co, to = _oracles()
    tdt = TORCH_DT[dt]
    tile = nat.lib().f8mi_amax_tile_elems(nat._DT[tdt])
    sizes = [1, 7, 8, 9, 0, tile - 1, tile, tile + 1, 3 * tile, 3 * tile + 5, 1000003, 5 * tile - 8, 2, 20 * tile + 3]
    hosts = [heavy((n,), tdt, 10 + i) * (0.01 * (i + 1)) for i, n in enumerate(sizes)]
    hosts[5][-1] = float("nan")          # in the partial last tile
    hosts[8][tile + 17] = float("-inf")  # in a whole tile
    hosts[9][-1] = 3.0e4                 # the maximum sits in the < 16-byte tail
    devs = [h.to(DEV) for h in hosts]
    for fmt, (code, f8dt) in F8.items():
        amaxes, scales = nat.amax_scale_multi(devs, f8dt)
        assert amaxes.shape == scales.shape == (len(sizes),)
        for i, (h, d) in enumerate(zip(hosts, devs)):
            a1, s1 = nat.amax_scale(d, f8dt)
            assert amaxes[i].view(torch.int32).item() == a1.view(torch.int32).item(), (dt, fmt, sizes[i])
            assert scales[i].view(torch.int32).item() == s1.view(torch.int32).item(), (dt, fmt, sizes[i])
            if h.numel() and not torch.isnan(h).any():
                assert amaxes[i].item() == to.tensor_to_amax(h).float().item()
                assert scales[i].cpu().view(torch.int32).item() == to.tensor_to_scale(h, f8dt).view(torch.int32).item()
        assert torch.isnan(amaxes[5]).item() and torch.isnan(scales[5]).item()
        assert amaxes[8].item() == float("inf") and scales[8].item() == 0.0
    # the same list again (cached table) after the data changed
    devs[0].fill_(5.0)
    amaxes, _ = nat.amax_scale_multi(devs, torch.float8_e4m3fn)
    assert amaxes[0].item() == 5.0


def test_amax_of_more_tensors_than_one_call_takes(nat):
    n = nat.lib().f8mi_workspace_bytes() // 4 + 300
    torch.manual_seed(5)
    big = torch.randn(n, 24, device=DEV).to(torch.bfloat16)  # rows of 48 bytes: 16-byte aligned
    rows = [big[i] for i in range(n)]
    amaxes, scales = nat.amax_scale_multi(rows, torch.float8_e5m2)
    want = big.abs().amax(dim=1).float()
    assert torch.equal(amaxes, want)
    _, s = nat.amax_scale(rows[n - 1], torch.float8_e5m2)
    assert scales[n - 1].item() == s.item()


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
def test_scale_math_sweep_16bit(nat, dt):
    """Scale arithmetic in the tensor's own dtype over a sweep of amax bit patterns."""
    co, to = _oracles()
    top = 0x7C00 if dt == "fp16" else 0x7F80
    pats = np.unique(np.concatenate([np.arange(0, top, 37), np.array([0, 1, 2, top - 1, 0x3F80, 0x3C00])])).astype(np.uint16)
    for fmt, (code, tdt) in F8.items():
        for p in pats[:: 1 if dt == "bf16" else 2]:
            x = torch.from_numpy(np.array([0, p, 0], np.uint16).view(np.int16)).view(TORCH_DT[dt]).to(DEV)
            a, s = nat.amax_scale(x, tdt)
            want = co.amax_to_scale(a.item(), CODE_DT[dt], code, dt == "fp16")
            assert np.float32(s.item()).view(np.uint32) == np.float32(want).view(np.uint32), (dt, fmt, hex(int(p)))


# ------------------------------------------------------------------ K2 cast


def _ref_cast(x_cpu, scale_cpu, tdt, delayed):
    _, to = _oracles()
    s = scale_cpu.reshape(1) if delayed else scale_cpu.reshape(())
    return fp8_bytes(to.cast_to_fp8(x_cpu, s, tdt))


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_cast_every_16bit_pattern(nat, dt, fmt):
    code, tdt = F8[fmt]
    allb = np.arange(65536, dtype=np.uint16)
    x = torch.from_numpy(allb.view(np.int16).copy()).view(TORCH_DT[dt]).reshape(256, 256)
    xd = x.to(DEV)
    scales = [1.0, 448.0 / 3.0, 0.0123, 57344.0 / 0.011, 1e-6, 3.3e4, 2.0**-20, 1.7]
    for s in scales:
        for delayed in (False, True):
            sc = torch.tensor(s, dtype=torch.float32)
            if dt == "fp16" and not delayed and s > 65504:
                continue
            want = _ref_cast(x, sc, tdt, delayed)
            out, out_t = nat.cast(xd, sc.to(DEV), tdt, product_dtype=torch.float32 if delayed else TORCH_DT[dt],
                                  want_out_t=True)
            got = fp8_bytes(out)
            assert same_bytes_mod_nan_sign(got, want), (dt, fmt, s, delayed, int((got != want).sum()))
            assert np.array_equal(fp8_bytes(out_t), got.T)


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_cast_fp32_bit_patterns(nat, fmt):
    code, tdt = F8[fmt]
    rng = np.random.default_rng(5)
    bits = np.concatenate([np.arange(0, 2**32, 8191, dtype=np.uint64).astype(np.uint32)[: 512 * 1024],
                           rng.integers(0, 2**32, size=512 * 1024, dtype=np.uint64).astype(np.uint32)])
    x = torch.from_numpy(bits.view(np.float32).copy()).reshape(1024, 1024)
    xd = x.to(DEV)
    for s in (1.0, 0.37, 1234.5):
        sc = torch.tensor(s, dtype=torch.float32)
        want = _ref_cast(x, sc, tdt, True)
        out, out_t = nat.cast(xd, sc.to(DEV), tdt, want_out_t=True)
        assert same_bytes_mod_nan_sign(fp8_bytes(out), want)
        assert np.array_equal(fp8_bytes(out_t), fp8_bytes(out).T)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_cast_bit_patterns_within_the_largest_code(nat, dt, fmt):
    """The same where no wave needs the clamp, as it takes other instructions: every 16-bit pattern, and fp32 patterns of every
    exponent, whose product stays below the largest code, under scales from tiny to large; products in either type."""
    _, tdt = F8[fmt]
    if dt == "fp32":
        rng = np.random.default_rng(7)
        bits = np.concatenate([np.arange(0, 2**32, 16381, dtype=np.uint64).astype(np.uint32), rng.integers(0, 2**32, size=256 * 1024, dtype=np.uint64).astype(np.uint32)])
        every = torch.from_numpy(bits.view(np.float32).copy())
    else:
        every = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(TORCH_DT[dt])
    for s in (1.0, -1.0, 0.37, 1234.5, 2.0**-30, 2.0**20):
        sc = torch.tensor(s, dtype=torch.float32)
        x = every[(every.float() * s).abs() <= (440.0 if fmt == "e4m3" else 56000.0)]
        x = torch.nn.functional.pad(x, (0, -x.numel() % 256)).reshape(-1, 256)
        for delayed in (False, True):
            out, out_t = nat.cast(x.to(DEV), sc.to(DEV), tdt, product_dtype=torch.float32 if delayed else TORCH_DT[dt], want_out_t=True)
            assert np.array_equal(fp8_bytes(out), np.asarray(_ref_cast(x, sc, tdt, delayed)).reshape(x.shape)), (s, delayed)
            assert np.array_equal(fp8_bytes(out_t), fp8_bytes(out).T)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_cast_of_tiles_around_the_largest_code(nat, dt, fmt):
    """A wave leaves the clamp out where its products stay below the middle past the largest code: one magnitude a tile, below, at
    and above that line, of either sign, under scales of either sign, and tiles of it with one larger, infinite or NaN element."""
    code, tdt = F8[fmt]
    top = 448.0 if fmt == "e4m3" else 57344.0
    edge = [0.98, 1.0, 1.01, 460 / 448, 462 / 448, 464 / 448, 466 / 448, 480 / 448, 60000 / 57344, 61440 / 57344, 61696 / 57344, 1.15]
    x = torch.empty(len(edge), 128, 4, 128)
    for i, e in enumerate(edge):
        x[i] = top * e / 8
        x[i, ::2, :, 1::2] *= -1
        x[i, 17, 1, 5], x[i, 99, 2, 127], x[i, 64, 3, 0] = top / 2, float("-inf"), float("nan")
    x = x.reshape(len(edge) * 128, 512).to(TORCH_DT[dt])
    for s in (8.0, -8.0, 8.5):
        sc = torch.tensor(s, dtype=torch.float32)
        for delayed in (False, True):
            want = _ref_cast(x, sc, tdt, delayed)
            amax = torch.zeros((), dtype=torch.float32, device=DEV) if delayed else None
            out, out_t = nat.cast(x.to(DEV), sc.to(DEV), tdt, product_dtype=torch.float32 if delayed else TORCH_DT[dt], want_out_t=True, amax_out=amax)
            assert same_bytes_mod_nan_sign(fp8_bytes(out), want), (s, delayed)
            assert np.array_equal(fp8_bytes(out_t), fp8_bytes(out).T)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1), (1, 129), (129, 1), (16, 16), (33, 47), (128, 128), (257, 131), (130, 1000),
                                   (1000, 136), (4099, 1000), (2, 3, 40)])
def test_cast_shapes_dynamic_and_delayed(nat, dt, shape):
    co, to = _oracles()
    x = heavy(shape, TORCH_DT[dt], 2)
    xd = x.to(DEV)
    x2 = x.reshape(-1, shape[-1])
    for fmt, (code, tdt) in F8.items():
        s = to.tensor_to_scale(x, tdt)
        # dynamic: product in the tensor's dtype
        out, out_t = nat.cast(xd, s.to(DEV), tdt, want_out_t=True)
        want = fp8_bytes(to.cast_to_fp8(x, s, tdt))
        assert out.shape == x.shape and out_t.shape == (x2.shape[1], x2.shape[0])
        assert np.array_equal(fp8_bytes(out), want), (dt, fmt, shape)
        assert np.array_equal(fp8_bytes(out_t), want.reshape(x2.shape).T)
        # delayed: [1]-shaped scale that saturates part of the tensor, amax fused
        s1 = (s * 2.5).reshape(1)
        amax = torch.full((1,), -1.0, dtype=torch.float32, device=DEV)
        out, out_t = nat.cast(xd, s1.to(DEV), tdt, product_dtype=torch.float32, want_out_t=True, amax_out=amax)
        want = fp8_bytes(to.cast_to_fp8(x, s1, tdt))
        assert np.array_equal(fp8_bytes(out), want), (dt, fmt, shape, "delayed")
        assert np.array_equal(fp8_bytes(out_t), want.reshape(x2.shape).T)
        assert amax.item() == to.tensor_to_amax(x).float().item()
        # only the transposed copy
        _, only_t = nat.cast(xd, s1.to(DEV), tdt, product_dtype=torch.float32, want_out=False, want_out_t=True)
        assert np.array_equal(fp8_bytes(only_t), want.reshape(x2.shape).T)


@pytest.mark.parametrize("dt", ["bf16", "fp32"])
@pytest.mark.parametrize("shape", [(64, 64), (128, 192), (448, 384), (320, 1024), (1000, 128), (192, 1000), (4, 96, 256)])
def test_cast_kblocked_layout_is_a_permutation_of_the_row_major_bytes(nat, dt, shape):
    """k-blocked outputs ([k/64][rows][64]) hold exactly the row-major result's bytes, re-placed; where a
    dimension is not a multiple of 64 the request is refused."""
    co, to = _oracles()
    x = heavy(shape, TORCH_DT[dt], 5)
    xd = x.to(DEV)
    rows, cols = x.numel() // shape[-1], shape[-1]
    tdt = torch.float8_e4m3fn
    s = to.tensor_to_scale(x, tdt).to(DEV)
    ref, ref_t = nat.cast(xd, s, tdt, want_out_t=True)
    ref_b, ref_tb = fp8_bytes(ref).reshape(rows, cols), fp8_bytes(ref_t)
    row_ok, t_ok = cols % 64 == 0, rows % 64 == 0
    amax = torch.zeros(1, dtype=torch.float32, device=DEV)
    out, out_t = nat.cast(xd, s, tdt, want_out=row_ok, want_out_t=t_ok, out_kblock=row_ok, out_t_kblock=t_ok,
                          amax_out=amax if (row_ok or t_ok) else None) if (row_ok or t_ok) else (None, None)
    if row_ok:
        assert out.shape == (cols // 64, rows, 64)
        assert np.array_equal(fp8_bytes(out), ref_b.reshape(rows, cols // 64, 64).transpose(1, 0, 2))
        # mixed: k-blocked out with a row-major transpose
        o2, t2 = nat.cast(xd, s, tdt, want_out_t=True, out_kblock=True)
        assert np.array_equal(fp8_bytes(o2), fp8_bytes(out)) and np.array_equal(fp8_bytes(t2), ref_tb)
    else:
        with pytest.raises(AssertionError):
            nat.cast(xd, s, tdt, out_kblock=True)
    if t_ok:
        assert out_t.shape == (rows // 64, cols, 64)
        assert np.array_equal(fp8_bytes(out_t), ref_tb.reshape(cols, rows // 64, 64).transpose(1, 0, 2))
    else:
        with pytest.raises(AssertionError):
            nat.cast(xd, s, tdt, want_out=False, want_out_t=True, out_t_kblock=True)
    if row_ok or t_ok:
        assert amax.item() == to.tensor_to_amax(x).float().item()


def test_cast_kblocked_refused_by_the_library_when_not_a_multiple_of_64(nat):
    x = torch.ones(100, 96, dtype=torch.bfloat16, device=DEV)
    s = torch.ones((), device=DEV)
    out = torch.empty(100 * 96, dtype=torch.uint8, device=DEV)
    L = nat.lib()
    rc = L.f8mi_cast_layout(x.data_ptr(), 100, 96, 96, 0, s.data_ptr(), 0, 0, out.data_ptr(), 1, None, 0, None, None)
    assert rc != 0 and b"64" in L.f8mi_last_error()
    rc = L.f8mi_cast_layout(x.data_ptr(), 100, 96, 96, 0, s.data_ptr(), 0, 0, None, 0, out.data_ptr(), 1, None, None)
    assert rc != 0
    rc = L.f8mi_cast_layout(x.data_ptr(), 100, 96, 96, 0, s.data_ptr(), 0, 0, out.data_ptr(), 7, None, 0, None, None)
    assert rc != 0


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
def test_delayed_cast_with_workspace_equals_the_cast_without(nat, dt):
    """f8mi_cast_delayed folds the amax of more than 2048 tiles into the 1024 words of its workspace and a second launch reduces them;
    up to 2048 its launch collects the amax and leaves the workspace alone: same bytes and the same amax as
    f8mi_cast_layout with amax_dev, the oracle's amax (NaN, inf, all-zero and all-negative-zero tensors included), and the
    workspace is all zero again after every call -- also on the next call with a smaller amax, of either kind."""
    co, to = _oracles()
    L = nat.lib()
    assert L.f8mi_delayed_workspace_bytes() == 4096
    tdt = torch.float8_e4m3fn
    cases = [heavy((777, 1031), TORCH_DT[dt], 3), heavy((4, 8), TORCH_DT[dt], 4), heavy((2048, 4096), TORCH_DT[dt], 5),
             torch.zeros(300, 200, dtype=TORCH_DT[dt]), -torch.zeros(130, 70, dtype=TORCH_DT[dt])]
    nan = heavy((257, 513), TORCH_DT[dt], 6)
    nan[100, 17] = float("nan")
    inf = heavy((129, 257), TORCH_DT[dt], 7)
    inf[5, 5] = float("-inf")
    cases += [nan, inf]
    big = heavy((65, 4096), TORCH_DT[dt], 8).repeat(127, 1)  # 65 x 32 tiles: the workspace
    nan_big = big.clone()
    nan_big[5000, 17] = float("nan")
    cases = [nan_big, big, big[:8193] * 0.25, torch.zeros_like(big), big] + cases
    ws = nat.delayed_workspace(torch.device(DEV))
    for x in cases:
        xd = x.to(DEV)
        s1 = torch.tensor([1.7], device=DEV)
        a_new = torch.full((1,), -1.0, device=DEV)
        a_old = torch.full((1,), -1.0, device=DEV)
        out, out_t = nat.cast(xd, s1, tdt, product_dtype=torch.float32, want_out_t=True, amax_out=a_new)   # f8mi_cast_delayed
        o2 = torch.empty_like(out)
        t2 = torch.empty_like(out_t)
        rc = L.f8mi_cast_layout(xd.data_ptr(), x.shape[0], x.shape[1], x.shape[1], CODE_DT[dt], s1.data_ptr(), 2, 0, o2.data_ptr(), 0,
                                t2.data_ptr(), 0, a_old.data_ptr(), None)
        assert rc == 0
        assert torch.equal(out.view(torch.uint8), o2.view(torch.uint8)) and torch.equal(out_t.view(torch.uint8), t2.view(torch.uint8))
        want = to.tensor_to_amax(x).float()
        for a in (a_new, a_old):
            assert (math.isnan(a.item()) and math.isnan(want.item())) or a.item() == want.item(), (dt, tuple(x.shape), a.item(), want.item())
        assert not ws.any().item(), "the workspace must be all zero after a call"


# One launch while every wave has a word (2048 tiles), which the workgroup started last collects: one tile, one more row or column,
# the last size and the first beyond; captured, the two launches.
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1), (128, 128), (129, 257), (1000, 3001), (8192, 4096), (8193, 4096)])
def test_delayed_cast_collects_the_maximum_in_its_launch(nat, dt, shape):
    tdt = TORCH_DT[dt]
    x = heavy(shape, tdt, 24).to(DEV)
    scale = torch.tensor([3.0], device=DEV)
    for at, value in ((0, 1e4), (-1, -2e4), (x.numel() // 2, float("nan")), (0, float("-inf"))):
        v = x.clone()
        v.view(-1)[at] = value
        amax = torch.full((1,), -1.0, device=DEV)
        o, _ = nat.cast(v, scale, torch.float8_e4m3fn, product_dtype=torch.float32, amax_out=amax)
        want, _ = nat.amax_scale(v, torch.float8_e4m3fn, want_scale=False)
        assert torch.equal(amax.view(()).isnan(), want.isnan()) and (torch.isnan(want) or amax.item() == want.item()), (at, value)
        plain, _ = nat.cast(v, scale, torch.float8_e4m3fn, product_dtype=torch.float32)
        assert torch.equal(o.view(torch.uint8), plain.view(torch.uint8))
    if shape != (129, 257):
        return
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        nat.cast(x, scale, torch.float8_e4m3fn, product_dtype=torch.float32, amax_out=amax)
    for _ in range(3):
        x.mul_(0.5)
        graph.replay()
        assert amax.item() == x.abs().max().item()


def _unblock(t_kb):
    """[kc/64, rows, 64] k-blocked bytes -> [rows, kc] row-major (numpy)."""
    b = fp8_bytes(t_kb)
    return b.transpose(1, 0, 2).reshape(b.shape[1], b.shape[0] * 64)


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1), (33, 47), (128, 128), (257, 131), (130, 1000), (1000, 136), (4099, 1000), (200, 4097),
                                   (3, 50, 70)])
def test_cast_zero_padded_kblocked_layout(nat, dt, shape):
    """F8MI_LAYOUT_KBLOCK64_PAD128 takes any shape: the output holds the row-major result's bytes, k-blocked after the
    contraction has been extended to a multiple of 128, and every byte of the extension is zero -- with a dynamic
    scale, a delayed one (amax fused), for both fp8 formats, for rows at an unaligned pitch, and under a NaN scale."""
    co, to = _oracles()
    x = heavy(shape, TORCH_DT[dt], 11)
    rows, cols = x.numel() // shape[-1], shape[-1]
    rp, cp = nat.padded_k(rows), nat.padded_k(cols)
    xd = x.to(DEV)

    def check(out, out_t, want, what):
        assert out.shape == (cp // 64, rows, 64) and out_t.shape == (rp // 64, cols, 64), what
        o, t = _unblock(out), _unblock(out_t)
        assert np.array_equal(o[:, :cols], want) and not o[:, cols:].any(), what
        assert np.array_equal(t[:, :rows], want.T) and not t[:, rows:].any(), what

    for fmt, (code, tdt) in F8.items():
        s = to.tensor_to_scale(x, tdt)
        want = fp8_bytes(to.cast_to_fp8(x, s, tdt)).reshape(rows, cols)
        out, out_t, sc = nat.cast_dynamic(xd, tdt, want_out_t=True, out_kblock=nat.KBLOCK_PAD, out_t_kblock=nat.KBLOCK_PAD)
        assert sc.item() == s.item()
        check(out, out_t, want, (dt, fmt, shape, "dynamic"))
        s1 = (s * 2.5).reshape(1)
        amax = torch.full((1,), -1.0, dtype=torch.float32, device=DEV)
        out, out_t = nat.cast(xd, s1.to(DEV), tdt, product_dtype=torch.float32, want_out_t=True, amax_out=amax,
                              out_kblock=nat.KBLOCK_PAD, out_t_kblock=nat.KBLOCK_PAD)
        check(out, out_t, fp8_bytes(to.cast_to_fp8(x, s1, tdt)).reshape(rows, cols), (dt, fmt, shape, "delayed"))
        assert amax.item() == to.tensor_to_amax(x).float().item()
    # one padded and one row-major output in the same call
    tdt = torch.float8_e4m3fn
    s = to.tensor_to_scale(x, tdt)
    want = fp8_bytes(to.cast_to_fp8(x, s, tdt)).reshape(rows, cols)
    out, out_t = nat.cast(xd, s.to(DEV), tdt, want_out_t=True, out_kblock=nat.KBLOCK_PAD)
    assert np.array_equal(_unblock(out)[:, :cols], want) and np.array_equal(fp8_bytes(out_t), want.T)
    out, out_t = nat.cast(xd, s.to(DEV), tdt, want_out_t=True, out_t_kblock=nat.KBLOCK_PAD)
    assert np.array_equal(fp8_bytes(out).reshape(rows, cols), want) and np.array_equal(_unblock(out_t)[:, :rows], want.T)
    # a NaN scale turns every element into a NaN code and leaves the padding zero
    out, out_t = nat.cast(xd, torch.full((), float("nan"), device=DEV), tdt, want_out_t=True, out_kblock=nat.KBLOCK_PAD,
                          out_t_kblock=nat.KBLOCK_PAD)
    o, t = _unblock(out), _unblock(out_t)
    assert ((o[:, :cols] & 0x7f) == 0x7f).all() and not o[:, cols:].any()
    assert ((t[:, :rows] & 0x7f) == 0x7f).all() and not t[:, rows:].any()
    # rows at a pitch that is no multiple of 16 bytes (a column slice of a wider tensor)
    if x.dim() == 2 and cols > 9:
        v, vd = x[:, 3:cols - 2], xd[:, 3:cols - 2]
        s = to.tensor_to_scale(v, tdt)
        want = fp8_bytes(to.cast_to_fp8(v, s, tdt)).reshape(rows, cols - 5)
        out, out_t, sc = nat.cast_dynamic(vd, tdt, want_out_t=True, out_kblock=nat.KBLOCK_PAD, out_t_kblock=nat.KBLOCK_PAD)
        o, t = _unblock(out), _unblock(out_t)
        assert sc.item() == s.item() and np.array_equal(o[:, :cols - 5], want) and not o[:, cols - 5:].any()
        assert np.array_equal(t[:, :rows], want.T) and not t[:, rows:].any()


def test_cast_row_strided_and_c_oracle(nat):
    co, to = _oracles()
    base = heavy((70, 400), torch.bfloat16, 4)
    x, xd = base[:, 8:264], base.to(DEV)[:, 8:264]     # 16-byte aligned rows, ld != cols
    y, yd = base[3:, 5:206], base.to(DEV)[3:, 5:206]   # unaligned
    for t, td in ((x, xd), (y, yd)):
        s = to.tensor_to_scale(t, torch.float8_e4m3fn)
        out, out_t = nat.cast(td, s.to(DEV), torch.float8_e4m3fn, want_out_t=True)
        want_c, want_ct = co.cast(np_for_c(t), co.BF16, s.item(), co.BF16, co.E4M3FN, transpose=True)
        assert np.array_equal(fp8_bytes(out), want_c) and np.array_equal(fp8_bytes(out_t), want_ct)


def test_cfg1_dy_ones(nat):
    """Benchmark configuration 1: dY = ones -> scale 57344, every e5m2 byte 0x7B."""
    dy = torch.ones(2048, 4096, dtype=torch.bfloat16, device=DEV)
    a, s = nat.amax_scale(dy, torch.float8_e5m2)
    assert a.item() == 1.0 and s.item() == 57344.0
    out, out_t = nat.cast(dy, s, torch.float8_e5m2, want_out_t=True)
    assert bool((out.view(torch.uint8) == 0x7B).all()) and bool((out_t.view(torch.uint8) == 0x7B).all())


@pytest.mark.parametrize("shape,strides", [((2048, 4096), (0, 0)), ((2048, 4096), (0, 1)), ((4, 300, 1000), (0, 0, 1)),
                                           ((40, 512), (0, 1))])
def test_expanded_gradient_is_cast_without_being_materialised(nat, shape, strides):
    """dY of ``y.sum().backward()`` is an expanded tensor (reference float8_scaling_utils.py:204-216 casts it like any
    other): amax, scale and bytes equal those of the materialised tensor, and the binding passes one row with row
    stride 0 instead of copying rows x cols elements."""
    torch.manual_seed(9)
    cols = shape[-1]
    base = (torch.ones(1, device=DEV) if strides[-1] == 0 else torch.randn(cols, device=DEV) * 0.3).to(torch.bfloat16)
    dy = torch.as_strided(base, shape, strides)
    full = dy.contiguous()
    read, rows, c, ld = nat._as_2d(dy)
    assert ld == 0 and read.numel() == cols and rows * c == full.numel()
    for f8, kb in ((torch.float8_e5m2, False), (torch.float8_e4m3fn, True)):
        kb = kb and cols % 64 == 0 and rows % 64 == 0
        a0, s0 = nat.amax_scale(full, f8)
        a1, s1 = nat.amax_scale(dy, f8)
        assert a0.item() == a1.item() and s0.item() == s1.item()
        o0, t0 = nat.cast(full.reshape(rows, cols), s0, f8, want_out_t=True, out_kblock=kb, out_t_kblock=kb)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        o1, t1 = nat.cast(dy.reshape(rows, cols) if dy.dim() > 2 else dy, s1, f8, want_out_t=True, out_kblock=kb, out_t_kblock=kb)
        torch.cuda.synchronize()
        assert torch.cuda.max_memory_allocated() - before < 2 * full.numel() + (1 << 20)  # the two fp8 outputs, no bf16 copy
        assert torch.equal(o0.view(torch.uint8), o1.view(torch.uint8)) and torch.equal(t0.view(torch.uint8), t1.view(torch.uint8))
        o2, _, s2 = nat.cast_dynamic(dy.reshape(rows, cols) if dy.dim() > 2 else dy, f8, out_kblock=kb)
        assert s2.item() == s0.item() and torch.equal(o2.view(torch.uint8), o0.view(torch.uint8))
        amax = torch.zeros(1, device=DEV)
        one = torch.ones(1, device=DEV)
        nat.cast(dy, one, f8, product_dtype=torch.float32, amax_out=amax)  # the delayed-scaling cast records the amax
        assert amax.item() == a0.item()
    if strides[-1] == 0:  # dY = ones: scale 57344, every e5m2 byte 0x7B
        o, _, s = nat.cast_dynamic(dy, torch.float8_e5m2)
        assert s.item() == 57344.0 and bool((o.view(torch.uint8) == 0x7B).all())


def test_golden_cast_fixtures_on_gpu(nat):
    from tests.helpers import from_bits, load

    g = load("casts")
    for case in sorted({k[:-2] for k in g.files if k.endswith(".x")}):
        dt = case.split(".")[0]
        x = from_bits(g[case + ".x"], dt).to(DEV)
        for fmt, (code, tdt) in F8.items():
            a, s = nat.amax_scale(x, tdt)
            assert np.float32(s.item()).view(np.uint32) == g[f"{case}.{fmt}.scale"].view(np.uint32), (case, fmt)
            out, _ = nat.cast(x, s, tdt)
            assert np.array_equal(fp8_bytes(out), g[f"{case}.{fmt}.dyn"]), (case, fmt)
            s1 = torch.from_numpy(g[f"{case}.{fmt}.scale1"].copy()).to(DEV)
            out, _ = nat.cast(x, s1, tdt, product_dtype=torch.float32)
            assert np.array_equal(fp8_bytes(out), g[f"{case}.{fmt}.del"]), (case, fmt)


# ------------------------------------------------------------------ K3 gemm


@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 8), (1, 8192), (3, 1000), (4, 8192), (16, 8192), (64, 512), (37, 129), (128, 1024),
                                   (200, 700), (5, 7, 64), (4096, 1), (4097, 3), (512, 4096)])
def test_cast_dynamic_equals_amax_scale_then_cast(nat, dt, shape):
    """f8mi_cast_dynamic (one workgroup up to 32 K elements, the two kernels beyond): scale and bytes of every output layout
    equal those of f8mi_amax_scale followed by f8mi_cast, bit for bit; NaN and all-zero tensors included."""
    tdt = TORCH_DT[dt]
    x = heavy(shape, tdt, 21).to(DEV)
    variants = [x]
    if len(shape) == 2 and shape[1] >= 64:
        variants.append(x[:, 3:shape[1] - 2])          # unaligned, strided rows
        z = torch.zeros_like(x)
        variants.append(z)
        n = x.clone()
        n[-1, -1] = float("nan")
        variants.append(n)
    for v in variants:
        rows, cols = v.reshape(-1, v.shape[-1]).shape
        for fmt, (code, f8dt) in F8.items():
            _, s_want = nat.amax_scale(v, f8dt, want_amax=False)
            kb, tkb = cols % 64 == 0, rows % 64 == 0
            for okb, otkb in {(False, False), (kb, tkb)}:
                o_want, t_want = nat.cast(v, s_want, f8dt, want_out_t=True, out_kblock=okb, out_t_kblock=otkb)
                o, t, s = nat.cast_dynamic(v, f8dt, want_out_t=True, out_kblock=okb, out_t_kblock=otkb)
                assert s.view(torch.int32).item() == s_want.view(torch.int32).item() or (torch.isnan(s) and torch.isnan(s_want))
                assert same_bytes_mod_nan_sign(fp8_bytes(o), fp8_bytes(o_want)), (dt, shape, fmt, okb)
                assert same_bytes_mod_nan_sign(fp8_bytes(t), fp8_bytes(t_want)), (dt, shape, fmt, otkb)
    o, t, s = nat.cast_dynamic(torch.empty(0, 64, device=DEV, dtype=tdt), torch.float8_e4m3fn, want_out_t=True)
    assert o.shape == (0, 64) and t.shape == (64, 0)
    _, s_want = nat.amax_scale(torch.empty(0, 64, device=DEV, dtype=tdt), torch.float8_e4m3fn)
    assert s.item() == s_want.item()


# One copy of more than 32 K elements and at most 512 KB: one launch, whose workgroups take 8192 elements each.  The first such
# size, a whole number of workgroups, one item more and less, the largest of 16-bit and of 32-bit types, the first beyond.
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 32776), (4097, 8), (5, 8192), (1, 40968), (3, 13656), (16, 4096), (16, 14336), (1, 131072), (1, 131080),
                                   (64, 4096), (1, 262144), (1, 262152)])
def test_cast_dynamic_one_copy_equals_amax_scale_then_cast(nat, dt, shape):
    tdt = TORCH_DT[dt]
    x = heavy(shape, tdt, 22).to(DEV)
    shifted = torch.zeros(x.numel() + 1, device=DEV, dtype=tdt)[1:].view(shape)  # rows start at odd multiples of the element size
    shifted.copy_(x)
    wide = torch.cat([x, x], dim=1)[:, :shape[1]]  # more than one row: strided, the two kernels
    first, last = x.clone(), x.clone()
    first.view(-1)[0], last.view(-1)[-1] = float("inf"), float("nan")
    for v in (x, shifted, wide, first, last, torch.zeros_like(x)):
        for fmt, (code, f8dt) in F8.items():
            _, s_want = nat.amax_scale(v, f8dt, want_amax=False)
            for kb in {False, shape[1] % 64 == 0}:
                o_want, _ = nat.cast(v, s_want, f8dt, out_kblock=kb)
                o, _, s = nat.cast_dynamic(v, f8dt, out_kblock=kb)
                assert s.view(torch.int32).item() == s_want.view(torch.int32).item() or (torch.isnan(s) and torch.isnan(s_want))
                assert same_bytes_mod_nan_sign(fp8_bytes(o), fp8_bytes(o_want)), (dt, shape, fmt, kb)


# The line between the kernels that read such a tensor once and once a workgroup, on either side; captured, the latter again.
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(40, 4096), (41, 4096), (15, 14336), (16, 14336), (20, 4096), (21, 4096), (15, 8192), (16, 8192), (64, 4096), (11, 20480), (12, 20480)])
def test_cast_dynamic_either_side_of_the_flat_kernel(nat, dt, shape):
    x = heavy(shape, TORCH_DT[dt], 33).to(DEV)
    for fmt, (code, f8dt) in F8.items():
        s_want = nat.amax_scale(x, f8dt, want_amax=False)[1]
        for layout in (0, 1):
            want = nat.cast(x, s_want, f8dt, out_kblock=layout)[0]
            got, _, s = nat.cast_dynamic(x, f8dt, out_kblock=layout)
            assert torch.equal(s, s_want) and torch.equal(got.view(torch.uint8), want.view(torch.uint8))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q, _, sq = nat.cast_dynamic(x, torch.float8_e4m3fn)
    for _ in range(3):
        x.mul_(0.5)
        graph.replay()
        assert torch.equal(sq, nat.amax_scale(x, torch.float8_e4m3fn, want_amax=False)[1])
        assert torch.equal(q.view(torch.uint8), nat.cast(x, sq, torch.float8_e4m3fn)[0].view(torch.uint8))


# The one-launch cast of a tensor that the chip holds: a single tile, tiles of 64 rows and of 128, one row or column into the next tile,
# the last size of either kind and the largest of all; nobody waits (every workgroup finds the maximum itself) or as shipped.
@pytest.mark.parametrize("dt", ["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1), (64, 128), (65, 129), (200, 1000), (513, 1031), (2048, 2048), (2049, 2048), (1000, 3001), (4096, 4096)])
def test_cast_dynamic_resident_equals_amax_scale_then_cast(nat, dt, shape):
    tdt = TORCH_DT[dt]
    x = heavy(shape, tdt, 23).to(DEV)
    rows, cols = shape
    big = rows * cols > 1 << 22
    first, last = x.clone(), x.clone()
    first.view(-1)[0], last.view(-1)[-1] = float("-inf"), float("nan")
    odd = torch.zeros(rows, cols + 5, device=DEV, dtype=tdt)[:, 3:cols + 3]  # rows at any multiple of the element size
    odd.copy_(x)
    variants = [x, last] if big else [x, first, last, odd, x[:1].expand(rows, cols), torch.zeros_like(x)]
    for v in variants:
        for fmt, (code, f8dt) in F8.items():
            _, s_want = nat.amax_scale(v, f8dt, want_amax=False)
            for layout in {0, nat.KBLOCK_PAD}:
                want = nat.cast(v.contiguous(), s_want, f8dt, want_out_t=True, out_kblock=layout, out_t_kblock=layout)
                for ticks in (0, 200000) if not big or layout == 0 and v is x and dt == "bf16" and shape[0] < 4096 else (200000,):
                    got = [torch.zeros_like(w.view(torch.uint8)) for w in want]
                    s = torch.zeros((), device=DEV)
                    rc = nat.lib().f8mi_cast_dynamic_resident(v.data_ptr(), rows, cols, v.stride(0), nat._DT[tdt], code, s.data_ptr(), got[0].data_ptr(),
                                                              layout, got[1].data_ptr(), layout, ticks, nat._stream(x))
                    assert rc == 0, nat.lib().f8mi_last_error()
                    assert s.view(torch.int32).item() == s_want.view(torch.int32).item() or (torch.isnan(s) and torch.isnan(s_want))
                    for g, w in zip(got, want):
                        assert same_bytes_mod_nan_sign(fp8_bytes(g), fp8_bytes(w)), (dt, shape, fmt, layout, ticks)


def test_cast_dynamic_resident_on_several_streams_and_what_it_refuses(nat):
    streams = [torch.cuda.Stream() for _ in range(4)]
    xs = [heavy((1024, 1024), torch.bfloat16, 30 + i).to(DEV) for i in range(4)]
    want = [nat.cast(x, nat.amax_scale(x, torch.float8_e4m3fn, want_amax=False)[1], torch.float8_e4m3fn)[0] for x in xs]
    torch.cuda.synchronize()
    got = []
    for _ in range(20):
        for st, x in zip(streams, xs):
            with torch.cuda.stream(st):
                got.append(nat.cast_dynamic(x, torch.float8_e4m3fn)[0])
    torch.cuda.synchronize()
    for i, g in enumerate(got):
        assert torch.equal(g.view(torch.uint8), want[i % 4].view(torch.uint8))
    big = torch.zeros(4097, 4096, device=DEV, dtype=torch.bfloat16)
    o, s = torch.empty(4097, 4096, device=DEV, dtype=torch.uint8), torch.empty((), device=DEV)
    call = lambda stream, rows=4096: nat.lib().f8mi_cast_dynamic_resident(big.data_ptr(), rows, 4096, 4096, 0, 0, s.data_ptr(), o.data_ptr(), 0, None, 0, 100,
                                                                          stream.cuda_stream)
    assert call(torch.cuda.current_stream(), 4097) == -2
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):  # its word would be the same on every replay: the two launches instead
        assert call(torch.cuda.current_stream()) == -2
        q, _, sq = nat.cast_dynamic(xs[0], torch.float8_e4m3fn)
    for _ in range(3):
        xs[0].mul_(0.5)
        graph.replay()
        assert torch.equal(sq, nat.amax_scale(xs[0], torch.float8_e4m3fn, want_amax=False)[1])
        assert torch.equal(q.view(torch.uint8), nat.cast(xs[0], sq, torch.float8_e4m3fn)[0].view(torch.uint8))


def test_cast_dynamic_resident_serves_every_stream(nat):
    """64 streams of a device have words of their own; those of streams that are gone go to new ones.  One handle is a stream of its
    own in every thread."""
    import threading

    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    x = heavy((1024, 1024), torch.bfloat16, 35).to(DEV)
    want = nat.cast(x, nat.amax_scale(x, torch.float8_e4m3fn, want_amax=False)[1], torch.float8_e4m3fn)[0].view(torch.uint8)
    torch.cuda.synchronize()

    def cast(out, scale, stream):
        rc = nat.lib().f8mi_cast_dynamic_resident(x.data_ptr(), 1024, 1024, 1024, 0, 0, scale.data_ptr(), out.data_ptr(), 0, None, 0, 200000, stream)
        assert rc == 0, nat.lib().f8mi_last_error()

    outs = [torch.zeros_like(want) for _ in range(8)]
    scales = [torch.zeros((), device=DEV) for _ in outs]
    for _ in range(3):
        streams = [ctypes.c_void_p() for _ in range(40)]
        for stream in streams:
            assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
        for i, stream in enumerate(streams):
            cast(outs[i % 8], scales[i % 8], stream)
        torch.cuda.synchronize()
        assert all(torch.equal(o, want) for o in outs)
        for o in outs:
            o.zero_()
        torch.cuda.synchronize()
        assert all(hip.hipStreamDestroy(stream) == 0 for stream in streams)

    def work(i):
        torch.cuda.set_device(0)
        for _ in range(50):
            cast(outs[i], scales[i], ctypes.c_void_p(2))  # hipStreamPerThread

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs[:4])


def test_cast_dynamic_resident_costs_little_when_workgroups_are_late(nat):
    """Three launches of 1024 workgroups at once are more than the chip holds, so each waits for workgroups that have no room until
    the others' end: they read the missing tiles, and not the whole tensor each (1.4 - 2.4 ms for three casts that take 0.08 in turn).
    The same where nobody waits for anybody (13.8 ms)."""
    import time

    for dt in (torch.bfloat16, torch.float32):
        streams = [torch.cuda.Stream() for _ in range(3)]
        xs = [heavy((4096, 4096), dt, 90 + i).to(DEV) for i in range(3)]
        want = [nat.cast(x, nat.amax_scale(x, torch.float8_e4m3fn, want_amax=False)[1], torch.float8_e4m3fn)[0].view(torch.uint8) for x in xs]
        outs = [torch.empty(4096, 4096, device=DEV, dtype=torch.uint8) for _ in xs]
        scales = [torch.empty((), device=DEV) for _ in xs]

        def cast(i, stream, ticks=None):
            args = (xs[i].data_ptr(), 4096, 4096, 4096, nat._DT[dt], 0, scales[i].data_ptr(), outs[i].data_ptr(), 0, None, 0)
            if ticks is None:
                rc = nat.lib().f8mi_cast_dynamic(*args, nat.workspace(xs[i].device).data_ptr(), stream.cuda_stream)
            else:
                rc = nat.lib().f8mi_cast_dynamic_resident(*args, ticks, stream.cuda_stream)
            assert rc == 0, nat.lib().f8mi_last_error()

        def fastest(calls):  # of six rounds: one may be interrupted
            best = 1e9
            for _ in range(6):
                torch.cuda.synchronize()
                begin = time.perf_counter()
                calls()
                torch.cuda.synchronize()
                best = min(best, time.perf_counter() - begin)
            return best

        in_turn = fastest(lambda: [cast(i, streams[0]) for _ in range(20) for i in range(3)])
        at_once = fastest(lambda: [cast(i, streams[i]) for _ in range(20) for i in range(3)])
        assert at_once < 4 * in_turn, (dt, in_turn, at_once)
        for o, w in zip(outs, want):
            assert torch.equal(o, w)
            o.zero_()
        assert fastest(lambda: [cast(i, streams[0], 0) for i in range(3)]) < 3e-3
        assert all(torch.equal(o, w) for o, w in zip(outs, want))


class CastJob(ctypes.Structure):  # f8mi_cast_job
    _fields_ = ([("x", ctypes.c_void_p)] + [(f, ctypes.c_int64) for f in ("rows", "cols", "ld")] + [(f, ctypes.c_void_p) for f in ("scale", "out", "out_t", "amax")] +
                [(f, ctypes.c_int) for f in ("dtype", "layout", "layout_t")])


# The casts that exchange maxima in their launch, where nobody waits for anybody: the collecting workgroups find the maximum themselves, which
# has to be the same.  One tile, edges in both directions, several tiles a window of words; row-strided and repeated rows; NaN, infinity.
@pytest.mark.parametrize("dts", ["bf16 bf16", "fp16 fp16", "fp32 fp32", "bf16 fp32", "fp16 fp32"])
@pytest.mark.parametrize("shapes", [((1, 1), (1, 1)), ((129, 257), (64, 130)), ((1000, 3001), (513, 1031)), ((2048, 4096), (4096, 2048))])
def test_one_launch_casts_that_do_not_wait(nat, dts, shapes):
    f8dt = torch.float8_e4m3fn
    base = [heavy(s, TORCH_DT[d], 60 + i).to(DEV) for i, (s, d) in enumerate(zip(shapes, dts.split()))]
    special = [x.clone() for x in base]
    special[0].view(-1)[-1], special[1].view(-1)[0] = float("nan"), float("-inf")
    strided = [torch.zeros(x.shape[0], x.shape[1] + 5, device=DEV, dtype=x.dtype)[:, 3:x.shape[1] + 3].copy_(x) for x in base]
    repeated = [x[-1:].expand(x.shape) for x in base]
    for xs in (base, special, strided, repeated):
        for delayed in (False, True):
            want = []
            for x, s in zip(xs, (3.0, 700.0)):
                amax, s_dyn = nat.amax_scale(x.contiguous(), f8dt)
                scale = torch.tensor([s], device=DEV) if delayed else s_dyn
                q, qt = nat.cast(x.contiguous(), scale, f8dt, product_dtype=torch.float32 if delayed else None, want_out_t=True, out_kblock=2, out_t_kblock=2)
                want.append((q, qt, scale, amax))
            for which in ((0,), (1,), (0, 1)):
                jobs, got = (CastJob * 2)(), []
                for i in which:
                    x, job = xs[i], jobs[i]
                    q, qt = (torch.zeros_like(t.view(torch.uint8)) for t in want[i][:2])
                    scale, amax = want[i][2].clone() if delayed else torch.zeros((), device=DEV), torch.full((1,), -1.0, device=DEV)
                    got.append((q, qt, scale, amax))
                    job.x, job.rows, job.cols, job.ld, job.dtype = x.data_ptr(), *x.shape, x.stride(0), nat._DT[x.dtype]
                    job.scale, job.amax, job.layout, job.layout_t, job.out, job.out_t = scale.data_ptr(), amax.data_ptr(), 2, 2, q.data_ptr(), qt.data_ptr()
                rc = nat.lib().f8mi_cast_one_launch(ctypes.byref(jobs[which[0]]), ctypes.byref(jobs[1]) if len(which) == 2 else None, int(delayed), 0, nat._stream(xs[0]))
                assert rc == 0, nat.lib().f8mi_last_error()
                for i, (q, qt, scale, amax) in zip(which, got):
                    assert same_bytes_mod_nan_sign(fp8_bytes(q), fp8_bytes(want[i][0])) and same_bytes_mod_nan_sign(fp8_bytes(qt), fp8_bytes(want[i][1])), (which, delayed)
                    assert torch.equal(scale, want[i][2]) or (torch.isnan(scale).all() and torch.isnan(want[i][2]).all())
                    assert not delayed or amax.item() == want[i][3].item() or (math.isnan(amax.item()) and math.isnan(want[i][3].item()))


def test_one_launch_casts_refuse_what_is_larger(nat):
    x = torch.zeros(8193, 4096, device=DEV, dtype=torch.bfloat16)
    out, s, amax = torch.zeros(8193, 4096, device=DEV, dtype=torch.uint8), torch.ones(1, device=DEV), torch.zeros(1, device=DEV)
    job = CastJob(x.data_ptr(), 8193, 4096, 4096, s.data_ptr(), out.data_ptr(), None, amax.data_ptr(), 0, 0, 0)
    small = CastJob(x.data_ptr(), 64, 4096, 4096, s.data_ptr(), out.data_ptr(), None, amax.data_ptr(), 0, 0, 0)
    call = lambda *a: nat.lib().f8mi_cast_one_launch(*(ctypes.byref(j) if j else None for j in a[:2]), a[2], 0, nat._stream(x))
    assert [call(job, None, 0), call(job, None, 1), call(small, job, 0), call(small, job, 1)] == [-2] * 4
    small.amax = None
    assert call(small, None, 0) == 0 and call(small, None, 1) == -1 and call(None, None, 0) == -1


# Two tensors in one call: tiny, tiles of 64 and of 128 rows, the most that one launch takes together (1024 tiles, delayed 2048) and one row
# more, one or both too large for it, ragged and row-strided.
@pytest.mark.parametrize("dts", ["bf16 bf16", "fp16 fp16", "fp32 fp32", "bf16 fp32", "fp16 fp32", "fp32 bf16"])
@pytest.mark.parametrize("shapes", [((1, 1), (1, 1)), ((64, 128), (65, 129)), ((512, 1024), (1024, 1024)), ((2048, 2048), (6144, 2048)), ((2049, 2048), (6144, 2048)),
                                    ((8192, 2048), (8193, 1024)), ((8192, 4096), (300, 4096)), ((4099, 4097), (1001, 4097)), ((4099, 4096), (4480, 4096))])
def test_cast_of_two_tensors_equals_two_casts(nat, dts, shapes):
    f8dt, tdts = torch.float8_e4m3fn, [TORCH_DT[d] for d in dts.split()]
    base = [heavy(s, t, 40 + i).to(DEV) for i, (s, t) in enumerate(zip(shapes, tdts))]
    nan = [x.clone() for x in base]
    nan[1].view(-1)[-1] = float("nan")
    odd = [torch.zeros(r, c + 5, device=DEV, dtype=t)[:, 3:c + 3].copy_(x) for (r, c), t, x in zip(shapes, tdts, base)]
    for xs in (base, nan, odd):
        for layout, both in ((0, False), (nat.KBLOCK_PAD, True)):
            for delayed in (False, True):
                scales = [torch.tensor([s], device=DEV) if delayed else torch.zeros((), device=DEV) for s in (3.0, 700.0)]
                amaxes, outs, want = [torch.full((1,), -1.0, device=DEV) for _ in xs], [], []
                jobs = (CastJob * 2)()
                for x, s, a, job in zip(xs, scales, amaxes, jobs):
                    wa = torch.zeros((1,), device=DEV)
                    if delayed:
                        w = nat.cast(x, s, f8dt, product_dtype=torch.float32, want_out_t=both, amax_out=wa, out_kblock=layout, out_t_kblock=layout)
                        want.append((*w, s, wa))
                    else:
                        ws = nat.amax_scale(x, f8dt, want_amax=False)[1]
                        want.append((*nat.cast(x, ws, f8dt, want_out_t=both, out_kblock=layout, out_t_kblock=layout), ws, a))
                    o = [torch.zeros_like(t.view(torch.uint8)) if t is not None else None for t in want[-1][:2]]
                    outs.append(o)
                    job.x, job.rows, job.cols, job.ld, job.dtype = x.data_ptr(), *x.shape, x.stride(0), nat._DT[x.dtype]
                    job.scale, job.amax, job.layout, job.layout_t = s.data_ptr(), a.data_ptr(), layout, layout
                    job.out, job.out_t = o[0].data_ptr(), o[1].data_ptr() if both else None
                if delayed:
                    rc = nat.lib().f8mi_cast_delayed_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), nat.delayed_workspace(xs[0].device).data_ptr(), nat._stream(xs[0]))
                else:
                    rc = nat.lib().f8mi_cast_dynamic_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), nat.workspace(xs[0].device).data_ptr(), nat._stream(xs[0]))
                assert rc == 0, nat.lib().f8mi_last_error()
                for (w, wt, ws, wa), o, s, a in zip(want, outs, scales, amaxes):
                    assert same_bytes_mod_nan_sign(fp8_bytes(o[0]), fp8_bytes(w)), (dts, shapes, layout, delayed)
                    assert not both or same_bytes_mod_nan_sign(fp8_bytes(o[1]), fp8_bytes(wt))
                    assert torch.equal(s, ws) or (torch.isnan(s).all() and torch.isnan(ws).all())
                    assert torch.equal(a, wa) or (torch.isnan(a).all() and torch.isnan(wa).all())


# 16-bit pairs past what one tensor may have: ragged, one with more tiles than that by itself, the most tiles one launch takes together (1536) and a
# row more.  After 64 launches on this stream no other one counts.
@pytest.mark.parametrize("dts", ["bf16 bf16", "fp16 fp16", "bf16 fp32"])
@pytest.mark.parametrize("shapes", [((3000, 3000), (3100, 3001)), ((100, 100), (6000, 4090)), ((6000, 4090), (100, 100)), ((2048, 4096), (4096, 4096)),
                                    ((2049, 4096), (4096, 4096))])
def test_cast_of_two_tensors_of_up_to_six_tiles_a_cu(nat, dts, shapes):
    x, out, scale = torch.ones(64, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(64, 128, device=DEV, dtype=torch.uint8), torch.zeros((), device=DEV)
    job = CastJob(x.data_ptr(), 64, 128, 128, scale.data_ptr(), out.data_ptr(), None, None, nat._DT[x.dtype], 0, 0)
    for _ in range(64):
        assert nat.lib().f8mi_cast_one_launch(ctypes.byref(job), ctypes.byref(job), 0, 6000, nat._stream(x)) == 0
    test_cast_of_two_tensors_equals_two_casts(nat, dts, shapes)


# The same where nobody waits for anybody: more words than one tensor by itself may have, most of them missing.
@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("shapes", [((3000, 3000), (3100, 3001)), ((100, 100), (6000, 4090)), ((6000, 4090), (100, 100)), ((2048, 4096), (4096, 4096))])
def test_large_pairs_that_do_not_wait(nat, dt, shapes):
    f8dt = torch.float8_e4m3fn
    base = [heavy(s, TORCH_DT[dt], 70 + i).to(DEV) for i, s in enumerate(shapes)]
    special = [x.clone() for x in base]
    special[0].view(-1)[-1], special[1].view(-1)[0] = float("nan"), float("-inf")
    for xs in (base, special):
        jobs, got, want = (CastJob * 2)(), [], []
        for x, job in zip(xs, jobs):
            scale = nat.amax_scale(x, f8dt, want_amax=False)[1]
            want.append((*nat.cast(x, scale, f8dt, want_out_t=True, out_kblock=nat.KBLOCK_PAD, out_t_kblock=nat.KBLOCK_PAD), scale))
            got.append((*(torch.zeros_like(t.view(torch.uint8)) for t in want[-1][:2]), torch.zeros((), device=DEV)))
            job.x, job.rows, job.cols, job.ld, job.dtype, job.layout, job.layout_t = x.data_ptr(), *x.shape, x.stride(0), nat._DT[x.dtype], nat.KBLOCK_PAD, nat.KBLOCK_PAD
            job.out, job.out_t, job.scale = (t.data_ptr() for t in got[-1])
        assert nat.lib().f8mi_cast_one_launch(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), 0, 0, nat._stream(xs[0])) == 0, nat.lib().f8mi_last_error()
        for (q, qt, s), (wq, wqt, ws) in zip(got, want):
            assert same_bytes_mod_nan_sign(fp8_bytes(q), fp8_bytes(wq)) and same_bytes_mod_nan_sign(fp8_bytes(qt), fp8_bytes(wqt))
            assert torch.equal(s, ws) or (torch.isnan(s).all() and torch.isnan(ws).all())


def test_large_pairs_are_one_launch_on_two_streams_and_two_on_three(nat):
    """Three launches that fill three quarters of the chip each hold the places that the others' workgroups wait for.  A stream counts while
    it had one of the last 64 such launches."""
    xs = [heavy(s, torch.bfloat16, 90 + i).to(DEV) for i, s in enumerate([(2048, 4096), (4096, 4096), (64, 128), (64, 128)])]
    outs, scales = [torch.zeros(x.shape, device=DEV, dtype=torch.uint8) for x in xs], torch.zeros(len(xs), device=DEV)
    jobs = [CastJob(x.data_ptr(), *x.shape, x.stride(0), scales[i:].data_ptr(), outs[i].data_ptr(), None, None, nat._DT[x.dtype], 0, 0) for i, x in enumerate(xs)]
    want = [nat.cast(x, nat.amax_scale(x, torch.float8_e4m3fn)[1], torch.float8_e4m3fn)[0] for x in xs]
    streams, ws = [torch.cuda.Stream() for _ in range(3)], [torch.empty_like(nat.workspace(xs[0].device)) for _ in range(3)]
    torch.cuda.synchronize()

    def casts(first, i):
        assert nat.lib().f8mi_cast_dynamic_pair(ctypes.byref(jobs[first]), ctypes.byref(jobs[first + 1]), ws[i].data_ptr(), streams[i].cuda_stream) == 0

    def launches(i):
        nat.prof_reset()
        nat.prof_enable(True)
        try:
            casts(0, i)
        finally:
            nat.prof_enable(False)
        torch.cuda.synchronize()
        count = nat.prof_read(nat.K_CAST)[0]
        nat.prof_reset()
        for o, w in zip(outs[:2], want):
            assert torch.equal(o, w.view(torch.uint8))
            o.zero_()
        torch.cuda.synchronize()
        return count

    for _ in range(64):
        casts(2, 0)
    torch.cuda.synchronize()
    assert launches(0) == 1
    casts(2, 1)
    assert launches(0) == 1 and launches(1) == 1
    casts(2, 2)
    assert [launches(i) for i in range(3)] == [2, 2, 2]
    for _ in range(64):
        casts(2, 0)
    assert launches(0) == 1


def _rand_fp8(shape, tdt, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    v = torch.randn(shape, generator=g) * scale
    fmax = torch.finfo(tdt).max
    return v.clamp(-fmax, fmax).to(tdt)


def _gemm_check(nat, m, n, k, a_fmt, b_fmt, out_dt, seed=0, bias=False, sa=3.0, sb=0.5):
    co, to = _oracles()
    ta, tb = F8[a_fmt][1], F8[b_fmt][1]
    a = _rand_fp8((m, k), ta, seed, 4.0)
    bt = _rand_fp8((n, k), tb, seed + 1, 4.0)
    sa_t, sb_t = torch.tensor(sa), torch.tensor(sb)
    bias_t = (torch.randn(n, generator=torch.Generator().manual_seed(seed + 2)) * 3).to(out_dt) if bias else None
    got = nat.gemm_nt(a.to(DEV), sa_t.to(DEV), bt.to(DEV), sb_t.to(DEV), out_dt,
                      bias=bias_t.to(DEV) if bias else None).cpu().double()
    ad, bd = a.double() / sa, bt.double() / sb
    exact = ad @ bd.T
    if bias:
        exact = exact + bias_t.double()
    bound = ad.abs() @ bd.abs().T + (bias_t.double().abs() if bias else 0)  # elementwise magnitude of the sum
    eps_out = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-23}[out_dt]
    # stated tolerance: one output rounding + the matrix core's accumulation error.  The gfx950 fp8
    # MFMA aligns the products of a 64-deep block to the largest one and truncates below ~2^-14 of
    # it (measured; the vendor BLAS shows the same figures), so the error is bounded by 2^-13 of the
    # summed magnitudes of the terms.
    tol = eps_out * exact.abs() + 2.0**-13 * bound + 1e-30
    err = (got - exact).abs()
    worst = (err / tol).max().item()
    assert worst <= 1.0, (m, n, k, a_fmt, b_fmt, out_dt, worst)
    # and against the reference's emulated op itself (fp32 mm on CPU), north-star bar 1e-2
    emu = to.mm_emulated(a, sa_t, bt.t(), sb_t, out_dt)
    if bias:
        emu = emu + bias_t
    # (with a bias the emulated route rounds twice in the output dtype, product then sum: two output ulps of slack)
    allow = 1e-2 * (emu.double().abs() + 1e-2 * bound.max()) + (2 * eps_out * (emu.double().abs() + bias_t.double().abs()) if bias else 0)
    rel = ((got - emu.double()).abs() / allow).max().item()
    assert rel <= 1.0, (m, n, k, rel)


@pytest.mark.parametrize("m,n,k", [(256, 256, 128), (256, 256, 256), (512, 768, 384), (16, 32, 16), (1, 1, 1),
                                   (300, 520, 200), (257, 255, 129), (64, 4096, 1024), (1000, 3000, 4099 // 4 * 4),
                                   (129, 77, 4097), (40, 50, 1000), (2048, 512, 2048)])
def test_gemm_shapes(nat, m, n, k):
    _gemm_check(nat, m, n, k, "e4m3", "e4m3", torch.bfloat16, seed=m + n + k)


# The library has two GEMM kernels: 16-byte aligned operands with k % 64 == 0 and k >= 384 take the
# LDS-DMA kernel (compiled separately for an odd and an even count of 64-deep units), everything
# else the register-staged one.  k = 384 .. 704 walks the shortest pipelines of both parities,
# ragged m / n exercise the clamped edge rows, 8192 a long steady state.
@pytest.mark.parametrize("m,n,k", [(256, 256, 384), (256, 256, 448), (300, 200, 512), (257, 511, 576), (64, 96, 640),
                                   (512, 256, 704), (1, 1, 384), (520, 264, 8192), (256, 512, 8256)])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float32])
def test_gemm_dma_kernel_shapes(nat, m, n, k, out_dt):
    _gemm_check(nat, m, n, k, "e5m2", "e4m3", out_dt, seed=m + n + k, bias=(m % 2 == 0))


# Tiles of 256 x 224: whole ones, a last column of tiles of 2, 112, 114, 220 and 222 columns, ragged rows, an odd and an even number of steps,
# every output type, against 128-row tiles (the same order of additions, hence the same bits) of both ends of the rows.
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(2048, 14336, 512), (2000, 14112 + 2, 384), (2048, 14112 + 112, 384), (1801, 14112 + 114, 640), (2048, 14112 + 222, 512), (2047, 14332, 384)])
def test_gemm_narrow_tiles_equal_128_row_tiles_bitwise(nat, m, n, k, out_dt):
    assert nat.gemm_plan(m, n, k) == ("tiles256x224", 0, 0)
    a, bt = _rand_fp8((m, k), torch.float8_e5m2, 61).to(DEV), _rand_fp8((n, k), torch.float8_e4m3fn, 62).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.37, device=DEV)
    bias = torch.linspace(-1, 1, n).to(out_dt).to(DEV)
    for b in (None, bias):
        buf = torch.full((m + 1, n), 7.0, device=DEV, dtype=out_dt)
        got = nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b, out=buf[:m])
        assert (buf[m] == 7).all()
        for rows in (slice(0, 272), slice(m - 300, m)):
            for cols in (slice(0, 4096), slice(4096, 8192), slice(8192, 12288), slice(12288, n)):
                assert nat.gemm_plan(rows.stop - rows.start, cols.stop - cols.start, k)[0] == "tiles128"
                want = nat.gemm_nt(a[rows], sa, bt[cols], sb, out_dt, bias=None if b is None else b[cols].contiguous())
                assert torch.equal(got[rows, cols], want), (rows, cols)


# An odd number of columns: 1, 111, 113 and 223 in the last column of tiles.  The plan answers for a dense 16-bit C, whose odd rows are for the
# large tiles; fp32, and 16-bit rows at an even pitch, take these.
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(2048, 14112 + 1, 384), (2000, 14112 + 111, 512), (1801, 14112 + 113, 640), (2048, 14112 + 223, 384)])
def test_gemm_narrow_tiles_of_odd_columns(nat, m, n, k, out_dt):
    assert nat.gemm_plan(m, n + 1, k)[0] == "tiles256x224" and nat.gemm_plan(m, n, k)[0] == "tiles256"
    pitch = n if out_dt == torch.float32 else n + 1
    a, bt = _rand_fp8((m, k), torch.float8_e4m3fn, 63).to(DEV), _rand_fp8((n, k), torch.float8_e5m2, 64).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.37, device=DEV)
    bias = torch.linspace(-1, 1, n).to(out_dt).to(DEV)
    for b in (None, bias):
        buf = torch.full((m + 1, pitch), 7.0, device=DEV, dtype=out_dt)
        rc = nat.lib().f8mi_gemm_nt(a.data_ptr(), 0, k, bt.data_ptr(), 1, k, m, n, k, sa.data_ptr(), sb.data_ptr(), buf.data_ptr(), nat._DT[out_dt], pitch,
                                    None if b is None else b.data_ptr(), nat._stream(a))
        assert rc == 0, nat.lib().f8mi_last_error()
        assert (buf[m] == 7).all() and (buf[:m, n:] == 7).all()
        for rows in (slice(0, 272), slice(m - 300, m)):
            for cols in (slice(0, 4096), slice(4096, 8192), slice(8192, 12288), slice(12288, n)):
                want = nat.gemm_nt(a[rows], sa, bt[cols], sb, out_dt, bias=None if b is None else b[cols].contiguous())
                assert torch.equal(buf[rows, cols], want), (rows, cols)


# Rows of C that start at odd multiples of two bytes (an odd pitch, or a C that starts at one): every column remainder of a lane's eight
# and of a wave's 128, in tiles of 128 x 128, 128 x 256 and 256 x 256, against the same product in rows at multiples of four bytes.
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n", [(300, 384, n) for n in (1, 7, 8, 9, 63, 121, 127, 128, 129, 135, 255)] +
                         [(2100, 512, n) for n in (2041, 2049)] + [(4099, 384, n) for n in (4611, 4625, 4735)] + [(8192, 512, 4095)])
def test_gemm_rows_of_c_at_odd_addresses(nat, m, k, n, out_dt):
    a, bt = (_rand_fp8((k // 64, rows, 64), torch.float8_e4m3fn, 50 + i, 4.0).to(DEV) for i, rows in enumerate((m, n)))
    one, code = torch.ones((), device=DEV), nat._DT[out_dt]

    def product(pitch, start):
        buf = torch.full((m * pitch + start + 16,), 7.0, device=DEV, dtype=out_dt)
        rc = nat.lib().f8mi_gemm_nt_kb(a.data_ptr(), 0, bt.data_ptr(), 0, m, n, k, one.data_ptr(), one.data_ptr(), buf.data_ptr() + 2 * start, code, pitch, None,
                                       nat._stream(one))
        assert rc == 0, nat.lib().f8mi_last_error()
        c = buf[start:start + m * pitch].view(m, pitch)
        assert (buf[:start] == 7).all() and (buf[start + m * pitch:] == 7).all() and (c[:, n:] == 7).all()
        return c[:, :n]

    want = product((n + 1) // 2 * 2, 0)
    for pitch, start in {(n | 1, 0), (n | 1, 1), ((n + 1) // 2 * 2, 1), ((n + 4) | 1, 3)}:
        assert torch.equal(product(pitch, start), want), (pitch, start)


# Few rows (m <= 256, k % 128 == 0, aligned): the kernel that streams Bt straight into the matrix cores and splits k
# over the eight waves of a workgroup.  m around the 16-row tile edges, n ragged against the 32-column
# workgroups, k from one step (seven idle waves) over nine (uneven split) to a long one.
@pytest.mark.parametrize("m", [1, 5, 16, 17, 32, 33, 64, 65, 100, 128, 129, 200, 256])
@pytest.mark.parametrize("n,k", [(7, 128), (32, 256), (200, 1152), (1000, 1024), (96, 8192)])
def test_gemm_few_rows_shapes(nat, m, n, k):
    fm = [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")][(m + n) % 4]
    out_dt = [torch.bfloat16, torch.float32, torch.float16][(m + k // 128) % 3]
    _gemm_check(nat, m, n, k, fm[0], fm[1], out_dt, seed=m + n + k, bias=(m % 2 == 1))


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (16, 520, 2048), (48, 1000, 640), (64, 264, 8192), (120, 264, 1024), (250, 520, 2048)])
def test_gemm_few_rows_kblocked_equals_row_major_bitwise(nat, m, n, k):
    a = _rand_fp8((m, k), torch.float8_e4m3fn, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(2.0, device=DEV), torch.tensor(0.25, device=DEV)
    bias = torch.randn(n, device=DEV).to(torch.bfloat16)
    want = nat.gemm_nt(a, sa, bt, sb, torch.bfloat16, bias=bias)
    got = nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, torch.bfloat16, bias=bias)
    assert torch.equal(got, want)
    # rows are independent: any subset of A's rows gives the same rows of C, whichever tile count it lands in
    sub = nat.gemm_nt(a[: max(1, m // 3)].contiguous(), sa, bt, sb, torch.bfloat16, bias=bias)
    assert torch.equal(sub, want[: max(1, m // 3)])


# Outputs that at most 256 tiles of 128 x 128 or of 128 x 256 cover (k % 128 == 0), unless the few-row kernel is
# estimated to be faster, take those tiles.
@pytest.mark.parametrize("m,n,k", [(257, 128, 128), (300, 520, 1024), (512, 1000, 256), (1024, 2048, 640), (384, 8192, 2048),
                                   (4099, 500, 1152), (1024, 8192, 1024), (1000, 5000, 384), (2049, 3000, 128),
                                   (64, 28672, 512), (20, 16384, 256)])  # few rows, wide Bt: one partial row of tiles
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float32])
def test_gemm_mid_tile_kernel_shapes(nat, m, n, k, out_dt):
    fm = [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")][(m + n + k // 128) % 4]
    _gemm_check(nat, m, n, k, fm[0], fm[1], out_dt, seed=m + n + k, bias=(n % 2 == 0))


# One to eight 128-deep steps: shorter and longer than the three (128 x 256) and five (128 x 128) stages in flight.
@pytest.mark.parametrize("steps", range(1, 9))
@pytest.mark.parametrize("m,n,mid", [(257, 200, 1), (1300, 4008, 2)])
def test_gemm_mid_tile_kernel_step_counts(nat, m, n, mid, steps):
    assert nat.gemm_plan(m, n, 128 * steps) == ("tiles128", 0, mid)
    for out_dt in (torch.bfloat16, torch.float32):
        _gemm_check(nat, m, n, 128 * steps, "e4m3", "e5m2", out_dt, seed=m + steps, bias=True)


# Both tile widths of the 128-row kernel (1: 128 x 128, 2: 128 x 256) and large tiles with a sparse last round (0), edges at half
# a tile, three to nine steps (the stages in flight are five and three).
@pytest.mark.parametrize("m,n,k,mid", [(192, 320, 384, 1), (64, 64, 640, 1), (1024, 1088, 512, 1), (128, 4096, 1152, 1), (448, 8128, 768, 1),
                                       (1344, 4032, 384, 2), (2048, 2304, 512, 2), (1984, 4096, 640, 2), (1088, 6464, 1152, 2),
                                       (4352, 4096, 512, 0), (4416, 4032, 384, 0)])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float32])
def test_gemm_mid_tile_kernel_reads_transposed_operands(nat, m, n, k, mid, out_dt):
    """The same bits as on operands that are not transposed, for one and for both of them transposed."""
    rows = m if m > 256 else 272  # past the few-row kernel, for the operands that are not transposed
    plan = nat.gemm_plan(rows, n, k, split_k=False)
    assert plan[0] == ("tiles256_and_128" if mid == 0 else "tiles128") and (mid == 0 or plan[2] == mid)
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(2.0, device=DEV), torch.tensor(0.25, device=DEV)
    turned = lambda t: _to_kb(t.view(torch.uint8).t().contiguous().view(t.dtype))
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(out_dt).to(DEV)
    tall = torch.cat([a.view(torch.uint8), torch.zeros(rows - m, k, dtype=torch.uint8, device=DEV)]).view(a.dtype)
    want = nat.gemm_nt_kb(_to_kb(tall), sa, _to_kb(bt), sb, out_dt, bias=bias, split_k=False)[:m]
    assert torch.equal(nat.gemm_kb_ex(_to_kb(a), False, sa, turned(bt), True, sb, out_dt, bias=bias), want)
    assert torch.equal(nat.gemm_kb_ex(turned(a), True, sa, turned(bt), True, sb, out_dt, bias=bias), want)


class GemmJob(ctypes.Structure):  # f8mi_gemm_job
    _fields_ = ([(f, ctypes.c_void_p) for f in ("a", "bt")] + [(f, ctypes.c_int) for f in ("a_fmt", "b_fmt", "a_tr", "b_tr")] +
                [(f, ctypes.c_int64) for f in ("m", "n", "k")] + [(f, ctypes.c_void_p) for f in ("sa", "sb", "c")] +
                [("ldc", ctypes.c_int64), ("dtype", ctypes.c_int), ("ws", ctypes.c_void_p), ("ws_bytes", ctypes.c_int64)])


# Both products of a backward in one launch, on each of its tiles and by the rule: grad_input (tokens x features) and grad_weight of one gradient,
# operands read transposed (multiples of 128) or as they are (any size); one tile and edges of tiles, odd and even step counts on either
# side, which of the two is longer, more than one round of workgroups, more than eight tile rows.
@pytest.mark.parametrize("tokens,k,n", [(384, 384, 384), (512, 1024, 1024), (640, 384, 1152), (1408, 512, 640), (2432, 1280, 4864), (2304, 4096, 512),
                                        (385, 391, 413), (700, 1001, 391), (1025, 515, 4099), (4133, 739, 862)])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16, torch.float32])
def test_gemm_pair_equals_the_products_one_by_one(nat, tokens, k, n, out_dt):
    g = _rand_fp8((tokens, n), torch.float8_e5m2, tokens + n, 4.0).to(DEV)
    w = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    x = _rand_fp8((tokens, k), torch.float8_e4m3fn, tokens + k, 4.0).to(DEV)
    sg, sw, sx = (torch.tensor(s, device=DEV) for s in (2.0, 0.25, 0.5))
    transposed = tokens % 128 == 0 and k % 128 == 0 and n % 128 == 0
    turned = lambda t: t.view(torch.uint8).t().contiguous().view(t.dtype)
    pad = lambda v: -(-v // 128) * 128
    forms = [(False, [_to_kb_padded(t)[0] for t in (g, turned(w), turned(g), turned(x))])]
    if transposed:
        forms.append((True, [_to_kb(g), _to_kb(w), _to_kb(g), _to_kb(x)]))
    for tr, (a0, b0, a1, b1) in forms:
        shapes = (tokens, k, pad(n)), (n, k, pad(tokens))
        if tr:
            want = [nat.gemm_kb_ex(a0, False, sg, b0, True, sw, out_dt), nat.gemm_kb_ex(a1, True, sg, b1, True, sx, out_dt)]
        else:
            want = [nat.gemm_nt_kb(a0, sg, b0, sw, out_dt, split_k=False), nat.gemm_nt_kb(a1, sg, b1, sx, out_dt, split_k=False)]
        jobs, got = (GemmJob * 2)(), [torch.empty_like(t) for t in want]
        for job, a, b, sb, (rows, cols, kc), c, a_tr in zip(jobs, (a0, a1), (b0, b1), (sw, sx), shapes, got, (0, int(tr))):
            job.a, job.bt, job.a_fmt, job.b_fmt, job.a_tr, job.b_tr = a.data_ptr(), b.data_ptr(), nat.E5M2, nat.E4M3FN, a_tr, int(tr)
            job.m, job.n, job.k, job.sa, job.sb, job.c, job.ldc, job.dtype = rows, cols, kc, sg.data_ptr(), sb.data_ptr(), c.data_ptr(), cols, nat._DT[out_dt]
        for tiles in (0, *(p | q << 2 for p in (1, 2, 3) for q in (1, 2, 3))):
            for t in got:
                t.fill_(float("nan"))
            assert nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), tiles, nat._stream(g)) == 0, nat.lib().f8mi_last_error()
            assert all(torch.equal(a, b) for a, b in zip(got, want)), (tr, tiles)
        jobs[1].b_fmt = nat.E5M2  # what one launch does not take is two by the rule, and refused by name
        assert nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), 15, nat._stream(g)) == nat.ERR_UNSUPPORTED


# Results in the columns of a wider matrix: rows at even and odd pitches and addresses, the same and different ones for the two products (which one
# launch takes only from operands read transposed); the columns beside them are left alone.
@pytest.mark.parametrize("tokens,k,n", [(385, 391, 413), (512, 1024, 1024), (1408, 512, 640)])
@pytest.mark.parametrize("wider,at", [((3, 0), (0, 0)), ((1, 1), (1, 0)), ((2, 1), (0, 1)), ((2, 2), (1, 1)), ((2, 4), (0, 1))])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float32])
def test_gemm_pair_writes_into_wider_matrices(nat, tokens, k, n, wider, at, out_dt):
    g, w, x = (_rand_fp8(s, t, sum(s), 4.0).to(DEV) for s, t in (((tokens, n), torch.float8_e5m2), ((n, k), torch.float8_e4m3fn), ((tokens, k), torch.float8_e4m3fn)))
    sg, sw, sx = (torch.tensor(s, device=DEV) for s in (2.0, 0.25, 0.5))
    turned = lambda t: t.view(torch.uint8).t().contiguous().view(t.dtype)
    pad = lambda v: -(-v // 128) * 128
    forms = [(0, [_to_kb_padded(t)[0] for t in (g, turned(w), turned(g), turned(x))])]
    if tokens % 128 == 0 and k % 128 == 0 and n % 128 == 0:
        forms.append((1, [_to_kb(g), _to_kb(w), _to_kb(g), _to_kb(x)]))
    for tr, (a0, b0, a1, b1) in forms:
        if tr:
            want = [nat.gemm_kb_ex(a0, False, sg, b0, True, sw, out_dt), nat.gemm_kb_ex(a1, True, sg, b1, True, sx, out_dt)]
        else:
            want = [nat.gemm_nt_kb(a0, sg, b0, sw, out_dt, split_k=False), nat.gemm_nt_kb(a1, sg, b1, sx, out_dt, split_k=False)]
        jobs = (GemmJob * 2)()
        memory = [torch.empty(c.shape[0] * (c.shape[1] + more) + at_, device=DEV, dtype=out_dt) for c, more, at_ in zip(want, wider, at)]
        rows_of = lambda i: memory[i][at[i]:].view(want[i].shape[0], -1)
        for i, (job, a, b, sb, (rows, cols, kc), a_tr) in enumerate(zip(jobs, (a0, a1), (b0, b1), (sw, sx), ((tokens, k, pad(n)), (n, k, pad(tokens))), (0, tr))):
            job.a, job.bt, job.a_fmt, job.b_fmt, job.a_tr, job.b_tr = a.data_ptr(), b.data_ptr(), nat.E5M2, nat.E4M3FN, a_tr, tr
            job.m, job.n, job.k, job.sa, job.sb, job.c, job.ldc, job.dtype = rows, cols, kc, sg.data_ptr(), sb.data_ptr(), rows_of(i).data_ptr(), cols + wider[i], nat._DT[out_dt]
        odd = [out_dt is not torch.float32 and bool(job.ldc % 2 or job.c % 4) for job in jobs]
        for tiles in (0, 1 | 1 << 2, 2 | 2 << 2, 3 | 3 << 2):
            for t in memory:
                t.fill_(7.0)
            rc = nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), tiles, nat._stream(g))
            if tiles and not tr and odd[0] != odd[1]:
                assert rc == nat.ERR_UNSUPPORTED
                continue
            assert rc == 0, nat.lib().f8mi_last_error()
            for i, c in enumerate(want):
                assert torch.equal(rows_of(i)[:, :c.shape[1]], c) and (rows_of(i)[:, c.shape[1]:] == 7.0).all() and (memory[i][:at[i]] == 7.0).all(), (tr, tiles, i)


# By the rule, one launch where the estimate for it is clearly the lower one, two where it is within the estimates' error (measured slower: by 8 and
# 7 %) or higher.
@pytest.mark.parametrize("tokens,k,n,launches", [(512, 1024, 1024, 1), (2048, 4096, 4096, 1), (640, 18048, 5248, 2), (6656, 2048, 3584, 2), (4096, 4096, 4096, 2)])
def test_gemm_pair_is_one_launch_where_the_estimate_is_clear(nat, tokens, k, n, launches):
    g, w, x = (torch.zeros(a * b, device=DEV, dtype=torch.uint8) for a, b in ((tokens, n), (n, k), (tokens, k)))
    got, one = [torch.ones(a, k, device=DEV, dtype=torch.bfloat16) for a in (tokens, n)], torch.ones((), device=DEV)
    jobs = (GemmJob * 2)()
    for job, b, (rows, cols, kc), c, a_tr in zip(jobs, (w, x), ((tokens, k, n), (n, k, tokens)), got, (0, 1)):
        job.a, job.bt, job.a_fmt, job.b_fmt, job.a_tr, job.b_tr = g.data_ptr(), b.data_ptr(), nat.E5M2, nat.E4M3FN, a_tr, 1
        job.m, job.n, job.k, job.sa, job.sb, job.c, job.ldc, job.dtype = rows, cols, kc, one.data_ptr(), one.data_ptr(), c.data_ptr(), cols, nat._DT[torch.bfloat16]
    nat.prof_reset()
    nat.prof_enable(True)
    try:
        assert nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), 0, nat._stream(g)) == 0, nat.lib().f8mi_last_error()
    finally:
        nat.prof_enable(False)
    count = nat.prof_read(nat.K_GEMM)[0]
    nat.prof_reset()
    assert count == launches and not any(t.any() for t in got)


# grad_weight's 16-bit result stored in fp32, beside grad_input in one launch on each of the tiles and by itself (a first product that one launch
# does not take): 128 x 128, 128 x 256, 256 x 256 with and without a sparse last round, 256 x 224; odd and even step counts, odd rows of grad_input.
@pytest.mark.parametrize("tokens,k,n", [(384, 1024, 512), (512, 4096, 2048), (384, 4096, 4096), (512, 4096, 4352), (384, 14336, 2048), (512, 513, 700),
                                        (500, 4095, 2100), (390, 14301, 2000)])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16])
def test_gemm_pair_stores_a_16_bit_gradient_in_fp32(nat, tokens, k, n, out_dt):
    g = _rand_fp8((tokens, n), torch.float8_e5m2, tokens + n, 4.0).to(DEV)
    w = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    x = _rand_fp8((tokens, k), torch.float8_e4m3fn, tokens + k, 4.0).to(DEV)
    sg, sw, sx = (torch.tensor(s, device=DEV) for s in (2.0, 0.25, 0.5))
    turned = lambda t: t.view(torch.uint8).t().contiguous().view(t.dtype)
    pad = lambda v: -(-v // 128) * 128
    forms = [(0, [_to_kb_padded(t)[0] for t in (g, turned(w), turned(g), turned(x))])]
    if tokens % 128 == 0 and k % 128 == 0 and n % 128 == 0:
        forms.append((1, [_to_kb(g), _to_kb(w), _to_kb(g), _to_kb(x)]))
    for tr, (a0, b0, a1, b1) in forms:
        if tr:
            want = [nat.gemm_kb_ex(a0, False, sg, b0, True, sw, out_dt), nat.gemm_kb_ex(a1, True, sg, b1, True, sx, out_dt)]
        else:
            want = [nat.gemm_nt_kb(a0, sg, b0, sw, out_dt, split_k=False), nat.gemm_nt_kb(a1, sg, b1, sx, out_dt, split_k=False)]
        want[1] = want[1].float()
        jobs, got = (GemmJob * 2)(), [torch.empty_like(t) for t in want]
        wide = 3 if out_dt is torch.bfloat16 else 4  # F8MI_BF16_IN_FP32, F8MI_FP16_IN_FP32
        for job, a, b, sb, (rows, cols, kc), c, a_tr, dt in zip(jobs, (a0, a1), (b0, b1), (sw, sx), ((tokens, k, pad(n)), (n, k, pad(tokens))), got, (0, tr),
                                                                (nat._DT[out_dt], wide)):
            job.a, job.bt, job.a_fmt, job.b_fmt, job.a_tr, job.b_tr = a.data_ptr(), b.data_ptr(), nat.E5M2, nat.E4M3FN, a_tr, tr
            job.m, job.n, job.k, job.sa, job.sb, job.c, job.ldc, job.dtype = rows, cols, kc, sg.data_ptr(), sb.data_ptr(), c.data_ptr(), cols, dt
        for tiles in (0, *(p | q << 2 for p in (1, 2, 3) for q in (1, 2, 3)), None):
            for t in got:
                t.fill_(float("nan"))
            if tiles is None:
                jobs[0].b_fmt = nat.E5M2
            assert nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), tiles or 0, nat._stream(g)) == 0, nat.lib().f8mi_last_error()
            assert (tiles is None or torch.equal(got[0], want[0])) and torch.equal(got[1], want[1]), (tr, tiles)
        jobs[1].b_fmt = nat.E5M2  # no such kernel: refused, and nothing queued
        got[0].fill_(0.0)
        assert nat.lib().f8mi_gemm_pair(ctypes.byref(jobs[0]), ctypes.byref(jobs[1]), 0, nat._stream(g)) == nat.ERR_UNSUPPORTED
        assert not got[0].any()


# A bias added to the rounded product, on each of the tiles that take it: 128 x 128, 128 x 256, 256 x 256 with and without a sparse last round,
# 256 x 224, odd and even step counts and rows of C; refused where the product runs on other kernels.
@pytest.mark.parametrize("m,n,k,plan", [(300, 200, 512, "tiles128"), (257, 511, 384, "tiles128"), (2048, 4000, 640, "tiles128"), (2040, 3999, 384, "tiles128"),
                                        (4096, 4096, 384, "tiles256"), (4090, 4095, 512, "tiles256"), (4352, 4095, 640, "tiles256_and_128"),
                                        (2048, 14336, 512, "tiles256x224"), (2000, 14300, 384, "tiles256x224"), (16, 512, 512, None), (64, 2048, 8192, None)])
@pytest.mark.parametrize("out_dt,bias_dt", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                            (torch.float16, torch.float16), (torch.float32, torch.float32)])
def test_gemm_adds_a_bias_to_the_rounded_product(nat, m, n, k, plan, out_dt, bias_dt):
    a, bt = (_rand_fp8((r, k), torch.float8_e4m3fn, r + k + i, 4.0).to(DEV) for i, r in enumerate((m, n)))
    sa, sb = torch.tensor(2.0, device=DEV), torch.tensor(0.25, device=DEV)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(bias_dt).to(DEV)
    c, ka, kbt = torch.full((m, n), float("nan"), device=DEV, dtype=out_dt), _to_kb(a), _to_kb(bt)
    call = lambda dt: nat.lib().f8mi_gemm_kb_bias(ka.data_ptr(), kbt.data_ptr(), m, n, k, sa.data_ptr(), sb.data_ptr(), c.data_ptr(), nat._DT[out_dt], n,
                                                  bias.data_ptr(), dt, nat.GEMM_WORKSPACE_BYTES, nat._stream(a))
    if plan is None:
        assert call(nat._DT[bias_dt]) == nat.ERR_UNSUPPORTED
        return
    assert nat.gemm_plan(m, n, k)[0] == plan
    assert call(nat._DT[bias_dt]) == 0, nat.lib().f8mi_last_error()
    want = nat.gemm_nt_kb(ka, sa, kbt, sb, out_dt) + bias.to(out_dt)
    assert torch.equal(c, want)
    for more, at in ((1, 0), (2, 1), (3, 1)):  # into a wider matrix: rows at other pitches and addresses, which other tiles may take
        memory = torch.full((m * (n + more) + at,), 7.0, device=DEV, dtype=out_dt)
        rows = memory[at:].view(m, n + more)
        rc = nat.lib().f8mi_gemm_kb_bias(ka.data_ptr(), kbt.data_ptr(), m, n, k, sa.data_ptr(), sb.data_ptr(), rows.data_ptr(), nat._DT[out_dt], n + more,
                                         bias.data_ptr(), nat._DT[bias_dt], nat.GEMM_WORKSPACE_BYTES, nat._stream(a))
        assert rc == 0, nat.lib().f8mi_last_error()
        assert torch.equal(rows[:, :n], want) and (rows[:, n:] == 7.0).all() and (memory[:at] == 7.0).all()


# One row and one workgroup's rows with one more or less; columns that leave a lane some of its eight or four; several chunks; rows at any
# distance and alignment.  Any order of fp32 additions is within rows * 2^-24 of the sum of the magnitudes; then the rounding to x's type (half an
# ulp: 2^-8 of a number with 8 bits, 2^-11, 2^-24) and to the bias's.
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (31, 512), (32, 513), (33, 256), (129, 1031), (4096, 4096), (4099, 11007), (20000, 24), (700, 70001)])
@pytest.mark.parametrize("dt,out_dt", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float16, torch.float32), (torch.float32, torch.float32),
                                       (torch.float32, torch.bfloat16)])
def test_column_sum(nat, rows, cols, dt, out_dt):
    base = heavy((rows, cols + 5), torch.float32, rows + cols).clamp(-100, 100).to(dt).to(DEV)
    for x in (base[:, :cols].contiguous(), base[:, 3:cols + 3]):
        need = nat.lib().f8mi_column_sum_workspace_bytes(rows, cols, nat._DT[dt])
        ws, out = torch.empty(max(need // 4, 1), device=DEV), torch.full((cols,), float("nan"), device=DEV, dtype=out_dt)
        call = lambda t: nat.lib().f8mi_column_sum(t.data_ptr(), rows, cols, t.stride(0), nat._DT[dt], out.data_ptr(), nat._DT[out_dt], ws.data_ptr(), need, nat._stream(t))
        assert call(x) == 0, nat.lib().f8mi_last_error()
        want, half = x.double().sum(0), {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}
        bound = rows * 2.0**-24 * x.double().abs().sum(0)
        bound = bound + (want.abs() + bound) * (half[dt] + half[out_dt] * 1.01) + 2.0**-24  # (fp16: half of its smallest number)
        assert ((out.double() - want).abs() <= bound).all()
        again = out.clone()
        assert call(x) == 0 and torch.equal(out, again)  # a fixed order
    x = base[:, :cols].clone()
    x[rows // 2, cols // 2], x[0, 0] = float("inf"), float("nan")
    assert call(x) == 0 and torch.isnan(out[0]) and (cols == 1 or out[cols // 2] == float("inf") or cols // 2 == 0)
    assert call(x) == 0 and torch.isfinite(out).sum() == cols - len({0, cols // 2})


# Few rows: one to three 128-deep steps per wave and one more or less of them, on each block of rows and both widths.
@pytest.mark.parametrize("m,n,k", [(m, n, k) for m, n in ((1, 1000), (16, 4104), (17, 40), (32, 1000), (33, 40), (64, 1000))
                                   for k in (128, 896, 1024, 1152, 2048, 2176, 3200) if m <= 16 or k > 128])
def test_gemm_few_rows_step_counts(nat, m, n, k):
    assert nat.gemm_plan(m, n, k)[0] == "few_rows"
    for out_dt in (torch.bfloat16, torch.float32):
        _gemm_check(nat, m, n, k, "e5m2", "e4m3", out_dt, seed=m + k, bias=(k % 256 == 0))


# Few 128-row tiles and a long contraction: with the stream's scratch buffer k is split over workgroups and a second
# kernel adds the parts in a fixed order.
@pytest.mark.parametrize("m,n,k", [(256, 2048, 16384), (512, 1024, 8192), (100, 4096, 16384)])
def test_gemm_split_over_k(nat, m, n, k):
    a = _rand_fp8((m, k), torch.float8_e4m3fn, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e5m2, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(0.5, device=DEV), torch.tensor(4.0, device=DEV)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(torch.bfloat16).to(DEV)
    split32 = nat.gemm_nt(a, sa, bt, sb, torch.float32)
    whole32 = nat.gemm_nt(a, sa, bt, sb, torch.float32, split_k=False)
    # another summation order (else the split did not run) but the same sums to fp32 accuracy, every time the same bits,
    # whichever layout the operands come in
    assert not torch.equal(split32, whole32)
    scale = whole32.abs().max()
    assert ((split32 - whole32).abs().max() / scale).item() < 1e-5
    assert torch.equal(nat.gemm_nt(a, sa, bt, sb, torch.float32), split32)
    assert torch.equal(nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, torch.float32), split32)
    got = nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, torch.bfloat16, bias=bias)
    assert torch.equal(got, nat.gemm_nt(a, sa, bt, sb, torch.bfloat16, bias=bias))
    want = (split32 + bias.float()).to(torch.bfloat16)  # one rounding of the scaled sum plus bias
    assert ((got.float() - want.float()).abs() <= 2 * torch.finfo(torch.bfloat16).eps * want.float().abs() + 1e-6).all()
    _gemm_check(nat, m, n, k, "e4m3", "e5m2", torch.bfloat16, seed=m + n, bias=True)


def test_gemm_split_over_k_random_shapes(nat):
    """Seeded shapes around the limits of the split (rows, ragged n, parts of k): whatever the plan, the result with
    the scratch buffer agrees with the one without to fp32 accuracy, and some of the shapes do get split."""
    import random

    rng = random.Random(1234)
    sa, sb = torch.tensor(2.0, device=DEV), torch.tensor(0.25, device=DEV)
    split = 0
    for case in range(14):
        m = rng.choice([17, 33, 64, 100, 128, 129, 200, 256, 257, 384, 512, 640])
        n = 4 * rng.randint(64, 768)
        k = 128 * rng.choice([32, 40, 64, 96, 112, 128, 192])
        name, parts, _ = nat.gemm_plan(m, n, k)
        split += name == "tiles128_split_k"
        a = _rand_fp8((m, k), torch.float8_e4m3fn, case, 4.0).to(DEV)
        bt = _rand_fp8((n, k), torch.float8_e4m3fn, case + 100, 4.0).to(DEV)
        with_ws = nat.gemm_nt(a, sa, bt, sb, torch.float32)
        without = nat.gemm_nt(a, sa, bt, sb, torch.float32, split_k=False)
        tol = 1e-5 if nat.gemm_plan(m, n, k, split_k=False)[0] != "few_rows" or name == "tiles128_split_k" else 0.0
        err = ((with_ws - without).abs().max() / without.abs().max()).item()
        assert err <= max(tol, 1e-5), (m, n, k, name, parts, err)
        if name != "tiles128_split_k":
            assert torch.equal(with_ws, without), (m, n, k, name)
        assert torch.equal(nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, torch.float32), with_ws), (m, n, k, name)
    assert split >= 3, split


# More than one round of 256 x 256 tiles with few tiles in the last one: the last tile rows go to a 128-row-tile kernel.
@pytest.mark.parametrize("m,n,k,m_pad", [(4352, 4096, 512, 8192),      # 272 tiles: 16 of them as 128 x 128 tiles
                                         (8500, 2048, 384, 16384),     # ragged last tile row
                                         (6144, 4096, 640, 8192),      # 384 tiles: 128 of them as 128 x 256 tiles
                                         (16640, 4000, 384, 20480)])   # four full rounds, then 16 tiles; ragged columns
def test_gemm_split_of_a_sparse_last_round_changes_no_bit(nat, m, n, k, m_pad):
    """Reference: the same rows inside a matrix padded with zero rows to whole rounds, which the large-tile kernel
    computes alone."""
    a = _rand_fp8((m, k), torch.float8_e4m3fn, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e5m2, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(0.5, device=DEV), torch.tensor(4.0, device=DEV)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(torch.bfloat16).to(DEV)
    assert (m_pad // 256) * ((n + 255) // 256) % 256 == 0
    a_pad = torch.cat([a.view(torch.uint8), torch.zeros(m_pad - m, k, dtype=torch.uint8, device=DEV)]).view(a.dtype)
    for out_dt, b in ((torch.bfloat16, bias), (torch.float32, None)):
        want = nat.gemm_nt(a_pad, sa, bt, sb, out_dt, bias=b)[:m]
        assert torch.equal(nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b), want)
        assert torch.equal(nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, out_dt, bias=b), want)
    _gemm_check(nat, m, n, k, "e4m3", "e5m2", torch.bfloat16, seed=m + n, bias=True)


@pytest.mark.parametrize("m,n,k", [(300, 520, 1024), (1000, 264, 2048), (512, 1024, 384), (1100, 4500, 640),
                                   (200, 8192, 512),     # 129 - 256 rows and a wide Bt: the 128-row tiles, not the few-row kernel
                                   (100, 16384, 384)])   # so do 17 - 128 rows when Bt is wide enough
def test_gemm_mid_tile_kernel_equals_the_large_tile_kernel_bitwise(nat, m, n, k):
    """The same rows of A inside a matrix tall enough for the 256 x 256-tile kernel: identical bits (same accumulation
    order), row-major and k-blocked."""
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(2.0, device=DEV), torch.tensor(0.25, device=DEV)
    bias = (torch.randn(n, generator=torch.Generator().manual_seed(n)) * 3).to(torch.bfloat16).to(DEV)
    tall = 256 * (128 // ((n + 255) // 256) + 2)
    a_tall = torch.cat([a.view(torch.uint8), torch.zeros(tall - m, k, dtype=torch.uint8, device=DEV)]).view(a.dtype)
    for out_dt, b in ((torch.bfloat16, bias), (torch.float32, None)):
        want = nat.gemm_nt(a_tall, sa, bt, sb, out_dt, bias=b)[:m]
        assert torch.equal(nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b), want)
        if k >= 384:
            assert torch.equal(nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, out_dt, bias=b), want)


def test_gemm_random_sweep_over_all_dispatch_paths(nat):
    """Seeded random (m, n, k), formats, output types, bias, row strides and 16-byte misalignment: whichever kernel
    the library picks (few-row, 16x16x128 or 32x32x64 LDS-DMA, register-staged) the result is within the stated
    tolerance of the exact product, and equal bit for bit to the same call on a dense, aligned copy when both take
    the same kernel family."""
    rng = np.random.default_rng(2024)
    fmts = ["e4m3", "e5m2"]
    outs = [torch.bfloat16, torch.float32, torch.float16]
    one = None
    for case in range(48):
        kind = case % 6
        m = int(rng.choice([1, 3, 16, 40, 64, 100, 128, 129, 255, 256, 300, 513]))
        n = int(rng.choice([1, 8, 31, 64, 200, 256, 257, 520]))
        k = int(rng.choice([[16, 48, 100, 129, 250], [128, 256, 1152], [384, 640, 1024, 2048], [448, 576, 704],
                            [392, 1000, 4097], [128, 384, 512]][kind]))
        a_fmt, b_fmt = fmts[int(rng.integers(2))], fmts[int(rng.integers(2))]
        out_dt = outs[int(rng.integers(3))]
        _gemm_check(nat, m, n, k, a_fmt, b_fmt, out_dt, seed=1000 + case, bias=bool(rng.integers(2)))
        # the same product from operands with a padded row stride, and from operands shifted off 16-byte alignment
        ta, tb = F8[a_fmt][1], F8[b_fmt][1]
        a = _rand_fp8((m, k), ta, 2000 + case, 4.0).to(DEV)
        bt = _rand_fp8((n, k), tb, 3000 + case, 4.0).to(DEV)
        if one is None:
            one = torch.ones((), device=DEV)
        want = nat.gemm_nt(a, one, bt, one, torch.float32)
        pad = 16 * int(rng.integers(1, 5))
        a_p = torch.zeros(m, k + pad, dtype=torch.uint8, device=DEV).view(ta)
        b_p = torch.zeros(n, k + pad, dtype=torch.uint8, device=DEV).view(tb)
        a_p[:, :k].view(torch.uint8).copy_(a.view(torch.uint8))
        b_p[:, :k].view(torch.uint8).copy_(bt.view(torch.uint8))
        got = nat.gemm_nt(a_p[:, :k], one, b_p[:, :k], one, torch.float32)
        if k % 16 == 0:
            assert torch.equal(got, want), (case, m, n, k, "padded rows")  # same kernel: strides only
        else:
            torch.testing.assert_close(got, want, rtol=1e-3, atol=1e-2)
        a_o = torch.empty(m * k + 3, dtype=torch.uint8, device=DEV)[3:].view(ta).view(m, k)
        a_o.view(torch.uint8).copy_(a.view(torch.uint8))
        got = nat.gemm_nt(a_o, one, bt, one, torch.float32)   # unaligned: the register-staged kernel
        torch.testing.assert_close(got, want, rtol=1e-3, atol=1e-2 * max(1.0, k / 256))


def test_gemm_kernels_agree_bitwise(nat):
    """Same operands through the LDS-DMA kernel (aligned view) and the register-staged kernel (the same
    values at a 1-byte offset, which forces the unaligned path): identical accumulation order, identical bits."""
    m, n, k = 300, 520, 1024
    a = _rand_fp8((m, k), torch.float8_e4m3fn, 31, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, 32, 4.0).to(DEV)
    s1 = torch.ones((), device=DEV)
    fast = nat.gemm_nt(a, s1, bt, s1, torch.float32)
    a_off = torch.empty(m * k + 1, dtype=torch.uint8, device=DEV)[1:].view(torch.float8_e4m3fn).view(m, k)
    b_off = torch.empty(n * k + 1, dtype=torch.uint8, device=DEV)[1:].view(torch.float8_e4m3fn).view(n, k)
    a_off.copy_(a)
    b_off.copy_(bt)
    assert a_off.data_ptr() % 16 != 0
    slow = nat.gemm_nt(a_off, s1, b_off, s1, torch.float32)
    assert torch.equal(fast, slow)


def _to_kb(t):
    """[rows, k] fp8 -> k-blocked [k/64, rows, 64] (byte permutation on the device)."""
    rows, k = t.shape
    return t.view(torch.uint8).view(rows, k // 64, 64).permute(1, 0, 2).contiguous().view(t.dtype)


@pytest.mark.parametrize("m,n,k", [(256, 256, 384), (300, 200, 448), (257, 511, 576), (1, 7, 640), (520, 264, 8192), (1024, 768, 2048)])
def test_gemm_kblocked_equals_row_major_bitwise(nat, m, n, k):
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.5, device=DEV)
    bias = (torch.randn(n) * 3).to(torch.bfloat16).to(DEV)
    for out_dt, b in ((torch.bfloat16, bias), (torch.float32, None), (torch.float16, None)):
        want = nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b)
        got = nat.gemm_nt_kb(_to_kb(a), sa, _to_kb(bt), sb, out_dt, bias=b)
        assert torch.equal(got, want), (m, n, k, out_dt)


@pytest.mark.parametrize("m,n,k", [(256, 256, 384), (320, 192, 512), (64, 128, 640), (704, 448, 1024), (512, 256, 8192),
                                   (16384 // 8, 1024, 2048)])
def test_gemm_with_transposed_operands_equals_row_major_bitwise(nat, m, n, k):
    """f8mi_gemm_kb_ex: Bt, or A and Bt, given as the k-blocked copy of the transposed matrix (what the other
    GEMMs of a linear layer hold), read with LDS transpose loads: identical bits to the row-major GEMM."""
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k + 5, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k + 6, 4.0).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.5, device=DEV)
    a_tr = _to_kb(a.view(torch.uint8).t().contiguous().view(a.dtype))    # [m/64, k, 64]
    bt_tr = _to_kb(bt.view(torch.uint8).t().contiguous().view(bt.dtype))  # [n/64, k, 64]
    bias = (torch.randn(n) * 3).to(torch.bfloat16).to(DEV)
    # the row-major product from the tile kernels (up to 256 rows f8mi_gemm_nt takes the few-row kernel, which sums in
    # another order: pad A with zero rows past that limit and cut the result)
    a_ref = a if m > 256 else torch.cat([a.view(torch.uint8), torch.zeros(320 - m, k, dtype=torch.uint8, device=DEV)]).view(a.dtype)
    for out_dt, b in ((torch.bfloat16, bias), (torch.float32, None)):
        want = nat.gemm_nt(a_ref, sa, bt, sb, out_dt, bias=b, split_k=False)[:m]  # transposed operands are never split over k
        got = nat.gemm_kb_ex(_to_kb(a), False, sa, bt_tr, True, sb, out_dt, bias=b)
        assert torch.equal(got, want), (m, n, k, out_dt, "bt transposed")
        got = nat.gemm_kb_ex(a_tr, True, sa, bt_tr, True, sb, out_dt, bias=b)
        assert torch.equal(got, want), (m, n, k, out_dt, "both transposed")
        got = nat.gemm_kb_ex(_to_kb(a), False, sa, _to_kb(bt), False, sb, out_dt, bias=b)
        if m > 256:
            assert torch.equal(got, want)
        else:
            torch.testing.assert_close(got.float(), want.float(), rtol=2.0**-7, atol=1e-2)
    with pytest.raises(nat.Float8NativeError):
        nat.gemm_kb_ex(a_tr, True, sa, _to_kb(bt), False, sb, torch.bfloat16)


def _to_kb_padded(t):
    """[rows, k] fp8 -> zero-padded k-blocked [padded_k/64, rows, 64] and the row-major padded matrix (device)."""
    rows, k = t.shape
    kp = -(-k // 128) * 128
    padded = torch.zeros(rows, kp, dtype=torch.uint8, device=t.device)
    padded[:, :k] = t.view(torch.uint8)
    return padded.view(rows, kp // 64, 64).permute(1, 0, 2).contiguous().view(t.dtype), padded.view(t.dtype)


@pytest.mark.parametrize("m,n,k", [(300, 200, 385), (257, 511, 1000), (129, 77, 4097), (4099, 1000, 3000), (1000, 3000, 4099),
                                   (64, 8190, 2047), (20, 515, 8191)])
def test_gemm_on_zero_padded_kblocked_operands(nat, m, n, k):
    """A ragged contraction on the LDS-DMA kernels: operands k-blocked with the contraction zero-padded to a multiple of
    128 (what the cast writes with F8MI_LAYOUT_KBLOCK64_PAD128) give the bits of the row-major product over the padded
    length, and the value of the unpadded product (register-staged kernel) within the accumulation tolerance.  n and
    the row pitch of C are odd in most cases: C leaves in 16-byte stores at 2-byte alignment."""
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k, 4.0).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, n + k, 4.0).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.5, device=DEV)
    a_kb, a_pad = _to_kb_padded(a)
    b_kb, b_pad = _to_kb_padded(bt)
    bias = (torch.randn(n) * 3).to(torch.bfloat16).to(DEV)
    for out_dt, b in ((torch.bfloat16, bias), (torch.float32, None), (torch.float16, None)):
        got = nat.gemm_nt_kb(a_kb, sa, b_kb, sb, out_dt, bias=b, split_k=False)
        want = nat.gemm_nt(a_pad, sa, b_pad, sb, out_dt, bias=b, split_k=False)
        assert torch.equal(got, want), (m, n, k, out_dt)
        ragged = nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b, split_k=False).double()
        bound = (a.float().abs() @ bt.float().abs().t()).double() / 1.5
        eps_out = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-23}[out_dt]
        tol = 2 * eps_out * ragged.abs() + 2.0**-12 * bound + 1e-30
        assert ((got.double() - ragged).abs() <= tol).all(), (m, n, k, out_dt)
    _gemm_check(nat, m, n, k, "e5m2", "e4m3", torch.bfloat16, seed=m + n + k)


@pytest.mark.parametrize("m,n,k", [(16, 128, 48), (16, 128, 41), (2048, 4096, 2048), (4096, 2048, 384), (2112, 2176, 640),
                                   (2050, 4096, 1024), (4096, 2100, 1024), (16384, 8192, 8192)])
def test_scaled_mm_on_row_major_operands_equals_the_copy_route_bitwise(nat, m, n, k):
    """f8mi_gemm_ex / scaled_mm: a @ b with b row-major (the grad_input product) and with a column-major as well (the
    grad_weight product) gives the bits of gemm_nt on the copies preprocess_addmm would have made -- read transposed by
    the kernel where the product is large and aligned (checked through the return code), copied where it is not."""
    a = _rand_fp8((m, k), torch.float8_e5m2, m + k, 4.0).to(DEV)
    b = _rand_fp8((k, n), torch.float8_e4m3fn, n + k, 4.0).to(DEV)            # row-major [k, n]
    a_cm = a.view(torch.uint8).t().contiguous().view(a.dtype).t()               # the same matrix, column-major
    bt = b.view(torch.uint8).t().contiguous().view(b.dtype)                     # [n, k]: what gemm_nt takes
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.5, device=DEV)
    bias = (torch.randn(n) * 3).to(torch.bfloat16).to(DEV)
    for out_dt, bi in ((torch.bfloat16, bias), (torch.float32, None)):
        want = nat.gemm_nt(a, sa, bt, sb, out_dt, bias=bi, split_k=False)
        assert torch.equal(nat.scaled_mm(a, sa, b, sb, out_dt, bias=bi), want), (m, n, k, out_dt, "b row-major")
        assert torch.equal(nat.scaled_mm(a_cm, sa, b, sb, out_dt, bias=bi), want), (m, n, k, out_dt, "a column-major, b row-major")
        assert torch.equal(nat.scaled_mm(a, sa, bt.t(), sb, out_dt, bias=bi), want)
        assert torch.equal(nat.scaled_mm(a_cm, sa, bt.t(), sb, out_dt, bias=bi), want)   # (1, 0): a is copied
    # which of them the kernel took without a copy
    L = nat.lib()
    out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    fast_b = k % 128 == 0 and k >= 384 and n % 64 == 0 and -(-m // 128) * -(-n // 128) > 256
    rc = L.f8mi_gemm_ex(a.data_ptr(), 1, 0, k, b.data_ptr(), 0, 1, n, m, n, k, sa.data_ptr(), sb.data_ptr(), out.data_ptr(), 0, n, None, None)
    assert rc == (0 if fast_b else nat.ERR_UNSUPPORTED), (m, n, k, rc)
    rc = L.f8mi_gemm_ex(a_cm.data_ptr(), 1, 1, m, b.data_ptr(), 0, 1, n, m, n, k, sa.data_ptr(), sb.data_ptr(), out.data_ptr(), 0, n, None, None)
    assert rc == (0 if fast_b and m % 64 == 0 else nat.ERR_UNSUPPORTED), (m, n, k, rc)
    rc = L.f8mi_gemm_ex(a_cm.data_ptr(), 1, 1, m, bt.data_ptr(), 0, 0, k, m, n, k, sa.data_ptr(), sb.data_ptr(), out.data_ptr(), 0, n, None, None)
    assert rc == nat.ERR_UNSUPPORTED


def test_gemm_kblocked_refuses_short_or_ragged_k(nat):
    s1 = torch.ones((), device=DEV)
    for k in (64, 320):
        a = torch.zeros(k // 64, 8, 64, dtype=torch.float8_e4m3fn, device=DEV)
        with pytest.raises(nat.Float8NativeError):
            nat.gemm_nt_kb(a, s1, a, s1, torch.bfloat16)


@pytest.mark.parametrize("a_fmt,b_fmt", [("e4m3", "e4m3"), ("e5m2", "e4m3"), ("e4m3", "e5m2"), ("e5m2", "e5m2")])
@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16, torch.float32])
def test_gemm_formats_and_output_dtypes(nat, a_fmt, b_fmt, out_dt):
    _gemm_check(nat, 384, 320, 448, a_fmt, b_fmt, out_dt, seed=7, bias=(out_dt != torch.float16))


def test_gemm_closed_forms(nat):
    one4 = torch.tensor([1.0]).to(torch.float8_e4m3fn)
    # identity: A @ I = A exactly (every fp8 value is a bf16 value)
    a = _rand_fp8((300, 256), torch.float8_e4m3fn, 3, 50.0)
    eye = torch.eye(256).to(torch.float8_e4m3fn)
    s1 = torch.ones((), device=DEV)
    out = nat.gemm_nt(a.to(DEV), s1, eye.to(DEV), s1, torch.bfloat16)
    assert torch.equal(out.cpu().float(), a.float())
    # all ones: k / (sa * sb)
    a = torch.ones(70, 1000).to(torch.float8_e5m2)
    b = torch.ones(90, 1000).to(torch.float8_e4m3fn)
    out = nat.gemm_nt(a.to(DEV), torch.tensor(2.0, device=DEV), b.to(DEV), torch.tensor(4.0, device=DEV), torch.float32)
    assert bool((out == 125.0).all())
    # one-hot rows pick single columns (catches a transposed or permuted operand)
    a = torch.zeros(64, 512)
    idx = torch.arange(64) * 7 % 512
    a[torch.arange(64), idx] = 2.0
    bt = _rand_fp8((96, 512), torch.float8_e4m3fn, 9, 8.0)
    out = nat.gemm_nt(a.to(torch.float8_e4m3fn).to(DEV), s1, bt.to(DEV), s1, torch.float32).cpu()
    assert torch.equal(out, 2.0 * bt.float()[:, idx].t())
    # zero-padding the reduction changes nothing (reference test_base.py:477-552 pads to 16)
    a = _rand_fp8((50, 41), torch.float8_e4m3fn, 11)
    bt = _rand_fp8((128, 41), torch.float8_e4m3fn, 12)
    o1 = nat.gemm_nt(a.to(DEV), s1, bt.to(DEV), s1, torch.float32)
    ap = torch.nn.functional.pad(a.view(torch.uint8), (0, 7)).view(torch.float8_e4m3fn)
    bp = torch.nn.functional.pad(bt.view(torch.uint8), (0, 7)).view(torch.float8_e4m3fn)
    o2 = nat.gemm_nt(ap.to(DEV), s1, bp.to(DEV), s1, torch.float32)
    assert torch.equal(o1, o2)
    # k = 0: the empty sum
    o = nat.gemm_nt(torch.empty(5, 0, dtype=torch.float8_e4m3fn, device=DEV), s1,
                    torch.empty(6, 0, dtype=torch.float8_e4m3fn, device=DEV), s1, torch.bfloat16)
    assert o.shape == (5, 6) and bool((o == 0).all())


def test_gemm_strided_operands(nat):
    co, to = _oracles()
    a = _rand_fp8((200, 512), torch.float8_e4m3fn, 21)
    bt = _rand_fp8((300, 512), torch.float8_e4m3fn, 22)
    ad, bd = a.to(DEV), bt.to(DEV)
    s1 = torch.ones((), device=DEV)
    # row-strided views (ld > k), aligned and not
    for sl in (slice(0, 256), slice(16, 400), slice(3, 260)):
        out = nat.gemm_nt(ad[:, sl], s1, bd[:, sl], s1, torch.float32).cpu()
        want = a[:, sl].double() @ bt[:, sl].double().t()
        bound = a[:, sl].double().abs() @ bt[:, sl].double().abs().t()
        assert bool(((out.double() - want).abs() <= 2.0**-13 * bound).all())


@pytest.mark.parametrize("out_dt", [torch.bfloat16, torch.float16])
def test_gemm_epilogue_of_tiles_inside_c_equals_the_checked_one_bitwise(nat, out_dt):
    """A 256 x 256 tile that lies inside C is written without bounds checks, one on the edge of C with them.  Dropping
    the last 8 rows and columns of a product turns its last row and column of tiles from the first kind into the
    second; what both products share must not change by a bit."""
    m, n, k = 4096, 4096, 512
    assert nat.gemm_plan(m, n, k)[0] == "tiles256" and nat.gemm_plan(m - 8, n - 8, k)[0] == "tiles256"
    a = _rand_fp8((m, k), torch.float8_e5m2, 31).to(DEV)
    bt = _rand_fp8((n, k), torch.float8_e4m3fn, 32).to(DEV)
    sa, sb = torch.tensor(3.0, device=DEV), torch.tensor(0.37, device=DEV)
    bias = torch.linspace(-1, 1, n).to(out_dt).to(DEV)
    for b in (None, bias):
        whole = nat.gemm_nt(a, sa, bt, sb, out_dt, bias=b)
        part = nat.gemm_nt(a[:m - 8], sa, bt[:n - 8], sb, out_dt, bias=None if b is None else b[:n - 8].contiguous())
        assert torch.equal(whole[:m - 8, :n - 8], part)
        # and the tiles inside C against the exact product
        exact = (a[:512].cpu().double() @ bt[:512].cpu().double().t()) / (3.0 * 0.37) + (0 if b is None else b[:512].cpu().double())
        err = (whole[:512, :512].cpu().double() - exact).abs()
        assert bool((err <= {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[out_dt] * exact.abs() + 2.0**-12 * (
            a[:512].cpu().double().abs() @ bt[:512].cpu().double().abs().t()) / (3.0 * 0.37)).all())


# ------------------------------------------------------------------ K4 sync


def test_sync_and_init_match_oracle(nat):
    co, to = _oracles()
    rng = np.random.default_rng(0)
    n, H = 999, 16
    amax = (np.abs(rng.standard_normal(n)) * 10.0 ** rng.integers(-14, 5, n)).astype(np.float32)
    hist = (np.abs(rng.standard_normal((n, H))) * 10.0 ** rng.integers(-14, 5, (n, 1))).astype(np.float32)
    hist[::7] = 0
    amax[:3] = [0.0, 448.0, np.nan]
    fmts = rng.integers(0, 2, n)
    for fp16 in (False, True):
        for wb in (False, True):
            a_d = torch.from_numpy(amax.copy()).to(DEV).reshape(n, 1)
            h_d = torch.from_numpy(hist.copy()).to(DEV)
            s_d = torch.zeros(n, 1, device=DEV)
            entries = [(a_d[i], h_d[i], s_d[i], (torch.float8_e4m3fn, torch.float8_e5m2)[fmts[i]]) for i in range(n)]
            nat.sync(nat.sync_table(entries, torch.device(DEV)), H, fp16, wb)
            got_s, got_h = s_d.cpu().numpy().reshape(-1), h_d.cpu().numpy()
            # the same through the entry point that takes the entries as kernel arguments (32 per launch: 999 = 31 * 32 + 7)
            h2_d = torch.from_numpy(hist.copy()).to(DEV)
            s2_d = torch.zeros(n, 1, device=DEV)
            nat.sync_host([(a_d[i], h2_d[i], s2_d[i], e[3]) for i, e in enumerate(entries)], H, fp16, wb)
            assert torch.equal(s2_d.view(torch.int32), s_d.view(torch.int32)) and torch.equal(h2_d.view(torch.int32), h_d.view(torch.int32))
            for i in range(n):
                h = hist[i].copy()
                want = co.sync_entry(amax[i], h, int(fmts[i]), fp16, wb)
                assert np.float32(got_s[i]).view(np.uint32) == np.float32(want).view(np.uint32) or (np.isnan(want) and np.isnan(got_s[i])), i
                assert np.array_equal(got_h[i], h, equal_nan=True), (i, wb)
    # init
    for i in range(0, 60):
        h = hist[i].copy()
        a_d = torch.tensor([amax[i]], device=DEV)
        h_d = torch.from_numpy(h.copy()).to(DEV)
        s_d = torch.zeros(1, device=DEV)
        nat.delayed_init(a_d, h_d, s_d, (torch.float8_e4m3fn, torch.float8_e5m2)[fmts[i]], False)
        want = co.delayed_init(amax[i], h, int(fmts[i]), False)
        assert np.array_equal(h_d.cpu().numpy(), h, equal_nan=True)
        assert np.float32(s_d.item()).view(np.uint32) == np.float32(want).view(np.uint32) or np.isnan(want)


# ------------------------------------------- full-size properties (config 2)


def test_full_size_properties_llama70b_wo(nat):
    """M=16384, K=N=8192: size-independent properties where the oracle is too slow."""
    torch.manual_seed(0)
    M, K, N = 16384, 8192, 8192
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = (torch.rand(N, K, device=DEV, dtype=torch.float32) * 2 - 1).mul_(K**-0.5).to(torch.bfloat16)
    ax, sx = nat.amax_scale(x, torch.float8_e4m3fn)
    aw, sw = nat.amax_scale(w, torch.float8_e4m3fn)
    assert ax.item() == x.abs().max().float().item() and aw.item() == w.abs().max().float().item()
    x8, x8t = nat.cast(x, sx, torch.float8_e4m3fn, want_out_t=True)
    w8, w8t = nat.cast(w, sw, torch.float8_e4m3fn, want_out_t=True)
    assert torch.equal(x8t.view(torch.uint8), x8.view(torch.uint8).t().contiguous())
    assert torch.equal(w8t.view(torch.uint8), w8.view(torch.uint8).t().contiguous())
    # the cast is the same function of (x, scale) everywhere: torch's own ops on the GPU agree byte for byte
    ref = (x * sx).clamp(-448, 448).to(torch.float8_e4m3fn)
    assert torch.equal(ref.view(torch.uint8), x8.view(torch.uint8))
    # idempotence: re-casting the dequantised tensor at scale 1 gives the same bytes
    one = torch.ones((), device=DEV)
    again, _ = nat.cast(x8.to(torch.bfloat16), one, torch.float8_e4m3fn)
    assert torch.equal(again.view(torch.uint8), x8.view(torch.uint8))
    # GEMM: checksum of checksums in fp64, and exact linearity in power-of-two scales
    y = nat.gemm_nt(x8, sx, w8, sw, torch.float32)
    col = (x8.double().sum(0) / sx.double()) @ (w8.double().t() / sw.double())
    torch.testing.assert_close(y.double().sum(0), col, rtol=1e-4, atol=1e-4 * col.abs().max().item())
    row = (x8.double() / sx.double()) @ (w8.double().sum(0) / sw.double())
    torch.testing.assert_close(y.double().sum(1), row, rtol=1e-4, atol=1e-4 * row.abs().max().item())
    y2 = nat.gemm_nt(x8, sx * 2, w8, sw * 4, torch.float32)
    assert torch.equal(y2 * 8, y)
    # a 64 x 64 corner against the emulated product computed in fp64
    sub = (x8[:64].double() / sx.double()) @ (w8[:64].double().t() / sw.double())
    torch.testing.assert_close(y[:64, :64].double(), sub, rtol=1e-4, atol=1e-4)
    # grad_weight-shaped product from the transposed copies: (x^T x)[i][j], symmetric by construction
    g = nat.gemm_nt(x8t[:512], sx, x8t[:768], sx, torch.float32)
    torch.testing.assert_close(g[:, :512], g[:, :512].t(), rtol=1e-5, atol=1e-3)


def test_tensors_of_more_than_2_31_elements(nat):
    """Index arithmetic past 32 bits: amax, cast (all layouts) and the GEMM's output addressing on a tensor of
    2.29e9 elements, checked on slices against torch's own ops on the GPU (the cast is the same function of
    (x, scale) everywhere, so slices pin it) and on planted maxima."""
    rows, cols = 70000, 32768
    assert rows * cols > 2**31
    g = torch.Generator(device=DEV).manual_seed(11)
    x = torch.empty(rows, cols, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    x[rows - 1, cols - 3] = 1000.0   # the maximum sits past element 2^31
    amax, scale = nat.amax_scale(x, torch.float8_e4m3fn)
    assert amax.item() == 1000.0
    x[rows - 1, cols - 3] = 0.5
    x[17, 5] = -2000.0
    amax, scale = nat.amax_scale(x, torch.float8_e4m3fn)
    assert amax.item() == 2000.0
    ams, _ = nat.amax_scale_multi([x[:3], x], torch.float8_e4m3fn)
    assert ams[1].item() == 2000.0
    ref_rows = [0, 1, 127, 128, 32767, 65535, 65536, rows - 129, rows - 2, rows - 1]
    want = (x[ref_rows] * scale).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    out, out_t = nat.cast(x, scale, torch.float8_e4m3fn, want_out_t=True)
    assert torch.equal(out[ref_rows].view(torch.uint8), want)
    assert torch.equal(out_t[:, ref_rows].view(torch.uint8), want.t())
    del out_t
    okb, _ = nat.cast(x, scale, torch.float8_e4m3fn, out_kblock=True)  # [cols/64, rows, 64]
    assert torch.equal(okb[:, ref_rows, :].view(torch.uint8).permute(1, 0, 2).reshape(len(ref_rows), cols), want)
    del okb
    # GEMM with more than 2^31 outputs: C = out[:, :384] (70000 x 384) times a 32768 x 384 matrix
    a8 = out[:, :384].contiguous()
    b8 = _rand_fp8((cols, 384), torch.float8_e4m3fn, 3, 2.0).to(DEV)
    one = torch.ones((), device=DEV)
    c = nat.gemm_nt(a8, one, b8, one, torch.bfloat16)
    assert c.numel() > 2**31
    for r0 in (0, 65536 - 128, rows - 256):
        ref = nat.gemm_nt(a8[r0:r0 + 256].contiguous(), one, b8, one, torch.bfloat16)
        assert torch.equal(c[r0:r0 + 256], ref), r0
    exact = a8[rows - 64:].double() @ b8.double().t()
    torch.testing.assert_close(c[rows - 64:].double(), exact, rtol=2.0**-7, atol=0.5)
