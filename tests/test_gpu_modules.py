"""The call-site classes of the reference's model.py:96-153 and their bf16-activation siblings on the GPU:
SpBitLinear, BF16BitLinear (the reference's dense golden mode, `--BF16`), SpBitLinearBF16 and
TernaInfer_linear_bf16, each against the CPU oracle, and the sparse module against the dense one."""
import numpy as np
import pytest
import torch

from oracle import terna_oracle as O
from tests._util import check_against_fp64, make_bf16_activations, make_ternary

pytestmark = pytest.mark.gpu


def bits(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def checkpoint_entry(w, scales, key="l"):
    """What the converter writes for one linear: the four format tensors, the 4-slot bf16 weight_scale, and the
    dense bf16 matrix ternary * scale of the bf16 checkpoint (convert_TernaInfer.py:112-114, 159-194)."""
    import ternainfer_amd as T
    n = w.shape[0]
    vals, off, med, bm = T.compress_weight(torch.from_numpy(w))
    ws = T.pack_weight_scale([torch.tensor(v, dtype=torch.bfloat16) for v in scales])
    groups = O.ws_group_decode(np.arange(n), n, len(scales))
    dense = (torch.from_numpy(w).float() * ws.float()[torch.from_numpy(groups)][:, None]).to(torch.bfloat16)
    return {f"{key}.weight_compressed_val": vals, f"{key}.weight_TileOffsets_global": off,
            f"{key}.weight_TileOffsets_median": med, f"{key}.weight_bitmap": bm, f"{key}.weight_scale": ws,
            f"{key}.weight": dense}, ws


def _check(got_bits, ref, max_rel=1e-2, med_ulp_max=1):
    max_err, max_ref, med_ulp, _ = check_against_fp64(got_bits, ref)
    assert max_err <= max_rel * max_ref and med_ulp <= med_ulp_max, (max_err, max_ref, med_ulp)


@pytest.mark.parametrize("m,n,k,scales", [(5, 384, 256, [1.59375, 0.8125]), (8, 2560, 2560, [1.25]),
                                          (1, 3840, 2560, [0.75, 1.5, 1.125]), (96, 512, 320, [0.5])])
def test_bf16bitlinear_dense_mode_against_oracle_and_sparse_module(m, n, k, scales):
    """BF16BitLinear (model.py:135-153) within the bf16-GEMM bar of the float64 evaluation of its formula, and
    SpBitLinear on the compressed form of the same weights within a bf16 step or two of it: the dense mode is
    the reference's own golden for the sparse path (README `--BF16`)."""
    import ternainfer_amd as T
    w = make_ternary(n, k, 0.40, 700 + m + n)
    dic, ws = checkpoint_entry(w, scales)
    x_bits = make_bf16_activations(m, k, 710 + m + k)
    x = torch.from_numpy(x_bits.view(np.int16)).view(torch.bfloat16).cuda()
    print(f"[case] BF16BitLinear / SpBitLinear M={m} N={n} K={k} groups={len(scales)}", flush=True)
    dense_mod = T.BF16BitLinear(k, n, dic, "l")
    got = dense_mod(x)
    torch.cuda.synchronize()
    assert got.shape == (m, n) and got.dtype == torch.bfloat16
    ref = O.bf16_bitlinear_golden(x_bits, bits(dic["l.weight"]))
    _check(bits(got), ref)
    # the module's quantiser is the library's one definition
    q, s = dense_mod.quant_input(x)
    q_want, s_want = O.quant_input(x_bits)
    assert (q.cpu().numpy() == q_want).all() and (bits(s).reshape(-1) == s_want).all()
    sparse = T.SpBitLinear(k, n, dic, "l")(x)
    torch.cuda.synchronize()
    _check(bits(sparse), ref)
    # bit-exact against the integer oracle with the epilogue rule the row count selects
    want = O.spmm_i8(q_want, w, s_want, bits(ws), len(scales), 0 if max(8, 1 << (m - 1).bit_length()) <= 64 else 1)
    assert (bits(sparse) == want).all()


@pytest.mark.parametrize("shape,n,k,scales", [((3, 320), 256, 320, [0.7, 1.9]), ((2, 5, 320), 256, 320, [1.3]),
                                              ((8, 2560), 2560, 2560, [1.37]), ((300, 192), 384, 192, [0.9, 1.1])])
def test_spbitlinear_bf16_module_and_call_site(shape, n, k, scales):
    """SpBitLinearBF16 and TernaInfer_linear_bf16 (auto / forced routes; 2-D and 3-D inputs keep their leading
    dimensions) against the float64 golden of the bf16-activation family."""
    import ternainfer_amd as T
    w = make_ternary(n, k, 0.40, 720 + n + len(shape))
    dic, ws = checkpoint_entry(w, scales)
    m = int(np.prod(shape[:-1]))
    x_bits = make_bf16_activations(m, k, 730 + m, outlier_frac=0.01 if m > 64 else 0.0)
    x = torch.from_numpy(x_bits.view(np.int16)).view(torch.bfloat16).reshape(shape).cuda()
    scale = ws.float().numpy()
    ref = O.spmm_bf16_golden(x_bits, w, scale[:len(scales)], len(scales))
    print(f"[case] SpBitLinearBF16 / TernaInfer_linear_bf16 shape={shape} N={n} K={k}", flush=True)
    mod = T.SpBitLinearBF16(k, n, dic, "l")
    assert mod.ws_num == len(scales)
    got = mod(x)
    torch.cuda.synchronize()
    assert tuple(got.shape) == tuple(shape[:-1]) + (n,) and got.dtype == torch.bfloat16
    _check(bits(got).reshape(m, n), ref)
    dev = lambda t: t.cuda()
    for route in ("auto", "decode", "prefill"):
        out = T.TernaInfer_linear_bf16(x, dev(dic["l.weight_compressed_val"]), dev(dic["l.weight_TileOffsets_global"]),
                                       dev(dic["l.weight_TileOffsets_median"]), dev(dic["l.weight_bitmap"]),
                                       dev(ws.float()), len(scales), n, route=route)
        torch.cuda.synchronize()
        assert tuple(out.shape) == tuple(shape[:-1]) + (n,)
        _check(bits(out).reshape(m, n), ref)


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (1, 2560, 2560), (2, 192, 8192), (3, 2560, 6912), (4, 320, 4160), (5, 3840, 320), (8, 13824, 2560),
                                   (8, 256, 3584), (8, 256, 3648), (9, 256, 512)])
def test_spbitlinear_few_rows_in_one_launch(m, n, k):
    """Quantisation and linear of a few rows in one launch (terna_quant_linear_kernel; the last two cases and the widest matrix are beyond it):
    the integer oracle's bits with a repacked weight and, through the library's cached copy, on the reference format."""
    import ternainfer_amd as T
    from ternainfer_amd import _lib
    lib = _lib.load()
    w = make_ternary(n, k, 0.40, 800 + m + n + k)
    scales = [0.75, 1.5, 1.125] if n == 3840 else [1.375]
    dic, ws = checkpoint_entry(w, scales)
    x_bits = make_bf16_activations(m, k, 810 + m + k, outlier_frac=0.01)
    x_bits[m // 2, : k // 2] = 0
    x = torch.from_numpy(x_bits.view(np.int16)).view(torch.bfloat16).cuda()
    print(f"[case] quantise + linear in one launch M={m} N={n} K={k}", flush=True)
    q, s = O.quant_input(x_bits)
    want = O.spmm_i8(q, w, s, bits(ws), len(scales), 0)
    assert (bits(T.SpBitLinear(k, n, dic, "l", repack=True)(x)) == want).all()
    was = lib.ternaspmm_repack_cache_enable(1)
    try:
        lib.ternaspmm_repack_cache_clear()
        module = T.SpBitLinear(k, n, dic, "l")
        for _ in range(2):                        # first sight makes the copy, both calls run on it
            assert (bits(module(x)) == want).all()
    finally:
        lib.ternaspmm_repack_cache_clear()
        lib.ternaspmm_repack_cache_enable(was)


def _with_broken_rows(x_bits, kind):
    """NaN, infinities or both in some rows: -> (bits, rows with a NaN, rows with infinities only)."""
    m, k = x_bits.shape
    x = x_bits.copy()
    nan, inf, neg = 0x7FC0, 0x7F80, 0xFF80
    if m < 4:
        x[m - 1, k - 1] = {"nan": nan, "inf": inf, "-inf": neg}[kind]
        return (x, [m - 1], []) if kind == "nan" else (x, [], [m - 1])
    x[0, k - 1], x[1, 3], x[m - 1, k // 2], x[m - 1, 1] = nan, inf, neg, 0xFFC0
    x[2, k - 8:] = neg
    return x, [0, m - 1], [1, 2]


@pytest.mark.parametrize("m", [1, 2, 5, 8, 9, 70])
def test_every_half_is_quantised_to_its_even_neighbour(m):
    """Rows of all multiples of a half up to 127 times a power of two, whose scale is that power's inverse: half of the products
    are ties.  Through an identity matrix the outputs are the integers themselves (up to 8 rows quantised inside the linear, above
    in front of it): exact."""
    import ternainfer_amd as T
    k = 512
    entry, _ = checkpoint_entry(np.eye(k, dtype=np.int8), [1.0])
    module = T.SpBitLinear(k, k, entry, "l")
    halves = torch.zeros(k)
    halves[:509] = torch.arange(-254, 255) / 2
    power = 2.0 ** (torch.arange(m) % 7 - 3)[:, None]
    x = torch.stack([halves.roll(37 * i) for i in range(m)]) * power
    want = torch.round(x / power) * power                                     # torch.round: ties to even
    got = module(x.to(torch.bfloat16).cuda())
    assert torch.equal(got.float().cpu(), want)


@pytest.mark.parametrize("m,kind", [(1, "nan"), (1, "inf"), (1, "-inf"), (2, "nan"), (3, "inf"), (4, ""), (8, ""), (9, ""), (64, ""), (65, ""), (300, "")])
@pytest.mark.parametrize("k", [192, 2560])
def test_spbitlinear_broken_activations_show_in_the_output(m, kind, k):
    """A NaN in a row makes the row's scale and with it all of its outputs NaN; an infinity makes the scale 0 and the integers 0,
    hence outputs 0 / 0 under the rule of up to 64 rows and 0 above (s == 0, epilogue_visitor_scale_ws.h:180-191): on every
    route, in every quantisation mode, and the other rows keep their bits."""
    import ternainfer_amd as T
    from ternainfer_amd import _lib, linear as L
    lib = _lib.load()
    n = 256
    w = make_ternary(n, k, 0.40, 900 + m + k)
    dic, ws = checkpoint_entry(w, [1.375])
    x_bits, nan_rows, inf_rows = _with_broken_rows(make_bf16_activations(m, k, 910 + m + k), kind)
    good = [r for r in range(m) if r not in nan_rows + inf_rows]
    x = torch.from_numpy(x_bits.view(np.int16)).view(torch.bfloat16).cuda()
    print(f"[case] broken activations M={m} K={k} {kind}", flush=True)
    q, s = L.quant_input(x)
    assert torch.isnan(s[nan_rows]).all() and (s[inf_rows] == 0).all() and (q[nan_rows + inf_rows] == 0).all()
    was = lib.ternaspmm_quant_mode(-1)
    try:
        for mode in (L.QUANT_ROUNDED, L.QUANT_COMPILED, L.QUANT_EAGER):
            lib.ternaspmm_quant_mode(mode)
            qm, sm = L.quant_input(x)
            want_q, want_s = L.quant_input(x.float(), mode)      # (another activation type: the torch lines)
            assert torch.equal(qm, want_q) and torch.equal(sm.nan_to_num(nan=-1.0), want_s.to(torch.bfloat16).nan_to_num(nan=-1.0)), mode
    finally:
        lib.ternaspmm_quant_mode(was)
    q_good, s_good = O.quant_input(x_bits[good]) if good else (None, None)
    for repack in (False, True):
        out = T.SpBitLinear(k, n, dic, "l", repack=repack)(x)
        torch.cuda.synchronize()
        assert torch.isnan(out[nan_rows]).all()
        assert torch.isnan(out[inf_rows]).all() if m <= 64 else (out[inf_rows] == 0).all()
        if good:
            assert (bits(out[good]) == O.spmm_i8(q_good, w, s_good, bits(ws), 1, 0 if m <= 64 else 1)).all()


@pytest.mark.parametrize("m", [4, 8, 12, 70])
def test_broken_rows_behind_a_norm_are_nan_on_every_route(m):
    """NaN and infinities in a row in front of a norm: all of the row's outputs are NaN, whether the norm takes its statistics
    itself or from partials (also where the norm's weight of an infinite element is 0), and the other rows keep their bits."""
    import ternainfer_amd as T
    from ternainfer_amd import linear as L
    n, k = 256, 512
    w = make_ternary(n, k, 0.40, 930 + m)
    dic, ws = checkpoint_entry(w, [1.375])
    dev = lambda b: torch.from_numpy(b.view(np.int16)).view(torch.bfloat16).cuda()
    packed = L.repack_weight(*(dic["l.weight" + p].cuda() for p in ("_compressed_val", "_TileOffsets_global", "_TileOffsets_median", "_bitmap")), n, k)
    clean = make_bf16_activations(m, k, 940 + m)
    broken, nan_rows, inf_rows = _with_broken_rows(clean, "")
    bad = nan_rows + inf_rows
    good = [r for r in range(m) if r not in bad]
    g = torch.rand(k, device="cuda").to(torch.bfloat16) + 0.5
    g[3] = 0                                      # (the infinity of row 1)
    scale = ws.cuda()
    zeros = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
    ones = torch.ones(n, dtype=torch.bfloat16, device="cuda")

    def with_stats(x):
        st = L.row_stats(x, g)
        q, s = L.quant_from_stats(x, st, g, 1e-5)
        outs = [L.TernaInfer_linear_packed(q, packed, s, scale, 1, n)]
        if m <= 8:
            outs.append(L.fused_linear(x, g, 1e-5, packed, scale, 1, n, k, stats=st)[0])
        if m <= 16:
            r = L.fused_linear(q, None, 1e-5, packed, scale, 1, n, k, quantised=s, epilogue=L.EPILOGUE_RESIDUAL, residual=zeros, next_norm_weight=ones)
            outs += [r[0], r[1].reshape(m, -1)]       # the stream and its partials
        return outs

    def with_norm(x):
        q, s, _ = L.rmsnorm_quant(x, g, 1e-5)
        return [L.TernaInfer_linear_packed(q, packed, s, scale, 1, n), L.rmsnorm_linear_packed(x, g, 1e-5, packed, scale, 1, n)[0]]

    def gated(x):
        x13 = torch.cat([x, torch.ones_like(x)], dim=1)
        q, s = L.relu2_mul_rmsnorm_quant(x13, g, 1e-5)
        return [L.TernaInfer_linear_packed(q, packed, s, scale, 1, n), L.relu2_mul_rmsnorm_linear_packed(x13, g, 1e-5, packed, scale, 1, n)]

    print(f"[case] broken rows behind a norm M={m}", flush=True)
    for route in (with_stats, with_norm, gated):
        rows = [r for r in bad if not (route is gated and r == 2)]     # (relu of -infinity is 0: that row is whole)
        for i, (got, want) in enumerate(zip(route(dev(broken)), route(dev(clean)))):
            torch.cuda.synchronize()
            assert torch.isnan(got[rows]).all(), (route.__name__, i)
            assert torch.equal(got[good], want[good]), (route.__name__, i)


# decode kernels; the kernel for 17 rows .. a few hundred (K in chunks of 256 columns); the MFMA-tiled ones (in stages of 128)
@pytest.mark.parametrize("m,n,k", [(1, 256, 320), (16, 256, 320), (17, 256, 320), (37, 256, 64), (37, 2560, 2624), (100, 3840, 448), (100, 512, 192), (300, 2560, 2560),
                                   (500, 2560, 192), (500, 2560, 320), (500, 2560, 256), (1000, 2560, 64), (1000, 2560, 448), (2048, 2560, 320)])
def test_infinite_bf16_activations_at_the_end_of_a_row(m, n, k):
    """bf16 linears: an infinity in the last columns gives +-infinity where its weight is not 0 (0 times it is NaN) and nowhere
    else, whatever part of a kernel's last piece of K the row leaves empty."""
    import ternainfer_amd as T
    from ternainfer_amd import _lib, linear as L
    w = make_ternary(n, k, 0.40, 950 + m + k)
    dic, ws = checkpoint_entry(w, [1.25])
    packed = L.repack_weight(*(dic["l.weight" + p].cuda() for p in ("_compressed_val", "_TileOffsets_global", "_TileOffsets_median", "_bitmap")), n, k)
    x_bits = make_bf16_activations(m, k, 960 + m + k)
    x_bits[0, k - 1] = 0x7F80
    x_bits[m // 2, k - 8] = 0xFF80
    x_bits[m - 1, k - 20] = 0x7F80
    x = torch.from_numpy(x_bits.view(np.int16)).view(torch.bfloat16)
    print(f"[case] infinite bf16 activations M={m} N={n} K={k}", flush=True)
    got = _lib.native().linear_bf16_packed(x.cuda(), packed, torch.tensor([1.25], device="cuda"), 1, n, None)
    torch.cuda.synchronize()
    got = got.cpu().double()
    broken = sorted({0, m // 2, m - 1})
    xw = x.double()
    want = (xw @ torch.from_numpy(w).double().t()) * 1.25
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])
    assert torch.isinf(want[broken]).any(dim=1).all() and torch.isfinite(want).any(dim=1).sum() == m - len(broken)
    whole = torch.isfinite(want)
    if whole.any():
        assert (got[whole] - want[whole]).abs().max() <= 1e-2 * want[whole].abs().max()


def test_other_threads_run_while_a_module_call_waits():
    """The first sight of a weight waits for the device inside the module's call (the library makes its copy): meanwhile other
    Python threads go on."""
    import threading
    import time
    import ctypes
    import ternainfer_amd as T
    from ternainfer_amd import _lib
    lib = _lib.load()
    n, k, wait = 256, 320, 0.5
    dic, _ = checkpoint_entry(make_ternary(n, k, 0.40, 970), [1.25])
    module = T.SpBitLinear(k, n, dic, "l")
    x = torch.ones((3, k), dtype=torch.bfloat16, device="cuda")
    was = lib.ternaspmm_repack_cache_enable(1)
    try:
        module(x)                                 # whatever is loaded or allocated once
        lib.ternaspmm_repack_cache_clear()
        torch.cuda.synchronize()
        print("[case] a module call that waits for the device, and another thread", flush=True)
        done = []

        def call():
            stream = torch.cuda.current_stream()
            lib.gpu_sleep(wait * 1e6, ctypes.c_void_p(stream.cuda_stream))
            start = time.monotonic()
            module(x)
            done.append(time.monotonic() - start)

        thread = threading.Thread(target=call)
        thread.start()
        longest, last = 0.0, time.monotonic()
        while thread.is_alive():
            time.sleep(0.002)
            now = time.monotonic()
            longest, last = max(longest, now - last), now
        thread.join()
        assert done and done[0] > wait / 2        # the call did wait ...
        assert longest < wait / 2                 # ... and this thread did not
    finally:
        torch.cuda.synchronize()
        lib.ternaspmm_repack_cache_clear()
        lib.ternaspmm_repack_cache_enable(was)
