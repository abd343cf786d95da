"""The conversions of checkpoints and fp32 import/export over lists of tensors (csrc/fo_codec.hip: convert_kernel),
against the oracle or the eager sequence they stand for.  Every value is exact: the same IEEE operations, one rounding to
the output type."""

import pytest
import torch

from oracle import c_oracle as C
from tests import parity

pytestmark = pytest.mark.gpu
DEV = "cuda"

# lanes, spans and workgroups of every kernel end at these lengths (8 / 4 elements, 512 / 256, 2048 / 1024), and around them
LENGTHS = [1, 7, 8, 9, 31, 33, 255, 257, 511, 512, 513, 1023, 1025, 2047, 2048, 2049, 4097, 70001]


def _lengths(many: bool):
    """`many`: more tensors than one launch takes, an empty one among them."""
    return LENGTHS + ([0] + [3 * i + 1 for i in range(90)] if many else [])


def _at(values: torch.Tensor, offset: int) -> torch.Tensor:
    """`values` on the GPU, `offset` elements into a larger buffer (offset 1: no vector access is aligned)."""
    buf = torch.zeros(values.numel() + offset, dtype=values.dtype, device=DEV)
    buf[offset:].copy_(values)
    return buf[offset:]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("signed,sqrt,softsign", [(True, False, True), (False, True, False), (True, True, False), (False, False, True)])
def test_dequantize_to_bf16_over_a_list(signed, sqrt, softsign, offset):
    from flashoptim_amd.kernels import ConversionBatch, dequantize

    g = torch.Generator().manual_seed(5)
    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        codes = torch.randint(0, 256, (n,), generator=g, dtype=torch.int32).to(torch.uint8)
        codes = codes.view(torch.int8) if signed else codes
        scales = torch.randn((n + 31) // 32, generator=g).abs().to(torch.float16)
        if n > 512:
            scales[1], codes[33] = float("inf"), 0  # inf * 0
        dev = _at(codes, offset), scales.to(DEV)
        cases.append((codes, scales, dev, batch.dequantize_bf16(*dev, signed, sqrt, softsign)))
    batch.launch()
    for codes, scales, dev, got in cases:
        eager = dequantize(*dev, signed=signed, sqrt=sqrt, softsign=softsign).to(torch.bfloat16)
        assert torch.equal(got.view(torch.int16), eager.view(torch.int16)), codes.numel()  # NaN bits too
        ref = C.dequantize(codes, scales, signed, sqrt, softsign).to(torch.bfloat16)
        assert torch.equal(got.cpu().nan_to_num(7.0), ref.nan_to_num(7.0)), codes.numel()  # a CPU's own NaN has a sign


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_widen_int8_over_a_list(dtype, offset):
    from flashoptim_amd.kernels import ConversionBatch

    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        values = (torch.arange(n) * 37 % 256 - 128).to(torch.int8)
        cases.append((values, batch.widen_int8(_at(values, offset), dtype)))
    batch.launch()
    for values, got in cases:
        assert parity.bits_equal(got, values.to(dtype)), values.numel()


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("signed,sqrt,softsign", [(True, False, True), (False, True, False), (True, False, False), (False, True, True)])
def test_quantize_over_a_list(signed, sqrt, softsign, dtype, offset):
    """Continuous values, bf16 lattices, values on rounding boundaries and groups beyond the quick forms' range."""
    from flashoptim_amd.kernels import ConversionBatch

    g = torch.Generator().manual_seed(6)
    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        x = torch.randn(n, generator=g) * 10.0 ** (n % 7 - 4)
        if n % 3 == 0:
            x = torch.randint(-127, 128, (n,), generator=g).float() / 127
        x = (x if signed else x.abs()).to(dtype)
        if n > 1024:
            x[40], x[70], x[100] = torch.finfo(dtype).max, torch.finfo(dtype).tiny, 0.0
            x[130:160] = 0.0
        cases.append((x, batch.quantize(_at(x, offset), signed, sqrt, softsign)))
    batch.launch()
    for x, (codes, scales) in cases:
        rc, rs = C.quantize(x, signed, sqrt, softsign)
        assert torch.equal(codes.cpu(), rc), (x.numel(), "codes")
        assert parity.bits_equal(scales, rs), (x.numel(), "scales")


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_narrow_to_int8_over_a_list(dtype, offset):
    from flashoptim_amd.kernels import ConversionBatch

    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        values = ((torch.arange(n) * 37 % 1021) / 4 - 127.75).clamp(-128, 127).to(dtype)
        cases.append((values, batch.narrow_to_int8(_at(values, offset))))
    batch.launch()
    for values, got in cases:
        assert torch.equal(got.cpu(), values.float().trunc().to(torch.int8)), values.numel()


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ecc_dtype", [torch.int8, torch.int16])
def test_import_fp32_over_a_list(ecc_dtype, dtype, offset):
    """Against the cast, the copy and the split it stands for, over magnitudes down to subnormals, infinities and NaN."""
    from flashoptim_amd.kernels import ConversionBatch, compute_ecc_bits

    g = torch.Generator().manual_seed(8)
    special = torch.tensor([0.0, -0.0, 1e-40, 3e38, float("inf"), -float("inf"), float("nan"), 1 + 2.0 ** -8, -(1 + 2.0 ** -9)])
    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        x = torch.exp(torch.empty(n).uniform_(-90, 12, generator=g)) * torch.where(torch.rand(n, generator=g) < 0.5, -1.0, 1.0)
        x[: min(n, 9)] = special[: min(n, 9)]
        x = _at(x, offset)
        narrow = _at(torch.zeros(n, dtype=dtype), offset)
        cases.append((x, narrow, batch.import_fp32(x, narrow, torch.empty(n, dtype=ecc_dtype, device=DEV))))
    batch.launch()
    for x, narrow, ecc in cases:
        want = x.to(dtype)
        assert torch.equal(narrow.view(torch.int16), want.view(torch.int16)), x.numel()
        assert ecc.dtype == ecc_dtype
        assert torch.equal(ecc, compute_ecc_bits(x, want, master_bytewidth=2 + ecc.element_size())), x.numel()


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ecc_dtype", [torch.int8, torch.int16])
def test_export_fp32_over_a_list(ecc_dtype, dtype, offset):
    from flashoptim_amd.kernels import ConversionBatch

    g = torch.Generator().manual_seed(9)
    special = torch.tensor([0.0, -0.0, 1e-40, 6e-8, float("inf"), -float("inf")])
    top = torch.iinfo(ecc_dtype).max
    batch, cases = ConversionBatch(), []
    for n in _lengths(many=offset == 0):
        w = torch.randn(n, generator=g) * 10.0 ** (n % 9 - 5)
        w[: min(n, 6)] = special[: min(n, 6)]
        w = w.to(dtype)
        ecc = torch.randint(-top, top + 1, (n,), generator=g).to(ecc_dtype)
        cases.append((w, ecc, batch.reconstruct_fp32(_at(w, offset), _at(ecc, offset))))
    batch.launch()
    for w, ecc, got in cases:
        want = C.ecc_join(w, ecc)
        assert torch.equal(got.cpu().nan_to_num(7.0), want.nan_to_num(7.0)), w.numel()


def test_fp32_export_of_a_module_with_buffers_tied_and_fp32_weights():
    """Keys, their order and every value as the per-tensor sequence gives them: parameters with a correction term as their
    masters (a tied one under its first name only), everything else cast."""
    import flashoptim_amd as fo

    m = torch.nn.Module()
    m.a = torch.nn.Parameter(torch.randn(33, 70, device=DEV).to(torch.bfloat16))
    m.b = torch.nn.Parameter(torch.randn(1000, device=DEV))
    m.c = torch.nn.Parameter(torch.randn(40, 25, device=DEV).to(torch.bfloat16).t())  # not contiguous: never stepped
    m.register_buffer("buf", torch.arange(5, device=DEV))
    m.tied = m.a
    m.d = torch.nn.Parameter(torch.zeros(0, device=DEV, dtype=torch.bfloat16))
    opt = fo.FlashAdamW(m.parameters(), lr=1e-3)
    for p in (m.a, m.b, m.d):
        p.grad = torch.randn_like(p)
    opt.step()
    opt.state[m.c]["error_bits"] = torch.randint(-127, 128, m.c.shape, device=DEV, dtype=torch.int8)
    want = {k: v.detach().float() for k, v in m.state_dict().items()}
    for k, p in (("a", m.a), ("c", m.c), ("d", m.d)):
        want[k] = C.ecc_join(p.detach().contiguous().cpu(), opt.state[p]["error_bits"].contiguous().cpu()).view(p.shape).to(DEV)
    got = opt.get_fp32_model_state_dict(m)
    assert list(got) == list(want)
    for k, v in want.items():
        assert got[k].dtype == torch.float32 and got[k].shape == v.shape and torch.equal(got[k], v), k


def test_import_fp32_declines_what_it_would_write_wrongly():
    from flashoptim_amd.kernels import ConversionBatch

    x, e = torch.zeros(8, 6, device=DEV), torch.zeros(8, 6, device=DEV, dtype=torch.int8)
    p = torch.zeros(8, 6, device=DEV, dtype=torch.bfloat16)
    declined = [(x.t(), p, e), (x, p.t(), e), (x[:1], p, e), (x.view(48), p, e), (x.cpu(), p, e), (x, x, e), (x.half(), p, e)]
    assert all(ConversionBatch().import_fp32(*args) is None for args in declined)


def test_imports_that_share_memory_keep_their_order():
    """Two parameters over one memory (the last import wins), and a value that lives in a parameter imported later."""
    import flashoptim_amd as fo

    class Holder(torch.nn.Module):
        def __init__(self):
            super().__init__()
            n = 5000
            self.a = torch.nn.Parameter(torch.zeros(n, device=DEV, dtype=torch.bfloat16))
            self.b = torch.nn.Parameter(torch.zeros(0, device=DEV, dtype=torch.bfloat16))
            self.b.data = self.a.data
            self.c = torch.nn.Parameter(torch.full((n,), 3.0, device=DEV))

    m = Holder()
    opt = fo.FlashAdamW(m.parameters(), lr=1e-3)
    for p in m.parameters():
        p.grad = torch.zeros_like(p)
    opt.step()
    n = m.a.numel()
    opt.set_fp32_model_state_dict(m, {"a": m.c.data, "b": torch.full((n,), 2.0, device=DEV), "c": torch.full((n,), 9.0, device=DEV)})
    assert (m.a == 2.0).all() and (m.b == 2.0).all() and (m.c == 9.0).all()
    opt.set_fp32_model_state_dict(m, {"b": m.c.data, "c": torch.full((n,), 4.0, device=DEV)})
    assert (m.b == 9.0).all() and (m.c == 4.0).all()


def test_imports_into_overlapping_spans_keep_their_order():
    """Two parameters that overlap in one buffer: the later import wins where they do, by the one-pass kernel and by the
    general path (a value that is not contiguous); and a value that lives in a parameter imported before it."""
    import flashoptim_amd as fo

    n, shift = 6000, 2048
    flat = torch.zeros(n + shift, device=DEV, dtype=torch.bfloat16)
    m = torch.nn.Module()
    m.a, m.b = torch.nn.Parameter(flat[:n]), torch.nn.Parameter(flat[shift:])
    m.c, m.d = torch.nn.Parameter(torch.zeros(n, device=DEV, dtype=torch.bfloat16)), torch.nn.Parameter(torch.zeros(n // 2, device=DEV))
    opt = fo.FlashAdamW(m.parameters(), lr=1e-3)
    for p in m.parameters():
        p.grad = torch.zeros_like(p)
        opt.step_param(p)  # one after the other: a and b overlap
    value = lambda v: torch.full((n,), v, device=DEV)  # noqa: E731
    for late in (value(2.0), torch.full((2 * n,), 2.0, device=DEV)[::2]):
        opt.set_fp32_model_state_dict(m, {"a": value(1.0), "b": late})
        assert (flat[:shift] == 1.0).all() and (flat[shift:] == 2.0).all()
    words = torch.zeros(n // 2, device=DEV)  # c's memory read as 32-bit words is d's value
    m.c.data = words.view(torch.bfloat16)
    opt.set_fp32_model_state_dict(m, {"c": value(5.0), "d": words})
    assert (m.c == 5.0).all() and torch.equal(m.d.data, m.c.data.view(torch.float32))


def _peak_above_start(call):
    torch.cuda.synchronize()
    start = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    call()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - start


def _stepped(n_tensors, n, dtype, **kw):
    import flashoptim_amd as fo

    m = torch.nn.ParameterList([torch.nn.Parameter(torch.randn(n, device=DEV).to(dtype)) for _ in range(n_tensors)])
    opt = fo.FlashAdamW(m.parameters(), lr=1e-3, **kw)
    for p in m:
        p.grad = torch.randn_like(p)
    opt.step()
    return m, opt


def test_import_of_host_masters_holds_few_of_them_on_the_device(monkeypatch):
    """The device copies of a list of host tensors do not add up: beside the new correction codes at most the batch's
    budget and the value at hand are alive."""
    from flashoptim_amd import kernels

    budget = 8 << 20
    monkeypatch.setattr(kernels, "_COPIES_HELD", budget, raising=False)
    n_tensors, n = 24, 1 << 20
    m, opt = _stepped(n_tensors, n, torch.bfloat16)
    masters = {k: torch.randn(n) for k, _ in m.named_parameters()}
    peak = _peak_above_start(lambda: opt.set_fp32_model_state_dict(m, masters))
    # the new codes (the launch plan of the last step keeps the old ones), the copies, the value at hand
    assert peak <= n_tensors * n + budget + 4 * n, peak
    for k, p in m.named_parameters():
        want = masters[k].to(torch.bfloat16)
        assert torch.equal(p.detach().cpu(), want), k
        assert torch.equal(opt.state[p]["error_bits"], kernels.compute_ecc_bits(masters[k].to(DEV), p.detach(), 3)), k


@pytest.mark.parametrize("compress", [False, True])
def test_load_of_a_host_checkpoint_frees_what_it_has_converted(compress, monkeypatch):
    """torch brings the whole checkpoint to the device in the parameters' dtype first; each part is freed once it is
    converted, give or take the batch's budget.  A checkpoint on the device stays whole in one launch."""
    from flashoptim_amd import kernels

    budget = 8 << 20
    monkeypatch.setattr(kernels, "_COPIES_HELD", budget, raising=False)
    n_tensors, n = 24, 1 << 20
    m, opt = _stepped(n_tensors, n, torch.bfloat16, compress_state_dict=compress)
    saved = opt.state_dict()
    host = {"state": {i: {k: v.cpu() if isinstance(v, torch.Tensor) else v for k, v in st.items()} for i, st in saved["state"].items()},
            "param_groups": saved["param_groups"]}
    cast = 6 * n_tensors * n  # both moments and the correction codes, two bytes each
    peak = _peak_above_start(lambda: opt.load_state_dict(host))
    assert peak <= cast + cast // 32 + budget + 8 * n, peak
    states = lambda: [t for p in m for st in [opt.state[p]] for t in (  # noqa: E731
        st["exp_avg"].quantized, st["exp_avg"].scales, st["exp_avg_sq"].quantized, st["exp_avg_sq"].scales, st["error_bits"])]
    loaded, launches, issue = states(), [], kernels.ConversionBatch.launch
    monkeypatch.setattr(kernels.ConversionBatch, "launch", lambda self: (launches.append(len(self._jobs)), issue(self)))
    opt.load_state_dict(saved)
    assert len(launches) == 1
    assert all(torch.equal(a, b) for a, b in zip(loaded, states()))


def test_values_with_a_negation_put_off_are_converted_as_what_they_stand_for():
    import flashoptim_amd as fo
    from flashoptim_amd.kernels import ConversionBatch, compute_ecc_bits

    m = torch.nn.Module()
    m.w = torch.nn.Parameter(torch.zeros(700, device=DEV, dtype=torch.bfloat16))
    opt = fo.FlashAdamW(m.parameters(), lr=1e-3)
    m.w.grad = torch.zeros_like(m.w)
    opt.step()
    master = torch.randn(700, device=DEV)
    opt.set_fp32_model_state_dict(m, {"w": torch._neg_view(master)})
    assert torch.equal(m.w.detach(), (-master).to(torch.bfloat16))
    assert torch.equal(opt.state[m.w]["error_bits"], compute_ecc_bits(-master, m.w.detach(), 3))
    batch, codes = ConversionBatch(), torch.arange(-100, 100, device=DEV, dtype=torch.int8)
    narrow, wide = batch.narrow_to_int8(torch._neg_view(codes.to(torch.bfloat16))), batch.widen_int8(torch._neg_view(codes), torch.bfloat16)
    batch.launch()
    assert torch.equal(narrow, -codes) and torch.equal(wide, -codes.to(torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("second_moment", [False, True])
def test_quantize_of_values_that_are_not_finite_or_negative(second_moment, dtype):
    """The two kinds of state whose codes take a quick form, against the formula in IEEE arithmetic: NaN, infinities and
    negative second moments (a NaN after the root), alone in a lane and beside ordinary values, at every place of it.  A NaN
    takes no part in the group's maximum and its code is 0, what the conversion instruction makes of it."""
    from flashoptim_amd.kernels import ConversionBatch

    nan, inf = float("nan"), float("inf")
    g = torch.Generator().manual_seed(11)
    odd = [nan, -nan, inf, -inf, -1.0, -0.0, 1e-30]
    rows = []
    for value in odd:
        for at in range(32):  # one of them at each place of a group
            row = torch.randn(32, generator=g).abs()
            row[at] = value
            rows.append(row)
        rows.append(torch.where(torch.arange(32) % 8 == 3, torch.randn(32, generator=g).abs(), torch.tensor(value)))
        rows.append(torch.full((32,), value))
    x = torch.cat(rows)
    if not second_moment:
        x = torch.where((torch.rand(x.shape, generator=g) < 0.5) & x.isfinite(), -x, x)
    x = x.to(dtype)
    batch = ConversionBatch()
    codes, scales = batch.quantize(x.to(DEV), not second_moment, second_moment, not second_moment)
    batch.launch()
    v = x.float().view(-1, 32)
    v = v.sqrt() if second_moment else v
    top = v.abs().nan_to_num(0.0, posinf=inf).amax(1, keepdim=True).clamp(min=1e-12)
    t = v / top
    if second_moment:
        q = (t * 255 + 0.5).floor()
    else:
        q = ((2 * t) / (1 + t.abs()) * 127 + 0.5).floor()
    want = q.nan_to_num(0.0).to(torch.int32).view(-1).to(codes.dtype)
    assert torch.equal(codes.cpu(), want)
    assert parity.bits_equal(scales, top.view(-1).to(torch.float16))
