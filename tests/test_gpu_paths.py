"""GPU: the sizes at which a launch takes another kernel or a kernel another
branch (one-workgroup and sliced selection, one and several dot-product
chunks), against the oracle or a plain sort.  Bar: bit-exact."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import log

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# one workgroup of 1024 threads takes up to 32768 ratios, slices of 16384 more
@pytest.mark.parametrize("nb", [1, 2, 63, 1023, 1025, 32_767, 32_768, 32_769, 49_153, 70_001])
def test_thresholds_at_the_selection_sizes(nb):
    from turboadam_amd import costate as C

    log(f"thresholds nb={nb}")
    rng = np.random.default_rng(nb)
    base = np.abs(rng.standard_normal(nb)).astype(np.float32)
    two = np.where(np.arange(nb) < nb // 2, np.float32(0.5), np.float32(0.75)).astype(np.float32)
    nan = base.copy()
    nan[:: 3] = np.nan
    nan[1:: 7] = 0.0
    narrow = (np.float32(1.0).view(np.uint32) + rng.integers(0, 1 << 12, nb, dtype=np.uint32)).view(np.float32)
    for what, r in (("normal", base), ("two values", two), ("nan and zero", nan), ("narrow", narrow),
                    ("equal", np.full(nb, 0.37, np.float32))):
        for null_pct, amp_pct in ((0.1, 0.9), (0.05, 0.95), (0.0, 1.0)):
            k_lo, k_hi = O.ranks(nb, null_pct, amp_pct)
            keys = np.sort(r.view(np.uint32))
            got = [np.float32(x.item()).view(np.uint32) for x in C.compute_thresholds(_t(r), null_pct, amp_pct)]
            assert got == [keys[k_lo], keys[k_hi]], (what, null_pct)


# 8192 quarter-tile partials (of 512 elements) make one chunk of the dot products' tree
@pytest.mark.parametrize("n", [512 * 4, 512 * 1024 + 1, 512 * 8192, 512 * 8192 + 1, 512 * 8192 * 2 + 12_345])
def test_alpha_at_the_chunk_sizes(n):
    from turboadam_amd import costate as C

    log(f"alpha n={n}")
    rng = np.random.default_rng(n)
    g = rng.standard_normal(n, dtype=np.float32) * np.float32(1e-3)
    m = np.float32(0.4) * g + rng.standard_normal(n, dtype=np.float32) * np.float32(1e-4)
    delta_o = np.empty(n, np.float32)
    alpha_o = O.lib().or_decompose(O.ptr(m), O.ptr(g), n, O.ptr(delta_o))
    alpha, delta = C.decompose(_t(m), _t(g))
    assert np.float32(alpha.item()) == np.float32(alpha_o)
    assert np.array_equal(delta.cpu().numpy().view(np.uint32), delta_o.view(np.uint32))


def _np(t):
    t = t.detach().cpu()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.float16 else t.numpy()


def _values(n, seed):
    """A positive v with what the certified index must hand to the exact path:
    values on a block's index boundaries, zeros, negatives, NaN and infinities."""
    rng = np.random.default_rng(seed)
    v = np.exp(rng.uniform(-30, -12, n)).astype(np.float32)
    nb = n // 128
    for b in range(0, nb, 3):  # log-equidistant: every index boundary of 16 levels is hit
        v[128 * b:128 * (b + 1)] = np.exp(np.linspace(-20, -12, 129)[:128]).astype(np.float32)
        v[128 * b + 127] = np.float32(np.exp(-12.0))
    for b in range(1, nb, 5):
        v[128 * b + 3] = 0.0
    if nb > 6:
        v[128 * 2 + 7] = -1.0
        v[128 * 4 + 9] = np.nan
        v[128 * 5 + 1] = np.inf
        v[128 * 6:128 * 7] = np.float32(0.25)  # no span
    return v


# a unit is 8 blocks (1024 elements) of one wave
@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("bits", [2, 3, 4, 6, 8])
@pytest.mark.parametrize("n", [128, 128 * 7, 1024, 1024 * 4 + 128, 1024 * 40])
def test_quantize_units(n, bits, stochastic):
    from turboadam_amd import quantize as Q

    log(f"quantize n={n} bits={bits} stochastic={stochastic}")
    v = _values(n, n + bits)
    idx_o, sc_o = np.empty(n, np.uint8), np.empty(n // 64, np.uint16)
    O.lib().or_quantize_logscale(O.ptr(v), n, bits, int(stochastic), 3, 4, 99, O.ptr(idx_o), O.ptr(sc_o))
    idx, sc, _ = Q.quantize_logscale_nbits(_t(v), bits, stochastic_round=stochastic, tensor_id=3, step=4, seed=99)
    assert np.array_equal(_np(idx), idx_o)
    nan = np.isnan(sc_o.view(np.float16))
    got = _np(sc).reshape(-1)
    assert np.array_equal(np.isnan(got.view(np.float16)), nan) and np.array_equal(got[~nan], sc_o[~nan])
    # a view that is aligned to its elements only
    base = torch.zeros(n + 1, device=DEV)
    base[1:] = _t(v)
    idx2, _, _ = Q.quantize_logscale_nbits(base[1:], bits, stochastic_round=stochastic, tensor_id=3, step=4, seed=99)
    assert torch.equal(idx, idx2)


@pytest.mark.parametrize("stochastic", [False, True])
@pytest.mark.parametrize("what", ["plain", "zero", "nan"])
@pytest.mark.parametrize("n", [1, 64, 127, 129, 1024 + 5, 128 * 33 + 90])
def test_compress_partial_block(n, what, stochastic):
    """The last block's missing elements take max(min(v), 1e-38) of the whole
    tensor, NaN when it holds one."""
    from turboadam_amd import oneq

    log(f"compress n={n} {what} stochastic={stochastic}")
    v = np.exp(np.random.default_rng(n).uniform(-30, -12, n)).astype(np.float32)
    if what != "plain":
        v[n // 3] = 0.0 if what == "zero" else np.nan
    nb = (n + 127) // 128
    pad = np.full(nb * 128, np.nan if what == "nan" else max(v.min(), np.float32(1e-38)), np.float32)
    pad[:n] = v
    idx_o, sc_o = np.empty(nb * 128, np.uint8), np.empty(nb * 2, np.uint16)
    O.lib().or_quantize_logscale(O.ptr(pad), nb * 128, 4, int(stochastic), 0, 1, 7, O.ptr(idx_o), O.ptr(sc_o))
    c = oneq.compress_v_logscale(_t(v), 4, stochastic_round=stochastic, seed=7)
    assert np.array_equal(_np(c["indices"]), idx_o)
    nan = np.isnan(sc_o.view(np.float16))
    got = _np(c["scales"]).reshape(-1)
    assert np.array_equal(np.isnan(got.view(np.float16)), nan) and np.array_equal(got[~nan], sc_o[~nan])


@pytest.mark.parametrize("n", [1, 256, 300])
def test_compress_of_a_negated_view(n):
    """A tensor with torch's negative bit (the imaginary part of a conjugate) means
    the negated values of its memory."""
    from turboadam_amd import oneq

    log(f"compress a negated view, n={n}")
    v = torch.rand(n, device=DEV) + 1e-3
    neg = torch._neg_view(-v)
    assert neg.is_neg() and torch.equal(neg, v)
    a, b = oneq.compress_v_logscale(v, 4), oneq.compress_v_logscale(neg, 4)
    assert torch.equal(a["indices"], b["indices"]) and torch.equal(a["scales"], b["scales"])


@pytest.mark.parametrize("bits", [2, 3, 4, 6, 8])
@pytest.mark.parametrize("n", [1, 128, 1023, 1024, 1025, 1024 * 5 + 77])
def test_dequantize_units(n, bits):
    from turboadam_amd import quantize as Q

    log(f"dequantize n={n} bits={bits}")
    rng = np.random.default_rng(n + bits)
    nb = (n + 127) // 128
    lo = rng.uniform(-60, 10, nb).astype(np.float32)
    sc = np.stack([lo, lo + rng.uniform(0, 9, nb).astype(np.float32)], 1).astype(np.float16)
    for top in (1 << bits, 256):  # in range, and beyond it (decoded by the same formula)
        idx = rng.integers(0, top, nb * 128).astype(np.uint8)
        want = O.dequantize(idx, sc.view(np.uint16).reshape(-1), n, bits)
        got = Q.dequantize_logscale_nbits(_t(idx), _t(sc), bits, original_numel=n)
        assert np.array_equal(_np(got).view(np.uint32), want.view(np.uint32)), top
        base = torch.zeros(nb * 128 + 1, dtype=torch.uint8, device=DEV)
        base[1:] = _t(idx)
        assert torch.equal(Q.dequantize_logscale_nbits(base[1:], _t(sc), bits, original_numel=n), got)


@pytest.mark.parametrize("bits,dt", [(4, torch.float32), (2, torch.bfloat16), (8, torch.float16), (6, torch.bfloat16)])
@pytest.mark.parametrize("n", [1, 513, 1024, 1025, 1024 * 4 + 640])
def test_fused_v_units(n, bits, dt):
    from turboadam_amd import quantize as Q

    log(f"fused_v_update n={n} bits={bits} {dt}")
    rng = np.random.default_rng(n + bits)
    nb = (n + 127) // 128
    idx = rng.integers(0, 1 << bits, nb * 128).astype(np.uint8)
    lo = rng.uniform(-25, -15, nb).astype(np.float32)
    sc = np.stack([lo, lo + rng.uniform(0, 6, nb).astype(np.float32)], 1).astype(np.float16).view(np.uint16)
    base = torch.zeros(n + 1, dtype=dt)  # the gradient is a view one element into it
    base[1:] = (torch.from_numpy(rng.standard_normal(n).astype(np.float32)) * 1e-3).to(dt)
    g32 = base[1:].float().numpy().copy()
    idx_o, sc_o, v_o = idx.copy(), sc.reshape(-1).copy(), np.empty(n, np.float32)
    O.lib().or_fused_v_update(O.ptr(idx_o), O.ptr(sc_o), O.ptr(g32), n, bits, O.f32(0.999), O.f32(1.0 - 0.999),
                              5, 9, 1234, O.ptr(v_o))
    ni, ns, v = Q.fused_v_update(_t(idx), _t(sc.view(np.float16)), base.to(DEV)[1:], 0.999, bits, tensor_id=5, step=9,
                                 seed=1234)
    assert np.array_equal(_np(ni), idx_o) and np.array_equal(_np(ns).reshape(-1), sc_o)
    assert np.array_equal(_np(v).view(np.uint32), v_o.view(np.uint32))


# a tensor's last tile may hold quarters past its end, whose partial sums no kernel writes
@pytest.mark.parametrize("dt", [O.DT_F32, O.DT_BF16])
def test_step_reads_no_workspace_it_did_not_write(dt, monkeypatch):
    from tests.helpers import run_side_by_side
    from turboadam_amd import optimizer

    sizes = [1024 * 5, 1024 * 9, 4096 + 77, 512 * 9, 512 * 11 + 3, 2048 * 3, 128 * 33, 700]
    log(f"step on a workspace of NaN bytes, dtype {dt}")
    plain = optimizer._DeviceBuffers.workspace

    def poisoned(self, nbytes):
        ws = plain(self, nbytes)
        ws.fill_(255)
        return ws

    monkeypatch.setattr(optimizer._DeviceBuffers, "workspace", poisoned)
    for ef in (False, True):
        bad = run_side_by_side(sizes, [dt] * len(sizes), steps=3, error_feedback=ef)
        assert not bad, "\n".join(bad[:10])


# units of 1024 elements, then quarters of 512; one dot-product chunk up to 4194304
@pytest.mark.parametrize("ef", [False, True])
@pytest.mark.parametrize("n,dt", [(1, torch.float32), (513, torch.bfloat16), (1024, torch.float16),
                                  (1025, torch.float32), (1024 * 9 + 640, torch.bfloat16),
                                  (512 * 8192 + 1000, torch.float32)])
def test_costate_update_units(n, dt, ef):
    from turboadam_amd import costate as C

    log(f"CoStateManager.update n={n} {dt} ef={ef}, 3 steps")
    rng = np.random.default_rng(n)
    nb = (n + 127) // 128
    labels, signs = np.zeros(nb, np.uint8), np.zeros((n + 7) // 8, np.uint8)
    norms, amp, alpha, res = (np.zeros(nb, np.float32), np.zeros(nb, np.uint16), np.zeros(1, np.float32),
                              np.zeros(n, np.float32))
    mgr = C.CoStateManager(error_feedback=ef)
    # state arrays that the kernels cannot take as they are are updated through copies
    mgr.allocate(n, DEV)
    mgr._encoded["block_norms"] = torch.zeros(nb, dtype=torch.float64, device=DEV)
    mgr._encoded["sign_packed"] = torch.zeros(signs.size + 1, dtype=torch.uint8, device=DEV)[1:]
    k_lo, k_hi = O.ranks(nb, 0.10, 0.90)
    kept = None
    for s in range(3):
        g = (torch.from_numpy(rng.standard_normal(n).astype(np.float32)) * 1e-3).to(dt)
        g32, m_o = g.float().numpy().copy(), np.empty(n, np.float32)
        O.lib().or_costate_update_ef(O.ptr(g32), n, O.f32(0.9), O.f32(1.0 - 0.9), float(np.float32(np.sqrt(128.0))),
                                     k_lo, k_hi, int(s > 0), O.ptr(labels), O.ptr(signs), O.ptr(norms), O.ptr(amp),
                                     O.ptr(alpha), int(ef), int(ef and s > 0), O.ptr(res), O.ptr(m_o))
        before = (kept, kept.clone()) if kept is not None else None
        m = mgr.update(g.to(DEV), 0.9)
        enc = mgr._encoded
        got = {"m": m, "labels": enc["labels"], "signs": enc["sign_packed"], "norms": enc["block_norms"].float(),
               "amp": enc["scales"], "alpha": mgr._alpha.reshape(1)}
        want = {"m": m_o, "labels": labels, "signs": signs, "norms": norms, "amp": amp, "alpha": alpha}
        if ef:
            got["residual"], want["residual"] = mgr._ef_residual, res
            if before is not None:  # the previous residual tensor is left as it was
                assert torch.equal(*before)
            kept = mgr._ef_residual
        for k, t in got.items():
            a, b = np.ascontiguousarray(_np(t)), want[k]
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"step {s}: {k}"


def test_fp32_update_square_root_and_reciprocal_on_every_input():
    """The fp32 update's own square root and reciprocal equal the correctly
    rounded ones on every input of the ranges it uses them on."""
    from turboadam_amd import _lib

    lib, chunk = _lib.load(), 1 << 27
    out = torch.empty(chunk, dtype=torch.float32, device=DEV)
    # (function, first and last bit pattern): sqrt on [2^-62, 2^127], 1/x on [2^-126, 2^126]
    for fn, lo, hi in ((9, 0x20800000, 0x7F000001), (10, 0x00800000, 0x7E800001)):
        wrong = 0
        for start in range(lo, hi, chunk):
            n = min(chunk, hi - start)
            x = torch.arange(start, start + n, dtype=torch.int64, device=DEV).to(torch.int32).view(torch.float32)
            _lib.check(lib.tam_math_eval(fn, x.data_ptr(), out.data_ptr(), n, _lib.stream_of(DEV)), "tam_math_eval")
            # rounding fp64's correctly rounded result once more gives the fp32 one (sqrt and 1/x of
            # 24-bit values stay 2^-50 away from a rounding boundary)
            want = (x.double().sqrt() if fn == 9 else 1.0 / x.double()).float()
            wrong += int((out[:n] != want).sum())
        log(f"function {fn}: {hi - lo} inputs, {wrong} wrong")
        assert wrong == 0


@pytest.mark.parametrize("what", ["random", "near midpoints", "all ones and powers of two", "range ends"])
def test_fp32_update_quotient(what):
    """The fp32 update's own quotient a/x equals the correctly rounded one where it
    is used: |a| >= 2^-100, x from 2^-32 to 2^80, the quotient from 2^-100 to 2^100."""
    from turboadam_amd import _lib

    lib, n = _lib.load(), 1 << 24
    gen = torch.Generator(device=DEV)
    gen.manual_seed(11)

    def ints(lo, hi):
        return torch.randint(lo, hi, (n,), generator=gen, device=DEV, dtype=torch.int64)

    def power(e):
        return torch.ldexp(torch.ones((), device=DEV, dtype=torch.float64), e)

    for rnd in range(8):
        sig_a, sig_x = ints(1 << 23, 1 << 24).double(), ints(1 << 23, 1 << 24).double()
        exp_x = ints(-32, 80)
        exp_a = ints(-100, 120)
        if what == "near midpoints":  # a next to x times a 25-bit odd significand
            exact = sig_x * (2 * ints(1 << 23, 1 << 24) + 1).double()  # 49 bits
            a = (exact * 2.0 ** -25).float() if rnd % 2 else exact.float() * 2.0 ** -25
            step = ints(-2, 3).to(torch.int32)
            sig_a = (a.view(torch.int32) + step).view(torch.float32).double()
        elif what == "all ones and powers of two":
            edge = torch.tensor([1 << 23, (1 << 23) + 1, (1 << 24) - 1, (1 << 24) - 2, 3 << 22], device=DEV).double()
            sig_x = edge[ints(0, 5)]
            if rnd % 2:
                sig_a = edge[ints(0, 5)]
        elif what == "range ends":
            ends = torch.tensor([-32, -31, 78, 79], device=DEV)
            exp_x = ends[ints(0, 4)]
            exp_a = torch.where(ints(0, 2) == 0, ints(-100, -97), exp_x + ints(-101, -96))
            if rnd % 2:
                exp_a = exp_x + ints(96, 101)
        a = (sig_a * 2.0 ** -23 * power(exp_a)).float()
        a = torch.where(ints(0, 2) == 0, a, -a)
        x = (sig_x * 2.0 ** -23 * power(exp_x)).float()
        q = a.double() / x.double()
        ok = (a.abs() >= 2.0 ** -100) & torch.isfinite(a) & (q.abs() >= 2.0 ** -100) & (q.abs() < 2.0 ** 100)
        pairs = torch.stack([a, x], 1)[ok].contiguous()
        want = q[ok].float()  # 53 bits >= 2 * 24 + 2: the second rounding changes nothing
        out = torch.empty_like(want)
        _lib.check(lib.tam_math_eval(11, pairs.data_ptr(), out.data_ptr(), out.numel(), _lib.stream_of(DEV)),
                   "tam_math_eval")
        wrong = int((out != want).sum())
        log(f"quotient, {what}: {out.numel()} pairs, {wrong} wrong")
        assert out.numel() > n // 20 and wrong == 0


@pytest.mark.parametrize("kw", [dict(eps=1e-8), dict(eps=0.0), dict(eps=1e-30), dict(eps=1e4), dict(lr=0.0),
                                dict(betas=(0.9, 0.5)), dict(betas=(0.0, 0.999), weight_decay=0.1)])
def test_fp32_update_ranges(kw):
    """Parameters around 2^-40, zeros, huge and infinite ones, gradients from
    subnormal to overflowing: lanes of the fast update and of the other one."""
    from turboadam_amd import TurboAdam

    log(f"fp32 update ranges {kw}")
    rng = np.random.default_rng(3)
    sizes = [1024 * 6, 3000, 1024 * 2 + 77]
    for compress_v in (True, False):
        init = [(rng.standard_normal(n) * 0.02).astype(np.float32) for n in sizes]
        for p in init:
            p[64:128] *= np.float32(2.0 ** -34)
            p[130:140] = 0.0
            p[300:310] = np.float32(1e38)
            p[320] = np.inf
            p[330] = -np.nan
            p[340:360] = np.float32(2.0 ** -40)
        o_params = [a.copy() for a in init]
        params = [torch.nn.Parameter(_t(a)) for a in init]
        opt = TurboAdam(params, compress_v=compress_v, philox_seed=5, **kw)
        orc = O.OracleTurboAdam(o_params, dtypes=[O.DT_F32] * len(sizes), seed=5, compress_v=compress_v, **kw)
        for s in range(3):
            grads = [(rng.standard_normal(n) * np.exp(rng.uniform(-60, 2, n))).astype(np.float32) for n in sizes]
            for g in grads:
                g[200:260] = 0.0
                g[256:384] = 0.0
                g[400:404] = np.float32(1e-42)
                g[410] = np.float32(1e25)
            if s == 2:
                grads[0][500] = np.inf
            for p, g in zip(params, grads):
                p.grad = _t(g)
            opt.step()
            orc.step(grads)
            for i, p in enumerate(params):
                a, b = p.detach().cpu().numpy(), o_params[i].reshape(-1)
                assert np.array_equal(np.isnan(a), np.isnan(b)), (s, i)
                k = ~np.isnan(b)
                assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (s, i, compress_v)


@pytest.mark.parametrize("kw", [dict(), dict(lr=0.0), dict(lr=-1e-3), dict(weight_decay=0.1), dict(lr=1e-30),
                                dict(compress_m=False), dict(compress_v=False), dict(betas=(0.0, 0.999))])
def test_fp32_update_of_zero_parameters(kw):
    """Parameters of +0, -0 and below 2^-40 (pruned, masked, zero-initialised) among
    ordinary ones, kept there from step to step, with gradients of either zero,
    tiny, ordinary and large: the sign of a zero result and every last bit."""
    from turboadam_amd import TurboAdam

    log(f"fp32 update of zero parameters {kw}")
    rng = np.random.default_rng(9)
    kw = dict(dict(lr=1e-3), **kw)
    n = 1024 * 5
    small = np.float32([0.0, -0.0, 1e-45, -1e-45, 2.0 ** -126, -(2.0 ** -100), 2.0 ** -41, 2.0 ** -40, np.nan])
    init = (rng.standard_normal(n) * 0.02).astype(np.float32)
    at = np.concatenate([np.arange(1024, 2048), rng.choice(n, 700, replace=False)])
    init[at] = rng.choice(small, at.size, p=[0.4, 0.4] + [0.2 / 7] * 7)
    o_param = init.copy()
    p = torch.nn.Parameter(_t(init))
    opt = TurboAdam([p], philox_seed=6, **kw)
    orc = O.OracleTurboAdam([o_param], dtypes=[O.DT_F32], seed=6, **kw)
    some = np.float32([0.0, -0.0, 1e-42, 2.0 ** -110, -(2.0 ** -90), 1e-12, -1e-3, 1e3])
    for s in range(5):
        g = (rng.standard_normal(n) * 1e-3).astype(np.float32)
        pick = rng.choice(at, 1500)
        g[pick] = rng.choice(some, pick.size)
        g[1024 + 256:1024 + 384] = 0.0  # a block without gradients
        p.grad = _t(g)
        opt.step()
        orc.step([g])
        a, b = p.detach().cpu().numpy(), o_param.reshape(-1)
        assert np.array_equal(np.isnan(a), np.isnan(b)), s
        k = ~np.isnan(b)
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), s
        with torch.no_grad():  # pruned again: masked parameters go back to where they were
            p[_t(at)] = _t(init[at])
        o_param.reshape(-1)[at] = init[at]


# pass 0 has a kernel for each mode (fp32 first moment, fp32 second moment, error feedback, any), pass 2 for
# error feedback; mixed: tensors of two modes in one dtype
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("dt", [O.DT_F32, O.DT_BF16, O.DT_F16])
@pytest.mark.parametrize("kw", [dict(compress_m=False), dict(compress_v=False), dict(compress_m=False, compress_v=False),
                                dict(error_feedback=True), dict(error_feedback=True, compress_v=False),
                                dict(error_feedback=True, v_bits=8), dict(min_m_compress_elements=6000)])
def test_step_modes(kw, dt, offset):
    from tests.helpers import run_side_by_side

    log(f"step {kw} dtype {dt} offset {offset}")
    sizes = [1024 * 5 + 300, 4096, 1024 * 2, 700, 9000, 512 * 17]
    bad = run_side_by_side(sizes, [dt] * len(sizes), steps=3, offset=offset, **kw)
    assert not bad, "\n".join(bad[:10])
