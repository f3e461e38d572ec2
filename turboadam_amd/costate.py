"""CoState first-moment codec (reference src/turboadam/costate.py).

m = alpha*g + delta is stored as one fp32 alpha per tensor plus, per
128-element block, a label (0 null, 1 phase, 2 amplitude), the residual L2
norm (fp32), an fp16 amplitude scale and one sign bit per element (MSB first).

TurboAdam.step runs the whole update fused in its multi-tensor launches.
The reference's public functions are also available one tensor at a time,
with the same names and argument meaning, on the gfx950 kernels (the
step's arithmetic: fp32 lane partials and fp64 pairwise sums for the dot
products and block norms, exact radix selection).  Inputs must be on an
MI355X (HIP) device.
"""

import ctypes

import torch

from . import _lib
from .utils import BLOCK_SIZE, num_blocks


def _require_gpu(t: torch.Tensor, what: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(f"turboadam_amd.{what}: tensors must be on an MI355X (HIP) device, got {t.device}")


def _require_block_size(block_size: int) -> None:
    if block_size != BLOCK_SIZE:
        raise NotImplementedError("turboadam_amd supports block_size=128 only")


def _f32_flat(t: torch.Tensor) -> torch.Tensor:
    return t.reshape(-1).float().contiguous()


def _scalar_on(x, device) -> torch.Tensor:
    """A 1-element fp32 device tensor holding x (a Python number or a tensor)."""
    if isinstance(x, torch.Tensor):
        return x.reshape(1).to(device=device, dtype=torch.float32).contiguous()
    return torch.tensor([float(x)], dtype=torch.float32, device=device)


def decompose(m: torch.Tensor, g: torch.Tensor):
    """alpha = (m.g)/(g.g) (0 when g.g == 0) and delta = m - alpha*g
    (reference costate.py:22-43).  Returns (alpha 0-dim fp32, delta like m)."""
    _require_gpu(m, "decompose")
    lib = _lib.load()
    mf, gf = _f32_flat(m), _f32_flat(g)
    n = mf.numel()
    alpha = torch.empty(1, dtype=torch.float32, device=m.device)
    delta = torch.empty(n, dtype=torch.float32, device=m.device)
    ws = torch.empty(lib.tam_decompose_workspace(max(n, 1)), dtype=torch.uint8, device=m.device)
    with torch.cuda.device(m.device):
        _lib.check(lib.tam_decompose(mf.data_ptr(), gf.data_ptr(), n, alpha.data_ptr(), delta.data_ptr(),
                                     ws.data_ptr(), ws.numel(), _lib.stream_of(m.device)), "tam_decompose")
    return alpha.reshape(()), delta.reshape(m.shape)


def compute_block_ratios(delta: torch.Tensor, m: torch.Tensor, block_size: int = BLOCK_SIZE) -> torch.Tensor:
    """r_b = ||delta_b|| / ||m_b||, 0 where ||m_b|| == 0 (reference costate.py:51-86)."""
    _require_gpu(delta, "compute_block_ratios")
    _require_block_size(block_size)
    lib = _lib.load()
    df, mf = _f32_flat(delta), _f32_flat(m)
    n = df.numel()
    ratios = torch.empty(num_blocks(n), dtype=torch.float32, device=delta.device)
    with torch.cuda.device(delta.device):
        _lib.check(lib.tam_block_ratios(df.data_ptr(), mf.data_ptr(), n, ratios.data_ptr(),
                                        _lib.stream_of(delta.device)), "tam_block_ratios")
    return ratios


def threshold_ranks(nb: int, null_pct: float, amp_pct: float):
    """Sorted positions of the two thresholds (costate.py:115-117, Python double arithmetic)."""
    return max(0, int(null_pct * nb) - 1), min(nb - 1, int(amp_pct * nb))


def compute_thresholds(ratios: torch.Tensor, null_pct: float = 0.10, amp_pct: float = 0.90):
    """(tau0, tau1): the ratios at sorted positions max(0, int(null_pct*nb)-1) and
    min(nb-1, int(amp_pct*nb)), NaN sorting last (reference costate.py:94-118)."""
    _require_gpu(ratios, "compute_thresholds")
    lib = _lib.load()
    r = ratios.reshape(-1).float().contiguous()
    if r.data_ptr() % 16:
        r = r.clone()
    nb = r.numel()
    if nb == 0:
        raise IndexError("compute_thresholds: empty ratios")
    k_lo, k_hi = threshold_ranks(nb, null_pct, amp_pct)
    taus = torch.empty(2, dtype=torch.float32, device=r.device)
    ws = torch.empty(lib.tam_thresholds_workspace(nb), dtype=torch.uint8, device=r.device)
    with torch.cuda.device(r.device):
        _lib.check(lib.tam_thresholds(r.data_ptr(), nb, k_lo, k_hi, taus.data_ptr(), ws.data_ptr(), ws.numel(),
                                      _lib.stream_of(r.device)), "tam_thresholds")
    return taus[0], taus[1]


def classify_blocks(ratios: torch.Tensor, tau0, tau1) -> torch.Tensor:
    """label = 2 if r >= tau1, 1 if r >= tau0, else 0 (reference costate.py:126-149)."""
    _require_gpu(ratios, "classify_blocks")
    lib = _lib.load()
    r = ratios.reshape(-1).float().contiguous()
    taus = torch.cat([_scalar_on(tau0, r.device), _scalar_on(tau1, r.device)])
    labels = torch.empty(r.numel(), dtype=torch.uint8, device=r.device)
    with torch.cuda.device(r.device):
        _lib.check(lib.tam_classify(r.data_ptr(), r.numel(), taus.data_ptr(), labels.data_ptr(),
                                    _lib.stream_of(r.device)), "tam_classify")
    return labels


def encode_blocks(delta: torch.Tensor, labels: torch.Tensor, block_size: int = BLOCK_SIZE) -> dict:
    """Block norms, fp16 amplitudes and packed sign bits of delta; labels pass
    through (reference costate.py:213-258)."""
    _require_gpu(delta, "encode_blocks")
    _require_block_size(block_size)
    lib = _lib.load()
    df = _f32_flat(delta)
    n = df.numel()
    nb = num_blocks(n)
    dev = delta.device
    signs = torch.empty((n + 7) // 8, dtype=torch.uint8, device=dev)
    norms = torch.empty(nb, dtype=torch.float32, device=dev)
    amp = torch.empty(nb, dtype=torch.float16, device=dev)
    with torch.cuda.device(dev):
        _lib.check(lib.tam_costate_encode(df.data_ptr(), n, signs.data_ptr(), norms.data_ptr(), amp.data_ptr(),
                                          _lib.stream_of(dev)), "tam_costate_encode")
    return {"labels": labels, "sign_packed": signs, "block_norms": norms, "scales": amp}


_ENCODED_DTYPES = {"labels": torch.uint8, "sign_packed": torch.uint8, "block_norms": torch.float32,
                   "scales": torch.float16}


def _check_covers(encoded: dict, n: int) -> None:
    nb = num_blocks(n)
    if (encoded["labels"].numel() != nb or encoded["block_norms"].numel() != nb
            or encoded["scales"].numel() != nb or encoded["sign_packed"].numel() < (n + 7) // 8):
        raise ValueError(f"decode_blocks: the encoding does not cover {n} elements ({nb} blocks)")


def _in_form(t: torch.Tensor, dtype, device) -> torch.Tensor:
    """t itself when it is a contiguous array of dtype on device, aligned as the
    kernels need (4 bytes at most), else a copy that is."""
    c = t.to(device=device, dtype=dtype).contiguous()
    return c if c.data_ptr() % 4 == 0 else c.clone()


def decode_blocks(encoded: dict, alpha, g: torch.Tensor, block_size: int = BLOCK_SIZE,
                  original_numel: int = None) -> torch.Tensor:
    """m_hat = alpha*g + s_b*sign (s_b: 0, norm_b/sqrt(128) or the fp16
    amplitude by label), in fp32 with the shape of g (reference costate.py:261-324)."""
    _require_gpu(g, "decode_blocks")
    _require_block_size(block_size)
    n = g.numel() if original_numel is None else original_numel
    lib = _lib.load()
    dev = g.device
    gf = g.reshape(-1)
    if gf.dtype not in _lib.DTYPES:
        gf = gf.float()
    gf = gf.contiguous()
    if n != gf.numel():
        raise ValueError(f"decode_blocks: original_numel {n} does not match the gradient's {gf.numel()} elements")
    out = torch.empty(n, dtype=torch.float32, device=dev)
    _check_covers(encoded, n)
    labels = encoded["labels"].to(device=dev, dtype=torch.uint8).contiguous()
    signs = encoded["sign_packed"].to(device=dev, dtype=torch.uint8).contiguous()
    norms = encoded["block_norms"].to(device=dev, dtype=torch.float32).contiguous()
    amp = encoded["scales"].to(device=dev, dtype=torch.float16).contiguous()
    a = _scalar_on(alpha, dev)
    with torch.cuda.device(dev):  # a previous state, no EMA
        _lib.check(lib.tam_costate_decode(labels.data_ptr(), signs.data_ptr(), norms.data_ptr(), amp.data_ptr(),
                                          a.data_ptr(), gf.data_ptr(), _lib.DTYPES[gf.dtype], n, 1, 0, 0.0, 1.0,
                                          out.data_ptr(), _lib.stream_of(dev)), "tam_costate_decode")
    return out.reshape(g.shape)


class CoStateManager:
    """Per-tensor CoState state (same attributes as the reference, costate.py:332-365).

    TurboAdam keeps one per CoState parameter and updates it inside the fused
    step; update() runs the reference's per-tensor procedure on its own.
    """

    def __init__(self, block_size: int = BLOCK_SIZE, error_feedback: bool = False, null_pct: float = 0.10,
                 amp_pct: float = 0.90) -> None:
        self.block_size = block_size
        self._null_pct = null_pct
        self._amp_pct = amp_pct
        self._has_state = False
        self._alpha = 0.0
        self._encoded = None
        self._original_numel = 0
        self._error_feedback = error_feedback
        self._ef_residual = None

    def allocate(self, numel: int, device: torch.device) -> None:
        """Create the persistent device buffers (the reference clones them on its first update, :441-451)."""
        nb = num_blocks(numel, self.block_size)
        self._alpha = torch.zeros((), dtype=torch.float32, device=device)
        self._encoded = {
            "labels": torch.zeros(nb, dtype=torch.uint8, device=device),
            "sign_packed": torch.zeros((numel + 7) // 8, dtype=torch.uint8, device=device),
            "block_norms": torch.zeros(nb, dtype=torch.float32, device=device),
            "scales": torch.zeros(nb, dtype=torch.float16, device=device),
        }

    def ranks(self, nb: int):
        """Sorted positions of the two thresholds (costate.py:115-117)."""
        return threshold_ranks(nb, self._null_pct, self._amp_pct)

    def update(self, g: torch.Tensor, beta1: float) -> torch.Tensor:
        """One CoState step for gradient g (reference costate.py:367-464): decode
        the previous state (or zeros), m = beta1*m_hat + (1-beta1)*g, then
        decompose, ratios, thresholds, labels and encode into the persistent
        buffers, in the optimizer step's launches.  With error feedback
        (:409-437) the EMA takes g + residual and the residual then takes the
        encoding loss delta - decode(new, alpha=0) (its EMA after the first
        step).  Returns m (fp32, shape of g)."""
        _require_gpu(g, "CoStateManager.update")
        _require_block_size(self.block_size)
        n = g.numel()
        dev = g.device
        if self._encoded is None or self._encoded["labels"].device != dev:
            self.allocate(n, dev)
        lib = _lib.load()
        gf = g.reshape(-1)
        if gf.dtype not in _lib.DTYPES:
            gf = gf.float()
        gf = gf.contiguous()
        nb = num_blocks(n)
        if self._has_state:
            _check_covers(self._encoded, n)
        # the arrays the kernels update in place; a copy where one is not in
        # their form, written back after
        held = {k: _in_form(self._encoded[k], dt, dev) for k, dt in _ENCODED_DTYPES.items()}
        sizes = {"labels": nb, "sign_packed": (n + 7) // 8, "block_norms": nb, "scales": nb}
        if any(held[k].numel() != c for k, c in sizes.items()):
            raise RuntimeError(f"CoStateManager.update: the state arrays do not match {n} elements ({nb} blocks)")
        alpha = _scalar_on(self._alpha, dev)
        res = None
        if self._error_feedback:  # a new tensor each update, as the reference rebinds it
            old = self._ef_residual
            if old is None:
                res = torch.empty(n, dtype=torch.float32, device=dev)
            else:
                if old.numel() != n or old.device != dev:
                    raise RuntimeError("CoStateManager.update: the residual does not match the gradient")
                res = old.detach().reshape(-1).to(torch.float32, copy=True).contiguous()
        m = torch.empty(n, dtype=torch.float32, device=dev)
        ws = torch.empty(lib.tam_costate_update_workspace(n, int(res is not None)), dtype=torch.uint8, device=dev)
        k_lo, k_hi = self.ranks(nb)
        b1, ob1 = ctypes.c_float(beta1).value, ctypes.c_float(1.0 - beta1).value
        with torch.cuda.device(dev):
            _lib.check(lib.tam_costate_update(
                gf.data_ptr(), _lib.DTYPES[gf.dtype], n, held["labels"].data_ptr(), held["sign_packed"].data_ptr(),
                held["block_norms"].data_ptr(), held["scales"].data_ptr(), alpha.data_ptr(), int(self._has_state), b1,
                ob1, k_lo, k_hi, 0 if res is None else res.data_ptr(), int(self._ef_residual is not None),
                m.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(dev)), "tam_costate_update")
        for k, t in held.items():
            if t is not self._encoded[k]:
                self._encoded[k].copy_(t.reshape(self._encoded[k].shape))
        if not isinstance(self._alpha, torch.Tensor):
            self._alpha = alpha.reshape(())
        elif alpha.data_ptr() != self._alpha.data_ptr():
            self._alpha.copy_(alpha.reshape(self._alpha.shape))
        if res is not None:
            self._ef_residual = res.reshape(g.shape)
        self._original_numel = n
        self._has_state = True
        return m.reshape(g.shape)
