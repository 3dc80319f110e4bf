"""Source-weight gradients of the Abbe image, for source-mask optimisation.

The Abbe image (CalculateAerialImage.py:46-92) is an explicit function of
the lit source points' weights V:

    I(x) = (n / W) sum_s V_s J_s(x),   W = sum_s V_s,
    J_s  = sum_c sum_e |E_sce|^2  (unit-weight coherent field of point s),

so for a loss with image cotangent g,

    dL/dV_s = (n / W) <g, J_s> - <g, I> / W.

<g, J_s> is taken on a coarse grid: J_s is a trigonometric polynomial whose
band |q| <= B is one shifted pupil wide, so with gamma = the band of g
resampled to an L x L grid (L > 2B, L holding the spectrum window),

    <g, J_s>_(N grid) = (N^2 / L^2) sum_t gamma(t) J_s^L(t)

exactly.  All J_s^L come from one oi_coherent_image call on a direct L x L
plan with the roles of spectrum and kernels exchanged: the unit-weight
shifted pupils of the points are the "spectra" of a batch of Nsrc images with
one channel per polarisation component, and the field's windowed spectrum
(one kernel per field channel) is the "kernel set".  gamma and the sums against
it are float64 products and reductions on the device (oi_source_gradient).

``AbbeSourceImage`` wraps this as a torch.autograd.Function of V;
``abbe_source_problem`` sets up a fixed field and optics.  The reference has
no source gradient (it would differentiate its complex64 loop with torch
autograd); the float64 gradient of the oracle's I(V) pins this one.
"""
from __future__ import annotations

import torch

from . import _native as nat
from . import engine, optics
from .Scatter import _pitches

__all__ = ["AbbeSourceProblem", "AbbeSourceImage", "abbe_source_problem", "abbe_image_weighted"]


def _smooth_at_least(n: int) -> int:
    """Smallest 2,3,5-smooth even integer >= n."""
    m = max(2, n)
    while True:
        k = m
        for p in (2, 3, 5):
            while k % p == 0:
                k //= p
        if k == 1 and m % 2 == 0:
            return m
        m += 1


# image lengths with register transforms (csrc/oi_fastpath.hip)
_REGISTER_LENGTHS = {128, 256, 512, 1024, 2048}


def _coarse(need: int, n: int) -> int:
    """The library's coarse size for a band: the smallest 2,3,5-smooth multiple
    of 8 that is >= need, n when that reaches n."""
    m = _smooth_at_least(max(need, 8))
    while m % 8 and m < n:
        m = _smooth_at_least(m + 1)
    return min(m, n)


def _resampling(n: int, L: int, B: int, dev) -> torch.Tensor | None:
    """Kt[y][t] = (1/n) sum_{|q| <= B} cos(2 pi q (t/L - y/n)): the band |q| <= B
    of n samples on L points, or None where the axis keeps its points."""
    if n == L:
        return None
    Kt = torch.empty((n, L), dtype=torch.float64, device=dev)
    nat.check(nat.load().oi_source_resampling(n, L, B, nat.ptr(Kt), nat.stream()))
    return Kt


class AbbeSourceProblem:
    """A field and optics held fixed, the source weights V free.

    Positions, polarisation and the lit set come from ``source`` (the
    reference's Calc_SourceSimple selection); ``V0`` holds its weights."""

    def __init__(self, field, source, scatter, projector, numerics):
        self.vector = optics.imaging_mode(numerics)
        self.dev = nat.device()
        h = torch.as_tensor(field)
        self.ny, self.nx = int(h.shape[0]), int(h.shape[1])
        px, py = _pitches(scatter, projector, source)
        self.src = optics.source_set(source)
        self.V0 = self.src.V.clone()
        self.n_index = float(projector.IndexImage)
        self.ncomp = 3 if self.vector else 1
        k0r, wr, k0c, wc, br, bc = optics.abbe_window(self.src, py, px, self.ny, self.nx)
        self.win = (k0r, wr, k0c, wc)
        self.band = (br, bc)
        tens, kind, cin, live = engine.field_encoding(h)
        self.C = len(live)
        nsrc = self.src.n
        # The float64 gradient takes <g, I> from this float32 image: image lengths
        # without register transforms keep the general kernels (a coarse grid of
        # the caller's choice) and with them the rounding of that term.  Past a
        # coarse grid of 128 the sum always was the two-pass one.
        lr = lc = 0
        if 2 * max(br, bc) - 1 <= 128 and not {self.ny, self.nx} <= _REGISTER_LENGTHS:
            lr, lc = _coarse(2 * br - 1, self.ny), _coarse(2 * bc - 1, self.nx)
        self.plan = engine.Plan(self.ny, self.nx, k0r, wr, k0c, wc, nchan=self.C, max_batch=1,
                                band_r=br, band_c=bc, lr=lr, lc=lc, max_kernels=self.ncomp * nsrc)
        lib = nat.load()
        self.spec = torch.empty((1, self.C, wr, wc), dtype=torch.complex64, device=self.dev)
        cptr, keep = nat.int_array(live)
        nat.check(lib.oi_spectrum_window(self.plan.handle, nat.ptr(tens), kind, cin, cptr, 1,
                                         nat.ptr(self.spec), nat.stream()))
        del keep
        # unit-weight shifted pupils per focus, c64 [nsrc][ncomp][wr][wc]: a
        # point's components together, as point_intensities takes them
        ones = torch.ones(nsrc, dtype=torch.float64, device=self.dev)
        self.foci = optics.focus_values(projector)
        self.G = []
        for z in self.foci:
            opt = optics.optics_record(source, projector, z, py, px, self.vector)
            G = optics.pupil_kernels(self.src, opt, ones, k0r, wr, k0c, wc)
            self.G.append(G.permute(1, 0, 2, 3).contiguous())
        # coarse grid of the per-point intensities: holds the window and
        # twice a pupil's band
        need = max(2 * max(br, bc) - 1, 2 * max(-k0r, k0r + wr - 1, -k0c, k0c + wc - 1) + 2)
        L = _smooth_at_least(need)
        self.Lr = self.ny if L >= self.ny else L
        self.Lc = self.nx if L >= self.nx else L
        self.cplan = engine.Plan(self.Lr, self.Lc, k0r, wr, k0c, wc, nchan=self.ncomp, max_batch=nsrc,
                                 band_r=wr, band_c=wc, lr=self.Lr, lc=self.Lc, max_kernels=self.C)
        if not self.cplan.geo.direct:
            raise RuntimeError("per-point intensity plan is not direct")
        self.Kr = _resampling(self.ny, self.Lr, br - 1, self.dev)
        self.Kc = _resampling(self.nx, self.Lc, bc - 1, self.dev)

    @property
    def nsrc(self) -> int:
        return self.src.n

    def image(self, V: torch.Tensor) -> torch.Tensor:
        """Abbe intensities (nFocus, ny, nx) float32 for weights V (nsrc,)."""
        V = self._weights(V)
        lib = nat.load()
        out = torch.empty((len(self.foci), self.ny, self.nx), dtype=torch.float32, device=self.dev)
        for i, G in enumerate(self.G):
            K = torch.empty_like(G)                           # [ncomp][nsrc][wr][wc]
            nat.check(lib.oi_source_kernels(nat.ptr(G), nat.ptr(V), self.nsrc, self.ncomp,
                                            G.shape[2], G.shape[3], self.n_index, nat.ptr(K),
                                            nat.stream()))
            nat.check(lib.oi_coherent_image(self.plan.handle, nat.ptr(self.spec), 1, nat.ptr(K),
                                            K.shape[0] * K.shape[1], nat.ptr(out[i]), nat.stream()))
        return out

    def _weights(self, V: torch.Tensor) -> torch.Tensor:
        V = V.detach().to(self.dev, torch.float64).contiguous()
        if V.shape != (self.nsrc,):
            raise ValueError(f"V must hold {self.nsrc} source weights")
        return V

    def point_intensities(self, focus_index: int) -> torch.Tensor:
        """J_s on the coarse Lr x Lc grid, float32 (nsrc, Lr, Lc)."""
        out = torch.empty((self.nsrc, self.Lr, self.Lc), dtype=torch.float32, device=self.dev)
        nat.check(nat.load().oi_coherent_image(self.cplan.handle, nat.ptr(self.G[focus_index]),
                                               self.nsrc, nat.ptr(self.spec), self.C, nat.ptr(out),
                                               nat.stream()))
        return out

    def source_gradient(self, V: torch.Tensor, grad_image: torch.Tensor) -> torch.Tensor:
        """dL/dV (float64, nsrc) for image cotangents grad_image (nFocus, ny, nx);
        those past the problem's foci are not read.  Weights that sum to zero
        raise ZeroDivisionError, except while the stream is captured."""
        V = self._weights(V)
        g = grad_image.detach().to(self.dev, torch.float32).contiguous()
        if g.dim() != 3 or len(g) < len(self.foci) or g.shape[1:] != (self.ny, self.nx):
            raise ValueError("grad_image must have the image's shape")
        # The read costs 20 us of a call of 100 (one focus of 128 x 128, 120 points); a
        # pinned copy read behind the launches costs as much.
        if self.foci and not torch.cuda.is_current_stream_capturing() and float(V.sum()) == 0.0:
            raise ZeroDivisionError("the source weights sum to zero")
        img = self.image(V)
        lib = nat.load()
        # the first focus writes it; the sum over an empty focus range is zero
        out = (torch.empty if self.foci else torch.zeros)(self.nsrc, dtype=torch.float64, device=self.dev)
        work = torch.empty(int(lib.oi_source_gradient_work_bytes(self.nx, self.Lr, self.Lc)),
                           dtype=torch.uint8, device=self.dev)
        for i in range(len(self.foci)):
            J = self.point_intensities(i)
            nat.check(lib.oi_source_gradient(nat.ptr(g[i]), nat.ptr(img[i]), self.ny, self.nx,
                                             nat.ptr(self.Kr), self.Lr, nat.ptr(self.Kc), self.Lc,
                                             nat.ptr(J), self.nsrc, nat.ptr(V), self.n_index,
                                             int(i > 0), nat.ptr(work), nat.ptr(out), nat.stream()))
        return out


class AbbeSourceImage(torch.autograd.Function):
    """I(V) of an AbbeSourceProblem; backward = source_gradient."""

    @staticmethod
    def forward(ctx, V: torch.Tensor, problem: AbbeSourceProblem) -> torch.Tensor:
        ctx.problem = problem
        ctx.save_for_backward(V)
        return problem.image(V)

    @staticmethod
    def backward(ctx, grad_out: torch.Tensor):
        (V,) = ctx.saved_tensors
        g = ctx.problem.source_gradient(V, grad_out)
        return g.to(device=V.device, dtype=V.dtype), None


def abbe_source_problem(field, source, scatter, projector, numerics) -> AbbeSourceProblem:
    return AbbeSourceProblem(field, source, scatter, projector, numerics)


def abbe_image_weighted(V: torch.Tensor, problem: AbbeSourceProblem) -> torch.Tensor:
    """Differentiable Abbe intensities (nFocus, ny, nx) as a function of the
    source weights V (nsrc,)."""
    if V.dim() != 1 or V.numel() != problem.nsrc:
        raise ValueError(f"V must hold {problem.nsrc} source weights")
    return AbbeSourceImage.apply(V, problem)
