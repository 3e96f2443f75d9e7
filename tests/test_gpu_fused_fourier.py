"""The fused 3D transforms of the reference preparation (to_fourier, from_fourier, reconstruct) against torch.fft
in double precision: edges whose passes mix every radix, one workgroup tile of columns and ragged ones, both
tile widths below the widest, an odd number of rows, several boxes, oversampling 1; and boxes with other prime
factors, which take the hipFFT path.  The boxes of a batch are compared with the same boxes alone.

The bar: each of the log2(N) butterfly levels of each axis rounds to 2^-24 relative, in the 2-norm about
sqrt(3 log2 N) 2^-24 with the twiddles' rounding as much again: 1e-6 is five times that at N = 2048.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 8, 8), (2, 5, 10), (3, 7, 14), (1, 16, 32), (2, 9, 18), (1, 24, 36), (1, 21, 42), (2, 30, 60), (1, 42, 84),
         (1, 31, 70), (1, 64, 128), (1, 33, 162), (1, 100, 200), (1, 128, 256), (1, 10, 500), (1, 20, 512), (1, 6, 600),
         (1, 22, 44), (1, 13, 26)]


def _rel(a, b):
    return ((a.to(b.dtype) - b).norm() / b.norm()).item()


@pytest.mark.parametrize("B,n,N", CASES, ids=[f"B{b}_n{n}_N{N}" for b, n, N in CASES])
def test_fused_transforms_match_fft64(B, n, N, gpu):
    from torch_projectors import fourier as FM
    g = torch.Generator(device="cuda").manual_seed(1000 * n + N)
    os_ = N / n
    x = torch.randn(B, n, n, n, generator=g, device="cuda")
    print(f"[fused fourier] B={B} n={n} N={N}", flush=True)
    lo = (N - n) // 2
    pad = torch.nn.functional.pad(x.double(), (lo, N - n - lo) * 3)
    exp = torch.fft.rfftn(torch.fft.fftshift(pad, dim=(1, 2, 3)), dim=(1, 2, 3), norm="forward")
    del pad
    keep = x.clone()
    if FM.capi.padded_boxsize(n, os_) == N:
        spec = FM.to_fourier(x, os_)
        assert spec.shape == exp.shape and spec.is_contiguous() and torch.equal(x, keep)
        assert _rel(spec, exp) < 1e-6
        del spec
    data = torch.randn(B, N, N, N // 2 + 1, generator=g, device="cuda", dtype=torch.complex64)
    w = torch.randn(B, N, N, N // 2 + 1, generator=g, device="cuda")
    w[..., 0] = -1.0  # weights + reg <= 0: zero
    del exp
    if FM.capi.cropped_boxsize(N, os_) != n:
        return
    at = (N - n) // 2

    def real_of(v):
        y = torch.fft.ifftshift(torch.fft.irfftn(v, s=[N] * 3, dim=(1, 2, 3), norm="forward"), dim=(1, 2, 3))
        return y[:, at:at + n, at:at + n, at:at + n].contiguous()

    kept = data.clone()
    assert _rel(FM.from_fourier(data, os_, dim=3), real_of(data.to(torch.complex128))) < 1e-6
    assert torch.equal(data, kept)
    den = (w + 0.25).double()
    v = torch.where(den > 0, data.to(torch.complex128) / den, torch.zeros((), dtype=torch.complex128, device="cuda"))
    assert _rel(FM.reconstruct(data, w, os_, reg=0.25, dim=3), real_of(v)) < 1e-6
    assert torch.equal(data, kept)


# (box edge, padded edge, oversampling of the way back): odd and even edges, whose boxes end with a row
# without and with a partner; 85 is what an oversampling of 1.5 keeps of 128
BOXES = [(9, 18, 2.0), (8, 16, 2.0), (1, 2, 2.0), (63, 126, 2.0), (85, 128, 1.5), (33, 162, 162 / 33)]


@pytest.mark.parametrize("n,N,os_", BOXES, ids=[f"n{n}_N{N}" for n, N, _ in BOXES])
def test_boxes_of_a_batch_are_independent(n, N, os_, gpu):
    """Boxes of very different scale, one with a NaN and one with an infinity: every other box must come out
    bit for bit as it does alone, and within the bar of the double-precision transform."""
    from torch_projectors import fourier as FM
    g = torch.Generator(device="cuda").manual_seed(7000 + N)
    B = 5
    scale = torch.tensor([1.0, 1e6, 1e-6, 1.0, 1.0], device="cuda").view(B, 1, 1, 1)
    print(f"[fused fourier] boxes n={n} N={N}", flush=True)

    def check(batch, run, exact, what):
        out = run(batch)
        for b in range(B):
            alone = run(batch[b:b + 1])
            if b == 3 or b == 1:
                assert not torch.isfinite(torch.view_as_real(alone) if alone.is_complex() else alone).all()
                continue
            assert torch.equal(out[b:b + 1], alone), f"{what}: box {b} differs from the same box alone"
            assert _rel(alone, exact(batch[b:b + 1])) < 1e-6, f"{what}: box {b}"

    if FM.capi.padded_boxsize(n, os_) == N:
        x = torch.randn(B, n, n, n, generator=g, device="cuda") * scale
        x[1, 0, 0, 0] = float("nan")
        x[3, -1, -1, -1] = float("inf")
        lo = (N - n) // 2

        def spec64(v):
            v = torch.nn.functional.pad(v.double(), (lo, N - n - lo) * 3)
            return torch.fft.rfftn(torch.fft.fftshift(v, dim=(1, 2, 3)), dim=(1, 2, 3), norm="forward")
        check(x, lambda v: FM.to_fourier(v, os_), spec64, "to_fourier")
    if FM.capi.cropped_boxsize(N, os_) != n:
        return
    at = (N - n) // 2

    def real64(v):
        y = torch.fft.irfftn(v.to(torch.complex128), s=[N] * 3, dim=(1, 2, 3), norm="forward")
        return torch.fft.ifftshift(y, dim=(1, 2, 3))[:, at:at + n, at:at + n, at:at + n]
    d = torch.randn(B, N, N, N // 2 + 1, generator=g, device="cuda", dtype=torch.complex64) * scale
    d[1, 0, 0, 0] = float("nan")
    d[3, -1, -1, 0] = float("inf")
    check(d, lambda v: FM.from_fourier(v, os_, dim=3), real64, "from_fourier")
    one = torch.ones(1, N, N, N // 2 + 1, device="cuda")
    check(d, lambda v: FM.reconstruct(v, one.expand(v.shape).contiguous(), os_, dim=3), real64, "reconstruct")


def test_strided_inputs_and_grad(gpu):
    from torch_projectors import fourier as FM
    x = torch.randn(12, 12, 12, device="cuda").permute(2, 0, 1)
    assert torch.equal(FM.to_fourier(x, 2.0), FM.to_fourier(x.contiguous(), 2.0))
    y = x.contiguous().requires_grad_(True)
    assert FM.to_fourier(y, 2.0).requires_grad
    d = torch.randn(24, 24, 26, device="cuda", dtype=torch.complex64)[..., ::2]
    assert torch.equal(FM.from_fourier(d, 2.0), FM.from_fourier(d.contiguous(), 2.0))
    c = torch.randn(24, 24, 13, device="cuda", dtype=torch.complex64)
    assert torch.equal(FM.from_fourier(c.conj(), 2.0), FM.from_fourier(c.conj().resolve_conj(), 2.0))


@pytest.mark.parametrize("N", [1024, 1050, 2048])
def test_long_axes_against_the_sums(N, gpu):
    """The longest lines of each workgroup width, on a box of 3: values of the spectrum, and the map of a
    spectrum with few non-zero values, against their defining sums in double precision."""
    from torch_projectors import fourier as FM
    n, os_ = 3, N / 3
    print(f"[fused fourier] n={n} N={N}", flush=True)
    g = torch.Generator().manual_seed(N)
    x = torch.randn(n, n, n, generator=g)
    H = N // 2 + 1
    k = torch.stack([torch.randint(0, m, (2000,), generator=g) for m in (N, N, H)])
    # box element s of an axis is element (s + pad + N / 2) mod N of the shifted line
    s = torch.arange(n) + (N - n) // 2 + N // 2
    ph = [torch.polar(torch.ones(2000, n, dtype=torch.float64),
                      (-2 * torch.pi / N) * ((ka[:, None] * s) % N).double()) for ka in k]
    exp = torch.einsum("ki,kj,kl,ijl->k", *ph, x.to(torch.complex128)) / float(N) ** 3
    pb = FM.capi.padded_boxsize(n, os_)
    if pb == N:
        spec = FM.to_fourier(x.cuda(), os_)
        got = spec[tuple(i.cuda() for i in k)].cpu()
        del spec
        assert _rel(got, exp) < 1e-6
    c = torch.randn(2000, generator=g, dtype=torch.complex64)
    d = torch.zeros(N, N, H, dtype=torch.complex64, device="cuda")
    k[2] = 1 + k[2] % (H - 2)  # (their mirror images are not stored)
    flat = torch.unique((k[0] * N + k[1]) * H + k[2])
    c = c[:flat.numel()]
    d.view(-1)[flat.cuda()] = c.cuda()
    n2 = FM.capi.cropped_boxsize(N, os_)
    s = torch.arange(n2) + (N - n2) // 2 + N // 2
    ks = (flat // (N * H), flat // H % N, flat % H)
    ph = [torch.polar(torch.ones(flat.numel(), n2, dtype=torch.float64),
                      (2 * torch.pi / N) * ((ka[:, None] * s) % N).double()) for ka in ks]
    ref = 2 * torch.einsum("ki,kj,kl,k->ijl", *ph, c.to(torch.complex128)).real
    assert _rel(FM.from_fourier(d, os_, dim=3).cpu(), ref) < 1e-6
