// The reference preparation's 3D transforms with their padding, shifting,
// cropping and normalisation inside (fp32, boxes of even edge N <= 2048 whose
// only prime factors are 2, 3, 5 and 7; the others take hipFFT, tp_fourier.hip):
//
//   fused_to_fourier    spectrum = rfftn(fftshift(zero-pad(x)), norm="forward")
//   fused_from_fourier  x = crop(ifftshift(irfftn(v, norm="forward"))), v the
//                       spectrum, or data / (weights + reg) where that sum is
//                       positive and 0 elsewhere
//
// (the steps that the reference's helpers take one by one,
// tests/test_utils.py:174-293, README.md:106-143.)
//
// A transform along one axis is one kernel, and HBM bounds it.  A padded box
// of oversampling 2 is seven eighths zeros, and of the inverse only an eighth
// is kept, so each axis is transformed only where it can be non-zero (or is
// wanted): 256^3 -> 512^3 reads and writes 1.42 GB in three passes, where the
// pad, three rocFFT passes over the whole box and its layout took 3.5 GB; the
// way back 1.69 GB, with the normalisation in its first pass.  Measured at
// 256^3 <-> 512^3: to_fourier 1.57 -> 0.44 ms, reconstruct 1.78 -> 0.54 ms
// (about 3.2 TB/s; the rest is the barriers between a workgroup's passes).
//
// A workgroup transforms W lines at once in LDS: W neighbouring columns of a
// strided axis (64- or 128-byte rows in memory; workgroups next to each other
// in x run on one XCD, whose L2 joins the rows' shared cache lines), or W pairs
// of rows of the real axis (two real rows of one box make one complex line, and
// their spectra separate by Hermitian symmetry; the last row of a box of odd
// edge has a zero partner, never a row of the next box, whose NaNs or scale it
// would take on).  Lines stand in LDS as [N][W + 1]
// (the odd stride keeps both access orders free of bank conflicts) and go
// through Stockham passes of radix 8, 4, 2, 7, 5 and 3: a thread holds its
// butterflies' inputs (at most 14 values) in registers between two barriers,
// so one buffer does.  Twiddles come from a table exp(-2 pi i k / N) that a
// kernel fills in the call's workspace from double-precision sincospi: about
// 2e-7 from the exact transform, as rocFFT.
#include "tp_device.hh"
#include "tp_launch.hh"

namespace tp {

namespace {

constexpr int kFftThreads = 1024; // most lanes of a workgroup
constexpr int kFftPer = 8;        // line elements per lane
constexpr int kFftMaxN = 2048;
constexpr int kFftXcds = 8;

struct FftPlan {
    int N, nf;
    int f[12];          // radix of each pass
    unsigned magic[12];  // ceil(2^32 / Ns) of each pass: j / Ns = umulhi(j, magic) for j < 2^16 (Ns > 1)
    int W, T;           // lines and lanes per workgroup
    bool p2;            // N is a power of two
};

void set_width(FftPlan& p, int W) {
    p.W = W;
    p.T = ((p.N * W + kFftPer - 1) / kFftPer + 63) / 64 * 64;
}
// The plan of an axis of N points, false when it is not covered.
bool plan_axis(int64_t N, FftPlan& p) {
    if (N < 2 || N > kFftMaxN || N % 2) return false;
    p.N = int(N);
    p.nf = 0;
    int64_t m = N, ns = 1;
    for (int r : {8, 4, 2, 7, 5, 3})
        while (m % r == 0) {
            p.f[p.nf] = r;
            p.magic[p.nf] = ns > 1 ? unsigned(((int64_t(1) << 32) + ns - 1) / ns) : 0u;
            ++p.nf;
            ns *= r;
            m /= r;
        }
    if (m != 1) return false;
    p.p2 = (N & (N - 1)) == 0;
    // to_fourier and reconstruct together: 512^3 919 us with 8 lines, 1012 with 16; 1024^3 8.96 ms with 8
    // lines, 9.76 with 4; 640^3 3.22 and 3.50 (25.3 and 6.48 by way of hipFFT)
    set_width(p, N <= 256 ? 16 : (N <= 1024 ? 8 : 4));  // W * N <= kFftThreads * kFftPer
    return true;
}
// The plan for `lines` lines: narrower workgroups while there are too few of them to fill the GPU (the
// rows of a box of 84, padded, are 110 workgroups of 16 pairs).
FftPlan for_lines(FftPlan p, int64_t lines) {
    while (p.W > 4 && lines / p.W < 1024) set_width(p, p.W / 2);
    return p;
}

__global__ __launch_bounds__(kBlock) void k_twiddles(int N, Cx<float>* __restrict__ tw) {
    const int k = int(blockIdx.x) * kBlock + int(threadIdx.x);
    if (k >= N) return;
    double s, c;
    sincospi(-2.0 * double(k) / double(N), &s, &c);
    tw[k] = Cx<float>{float(c), float(s)};
}

// i * v for the forward sign of the transform, -i * v for the inverse one: v * exp(-+ pi i / 2)
template <bool INV> __device__ __forceinline__ Cx<float> turn(Cx<float> v) {
    return INV ? Cx<float>{-v.im, v.re} : Cx<float>{v.im, -v.re};
}
template <bool INV> __device__ __forceinline__ void dft2(Cx<float>* v) {
    const Cx<float> a = v[0];
    v[0] = cadd(a, v[1]);
    v[1] = csub(a, v[1]);
}
template <bool INV> __device__ __forceinline__ void dft4(Cx<float>* v) {
    const Cx<float> a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]), d = turn<INV>(csub(v[1], v[3]));
    v[0] = cadd(a, c);
    v[1] = cadd(b, d);
    v[2] = csub(a, c);
    v[3] = csub(b, d);
}
template <bool INV> __device__ __forceinline__ void dft8(Cx<float>* v) {
    Cx<float> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft4<INV>(e);
    dft4<INV>(o);
    constexpr float h = 0.70710678118654752440f;
    // o[k] * exp(-+ 2 pi i k / 8)
    const Cx<float> t1 = turn<INV>(o[1]), t3 = turn<INV>(o[3]);
    o[1] = cscale(cadd(o[1], t1), h);
    o[2] = turn<INV>(o[2]);
    o[3] = cscale(csub(t3, o[3]), h);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = cadd(e[k], o[k]);
        v[k + 4] = csub(e[k], o[k]);
    }
}
// Odd radix R: with s_q = v_q + v_(R-q) and d_q = v_q - v_(R-q), output k (and R - k) is
// v_0 + sum_q s_q cos(2 pi q k / R) -+ i sum_q d_q sin(2 pi q k / R).
template <int R> struct OddRoots;
template <> struct OddRoots<3> {
    static constexpr float c[2] = {1.f, -0.5f}, s[2] = {0.f, 0.86602540378443864676f};
};
template <> struct OddRoots<5> {
    static constexpr float c[3] = {1.f, 0.30901699437494742410f, -0.80901699437494742410f},
                           s[3] = {0.f, 0.95105651629515357212f, 0.58778525229247312917f};
};
template <> struct OddRoots<7> {
    static constexpr float c[4] = {1.f, 0.62348980185873353053f, -0.22252093395631440429f, -0.90096886790241912624f},
                           s[4] = {0.f, 0.78183148246802980871f, 0.97492791218182360702f, 0.43388373911755812048f};
};
template <int R, bool INV> __device__ __forceinline__ void dft_odd(Cx<float>* v) {
    constexpr int M = R / 2;
    Cx<float> s[M + 1], d[M + 1];
    const Cx<float> v0 = v[0];
    Cx<float> sum = v0;
#pragma unroll
    for (int q = 1; q <= M; ++q) {
        s[q] = cadd(v[q], v[R - q]);
        d[q] = csub(v[q], v[R - q]);
        sum = cadd(sum, s[q]);
    }
    v[0] = sum;
#pragma unroll
    for (int k = 1; k <= M; ++k) {
        Cx<float> a = v0, b = {0.f, 0.f};
#pragma unroll
        for (int q = 1; q <= M; ++q) {
            const int t = q * k % R, u = t <= M ? t : R - t;
            const float sn = t <= M ? OddRoots<R>::s[u] : -OddRoots<R>::s[u];
            a = cfma(s[q], OddRoots<R>::c[u], a);
            b = cfma(d[q], sn, b);
        }
        const Cx<float> tb = turn<INV>(b);
        v[k] = cadd(a, tb);
        v[R - k] = csub(a, tb);
    }
}
template <int R, bool INV> __device__ __forceinline__ void dft(Cx<float>* v) {
    if constexpr (R == 2) dft2<INV>(v);
    else if constexpr (R == 4) dft4<INV>(v);
    else if constexpr (R == 8) dft8<INV>(v);
    else dft_odd<R, INV>(v);
}

// What a pass loads for a line element, and the element.
struct FftWeighted {
    Cx<float> v;
    float d;
};
struct FftPadded {
    Cx<float> v;
    bool in;
};
__device__ __forceinline__ Cx<float> line_value(Cx<float> v) { return v; }
__device__ __forceinline__ Cx<float> line_value(FftWeighted x) {
    const Cx<float> q = {x.v.re / x.d, x.v.im / x.d};
    return x.d > 0.f ? q : Cx<float>{0.f, 0.f};
}
__device__ __forceinline__ Cx<float> line_value(FftPadded x) { return x.in ? x.v : Cx<float>{0.f, 0.f}; }

// One Stockham pass of radix R over the W lines: element i of line w comes from ld(i, w) and goes to
// st(i, w, value).  `mid`: both are the same LDS lines, so the lanes wait for one another in between.
template <int R, bool INV, typename LD, typename ST>
__device__ __forceinline__ void fft_pass(LD&& ld, ST&& st, bool mid, const Cx<float>* tw, const FftPlan& p, int Ns,
                                         unsigned magic) {
    constexpr int NB = (kFftPer + R - 1) / R;  // butterflies per lane: T * kFftPer >= N * W
    const int n = p.N / R, nb = n * p.W, lw = 31 - __clz(p.W), step = n / Ns;
    Cx<float> v[NB][R];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int b = int(threadIdx.x) + i * p.T;
        if (b >= nb) continue;
        const int w = b & (p.W - 1), j = b >> lw;
        decltype(ld(0, 0)) in[R];  // (all of them under way before the first is used)
#pragma unroll
        for (int q = 0; q < R; ++q) in[q] = ld(j + q * n, w);
#pragma unroll
        for (int q = 0; q < R; ++q) v[i][q] = line_value(in[q]);
        if (Ns > 1) {
            const int k = j - int(__umulhi(unsigned(j), magic)) * Ns;
#pragma unroll
            for (int q = 1; q < R; ++q) {
                Cx<float> t = tw[k * q * step];
                if (INV) t.im = -t.im;
                v[i][q] = Cx<float>{fmaf(v[i][q].re, t.re, -(v[i][q].im * t.im)), fmaf(v[i][q].re, t.im, v[i][q].im * t.re)};
            }
        }
    }
    if (mid) __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int b = int(threadIdx.x) + i * p.T;
        if (b >= nb) continue;
        const int w = b & (p.W - 1), j = b >> lw, g = Ns > 1 ? int(__umulhi(unsigned(j), magic)) : j;
        dft<R, INV>(v[i]);
#pragma unroll
        for (int q = 0; q < R; ++q) st(g * Ns * R + (j - g * Ns) + q * Ns, w, v[i][q]);
    }
}
// Pass number i with radix p.f[i].  P2: N is a power of two (without the odd radices' code the kernels
// take half the registers, so two or more workgroups of N = 512 share a CU and one's passes run beside
// another's loads).
template <bool INV, bool P2, typename LD, typename ST>
__device__ __forceinline__ void fft_pass_at(int i, LD&& ld, ST&& st, bool mid, const Cx<float>* tw, const FftPlan& p,
                                            int Ns) {
    const int r = p.f[i];
    const unsigned m = p.magic[i];
    if (r == 8) fft_pass<8, INV>(ld, st, mid, tw, p, Ns, m);
    else if (r == 4) fft_pass<4, INV>(ld, st, mid, tw, p, Ns, m);
    else if (r == 2) fft_pass<2, INV>(ld, st, mid, tw, p, Ns, m);
    else if (P2) return;
    else if (r == 3) fft_pass<3, INV>(ld, st, mid, tw, p, Ns, m);
    else if (r == 5) fft_pass<5, INV>(ld, st, mid, tw, p, Ns, m);
    else fft_pass<7, INV>(ld, st, mid, tw, p, Ns, m);
}
// The passes [i0, i1) within LDS (line element i of line w at buf[i * (W + 1) + w]); all lanes of the
// workgroup call it, the lines complete in LDS before and after.  Ns: product of the earlier radices.
template <bool INV, bool P2>
__device__ __forceinline__ void fft_lines(Cx<float>* buf, const Cx<float>* tw, const FftPlan& p, int i0, int i1,
                                          int& Ns) {
    const int WP = p.W + 1;
    for (int i = i0; i < i1; ++i) {
        fft_pass_at<INV, P2>(
            i, [&](int e, int w) { return buf[e * WP + w]; }, [&](int e, int w, Cx<float> x) { buf[e * WP + w] = x; },
            true, tw, p, Ns);
        __syncthreads();
        Ns *= p.f[i];
    }
}

// Work item of this workgroup, neighbouring items on one XCD (workgroups are dealt to the XCDs round-robin).
__device__ __forceinline__ int64_t xcd_block(int64_t items) {
    const int64_t per = (items + kFftXcds - 1) / kFftXcds;
    return (int64_t(blockIdx.x) % kFftXcds) * per + int64_t(blockIdx.x) / kFftXcds;
}
// (the grid is kFftXcds * per workgroups; those whose item is past the last leave at once)

// Geometry of a box: edge n of the real-space cube (offset `off`: pad_before, or crop_start) in the
// padded edge N, whose fftshift puts element s at (s + off + N / 2) mod N of an axis.
struct FftBox {
    int n, off;
};
__device__ __forceinline__ int box_to_line(const FftBox& b, int N, int s) {
    const int i = s + b.off + N / 2;
    return i >= N ? i - N : i;
}
__device__ __forceinline__ int line_to_box(const FftBox& b, int N, int i) {  // outside [0, n): padding
    const int i2 = i + N - N / 2;
    return (i2 >= N ? i2 - N : i2) - b.off;
}

// A strided axis: W columns x0 .. x0 + W - 1 of the `cols` contiguous ones of a plane or volume (the y
// axis: a row's; the z axis: a whole plane's, so that its workgroups' rows are whole aligned cache
// lines, which the rows of N / 2 + 1 values are not).  Forward: the box's n rows, padded, to all N,
// times `scale`.  Inverse: all N rows to the box's n, and with NORM each value is divided by
// weights + reg as it is read.
struct FftCols {
    int64_t items, in_outer, in_stride, out_outer, out_stride;
    int cols, tiles;
};
// Row pitch (values) of the y passes' other side, rounded up to cache lines.
int64_t pitch_of(int64_t H) { return (H + 15) / 16 * 16; }
template <bool INV, bool NORM, bool P2>
__global__ __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(P2 ? 6 : 4))) void k_fft_cols(FftPlan p, FftBox box, FftCols g,
                                                          const Cx<float>* __restrict__ in,
                                                          const float* __restrict__ weights, float reg,
                                                          const Cx<float>* __restrict__ twg,
                                                          Cx<float>* __restrict__ out, float scale) {
    extern __shared__ __align__(16) unsigned char smem[];
    Cx<float>* buf = reinterpret_cast<Cx<float>*>(smem);
    Cx<float>* tw = buf + p.N * (p.W + 1);
    const int64_t item = xcd_block(g.items);
    if (item >= g.items) return;
    const int64_t outer = item / g.tiles;
    const int x0 = int(item - outer * g.tiles) * p.W, WP = p.W + 1;
    const Cx<float>* ib = in + outer * g.in_outer + x0;
    const float* iw = NORM ? weights + outer * g.in_outer + x0 : nullptr;
    Cx<float>* ob0 = out + outer * g.out_outer + x0;
    for (int k = threadIdx.x; k < p.N; k += p.T) tw[k] = twg[k];
    // The first pass takes its inputs from memory and the last one sends its outputs there: a lane has
    // all of its loads under way at once (one after another, each waiting at its division: the
    // normalising pass of 512^3 465 instead of 355 us), and two barriers and LDS trips fall away.
    // (columns past the last and padding read some element inside instead of branching around the load)
    const int last = min(p.W, g.cols - x0) - 1;
    auto ld = [&](int i, int w) {
        const int x = min(w, last);
        if constexpr (NORM) {
            return FftWeighted{ib[i * g.in_stride + x], iw[i * g.in_stride + x] + reg};
        } else if constexpr (INV) {
            return ib[i * g.in_stride + x];
        } else {
            const int s = line_to_box(box, p.N, i);
            return FftPadded{ib[min(max(s, 0), box.n - 1) * g.in_stride + x], s >= 0 && s < box.n};
        }
    };
    auto st = [&](int i, int w, Cx<float> v) {
        if (x0 + w >= g.cols) return;
        if (INV) {
            const int j = line_to_box(box, p.N, i);
            if (j >= 0 && j < box.n) ob0[j * g.out_stride + w] = v;
        } else {
            ob0[i * g.out_stride + w] = cscale(v, scale);
        }
    };
    auto to_lds = [&](int i, int w, Cx<float> v) { buf[i * WP + w] = v; };
    auto from_lds = [&](int i, int w) { return buf[i * WP + w]; };
    if (p.nf == 1) {
        fft_pass_at<INV, P2>(0, ld, st, false, tw, p, 1);
        return;
    }
    fft_pass_at<INV, P2>(0, ld, to_lds, false, tw, p, 1);
    __syncthreads();
    int Ns = p.f[0];
    fft_lines<INV, P2>(buf, tw, p, 1, p.nf - 1, Ns);
    fft_pass_at<INV, P2>(p.nf - 1, from_lds, st, false, tw, p, Ns);
}

// The lines of the real axis: each box's `rows` rows in pairs, 2q and 2q + 1 as line q of its `pairs`.
struct FftRows {
    int lines, rows, pairs;
};
__device__ __forceinline__ void rows_of_line(const FftRows& r, int l, int64_t& ra, bool& has_a, bool& has_b) {
    const int b = l / r.pairs, q = l - b * r.pairs;
    ra = int64_t(b) * r.rows + 2 * q;
    has_a = l < r.lines;
    has_b = has_a && 2 * q + 1 < r.rows;
}
FftRows rows_in_pairs(int64_t batch, int64_t n) {
    const int64_t pairs = (n * n + 1) / 2;  // (batch * n * n stays below 2^23: fused_fft_work)
    return FftRows{int(batch * pairs), int(n * n), int(pairs)};
}

// The real axis, forward: a pair of rows of a box (n reals each) as one line; their spectra of
// H = N / 2 + 1 values to the same rows of `out` (`pitch` values apart).
template <bool P2>
__global__ __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(P2 ? 6 : 4))) void k_fft_rows_forward(FftPlan p, FftBox box, FftRows rows, int H, int64_t pitch,
                                                                  const float* __restrict__ in,
                                                                  const Cx<float>* __restrict__ twg,
                                                                  Cx<float>* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char smem[];
    Cx<float>* buf = reinterpret_cast<Cx<float>*>(smem);
    Cx<float>* tw = buf + p.N * (p.W + 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = p.T / 64, WP = p.W + 1;
    for (int k = threadIdx.x; k < p.N; k += p.T) tw[k] = twg[k];
    const int l0 = int(blockIdx.x) * p.W;
    for (int w = wave; w < p.W; w += waves) {
        int64_t ra;
        bool has_a, has_b;
        rows_of_line(rows, l0 + w, ra, has_a, has_b);
        const int64_t rb = ra + 1;
        for (int i = lane; i < p.N; i += 64) {
            const int s = line_to_box(box, p.N, i);
            const bool ok = s >= 0 && s < box.n;
            buf[i * WP + w] = Cx<float>{ok && has_a ? in[ra * box.n + s] : 0.f, ok && has_b ? in[rb * box.n + s] : 0.f};
        }
    }
    __syncthreads();
    int Ns = 1;
    fft_lines<false, P2>(buf, tw, p, 0, p.nf, Ns);
    for (int w = wave; w < p.W; w += waves) {
        int64_t ra;
        bool has_a, has_b;
        rows_of_line(rows, l0 + w, ra, has_a, has_b);
        const int64_t rb = ra + 1;
        for (int k = lane; k < H; k += 64) {
            const Cx<float> z = buf[k * WP + w], y = buf[(k == 0 ? 0 : p.N - k) * WP + w];
            if (has_a) out[ra * pitch + k] = Cx<float>{0.5f * (z.re + y.re), 0.5f * (z.im - y.im)};
            if (has_b) out[rb * pitch + k] = Cx<float>{0.5f * (z.im + y.im), 0.5f * (y.re - z.re)};
        }
    }
}

// The real axis, inverse: the half spectra of a pair of rows as one line, a + i b on the whole axis
// (their Hermitian halves filled in; the imaginary parts at k = 0 and N / 2 are ignored, as complex-to-
// real transforms do), to the box's n reals of each row.
template <bool P2>
__global__ __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(P2 ? 6 : 4))) void k_fft_rows_inverse(FftPlan p, FftBox box, FftRows rows, int H, int64_t pitch,
                                                                  const Cx<float>* __restrict__ in,
                                                                  const Cx<float>* __restrict__ twg,
                                                                  float* __restrict__ out) {
    extern __shared__ __align__(16) unsigned char smem[];
    Cx<float>* buf = reinterpret_cast<Cx<float>*>(smem);
    Cx<float>* tw = buf + p.N * (p.W + 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = p.T / 64, WP = p.W + 1;
    for (int k = threadIdx.x; k < p.N; k += p.T) tw[k] = twg[k];
    const int l0 = int(blockIdx.x) * p.W;
    for (int w = wave; w < p.W; w += waves) {
        int64_t ra;
        bool has_a, has_b;
        rows_of_line(rows, l0 + w, ra, has_a, has_b);
        const int64_t rb = ra + 1;
        for (int k = lane; k < H; k += 64) {
            Cx<float> a = {0.f, 0.f}, b = {0.f, 0.f};
            if (has_a) a = in[ra * pitch + k];
            if (has_b) b = in[rb * pitch + k];
            if (k == 0 || k == p.N / 2) a.im = b.im = 0.f;
            buf[k * WP + w] = Cx<float>{a.re - b.im, a.im + b.re};
            if (k > 0 && k < p.N / 2) buf[(p.N - k) * WP + w] = Cx<float>{a.re + b.im, b.re - a.im};
        }
    }
    __syncthreads();
    int Ns = 1;
    fft_lines<true, P2>(buf, tw, p, 0, p.nf, Ns);
    for (int w = wave; w < p.W; w += waves) {
        int64_t ra;
        bool has_a, has_b;
        rows_of_line(rows, l0 + w, ra, has_a, has_b);
        const int64_t rb = ra + 1;
        for (int j = lane; j < box.n; j += 64) {
            const Cx<float> z = buf[box_to_line(box, p.N, j) * WP + w];
            if (has_a) out[ra * box.n + j] = z.re;
            if (has_b) out[rb * box.n + j] = z.im;
        }
    }
}

size_t lds_bytes(const FftPlan& p) { return size_t(p.N) * (p.W + 2) * sizeof(Cx<float>); }
size_t aligned(size_t b) { return (b + 255) / 256 * 256; }

// Workgroups of a kernel over `items` in xcd_block's order.
unsigned xcd_grid(int64_t items) { return unsigned(kFftXcds * ((items + kFftXcds - 1) / kFftXcds)); }
constexpr int64_t kFftMaxItems = (int64_t(1) << 32) / kFftThreads - kFftXcds - 1;

template <bool INV, bool NORM>
hipError_t run_cols(const FftPlan& wide, const FftBox& box, FftCols g, int64_t outer, const void* in, const void* weights,
                    float reg, const Cx<float>* tw, void* out, float scale, hipStream_t s) {
    const FftPlan p = for_lines(wide, outer * g.cols);
    g.tiles = (g.cols + p.W - 1) / p.W;
    g.items = outer * g.tiles;
    const auto k = p.p2 ? k_fft_cols<INV, NORM, true> : k_fft_cols<INV, NORM, false>;
    hipLaunchKernelGGL(k, dim3(xcd_grid(g.items)), dim3(p.T), lds_bytes(p), s, p, box, g, (const Cx<float>*)in,
                       (const float*)weights, reg, tw, (Cx<float>*)out, scale);
    return hipGetLastError();
}

hipError_t run_twiddles(const FftPlan& p, Cx<float>* tw, hipStream_t s) {
    hipLaunchKernelGGL(k_twiddles, dim3((p.N + kBlock - 1) / kBlock), dim3(kBlock), 0, s, p.N, tw);
    return hipGetLastError();
}

}  // namespace

int64_t fused_fft_work(bool inverse, int64_t batch, int64_t n, int64_t N) {
    FftPlan p;
    if (batch < 1 || n < 1 || n > N || !plan_axis(N, p)) return 0;
    const int64_t H = N / 2 + 1, tiles = (H + 3) / 4;  // (of the narrowest workgroups)
    if (batch > kFftMaxItems / (N * tiles) || batch * n > kFftMaxItems / n) return 0;
    const size_t lines = aligned(size_t(batch) * n * N * H * 8);
    return int64_t(aligned(size_t(N) * 8) + lines + (inverse ? aligned(size_t(batch) * n * n * pitch_of(H) * 8) : 0));
}

hipError_t fused_to_fourier(int64_t batch, int64_t n, int64_t N, int64_t pad_before, const void* real, void* spectrum,
                            void* work, hipStream_t s) {
    FftPlan p;
    if (!plan_axis(N, p)) return hipErrorInvalidValue;
    const FftBox box{int(n), int(pad_before)};
    const int64_t H = N / 2 + 1;
    const FftRows rows = rows_in_pairs(batch, n);
    Cx<float>* tw = static_cast<Cx<float>*>(work);
    char* lines = static_cast<char*>(work) + aligned(size_t(N) * 8);
    hipError_t e = run_twiddles(p, tw, s);
    if (e != hipSuccess) return e;
    // the rows' spectra [batch, n, n, pitch] stand in the output's memory until the last pass overwrites it
    const int64_t pitch = n * n * pitch_of(H) <= N * N * H ? pitch_of(H) : H;
    const FftPlan pr = for_lines(p, rows.lines);
    const int64_t groups = (rows.lines + pr.W - 1) / pr.W;
    hipLaunchKernelGGL((p.p2 ? k_fft_rows_forward<true> : k_fft_rows_forward<false>), dim3(unsigned(groups)),
                       dim3(pr.T), lds_bytes(pr), s, pr, box, rows, int(H), pitch,
                       (const float*)real, tw, (Cx<float>*)spectrum);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    FftCols y{0, n * pitch, pitch, N * H, H, int(H), 0};
    e = run_cols<false, false>(p, box, y, batch * n, spectrum, nullptr, 0.f, tw, lines, 1.0f, s);
    if (e != hipSuccess) return e;
    FftCols z{0, n * N * H, N * H, N * N * H, N * H, int(N * H), 0};
    const float scale = float(1.0 / (double(N) * double(N) * double(N)));
    return run_cols<false, false>(p, box, z, batch, lines, nullptr, 0.f, tw, spectrum, scale, s);
}

hipError_t fused_from_fourier(int64_t batch, int64_t n, int64_t N, int64_t crop_start, const void* data,
                              const void* weights, double reg, void* real, void* work, hipStream_t s) {
    FftPlan p;
    if (!plan_axis(N, p)) return hipErrorInvalidValue;
    const FftBox box{int(n), int(crop_start)};
    const int64_t H = N / 2 + 1;
    const FftRows rows = rows_in_pairs(batch, n);
    Cx<float>* tw = static_cast<Cx<float>*>(work);
    char* lines = static_cast<char*>(work) + aligned(size_t(N) * 8);
    char* planes = lines + aligned(size_t(batch) * n * N * H * 8);
    hipError_t e = run_twiddles(p, tw, s);
    if (e != hipSuccess) return e;
    FftCols z{0, N * N * H, N * H, n * N * H, N * H, int(N * H), 0};
    e = weights ? run_cols<true, true>(p, box, z, batch, data, weights, float(reg), tw, lines, 1.0f, s)
                : run_cols<true, false>(p, box, z, batch, data, nullptr, 0.f, tw, lines, 1.0f, s);
    if (e != hipSuccess) return e;
    const int64_t pitch = pitch_of(H);
    FftCols y{0, N * H, H, n * pitch, pitch, int(H), 0};
    e = run_cols<true, false>(p, box, y, batch * n, lines, nullptr, 0.f, tw, planes, 1.0f, s);
    if (e != hipSuccess) return e;
    const FftPlan pr = for_lines(p, rows.lines);
    const int64_t groups = (rows.lines + pr.W - 1) / pr.W;
    hipLaunchKernelGGL((p.p2 ? k_fft_rows_inverse<true> : k_fft_rows_inverse<false>), dim3(unsigned(groups)),
                       dim3(pr.T), lds_bytes(pr), s, pr, box, rows, int(H), pitch,
                       (const Cx<float>*)planes, tw, (float*)real);
    return hipGetLastError();
}

}  // namespace tp
