// Transforms of any length: C2C, R2C and C2R lines whose length has a prime factor above 13
// (or needs more radix passes than a schedule holds), and real transforms of odd length.
// cuFFT and FFTW, the executors this library stands in for, accept every length
// (src/interfaces/fft/cufft/dtfft_executor_cufft_m.F90:77-93), and so must this one.
//
// A line of logical length n is carried through an M-point Stockham transform held in LDS
// (the passes of fft_tile in device/fft.hip):
//   CHIRP = false, M = n: the plain transform; real transforms of odd length take this
//     form, since the half-length complex trick of fft_r2c_kernel needs n even.
//   CHIRP = true, M >= 2n - 1 (Bluestein's chirp z-transform).  With jk = (j^2 + k^2 -
//     (k - j)^2) / 2 and the chirp c_j = exp(-i pi j^2 / n),
//       X_k = c_k sum_j (x_j c_j) conj(c_{k-j}),
//     a linear convolution that a cyclic one of length M >= 2n - 1 holds exactly:
//       X_k = c_k IDFT_M(DFT_M(a) DFT_M(b))_k,  a_j = x_j c_j (j < n, else 0),
//       b_j = conj(c_j) for j < n, b_{M-j} = conj(c_j) for 0 < j < n, else 0.
// KIND 0: C2C, complex in and out; the backward sign conjugates on load and store.
// KIND 1: R2C, n reals in, n/2 + 1 complex out (forward).
// KIND 2: C2R, n/2 + 1 complex in, n reals out (backward, FFTW c2r semantics: the input is
//         extended to the Hermitian spectrum X_{n-k} = conj X_k, Im X_0 and, for even n,
//         Im X_{n/2} do not contribute).
// Lines are addressed as in fft_tile, (l, b) with line start l * ls + b * bs, element
// stride ns, in units of the element type of each side (reals for the real side).
// A block's last read of global memory precedes its first write (a barrier between), so in
// place is safe.
// bh = DFT_M(b) / M is a table made once per (n, M); the inverse transform is
// conj(DFT_M(conj(.))), so both transforms run forward passes.  The second one runs the radices
// in reverse: the last pass of the first transform (radix R, span M / R) leaves elements
// b + s M / R in the registers of butterfly b, and the first pass of the second reads the same
// ones, so product and both butterflies take one trip through LDS.  The first pass reads global
// memory (its elements past n are zeros), the last one writes it: M = R0 R1 costs two LDS
// exchanges, M = R0 R1 R2 four.
#include "fft.hip"


// S: the schedule of M; SR: its radices in reverse (CHIRP only, with the table twr).
// IN_COLS / OUT_COLS: lines adjacent in memory on that side, so threads run across lines.
template <typename T, class S, class SR, int TPL, int LPB, int PAD, int KIND, bool CHIRP, bool IN_COLS, bool OUT_COLS>
__global__ void __launch_bounds__(TPL * LPB)
fft_any_kernel(const void* __restrict__ in_, void* __restrict__ out_,
               const typename tw_of<T>::type* __restrict__ tw_,
               const typename tw_of<T>::type* __restrict__ twr_,
               const typename tw_of<T>::type* __restrict__ chirp_,
               const typename tw_of<T>::type* __restrict__ bh_, dtfft::lines_desc d, int inv, int n) {
    typedef dtfft::line_passes<T, S, TPL, LPB> F;
    typedef dtfft::line_passes<T, SR, TPL, LPB> B;
    constexpr int NP = S::NP, LD = S::N + PAD;
    __shared__ cx<T> lds[LPB * LD];
    const bool iv = KIND == 2 ? true : (KIND == 1 ? false : inv != 0);
    const int nout = KIND == 1 ? n / 2 + 1 : n;
    for (i64 t = blockIdx.x; t < d.ntiles; t += gridDim.x) {
        const i64 l0 = t % d.ntl * LPB, bt = t / d.ntl;
        const i64 ibase = l0 * d.in_ls + bt * d.in_bs, obase = l0 * d.out_ls + bt * d.out_bs;
        const int lines = (int)(d.nl - l0 < LPB ? d.nl - l0 : LPB);
        const auto* tw = fresh(tw_);
        const auto* twr = fresh(twr_);
        const auto* chirp = fresh(chirp_);
        const auto* bh = fresh(bh_);
        auto gload = [&](int line, int m) {
            cx<T> v = mk((T)0, (T)0);
            if (m < n && line < lines) {
                const i64 lb = ibase + (i64)line * d.in_ls;
                if constexpr (KIND == 0) {
                    v = ((const cx<T>*)in_)[lb + (i64)m * d.in_ns];
                    if (iv) v = conj(v);
                } else if constexpr (KIND == 1) {
                    v = mk(((const T*)in_)[lb + (i64)m * d.in_ns], (T)0);
                } else {
                    const cx<T>* in = (const cx<T>*)in_;
                    if (m <= n / 2) v = in[lb + (i64)m * d.in_ns];
                    else v = conj(in[lb + (i64)(n - m) * d.in_ns]);
                    if (m == 0 || 2 * m == n) v.y = (T)0;
                    v = conj(v);  // backward = conj(forward(conj))
                }
                if constexpr (CHIRP) v = twmul(v, chirp[m]);
            }
            return v;
        };
        auto gstore = [&](int line, int k, cx<T> y) {
            if (k < nout && line < lines) {
                if constexpr (CHIRP) y = twmul(conj(y), chirp[k]);
                const i64 o = obase + (i64)line * d.out_ls + (i64)k * d.out_ns;
                if constexpr (KIND == 0) ((cx<T>*)out_)[o] = iv ? conj(y) : y;
                else if constexpr (KIND == 1) ((cx<T>*)out_)[o] = y;
                else ((T*)out_)[o] = y.x;  // real part; the conjugation leaves it unchanged
            }
        };
        auto sload = [&](int line, int m) { return lds[line * LD + m]; };
        auto sstore = [&](int line, int m, cx<T> y) { lds[line * LD + m] = y; };
        if constexpr (NP == 0) {  // one point
            for (int line = threadIdx.x; line < LPB; line += F::NT) gstore(line, 0, gload(line, 0));
        } else if constexpr (NP == 1) {  // direct only: a whole line in the registers of a thread
            F::template run<0, IN_COLS, true>(tw, gload, gstore);
        } else {
            F::template run<0, IN_COLS, false>(tw, gload, sstore);
            __syncthreads();
            F::template inner<1, NP - 1, LD>(tw, lds);
            if constexpr (CHIRP) {
                F::template turn<LD>(tw, bh, lds);
                __syncthreads();
                B::template inner<1, NP - 1, LD>(twr, lds);
                B::template run<NP - 1, OUT_COLS, false>(twr, sload, gstore);
            } else {
                F::template run<NP - 1, OUT_COLS, false>(tw, sload, gstore);
            }
        }
        __syncthreads();
    }
}

// Chirp c_j = exp(-i pi j^2 / n), j < n, with j^2 reduced mod 2n in integers so that the
// FP64 angle stays exact for every j.
__device__ __forceinline__ void store_tw(twf* t, i64 i, double c, double s) {
    twf w;
    w.rh = (float)c; w.rl = (float)(c - (double)w.rh);
    w.ih = (float)s; w.il = (float)(s - (double)w.ih);
    t[i] = w;
}
__device__ __forceinline__ void store_tw(cx<double>* t, i64 i, double c, double s) { t[i] = mk(c, s); }

template <typename T>
__global__ void gen_chirp(typename tw_of<T>::type* out, int n) {
    const i64 j = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const i64 r = (j * j) % (2 * (i64)n);
    double s, c;
    sincospi(-(double)r / (double)n, &s, &c);
    store_tw(out, j, c, s);
}

// bh_k = DFT_M(b)_k / M = (1 + 2 sum_{j=1}^{n-1} cos(2 pi j k / M) exp(i pi j^2 / n)) / M:
// the two halves of b pair up as exp(-2 pi i j k / M) + exp(+2 pi i j k / M).  One block per
// k, FP64 sums over j reduced through LDS; j k and j^2 are reduced in integers.
template <typename T>
__global__ void __launch_bounds__(256) gen_bluestein_bh(typename tw_of<T>::type* out, int n, int M) {
    const i64 k = blockIdx.x;
    double sr = 0.0, si = 0.0;
    for (i64 j = 1 + threadIdx.x; j < n; j += blockDim.x) {
        const i64 a = (j * k) % (i64)M;
        const i64 r = (j * j) % (2 * (i64)n);
        const double cw = cospi(2.0 * (double)a / (double)M);
        double s, c;
        sincospi((double)r / (double)n, &s, &c);
        sr += cw * c;
        si += cw * s;
    }
    __shared__ double red[2][256];
    red[0][threadIdx.x] = sr;
    red[1][threadIdx.x] = si;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            red[0][threadIdx.x] += red[0][threadIdx.x + w];
            red[1][threadIdx.x] += red[1][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) store_tw(out, k, (1.0 + 2.0 * red[0][0]) / (double)M, 2.0 * red[1][0] / (double)M);
}
