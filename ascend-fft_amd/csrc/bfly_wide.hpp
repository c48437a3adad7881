// bfly_wide.hpp -- the 32-points-per-thread Stockham core.
//
// Same passes as bfly_device.hpp with twice the points per thread and the
// exchanges between passes done one component at a time: every thread writes
// its real parts, reads back the ones the next pass needs, then does the same
// with the imaginary parts.  A transform then needs half the threads and half
// the LDS of the 16-point core (N floats instead of N complex values), so
// where a 16-point workgroup fills a CU by itself (its LDS), two or more
// 32-point ones share it and one's memory time hides behind another's passes.
// The data take 64 registers, so four waves per SIMD (128 VGPRs) leave no
// room for a prefetched transform: the overlap comes from the workgroups.
#pragma once
#include "bfly_device.hpp"

namespace bfly_dev {

constexpr int kWide = 32;  // points per thread

// Multiply by e^{DIR 2 pi i m / 32} (m a compile-time constant after unrolling).
__device__ __forceinline__ float cos32(int m) {
    switch (m & 31) {
        case 1: case 31: return 0.98078528040323044913f;
        case 3: case 29: return 0.83146961230254523708f;
        case 5: case 27: return 0.55557023301960222474f;
        case 7: case 25: return 0.19509032201612826785f;
        case 9: case 23: return -0.19509032201612826785f;
        case 11: case 21: return -0.55557023301960222474f;
        case 13: case 19: return -0.83146961230254523708f;
        case 15: case 17: return -0.98078528040323044913f;
        default: return cos16((m & 31) / 2);
    }
}
template <int DIR>
__device__ __forceinline__ float2 rot32(float2 a, int m) {
    m &= 31;
    if ((m & 1) == 0) return rot16<DIR>(a, m / 2);
    const float c = cos32(m), s = DIR < 0 ? -cos32(m - 8) : cos32(m - 8);
    return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
}

// 32 = 4 * 8 (see dft_split): Y[k1][n2] = W_32^{n2 k1} DFT_4 over n1 of
// x[8 n1 + n2], X[k1 + 4 k2] = DFT_8 over n2 of Y[k1][n2].
template <int DIR>
__device__ __forceinline__ void dft32(float2* v) {
    float2 t[32];
#pragma unroll
    for (int n2 = 0; n2 < 8; n2++) {
        float2 c[4];
#pragma unroll
        for (int n1 = 0; n1 < 4; n1++) c[n1] = v[8 * n1 + n2];
        dft4<DIR>(c);
#pragma unroll
        for (int k1 = 0; k1 < 4; k1++) t[8 * k1 + n2] = rot32<DIR>(c[k1], n2 * k1);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; k1++) {
        float2 c[8];
#pragma unroll
        for (int n2 = 0; n2 < 8; n2++) c[n2] = t[8 * k1 + n2];
        dft<8, DIR>(c);
#pragma unroll
        for (int k2 = 0; k2 < 8; k2++) v[k1 + 4 * k2] = c[k2];
    }
}
template <>
__device__ __forceinline__ void dft<32, -1>(float2* v) { dft32<-1>(v); }
template <>
__device__ __forceinline__ void dft<32, 1>(float2* v) { dft32<1>(v); }

// One component of an exchange: butterfly j = t + m T of the pass that ends
// (radix R, Ns points combined before it) writes its outputs, the threads
// read the operands of the next pass (radix R2).  COMP 0: x, 1: y.
template <int N, int T, int Ns, int R, int R2, int COMP>
__device__ __forceinline__ void exchange_half(float2 (&v)[kWide], float* lds, int t) {
#pragma unroll
    for (int m = 0; m < kWide / R; m++) {
        const int j = t + m * T, k = j & (Ns - 1);
        const int base = (j - k) * R + k;
        // Ns == 1: base is a multiple of R, a group starts on a pad boundary
        const int wb = (Ns == 1 || pad_aligned<Ns>()) ? lds_idx(base) : base;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int at = Ns == 1 ? wb + (R % 16 == 0 ? lds_idx(r) : r) : lx_wat<LX_PAD, Ns>(wb, r);
            lds[at] = COMP ? v[m * R + r].y : v[m * R + r].x;
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kWide / R2; m++) {
        const int rb = lx_rbase<LX_PAD, N / R2>(0, t + m * T);
#pragma unroll
        for (int r = 0; r < R2; r++) {
            const float x = lds[lx_rat<LX_PAD, N / R2>(rb, r)];
            if (COMP) v[m * R2 + r].y = x;
            else v[m * R2 + r].x = x;
        }
    }
    __syncthreads();
}

template <int N, int T, int Ns, int R, int R2>
__device__ __forceinline__ void exchange(float2 (&v)[kWide], float* lds, int t) {
    exchange_half<N, T, Ns, R, R2, 0>(v, lds, t);
    exchange_half<N, T, Ns, R, R2, 1>(v, lds, t);
}

// The twiddles of one butterfly, W_{Ns R}^{r k}.  `t1` holds the second
// pass's table stored [r Ns + k].  The third pass forms its 31 as powers of
// one, W_N^k, in FP64, whose multiply-adds issue at the rate of the FP32 ones
// here, and rounds each once.  As FP32 products of table entries (ten of two
// entries, the others of two such products) they added to the transform's
// error (relative L2 at 8192 / 16384 / 32768 points 1.362e-7 / 1.418e-7 /
// 1.486e-7; the kernels of 16 points per thread and the four-step chain have
// 1.315e-7 / 1.416e-7 / 1.414e-7; columns of 4096 points 1.381e-7 against
// 1.291e-7 in two passes).  So 1.294e-7 / 1.359e-7 / 1.432e-7 and 1.230e-7, in
// the same time or less (8192 x 512 14.1 -> 13.6 us, 32768 x 256 32.9 -> 32.7).
struct Wide64 {
    double x, y;
};
__device__ __forceinline__ Wide64 mul64(Wide64 a, Wide64 b) {
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// W_L^m
__device__ __forceinline__ Wide64 root64(int m, int L) {
    Wide64 w;
    sincospi(-2.0 * m / L, &w.y, &w.x);
    return w;
}
// W_N^k = tab[k % kWideLo] tab[kWideLo + k / kWideLo], k < N / 32.
constexpr int kWideLo = 32;
template <int N>
constexpr int kWideTab = kWideLo + N / kWide / kWideLo;
template <int N>
__device__ __forceinline__ void wide_table(Wide64* tab, int tid) {
    if (tid < kWideTab<N>) tab[tid] = root64(tid < kWideLo ? tid : (tid - kWideLo) * kWideLo, N);
}
// 32768 points multiply by the unrounded twiddles as well: the four-step chain
// reads all of its own from tables (1.432e-7 -> 1.405e-7; 8192 x 2048 would
// take 49.2 us instead of 48.5).
template <int N>
constexpr bool kProduct64 = N == 32768;
// Multiplies the MM butterflies v[m R ..] that share one k.
template <int N, int DIR, int First, int Ns, int R, int MM>
__device__ __forceinline__ void wide_twiddle(float2* v, const Wide64* tab, const float2* t1, int k) {
    if constexpr (Ns == First) {
#pragma unroll
        for (int r = 1; r < R; r++)
#pragma unroll
            for (int m = 0; m < MM; m++) v[m * R + r] = cmul_tw<DIR>(v[m * R + r], t1[r * Ns + k]);
    } else {
        static_assert(R == 32 && MM == 1 && Ns * R == N, "only a last radix-32 pass follows the second");
        // W^{r k} for r = b, b + 4, ..: few live at a time
        const Wide64 w1 = mul64(tab[k % kWideLo], tab[kWideLo + k / kWideLo]), w2 = mul64(w1, w1),
                     w4 = mul64(w2, w2);
        Wide64 first = w1;
#pragma unroll
        for (int b = 1; b <= 4; b++) {
            Wide64 w = first;
#pragma unroll
            for (int r = b; r < R; r += 4) {
                if constexpr (kProduct64<N>) {
                    const Wide64 p = mul64({v[r].x, v[r].y}, {w.x, DIR < 0 ? w.y : -w.y});
                    v[r] = make_float2((float)p.x, (float)p.y);
                } else {
                    v[r] = cmul_tw<DIR>(v[r], make_float2((float)w.x, (float)w.y));
                }
                if (r + 4 < R) w = mul64(w, w4);
            }
            if (b < 4) first = mul64(first, w1);
        }
    }
}

// Runs passes <R, Rest...> with Ns points combined; on entry v[m R + r] =
// x[t + m T + r N/R], on exit v[m RL + r] = X[t + m T + r N/RL].  First = the
// first pass's radix; `lds` = this transform's lds_len(N) floats; `tab`: of
// wide_table, unused by two passes.  Every LDS read has ended (a barrier
// passed) when an exchange returns.
template <int N, int T, int DIR, int First, int Ns, int R, int... Rest>
__device__ __forceinline__ void stockham_wide(float2 (&v)[kWide], float* lds, const Wide64* tab, const float2* t1,
                                              int t) {
    static_assert(kWide % R == 0 && N == T * kWide, "32 points per thread");
    constexpr int M = kWide / R;
    if constexpr (Ns > 1 && T % Ns == 0) {
        // every butterfly of the thread has the same k
        wide_twiddle<N, DIR, First, Ns, R, M>(v, tab, t1, t & (Ns - 1));
    }
#pragma unroll
    for (int m = 0; m < M; m++) {
        if constexpr (Ns > 1 && T % Ns != 0)
            wide_twiddle<N, DIR, First, Ns, R, 1>(&v[m * R], tab, t1, (t + m * T) & (Ns - 1));
        dft<R, DIR>(&v[m * R]);
        // one butterfly at a time: interleaved, their temporaries spill
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (sizeof...(Rest) > 0) {
        asm volatile("" : "+v"(t));
        constexpr int R2 = bfly_dev::First<Rest...>::value;
        exchange<N, T, Ns, R, R2>(v, lds, t);
        asm volatile("" : "+v"(t));
        stockham_wide<N, T, DIR, First, Ns * R, Rest...>(v, lds, tab, t1, t);
    }
}

}  // namespace bfly_dev
