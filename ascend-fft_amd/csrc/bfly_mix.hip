// bfly_mix.hip -- per-mode complex channel mixing of the 1-D spectral
// convolution on the matrix cores, in the layouts the mode-truncated R2C
// writes and the C2R reads (mode index fastest), so no transposed copy of the
// modes or of the weights is ever made.
//
//   C[m][n][k] = sum_r  opA(A)[m][r][k] * opB(B)[r][n][k],   k < K,
//
// complex64 interleaved, every operand with unit stride along the mode k and
// arbitrary strides along its two channel indices; opA / opB optionally
// conjugate.  The three products of the layer (forward, input gradient,
// weight gradient) are this one kernel with different strides.
//
// Per mode the product is a small complex GEMM, done as four real fp32
// v_mfma_f32_16x16x4_f32 products per 16x16 tile and 4-deep slice of r:
//   Cre += Are Bre,  Cre += (-Aim) Bim,  Cim += Are Bim,  Cim += Aim Bre
// (fp32 operands, fp32 accumulation).
//
// Workgroup: 8 modes x 16 MH rows (m) x 16 NH columns (n) of C, 512 threads;
// wave w owns mode w and all MH x NH 16x16 tiles of it.  The reduction runs
// in chunks of 8 r.  A chunk of A (8 r x 16 MH m x 8 k) and of B is read with
// two modes per lane (16 bytes, four lanes per 64-byte run along k) into
// registers two chunks ahead of its products, parked in one of two LDS
// buffers one chunk ahead, and read from there as matrix operands (lane l:
// row l % 16, r = 4 s + l / 16): one barrier per chunk, and a load has two
// chunks of products to arrive.  Results leave through the same LDS and are
// stored along the mode index (64-byte runs per (m, n)).
//
// Bound by the matrix cores at the layer's sizes: batch 64, 128 x 128
// channels, 256 modes are 2.15 GFLOP, 14 us at the 153 TFLOP/s that fp32
// matrix instructions reach here, against 67 MB of operands (11 us).  Measured
// there 24.3 us forward and input gradient, 25.6 weight gradient (38.0 and
// 35.3 with 4 waves of two modes, one LDS buffer, two barriers per chunk and
// nothing between the matrix instructions); without the loop's loads 23, so
// what is left is the launch, the first chunk's latency and the stores (about
// 8 us together).  Batch 16, 64 x 64 channels, 64 modes 12.4 -> 5.6 us, 255
// modes (rows not 16-byte aligned, 8-byte accesses before) 53.9 -> 26.7.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "bfly_device.hpp"
#include "bfly_kernels.hpp"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// two modes, 8-byte aligned (a 16-byte access all the same)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ float4 load_pair(const float2* p) {
    const f32x4u v = *reinterpret_cast<const f32x4u*>(p);
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void store_pair(float2* p, float4 c) {
    *reinterpret_cast<f32x4u*>(p) = f32x4u{c.x, c.y, c.z, c.w};
}

constexpr int kKT = 8;  // modes per workgroup, one per wave
constexpr int kRT = 8;  // reduction chunk: two 4-deep matrix steps
constexpr int kThreads = 64 * kKT;
constexpr uint64_t kMaxGridX = 1u << 22;

// LDS layout of a chunk: [r][row][4 slots of two modes], where modes 2 p, 2 p
// + 1 of (r, row) are in slot p ^ (row / 4 % 4), swapped for odd r: the 16
// rows of a matrix operand then lie in 16 different slots of the 64 banks
// and its even and odd r in different halves of a slot.
__device__ __forceinline__ int slot_of(int p, int row) { return p ^ ((row >> 2) & 3); }

// One operand's chunks of 16 H rows: pair q = (t + 512 j) / 4 is row q % (16
// H) at reduction index q / (16 H) of the chunk; lane t % 4 loads its modes 2
// (t % 4) and + 1.  `lead` = the row stride, `red` = the r stride.  Each lane
// keeps its pointers and steps them from chunk to chunk; an element outside
// the operand re-reads a real one and is masked where the chunk is parked, so
// no load sits under a branch (which would make the compiler wait for it).
// EDGE: the tile or the last chunk reaches past the operand.
template <int H, bool PAIRS, bool EDGE>
struct Operand {
    const float2* p[H];
    bool row_ok[H];
    uint64_t step;
    uint32_t R;
    bool pair_ok;
    int at;  // LDS complex index of the lane's first pair's even mode, minus its half
    int half;
    static __device__ __forceinline__ int q(int j, int t) { return (t + kThreads * j) / 4; }
    __device__ __forceinline__ void init(const float2* __restrict__ base, uint32_t rows, uint32_t R_, uint32_t K,
                                         uint64_t lead, uint64_t red, uint32_t row0, uint32_t k, int t) {
        R = R_;
        step = kRT * red;
        pair_ok = k + 1 < K;
#pragma unroll
        for (int j = 0; j < H; j++) {
            const uint32_t row = row0 + q(j, t) % (16 * H), r = q(j, t) / (16 * H);
            row_ok[j] = !EDGE || (row < rows && k < K);
            // an odd K's last mode is read as the second of the pair before it
            const uint32_t kk = PAIRS && EDGE && !pair_ok ? k - 1 : k;
            p[j] = base + (row_ok[j] ? (uint64_t)row * lead + kk : 0) + (uint64_t)(!EDGE || r < R ? r : R - 1) * red;
        }
        // pairs lie 128 apart: the same slot, and r of the same parity
        static_assert(128 % (16 * H) == 0 && 128 / (16 * H) % 2 == 0, "slot and parity of all pairs");
        at = q(0, t) * 8 + 2 * slot_of(t % 4, q(0, t) % (16 * H));
        half = (q(0, t) / (16 * H)) & 1;
    }
    // loads the chunk that starts at r0 and steps on
    __device__ __forceinline__ void load(float4 (&reg)[H], uint32_t r0, int t) {
#pragma unroll
        for (int j = 0; j < H; j++) {
            if constexpr (PAIRS) {
                reg[j] = load_pair(p[j]);
            } else {
                reg[j] = make_float4(p[j]->x, p[j]->y, 0.f, 0.f);
            }
            p[j] += r0 + kRT + (EDGE ? q(j, t) / (16 * H) : 0) < R ? step : 0;
        }
    }
    __device__ __forceinline__ void park(float2* __restrict__ lds, float4 (&reg)[H], uint32_t r0, int t) const {
#pragma unroll
        for (int j = 0; j < H; j++) {
            float2 a = make_float2(reg[j].x, reg[j].y), b = make_float2(reg[j].z, reg[j].w);
            if constexpr (EDGE) {
                const bool in0 = row_ok[j] && r0 + q(j, t) / (16 * H) < R, in1 = in0 && pair_ok;
                if (PAIRS && !pair_ok) a = b;
                a = make_float2(in0 ? a.x : 0.f, in0 ? a.y : 0.f);
                b = make_float2(in1 ? b.x : 0.f, in1 ? b.y : 0.f);
            }
            lds[at + half + kThreads * 2 * j] = a;
            lds[at + 1 - half + kThreads * 2 * j] = b;
        }
    }
};

// MH / NH = 16-row halves of the tile along m / n (tile 16 MH x 16 NH).
// CONJ: which operand is conjugated (0 none, 1 A, 2 B).
template <int MH, int NH, bool PAIRS, int CONJ, bool EDGE>
__device__ __forceinline__ void mix_tile(float4* lds, const float2* __restrict__ A, const float2* __restrict__ B,
                                         float2* __restrict__ C, uint32_t M, uint32_t N, uint32_t R, uint32_t K,
                                         uint64_t sam, uint64_t sar, uint64_t sbr, uint64_t sbn, uint64_t scm,
                                         uint64_t scn, uint32_t m0, uint32_t n0, uint32_t k0) {
    constexpr int TM = 16 * MH, TN = 16 * NH;
    constexpr int LA = kRT * TM * 8, LB = kRT * TN * 8;  // complex values per chunk
    const int t = threadIdx.x, lane = t % 64, w = t / 64;
    const uint32_t kl = k0 + 2 * (t % 4);  // first of this lane's two load modes
    f32x4 acc[MH][NH][2];  // [m half][n half][re, im]
#pragma unroll
    for (int i = 0; i < MH; i++)
#pragma unroll
        for (int j = 0; j < NH; j++)
#pragma unroll
            for (int c = 0; c < 2; c++) acc[i][j][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    Operand<MH, PAIRS, EDGE> oa;
    Operand<NH, PAIRS, EDGE> ob;
    oa.init(A, M, R, K, sam, sar, m0, kl, t);
    ob.init(B, N, R, K, sbn, sbr, n0, kl, t);
    float2* const As0 = reinterpret_cast<float2*>(lds);
    float4 ra[2][MH], rb[2][NH];
    auto load = [&](auto p, uint32_t r0) {
        oa.load(ra[decltype(p)::value], r0, t);
        ob.load(rb[decltype(p)::value], r0, t);
    };
    auto park = [&](auto p, uint32_t r0) {
        constexpr int P = decltype(p)::value;
        oa.park(As0 + P * (LA + LB), ra[P], r0, t);
        ob.park(As0 + P * (LA + LB) + LA, rb[P], r0, t);
    };
    const int lr = lane % 16, lq = lane / 16;
    const int op = 2 * slot_of(w / 2, lr) + ((w ^ lq) & 1);  // complex index inside a (r, row)
    // the operands of one chunk, and their products (`mma`s of the two halves
    // of the complex product use different accumulators, so consecutive
    // matrix instructions never wait on each other)
    float2 x[kRT / 4][MH], y[kRT / 4][NH];
    auto fetch = [&](auto p) {
        const float2* As = As0 + decltype(p)::value * (LA + LB) + op;
        const float2* Bs = As + LA;
#pragma unroll
        for (int s = 0; s < kRT / 4; s++) {
#pragma unroll
            for (int h = 0; h < MH; h++) x[s][h] = As[((4 * s + lq) * TM + 16 * h + lr) * 8];
#pragma unroll
            for (int h = 0; h < NH; h++) y[s][h] = Bs[((4 * s + lq) * TN + 16 * h + lr) * 8];
        }
    };
    auto products = [&]() {
        auto mma = [](float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); };
#pragma unroll
        for (int s = 0; s < kRT / 4; s++) {
#pragma unroll
            for (int i = 0; i < MH; i++)
#pragma unroll
                for (int j = 0; j < NH; j++) {
                    acc[i][j][0] = mma(x[s][i].x, y[s][j].x, acc[i][j][0]);
                    acc[i][j][1] = mma(CONJ == 2 ? -x[s][i].x : x[s][i].x, y[s][j].y, acc[i][j][1]);
                }
#pragma unroll
            for (int i = 0; i < MH; i++)
#pragma unroll
                for (int j = 0; j < NH; j++) {
                    acc[i][j][0] = mma(CONJ ? x[s][i].y : -x[s][i].y, y[s][j].y, acc[i][j][0]);
                    acc[i][j][1] = mma(CONJ == 1 ? -x[s][i].y : x[s][i].y, y[s][j].x, acc[i][j][1]);
                }
        }
    };
    constexpr std::integral_constant<int, 0> p0{};
    constexpr std::integral_constant<int, 1> p1{};
    load(p0, 0);
    load(p1, kRT);  // a chunk past the end re-reads real elements and is never multiplied
    park(p0, 0);
    load(p0, 2 * kRT);
    __syncthreads();
    auto weave = [] {
        __builtin_amdgcn_sched_group_barrier(0x100, MH + NH, 0);  // operands of the first matrix steps
#pragma unroll
        for (int i = 0; i < kRT / 4 * MH * NH * 2; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);  // matrix
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
            if (i >= kRT / 4 * MH * NH) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // load
        }
    };
    // step r0: fetch this chunk's operands, park the next chunk, load the
    // third next, multiply
    for (uint32_t r0 = 0; r0 < R; r0 += 2 * kRT) {
        fetch(p0);
        park(p1, r0 + kRT);
        load(p1, r0 + 3 * kRT);
        products();
        weave();
        __syncthreads();
        if (r0 + kRT < R) {
            fetch(p1);
            park(p0, r0 + 2 * kRT);
            load(p0, r0 + 4 * kRT);
            products();
            weave();
            __syncthreads();
        }
    }
    // Results leave through LDS ([m][n][4 slots], slots and halves chosen as
    // above with n for the row and m / 4 for r).  Lane l holds rows 4 (l / 16)
    // + v (v < 4) and column l % 16 of each 16x16 tile.
#pragma unroll
    for (int i = 0; i < MH; i++)
#pragma unroll
        for (int j = 0; j < NH; j++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int m = 16 * i + 4 * lq + v, n = 16 * j + lr;
                As0[(m * TN + n) * 8 + op] = make_float2(acc[i][j][0][v], acc[i][j][1][v]);
            }
    __syncthreads();
    const uint32_t ks = k0 + 2 * (t % 4);
#pragma unroll
    for (int e = 0; e < TM * TN * 4 / kThreads; e++) {
        const int q = (t + kThreads * e) / 4, ml = q / TN, nl = q % TN;
        const uint32_t m = m0 + ml, n = n0 + nl;
        float4 c = lds[q * 4 + slot_of(t % 4, nl)];
        if ((ml >> 2) & 1) c = make_float4(c.z, c.w, c.x, c.y);
        if (!EDGE || (m < M && n < N && ks < K)) {
            float2* dst = C + (uint64_t)m * scm + (uint64_t)n * scn + ks;
            if (!EDGE || ks + 1 < K) store_pair(dst, c);
            else dst[0] = make_float2(c.x, c.y);
        }
    }
}

template <int MH, int NH, bool PAIRS, int CONJ>
__global__ __launch_bounds__(kThreads) void k_mix(const float2* __restrict__ A, const float2* __restrict__ B,
                                                  float2* __restrict__ C, uint32_t M, uint32_t N, uint32_t R,
                                                  uint32_t K, uint64_t sam, uint64_t sar, uint64_t sbr,
                                                  uint64_t sbn, uint64_t scm, uint64_t scn, uint32_t mtiles,
                                                  uint32_t tiles, uint32_t blocks) {
    constexpr int TM = 16 * MH, TN = 16 * NH;
    // two chunks of both operands, or the staged results
    constexpr int LDS = 2 * kRT * (TM + TN) * 4 > TM * TN * 4 ? 2 * kRT * (TM + TN) * 4 : TM * TN * 4;
    __shared__ float4 lds[LDS];
    const uint32_t bid = blockIdx.y * gridDim.x + blockIdx.x;
    if (bid >= blocks) return;
    // tiles of one mode group are neighbours, and each XCD gets a contiguous
    // part of the list: the tiles that read the same operands, and the mode
    // groups that share their 128-byte lines, meet in one L2
    const uint32_t u = bfly_dev::xcd_window(bid, blocks, blocks >= 8 ? blocks / 8 : 1);
    const uint32_t tile = u % tiles, k0 = u / tiles * kKT;
    const uint32_t m0 = (tile % mtiles) * TM, n0 = (tile / mtiles) * TN;
    const bool edge = m0 + TM > M || n0 + TN > N || k0 + kKT > K || R % kRT != 0;  // uniform
    if (edge)
        mix_tile<MH, NH, PAIRS, CONJ, true>(lds, A, B, C, M, N, R, K, sam, sar, sbr, sbn, scm, scn, m0, n0, k0);
    else
        mix_tile<MH, NH, PAIRS, CONJ, false>(lds, A, B, C, M, N, R, K, sam, sar, sbr, sbn, scm, scn, m0, n0, k0);
}

template <int MH, int NH>
hipError_t launch_mix(const float2* A, const float2* B, float2* C, uint32_t M, uint32_t N, uint32_t R, uint32_t K,
                      uint64_t sam, uint64_t sar, uint64_t sbr, uint64_t sbn, uint64_t scm, uint64_t scn,
                      int conj, hipStream_t s) {
    const uint32_t kt = (K + kKT - 1) / kKT, mt = (M + 16 * MH - 1) / (16 * MH), nt = (N + 16 * NH - 1) / (16 * NH);
    const uint64_t blocks = (uint64_t)kt * mt * nt;
    if (blocks == 0 || blocks > 0x7FFFFFFFull) return hipErrorInvalidValue;
    // a grid dimension holds less than 2^32 threads: 2^23 workgroups of 512
    // (one row, column and channel of 2^26 modes) take a second one
    const uint32_t gx = (uint32_t)(blocks < kMaxGridX ? blocks : kMaxGridX), gy = (uint32_t)((blocks + gx - 1) / gx);
    auto go = [&](auto v, auto cj) {
        hipLaunchKernelGGL((k_mix<MH, NH, decltype(v)::value, decltype(cj)::value>), dim3(gx, gy), dim3(kThreads), 0, s,
                           A, B, C, M, N, R, K, sam, sar, sbr, sbn, scm, scn, mt, mt * nt, (uint32_t)blocks);
    };
    auto pick = [&](auto v) {
        if (conj == 0) go(v, std::integral_constant<int, 0>{});
        else if (conj == 1) go(v, std::integral_constant<int, 1>{});
        else go(v, std::integral_constant<int, 2>{});
    };
    // modes go in pairs; a single mode (K = 1) has none
    if (K > 1) pick(std::true_type{});
    else pick(std::false_type{});
    return hipGetLastError();
}

}  // namespace

namespace bfly_kern {

hipError_t mode_mix(int op, const float* a, const float* b, float* c, uint32_t batch, uint32_t c_in,
                    uint32_t c_out, uint32_t modes, hipStream_t s) {
    const uint64_t K = modes;
    uint32_t M, N, R;
    uint64_t sam, sar, sbr, sbn, scm, scn;
    int conj = 0;
    if (op == 0) {  // y[b][o] = sum_i x[b][i] w[i][o]
        M = batch, N = c_out, R = c_in;
        sam = c_in * K, sar = K, sbr = c_out * K, sbn = K, scm = c_out * K, scn = K;
    } else if (op == 1) {  // gx[b][i] = sum_o gy[b][o] conj(w[i][o])
        M = batch, N = c_in, R = c_out;
        sam = c_out * K, sar = K, sbr = K, sbn = c_out * K, scm = c_in * K, scn = K;
        conj = 2;
    } else if (op == 2) {  // gw[i][o] = sum_b conj(x[b][i]) gy[b][o]
        M = c_in, N = c_out, R = batch;
        sam = K, sar = c_in * K, sbr = c_out * K, sbn = K, scm = c_out * K, scn = K;
        conj = 1;
    } else {
        return hipErrorInvalidValue;
    }
    const auto* A = reinterpret_cast<const float2*>(a);
    const auto* B = reinterpret_cast<const float2*>(b);
    auto* C = reinterpret_cast<float2*>(c);
    // The largest tile that still gives every CU one (a larger tile re-reads
    // the operands less, a smaller one has more workgroups to hide each
    // other's loads): 32 x 32 / 16 x 32 / 16 x 16 at batch 64, 128 x 128
    // channels, 256 modes 24.6 / 24.3 / 28.1 us forward, 25.6 / 28.1 / 30.2
    // weight gradient; batch 16, 64 x 64 channels, 64 modes 12.9 / 7.5 / 5.6.
    auto tiles = [&](uint64_t tm, uint64_t tn) { return (K + kKT - 1) / kKT * ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
    if (tiles(32, 32) >= 256) return launch_mix<2, 2>(A, B, C, M, N, R, (uint32_t)K, sam, sar, sbr, sbn, scm, scn, conj, s);
    if (tiles(16, 32) >= 256) return launch_mix<1, 2>(A, B, C, M, N, R, (uint32_t)K, sam, sar, sbr, sbn, scm, scn, conj, s);
    return launch_mix<1, 1>(A, B, C, M, N, R, (uint32_t)K, sam, sar, sbr, sbn, scm, scn, conj, s);
}

}  // namespace bfly_kern
