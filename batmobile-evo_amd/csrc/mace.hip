// MACE-style interaction layer with per-edge radial weights (the baseline's
// configs[4]): Bessel radial basis -> MLP [8 -> 64 -> 34 C] -> channel-wise
// weighted CG product of X[src] with Y(v) -> scatter-add into destinations,
// and its gradient with respect to the positions.
//
// Pattern of reference benchmarks/benchmark_e2e_mace.py:281-434 (SH -> TP ->
// scatter, forces by backward through the edge vectors :412-420); the
// reference's own block shares one W[34, C, C] over edges, the per-edge radial
// weights are this configuration's.  Layer definition (fp32 here):
//   v_e = min_image(pos[dst_e] - pos[src_e]), r = |v|, u = v / r
//   B_k = sqrt(2/rc) sin(k pi r/rc) / r * f(r/rc),  f(d) = 1 - 28 d^6 + 48 d^7 - 21 d^8
//   h = silu(B W1 + b1), R[e, c, p] = (h W2)[p * C + c]
//   out[d, c, o] = sum_{e -> d} sum_p R[e,c,p] sum_{(a,b) in p -> o} CG x[src_e,c,a] Y_e[b]
//
// Work per edge: the MLP's second layer is a GEMM [edges x 64] x [64 x 34C]
// (557 kflop per edge at C = 128).  One kernel per pass runs it on the bf16 matrix
// cores (each fp32 operand as three bf16 parts, six products: common.h) and
// consumes each tile of per-edge weights R straight from the accumulators in
// the channel-wise CG product on the VALU, formed in the frame of the edge
// (aligned.h: about 340 operations per edge and channel against 1023), so R
// (26 GB at configs[4]) never reaches memory.  The backward forms R and its
// derivative along the edge length by the same GEMM, contracts both with the
// incoming gradient in the same frame, and ends in per-edge position gradients; forces are gathered per atom through
// the reverse-edge map of the symmetric edge list.  Every sum runs in a fixed
// order (deterministic, no atomics).
#include "aligned.h"
#include "batmobile_hip.h"

namespace bmhip {

constexpr int kNBasis = 8;
constexpr int kHidden = 64;

#pragma clang fp contract(off)
// v = pos[dst] - pos[src] with the minimum image of an orthorhombic box, in the
// neighbor list's operation order (so v equals its vectors negated, exactly)
__device__ __forceinline__ void edge_vector(const float* __restrict__ pos, int64_t s, int64_t d,
                                            const float* box, const float* inv, float* v) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float t = pos[d * 3 + k] - pos[s * 3 + k];
        const float q = t * inv[k];
        const float rr = rintf(q);
        const float m = rr * box[k];
        v[k] = t - m;
    }
}
#pragma clang fp contract(on)

struct MaceBox {
    float box[3];
    float inv[3];
};

__device__ __forceinline__ float sigmoidf(float z) { return 1.0f / (1.0f + expf(-z)); }

// ---------------------------------------------------------------------------
// fp32 GEMM on MFMA: C[M, N] = A[M, K] B, with B = [K, N] (row-major) or, when
// TB, given as B^T [N, K] (row-major).  Workgroup tile 128 x BN, K step 16,
// four waves in 2 x 2, each 64 x BN/2 (4 x BN/32 MFMA tiles of 16 x 16).  Both
// operands sit in LDS with k contiguous (sA[m][k], sB[n][k]), so one float4
// read gives a lane its A (or B) values for four k-steps: k-step s of lane
// group g = lane / 16 is k = 4 g + s, the same for A and B.
// ---------------------------------------------------------------------------
template <bool TB, int BN>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ A,
                                                       const float* __restrict__ B,
                                                       float* __restrict__ C, int M, int N, int K) {
    constexpr int BM = 128, BK = 16, WN = BN / 2, NT = WN / 16;
    constexpr int LD = BK + 4;  // row stride in floats (keeps float4 alignment)
    __shared__ __attribute__((aligned(16))) float sA[BM * LD];
    __shared__ __attribute__((aligned(16))) float sB[BN * LD];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wm = wv >> 1, wn = wv & 1;
    const int g4 = lane >> 4, i16 = lane & 15;
    const int64_t m0 = (int64_t)blockIdx.y * BM;
    const int n0 = blockIdx.x * BN;
    const bool k4 = (K & 3) == 0, n4 = (N & 3) == 0;  // float4 global loads possible
    v4f acc[4][NT];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < NT; ++ni) acc[mi][ni] = v4f{0.f, 0.f, 0.f, 0.f};
    // one float4 of a row-major [rows, K] matrix (zeros past the edges)
    auto ld_rowk = [&](const float* P, int64_t row, int64_t rows, int k) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < rows) {
            const float* q = P + row * K + k;
            if (k4 && k + 3 < K) {
                v = *reinterpret_cast<const float4*>(q);
            } else {
                v.x = k < K ? q[0] : 0.f;
                v.y = k + 1 < K ? q[1] : 0.f;
                v.z = k + 2 < K ? q[2] : 0.f;
                v.w = k + 3 < K ? q[3] : 0.f;
            }
        }
        return v;
    };
    for (int k0 = 0; k0 < K; k0 += BK) {
        __syncthreads();
#pragma unroll
        for (int it = 0; it < BM * BK / 4 / 256; ++it) {
            const int idx = tid + it * 256, m = idx >> 2, kq = idx & 3;
            *reinterpret_cast<float4*>(sA + m * LD + 4 * kq) = ld_rowk(A, m0 + m, M, k0 + 4 * kq);
        }
        if constexpr (TB) {
#pragma unroll
            for (int it = 0; it < BN * BK / 4 / 256; ++it) {
                const int idx = tid + it * 256, n = idx >> 2, kq = idx & 3;
                *reinterpret_cast<float4*>(sB + n * LD + 4 * kq) = ld_rowk(B, n0 + n, N, k0 + 4 * kq);
            }
        } else {
#pragma unroll
            for (int it = 0; it < BN * BK / 4 / 256; ++it) {
                const int idx = tid + it * 256, k = idx / (BN / 4), nq = idx % (BN / 4);
                const int kk = k0 + k, nn = n0 + 4 * nq;
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (kk < K) {
                    const float* q = B + (int64_t)kk * N + nn;
                    if (n4 && nn + 3 < N) {
                        v = *reinterpret_cast<const float4*>(q);
                    } else {
                        v.x = nn < N ? q[0] : 0.f;
                        v.y = nn + 1 < N ? q[1] : 0.f;
                        v.z = nn + 2 < N ? q[2] : 0.f;
                        v.w = nn + 3 < N ? q[3] : 0.f;
                    }
                }
                sB[(4 * nq + 0) * LD + k] = v.x;
                sB[(4 * nq + 1) * LD + k] = v.y;
                sB[(4 * nq + 2) * LD + k] = v.z;
                sB[(4 * nq + 3) * LD + k] = v.w;
            }
        }
        __syncthreads();
        float4 a[4];
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
            a[mi] = *reinterpret_cast<const float4*>(sA + (wm * 64 + mi * 16 + i16) * LD + 4 * g4);
#pragma unroll
        for (int ni = 0; ni < NT; ++ni) {
            const float4 b =
                *reinterpret_cast<const float4*>(sB + (wn * WN + ni * 16 + i16) * LD + 4 * g4);
#pragma unroll
            for (int mi = 0; mi < 4; ++mi) acc[mi][ni] = mfma4(a[mi], b, acc[mi][ni]);
        }
    }
    // D[4 g4 + r][i16] of tile (mi, ni)
#pragma unroll
    for (int ni = 0; ni < NT; ++ni) {
        const int n = n0 + wn * WN + ni * 16 + i16;
        if (n >= N) continue;
#pragma unroll
        for (int mi = 0; mi < 4; ++mi)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = m0 + wm * 64 + mi * 16 + 4 * g4 + r;
                if (m < M) C[m * N + n] = acc[mi][ni][r];
            }
    }
}

__device__ __forceinline__ void load_row16(const float* __restrict__ p, float* v) {
    const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 t = q[i];
        v[4 * i] = t.x;
        v[4 * i + 1] = t.y;
        v[4 * i + 2] = t.z;
        v[4 * i + 3] = t.w;
    }
}

// ---------------------------------------------------------------------------
// grad_pos[a] = sum_{e in row a} (g_v[e] - g_v[rev[e]]): v_e = pos[dst] -
// pos[src], and rev[e] is the edge with the roles of a and src_e swapped.
// ---------------------------------------------------------------------------
__global__ void mace_forces_kernel(const float* __restrict__ gv, const int64_t* __restrict__ row_ptr,
                                   const int64_t* __restrict__ rev, float* __restrict__ gpos,
                                   int64_t n) {
    const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= n) return;
    float f0 = 0.f, f1 = 0.f, f2 = 0.f;
    for (int64_t e = row_ptr[a]; e < row_ptr[a + 1]; ++e) {
        const int64_t t = rev[e];
        if (t < 0) continue;  // edge list not symmetric (reported by the reverse-edge build)
        f0 += gv[e * 3 + 0] - gv[t * 3 + 0];
        f1 += gv[e * 3 + 1] - gv[t * 3 + 1];
        f2 += gv[e * 3 + 2] - gv[t * 3 + 2];
    }
    gpos[a * 3 + 0] = f0;
    gpos[a * 3 + 1] = f1;
    gpos[a * 3 + 2] = f2;
}

// rev[e] for e = (src j -> dst i): the edge (src i -> dst j), found by binary
// search in row j (sources ascending); -1 if the edge list is not symmetric.
__global__ void mace_reverse_edges_kernel(const int64_t* __restrict__ row_ptr,
                                          const int64_t* __restrict__ src,
                                          int64_t* __restrict__ rev, int* __restrict__ missing,
                                          int64_t n, int64_t n_edges) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_edges) return;
    // destination of e: the row containing e
    int64_t lo = 0, hi = n;  // last row with row_ptr[row] <= e
    while (hi - lo > 1) {
        const int64_t mid = (lo + hi) >> 1;
        if (row_ptr[mid] <= e) lo = mid;
        else hi = mid;
    }
    const int64_t i = lo, j = src[e];
    int64_t a = row_ptr[j], b = row_ptr[j + 1];  // first position with src >= i
    while (a < b) {
        const int64_t mid = (a + b) >> 1;
        if (src[mid] < i) a = mid + 1;
        else b = mid;
    }
    const bool ok = a < row_ptr[j + 1] && src[a] == i;
    rev[e] = ok ? a : -1;
    if (!ok) atomicAdd(missing, 1);
}

// ---------------------------------------------------------------------------
// Fused layer kernels.
//
// Edges are taken in "positions": the destinations in the given order (a
// spatial order keeps shared source rows in cache), each destination's edges
// consecutive and ascending.  A prepass writes per position the direction, the
// source and destination, and the radial MLP's hidden layer h [E][64] in three
// bf16 parts (the backward also the length and s[E][64], below).
//
// A workgroup owns one quad of 4 channels c0..c0+3 and keeps that quad's slice
// of W2 in LDS, split into bf16 parts, as MFMA operand fragments (paths in 9 groups
// of 4, the last two slots zero).  Each of its waves walks its own range of positions
// (ranges end at destination boundaries) in tiles of 16 edges.  Per tile,
// v_mfma_f32_16x16x32_bf16 gives
//   D[4 ch + j][e] = sum_k W2[k][(4g + j) C + c0 + ch] h[e][k]  = R[e, c0 + ch, 4g + j]
// (A = the W2 fragments from LDS, B = h of the tile, K = 64 in 2 steps of 6 products,
// 9 groups: 108 MFMAs of 16 cycles, against 144 of 32 with fp32 MFMAs), and by the
// accumulator layout lane l = 16 ch + e holds the 34 weights of its own (edge e,
// channel c0 + ch) pair.  The lane then forms the message of that pair,
// sum_p R_p T_p(x[src, c], Y(u)), on the VALU (aligned.h).  R never leaves the registers.
//
// Bound: VALU + MFMA issue of the SIMD, which overlap little (a probe: 8 FMAs between
// 16-cycle MFMAs add their whole time with 4 waves per SIMD).  N = 50,000, C = 128,
// 1.5 M edges, forward / backward kernel: fp32 MFMAs and the product by CG entries 10.5 /
// 17.9 ms; bf16 parts 7.4 / 12.6 ms; product in the edge's frame and the length's
// derivative by S = s W2 instead of the transpose GEMM 5.1 / 9.7 ms.  The layer's pass
// with position gradients 29.1 -> 20.9 -> 15.7 ms, its error against 64 bits unchanged
// (1.0e-6; it comes from the radial basis).
//
// Each destination's messages are summed in ascending edge order by one lane
// after another along the tile (lane e adds lane e - 1's running sum when both
// belong to the same destination), the running sum of a destination that
// continues into the next tile carried in LDS.  The sum is therefore the same
// sequence of additions whatever the tiling, the order of the destinations or
// the launch shape; each output row is written once, with no atomics.
// ---------------------------------------------------------------------------
constexpr int kMaceFwdWaves = 16;                    // waves (position ranges) per workgroup
constexpr int kMaceBwdWaves = 12;
constexpr int kPG = 9;                               // groups of 4 paths (36 slots)
constexpr int kHSteps = kHidden / 32;                // K = 32 steps of the hidden layer
constexpr int kHRow = 3 * kHidden / 8;               // h of a position: 24 v4u, [part][k / 8]
constexpr int kW2Frags = kPG * kHSteps * 3;          // 1 KB operand fragments per channel quad
constexpr int kMaceMaxWorkers = 8192;                // position ranges (wstart entries - 1)

// The quad's W2 slice as MFMA operand fragments, sW[(g * 2 + s) * 3 + part][lane]: row
// lane % 16 = 4 ch + j of group g (path 4g + j of channel c0 + ch), hidden units
// 32 s + 8 (lane / 16) .. + 7 (zeros past path 33 and past channel C - 1).
__device__ __forceinline__ void mace_fill_w2(const float* __restrict__ w2, int C, int c0,
                                             v4u* sW) {
    for (int i = threadIdx.x; i < kPG * kHSteps * 64; i += blockDim.x) {
        const int lane = i & 63, s = (i >> 6) % kHSteps, g = (i >> 6) / kHSteps;
        const int c = c0 + ((lane & 15) >> 2), p = 4 * g + (lane & 3);
        const int k0 = 32 * s + 8 * (lane >> 4);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = p < kNumPaths && c < C ? w2[((int64_t)(k0 + j) * kNumPaths + p) * C + c] : 0.0f;
        const Bf3 b = bf16_split8(v);
        v4u* f = sW + (g * kHSteps + s) * 3 * 64 + lane;
        f[0] = b.h;
        f[64] = b.m;
        f[128] = b.l;
    }
}

// r_i[p] = sum_k W2[k][p C + c0 + ch] b_i[e][k] of the lane's pair, for NB right-hand
// sides: sA = sW + lane, b_i[part * 2 + s] = the part of b_i[e][32 s + 8 (lane / 16) .. + 7].
// The small products of both K steps go first, while the accumulator is small.
template <int NB>
__device__ __forceinline__ void mace_tile_weights(const v4u* sA, const v4u* const* b,
                                                  float* const* r) {
    // the W2 operands are the same for every tile: read them from LDS per tile (an
    // opaque base keeps the compiler from hoisting the reads out of the tile loop)
    int base = 0;
    asm volatile("" : "+v"(base));
    sA += base;
    static_for<kPG>([&](auto gg) {
        constexpr int g = decltype(gg)::value;
        v4u a[3 * kHSteps];
#pragma unroll
        for (int s = 0; s < kHSteps; ++s)
#pragma unroll
            for (int q = 0; q < 3; ++q) a[q * kHSteps + s] = sA[((g * kHSteps + s) * 3 + q) * 64];
        v4f acc[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
        constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};  // l h, h l, m m, ...
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int s = 0; s < kHSteps; ++s)
#pragma unroll
                for (int i = 0; i < NB; ++i)
                    acc[i] = mfma_bf16(a[kA[t] * kHSteps + s], b[i][kB[t] * kHSteps + s], acc[i]);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (4 * g + j < kNumPaths) r[i][4 * g + j] = acc[i][j];
        __builtin_amdgcn_sched_barrier(0);  // one group's fragments at a time
    });
}

// Lane reads within the 16-lane row.  Call them where every lane runs (a lane that
// reads a lane skipped by a branch, e.g. the right side of a short-circuit ||,
// gets no value).
__device__ __forceinline__ int dpp_prev_i(int v) {  // lane e - 1
    return __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
}
__device__ __forceinline__ int dpp_next_i(int v) {  // lane e + 1 of the 16-lane row
    return __builtin_amdgcn_update_dpp(0, v, 0x101, 0xF, 0xF, false);
}

// The frame of edge direction u = (cos f, sin f, c, s); c and s are also returned.
//
// An edge shorter than the length's lower bound kMinLength has u = v / kMinLength, of length
// rho < 1 (0 for a self loop), and Y_l(u) = rho^l Y_l(u / rho).  It is marked by a negative s
// (-0 counts) and stored as rho (c, -s).  Its weights r are taken times rho^l2.  In the backward
// (GRAD) the length is a constant there, so the gradient is that with respect to u alone, along
// u / rho as well as across: with r times rho^(l2 - 1) (0 for l2 = 0, whose Y is a constant) the
// torque is the part across times kMinLength, and s = l2 r / kMinLength gives the part along.
constexpr float kMinLength = 1e-10f;
template <bool GRAD>
__device__ __forceinline__ void mace_frame(const float4& u, float* r, float* s, AlignedFrame& f,
                                           float& c, float& sn) {
    c = u.z;
    sn = u.w;
    const bool tiny = __float_as_int(u.w) < 0;
    if (__any(tiny)) {
        const float rho = tiny ? sqrtf(c * c + sn * sn) : 1.0f;
        if (tiny) {
            c = rho > 0.0f ? c / rho : 1.0f;
            sn = rho > 0.0f ? -sn / rho : 0.0f;
        }
        const float pw[4] = {1.0f, rho, rho * rho, rho * rho * rho};
#pragma unroll
        for (int p = 0; p < kNumPaths; ++p) {
            const int l2 = kPathL[p][1];
            if constexpr (GRAD) {
                r[p] = l2 > 0 ? r[p] * pw[l2 > 0 ? l2 - 1 : 0] : (tiny ? 0.0f : r[p]);
                s[p] = tiny ? (float)l2 * r[p] / kMinLength : s[p];
            } else if (l2 > 0) {
                r[p] *= pw[l2];
            }
        }
    }
    aligned_frame(u.x, u.y, c, sn, f);
}

// One tile's per-position operands (pos clamped into the range by the caller).
struct MaceTileIn {
    v4u hb[3 * kHSteps];
    float4 u;  // direction (mace_frame)
    int s, d;
};

__device__ __forceinline__ void mace_load_tile(const float4* __restrict__ u4,
                                               const int* __restrict__ srcp,
                                               const int* __restrict__ dstp,
                                               const v4u* __restrict__ h, int64_t pos, int kk,
                                               MaceTileIn& t) {
    const v4u* hr = h + pos * kHRow + kk;
#pragma unroll
    for (int j = 0; j < 3 * kHSteps; ++j) t.hb[j] = hr[4 * j];
    t.u = u4[pos];
    t.s = srcp[pos];
    t.d = dstp[pos];
}

// Sum of the tile's messages over each destination, in ascending edge order.
// The 16 x 16 messages of a row (channel) go through LDS so that lane (row, o)
// holds component o of all 16 edges; it adds them one after another into acc,
// restarting at each destination's first edge (the tile's destination pattern
// is the same on every row, so it is one scalar bit mask), and stores acc when a
// destination closes.  acc carries a destination that continues into the next
// tile.  sT: [row (272 floats)][edge (16)][component, in quads rotated by
// edge / 4] (conflict-free 16-byte writes and 4-byte reads).
constexpr int kTRow = 272;
// messages to LDS: lane (row kk, edge e16) writes its 16 components
__device__ __forceinline__ void mace_stage_tile(const float* v, int e16, int kk, float* sT) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(sT + kk * kTRow + e16 * 16 + 4 * ((i + (e16 >> 2)) & 3)) =
            make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}
__device__ __forceinline__ void mace_scatter_tile(int d, bool valid, int e16, int kk, bool cok,
                                                  int64_t c, int C, const float* sT, float& acc,
                                                  int& carry_d, float* __restrict__ out) {
    const int dp = dpp_prev_i(d), dn = dpp_next_i(d);
    const uint64_t head = __ballot((e16 == 0) | (dp != d));
    const uint64_t ends = __ballot(valid & (e16 < 15) & (dn != d));
    const int d0 = __builtin_amdgcn_readfirstlane(d);  // lane 0 of a tile is always valid
    // component o = e16 of row kk for all 16 edges
    float col[16];
#pragma unroll
    for (int e = 0; e < 16; ++e)
        col[e] = sT[kk * kTRow + e * 16 + 4 * (((e16 >> 2) + (e >> 2)) & 3) + (e16 & 3)];
    float* orow = out + c * 16 + e16;  // + destination * C * 16
    if (carry_d >= 0 && d0 != carry_d && cok) orow[(int64_t)carry_d * C * 16] = acc;
    acc = (d0 == carry_d) ? acc + col[0] : col[0];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        if (e > 0) acc = ((head >> e) & 1) ? col[e] : acc + col[e];
        if ((ends >> e) & 1) {
            const int de = __builtin_amdgcn_readlane(d, e);
            if (cok) orow[(int64_t)de * C * 16] = acc;
        }
    }
    carry_d = __builtin_amdgcn_readlane(d, 15);  // -1: the tile's last lane is past the range
}

// Workgroup -> (channel quad, position range): consecutive workgroup ids go to
// consecutive XCDs, so (bid % 8, bid / 8) puts all quads of a position range on one
// XCD, whose L2 then serves the range's h rows to every quad.
struct MaceWg {
    int quad, wave_range;
};
template <int WAVES>
__device__ __forceinline__ MaceWg mace_wg(int n_quads, int ranges_per_xcd) {
    const int bid = blockIdx.x, xcd = bid & 7, k = bid >> 3;
    MaceWg w;
    w.quad = k % n_quads;
    w.wave_range = ((xcd * ranges_per_xcd + k / n_quads) * WAVES) + (threadIdx.x >> 6);
    return w;
}

// out[d, c, :] = sum_{e -> d} sum_p R[e, c, p] T_p(x[src_e, c], Y(u_e)) for every
// destination with an edge (out of the others is zeroed by the caller).
__global__ __launch_bounds__(64 * kMaceFwdWaves) __attribute__((amdgpu_waves_per_eu(4))) void
mace_fused_forward_kernel(const float4* __restrict__ u4, const int* __restrict__ srcp,
                          const int* __restrict__ dstp, const v4u* __restrict__ h,
                          const float* __restrict__ w2, const float* __restrict__ x,
                          const int64_t* __restrict__ wstart, float* __restrict__ out, int C,
                          int n_quads, int ranges_per_xcd) {
    __shared__ v4u sW[kW2Frags * 64];
    __shared__ __attribute__((aligned(16))) float sTAll[kMaceFwdWaves * 4 * kTRow];
    const MaceWg wg = mace_wg<kMaceFwdWaves>(n_quads, ranges_per_xcd);
    const int lane = threadIdx.x & 63, e16 = lane & 15, kk = lane >> 4;
    const int c0 = wg.quad * 4;
    mace_fill_w2(w2, C, c0, sW);
    __syncthreads();
    float* sT = sTAll + (threadIdx.x >> 6) * 4 * kTRow;
    const int64_t p0 = wstart[wg.wave_range], p1 = wstart[wg.wave_range + 1];
    const int c = c0 + kk;
    const bool cok = c < C;
    const int cc = cok ? c : C - 1;
    const v4u* sA = sW + lane;
    int carry_d = -1;
    float acc = 0.0f;
    MaceTileIn cur;
    if (p0 < p1) mace_load_tile(u4, srcp, dstp, h, min(p0 + e16, p1 - 1), kk, cur);
    for (int64_t t0 = p0; t0 < p1; t0 += 16) {
        const bool valid = t0 + e16 < p1;
        if (!valid) {
#pragma unroll
            for (int j = 0; j < 3 * kHSteps; ++j) cur.hb[j] = v4u{0, 0, 0, 0};
        }
        float rr[kNumPaths];
        const v4u* const hp[1] = {cur.hb};
        float* const rp[1] = {rr};
        mace_tile_weights<1>(sA, hp, rp);
        // source row of the pair (after the weights: before them its 16 registers spill;
        // the other waves of the SIMD cover its latency)
        float xs[16];
        load_row16(x + ((int64_t)cur.s * C + cc) * 16, xs);
        AlignedFrame f;
        float c1, s1;
        mace_frame<false>(cur.u, rr, nullptr, f, c1, s1);
        float m[16];
        aligned_message(f, xs, rr, m);
        mace_stage_tile(m, e16, kk, sT);
        const int dcur = valid ? cur.d : -1;
        // the next tile's operands (the other waves of the SIMD cover their latency)
        const int64_t t1 = t0 + 16;
        mace_load_tile(u4, srcp, dstp, h, t1 < p1 ? min(t1 + e16, p1 - 1) : p1 - 1, kk, cur);
        mace_scatter_tile(dcur, valid, e16, kk, cok, c, C, sT, acc, carry_d, out);
    }
    if (carry_d >= 0 && cok) out[((int64_t)carry_d * C + c) * 16 + e16] = acc;
}

// Backward.  The gradient with respect to the length runs back through the MLP as
//   g_r = sum_{c, p} gR[e, c, p] S[e, c, p],   S = s W2   (= dR/dr),
// with gR_p = g . T_p and s[e][k] = silu'(z_k) sum_b W1[b][k] dB_b/dr: the same GEMM as
// R = h W2 on the same operand fragments, consumed where it leaves the accumulators (the
// transpose GEMM of gR needs gR split per tile and a second copy of W2).  The gradient with
// respect to the direction is a torque (aligned_gradient).  Both are summed over the quad's
// channels, and the quad's share of the edge's position gradient,
//   g_v = g_r u + (torque x u) / r,
// goes to gv_part[quad][position].
__global__ __launch_bounds__(64 * kMaceBwdWaves) __attribute__((amdgpu_waves_per_eu(3))) void mace_fused_backward_kernel(
    const float4* __restrict__ u4, const int* __restrict__ srcp, const int* __restrict__ dstp,
    const v4u* __restrict__ h, const v4u* __restrict__ sg, const float* __restrict__ rl,
    const float* __restrict__ w2, const float* __restrict__ x, const float* __restrict__ gout,
    const int64_t* __restrict__ wstart, float* __restrict__ gv_part, int64_t n_pos, int C,
    int n_quads, int ranges_per_xcd) {
    __shared__ v4u sW[kW2Frags * 64];
    const MaceWg wg = mace_wg<kMaceBwdWaves>(n_quads, ranges_per_xcd);
    const int lane = threadIdx.x & 63, e16 = lane & 15, kk = lane >> 4;
    const int c0 = wg.quad * 4;
    mace_fill_w2(w2, C, c0, sW);
    __syncthreads();
    const int64_t p0 = wstart[wg.wave_range], p1 = wstart[wg.wave_range + 1];
    const int c = c0 + kk;
    const bool cok = c < C;
    const int cc = cok ? c : C - 1;
    const v4u* sA = sW + lane;
    float* gvq = gv_part + (int64_t)wg.quad * n_pos * 3;
    MaceTileIn cur;
    v4u sb[3 * kHSteps];
    auto load_s = [&](int64_t pos) {
        const v4u* sr = sg + pos * kHRow + kk;
#pragma unroll
        for (int j = 0; j < 3 * kHSteps; ++j) sb[j] = sr[4 * j];
    };
    if (p0 < p1) {
        const int64_t pos = min(p0 + e16, p1 - 1);
        mace_load_tile(u4, srcp, dstp, h, pos, kk, cur);
        load_s(pos);
    }
    for (int64_t t0 = p0; t0 < p1; t0 += 16) {
        const int64_t pos = t0 + e16;
        const bool valid = pos < p1;
        if (!valid) {
#pragma unroll
            for (int j = 0; j < 3 * kHSteps; ++j) cur.hb[j] = sb[j] = v4u{0, 0, 0, 0};
        }
        float rr[kNumPaths], ss[kNumPaths];
        const v4u* const hp[2] = {cur.hb, sb};
        float* const rp[2] = {rr, ss};
        mace_tile_weights<2>(sA, hp, rp);
        float xs[16], g[16];
        load_row16(x + ((int64_t)cur.s * C + cc) * 16, xs);
        load_row16(gout + ((int64_t)cur.d * C + cc) * 16, g);
        if (!(valid && cok)) {
#pragma unroll
            for (int o = 0; o < 16; ++o) g[o] = 0.0f;
        }
        AlignedFrame f;
        float c1, s1;
        mace_frame<true>(cur.u, rr, ss, f, c1, s1);
        float tx, tz, gr;
        aligned_gradient(f, xs, g, rr, ss, tx, tz, gr);
        // the next tile's operands, in flight during the reductions
        const float cf = cur.u.x, sf = cur.u.y;
        const int64_t t1 = t0 + 16, np = t1 < p1 ? min(t1 + e16, p1 - 1) : p1 - 1;
        mace_load_tile(u4, srcp, dstp, h, np, kk, cur);
        load_s(np);
        // summed over the quad's channels (rows of the wave)
        tx += __shfl_xor(tx, 16, 64);
        tz += __shfl_xor(tz, 16, 64);
        gr += __shfl_xor(gr, 16, 64);
        tx += __shfl_xor(tx, 32, 64);
        tz += __shfl_xor(tz, 32, 64);
        gr += __shfl_xor(gr, 32, 64);
        if (valid && kk == 0) {
            // in the aligned frame the unit vector moves by (-tz, 0, tx): back by the tilt and
            // the turn
            const float ir = 1.0f / rl[pos];
            const float ax = -tz * ir, az = c1 * tx * ir;
            float* o = gvq + pos * 3;
            o[0] = gr * s1 * sf + fmaf(ax, cf, az * sf);
            o[1] = gr * c1 - s1 * tx * ir;
            o[2] = gr * s1 * cf + fmaf(-ax, sf, az * cf);
        }
    }
}

// ---------------------------------------------------------------------------
// Positions: deg[i] = degree of order[i] (then an exclusive scan gives pos0[i]),
// perm[pos0[i] + j] = row_ptr[order[i]] + j.  Writes past n_edges are dropped
// (order must be a permutation of the rows for the layer to be correct; a
// malformed one cannot make these kernels read or write out of bounds).
// ---------------------------------------------------------------------------
__global__ void mace_order_degrees_kernel(const int64_t* __restrict__ row_ptr,
                                          const int64_t* __restrict__ order, int64_t n,
                                          int64_t* __restrict__ deg) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t d = order ? order[i] : i;
    d = d < 0 ? 0 : (d >= n ? n - 1 : d);
    deg[i] = row_ptr[d + 1] - row_ptr[d];
}

__global__ void mace_positions_kernel(const int64_t* __restrict__ row_ptr,
                                      const int64_t* __restrict__ order,
                                      const int64_t* __restrict__ pos0, int64_t n,
                                      int64_t n_edges, int64_t* __restrict__ perm) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int64_t d = order ? order[i] : i;
    d = d < 0 ? 0 : (d >= n ? n - 1 : d);
    const int64_t e0 = row_ptr[d], k = row_ptr[d + 1] - e0, p = pos0[i];
    for (int64_t j = 0; j < k && p + j < n_edges; ++j) perm[p + j] = e0 + j;
}

// wstart[w] = the first position of the first destination that starts at or after
// w * n_edges / n_workers (positions of whole destinations per worker), wstart[n_workers]
// = n_edges.
__global__ void mace_worker_starts_kernel(const int64_t* __restrict__ pos0, int64_t n,
                                          int64_t n_edges, int n_workers,
                                          int64_t* __restrict__ wstart) {
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w > n_workers) return;
    if (w == n_workers) {
        wstart[w] = n_edges;
        return;
    }
    const int64_t target = n_edges * w / n_workers;
    int64_t lo = 0, hi = n;  // smallest i in [0, n] with pos0[i] >= target (pos0[n] = total)
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (pos0[mid] < target) lo = mid + 1;
        else hi = mid;
    }
    wstart[w] = min(pos0[lo], n_edges);
}

// (a, b), of unit length but for rounding, closer to it: the rotations take up to the sixth
// power of what its length is off.
__device__ __forceinline__ void unit2(float& a, float& b) {
    const float big = fmaxf(fabsf(a), fabsf(b)), small = fminf(fabsf(a), fabsf(b));
    const float e = 0.5f * fmaf(-small, small, fmaf(-big, big, 1.0f));
    a = fmaf(a, e, a);
    b = fmaf(b, e, b);
}

// Per position p (edge e = perm[p]): direction (and length), source, destination,
// h = silu(B(r) W1 + b1); with sg, also s[k] = silu'(z_k) sum_b W1[b][k] dB_b/dr.
// Sixteen lanes per position: lane q evaluates Bessel function q % 8 (one sincos)
// and shares it with the position's other lanes, then forms hidden units
// 4q .. 4q + 3, so every store instruction writes whole 128-byte rows.
constexpr int kPrepPositions = 16;  // positions per 256-thread workgroup
__global__ __launch_bounds__(256) void mace_prep_kernel(
    const float* __restrict__ pos, MaceBox bx, const int64_t* __restrict__ src,
    const int64_t* __restrict__ dst, const int64_t* __restrict__ perm,
    const float* __restrict__ w1, const float* __restrict__ b1, float rc, int64_t n_edges,
    float4* __restrict__ u4, int* __restrict__ srcp, int* __restrict__ dstp,
    v4u* __restrict__ h, v4u* __restrict__ sg, float* __restrict__ rl) {
    __shared__ float sW[kNBasis * kHidden + kHidden];
    for (int i = threadIdx.x; i < kNBasis * kHidden + kHidden; i += blockDim.x)
        sW[i] = i < kNBasis * kHidden ? w1[i] : b1[i - kNBasis * kHidden];
    __syncthreads();
    const int q = threadIdx.x & 15;
    int64_t p = (int64_t)blockIdx.x * kPrepPositions + (threadIdx.x >> 4);
    const bool valid = p < n_edges;
    p = valid ? p : n_edges - 1;  // every lane takes part in the shuffles below
    int64_t e = perm[p];
    e = e < 0 ? 0 : (e >= n_edges ? n_edges - 1 : e);
    const int64_t s = src[e], d = dst[e];
    float v[3];
    edge_vector(pos, s, d, bx.box, bx.inv, v);
    const float r = normalize3(v[0], v[1], v[2]);
    if (valid && q == 0) {
        // direction (aligned.h): u = (s sin f, c, s cos f); along the axis any turn serves.
        // The off-axis part is scaled before it is squared: below 1e-19 its square is
        // subnormal, and (cos f, sin f) would not be of unit length.
        const float m = fmaxf(fabsf(v[0]), fabsf(v[2]));
        float cf = 1.0f, sf = 0.0f, c = v[1], s2 = fabsf(v[0] + v[2]);  // (0, or NaN)
        if (m > 0.0f) {
            sf = v[0] / m;
            cf = v[2] / m;
            const float h = sqrtf(cf * cf + sf * sf), ih = 1.0f / h;
            sf *= ih;
            cf *= ih;
            s2 = m * h;
        }
        if (r <= kMinLength) {  // (marked: mace_frame; also a NaN, which stays one)
            if (s2 < 1e-15f && fabsf(c) < 1e-15f) c = s2 = 0.0f;  // (its square is subnormal)
            s2 = copysignf(s2, -1.0f);
        } else {
            unit2(c, s2);
        }
        unit2(cf, sf);
        u4[p] = make_float4(cf, sf, c, s2);
        srcp[p] = (int)s;
        dstp[p] = (int)d;
        if (rl) rl[p] = r;
    }
    // Bessel function k = q % 8 of this position, with the envelope
    const float dd = r / rc;
    float f = 0.f, df = 0.f;
    if (dd < 1.0f) {
        const float d5 = dd * dd * dd * dd * dd, d6 = d5 * dd;
        f = 1.0f - 28.0f * d6 + 48.0f * d6 * dd - 21.0f * d6 * dd * dd;
        const float om = 1.0f - dd;
        df = -168.0f * d5 * om * om / rc;
    }
    const float norm = sqrtf(2.0f / rc), ir = 1.0f / r;
    const float w = (float)((q & 7) + 1) * 3.14159265358979323846f / rc;
    float sn, cs;
    sincosf(w * r, &sn, &cs);
    const float gk = norm * sn * ir;
    const float bk = gk * f;
    const float dbk = sg ? (norm * (w * cs * ir - sn * ir * ir)) * f + gk * df : 0.0f;
    const int base = (threadIdx.x & 63) & ~15;
    float B[kNBasis], dB[kNBasis];
#pragma unroll
    for (int k = 0; k < kNBasis; ++k) B[k] = __shfl(bk, base + k, 64);
    if (sg) {
#pragma unroll
        for (int k = 0; k < kNBasis; ++k) dB[k] = __shfl(dbk, base + k, 64);
    }
    float z[4], sd[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int j = 4 * q + t;
        float acc = sW[kNBasis * kHidden + j];
#pragma unroll
        for (int k = 0; k < kNBasis; ++k) acc = fmaf(B[k], sW[k * kHidden + j], acc);
        const float sgm = sigmoidf(acc);
        z[t] = acc * sgm;
        if (sg) {
            float qq = 0.0f;
#pragma unroll
            for (int k = 0; k < kNBasis; ++k) qq = fmaf(sW[k * kHidden + j], dB[k], qq);
            sd[t] = sgm * (1.0f + acc * (1.0f - sgm)) * qq;
        }
    }
    // h and s in three bf16 parts, [part][k] (hidden units 4q .. 4q + 3 of each part here)
    auto store = [&](v4u* row, const float* v) {
        const float v8[8] = {v[0], v[1], v[2], v[3], 0.f, 0.f, 0.f, 0.f};
        const Bf3 b = bf16_split8(v8);
        if (!valid) return;
        uint2* o = reinterpret_cast<uint2*>(row) + q;
        o[0] = make_uint2(b.h[0], b.h[1]);
        o[kHidden / 4] = make_uint2(b.m[0], b.m[1]);
        o[kHidden / 2] = make_uint2(b.l[0], b.l[1]);
    };
    store(h + p * kHRow, z);
    if (sg) store(sg + p * kHRow, sd);
}

// out rows of destinations without edges (the fused kernel writes the others)
__global__ void mace_zero_empty_rows_kernel(const int64_t* __restrict__ row_ptr, int64_t n,
                                            int C, float4* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t per = (int64_t)C * 4;
    if (i >= n * per) return;
    const int64_t d = i / per;
    if (row_ptr[d + 1] == row_ptr[d]) out[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// g_v[perm[p]] = sum over the channel quads, in order, of gv_part[quad][p]
__global__ void mace_gv_reduce_kernel(const float* __restrict__ gv_part,
                                      const int64_t* __restrict__ perm, int64_t n_edges,
                                      int n_quads, float* __restrict__ gv) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_edges) return;
    float a = 0.f, b = 0.f, c = 0.f;
    for (int q = 0; q < n_quads; ++q) {
        const float* s = gv_part + ((int64_t)q * n_edges + p) * 3;
        a += s[0];
        b += s[1];
        c += s[2];
    }
    int64_t e = perm[p];
    e = e < 0 ? 0 : (e >= n_edges ? n_edges - 1 : e);
    gv[e * 3 + 0] = a;
    gv[e * 3 + 1] = b;
    gv[e * 3 + 2] = c;
}

__global__ void mace_fill_zero_kernel(float* __restrict__ p, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) p[i] = 0.0f;
}

__global__ void mace_zero_int_kernel(int* __restrict__ p) { *p = 0; }

// Workspace of one pass (per-position arrays; the backward adds s, the quads'
// gradient shares and the per-edge gradient).
struct MaceWs {
    int64_t *deg, *pos0, *perm, *wstart;
    float4* u4;
    int *srcp, *dstp;
    v4u *h, *sg;
    float *rl, *gv_part, *gv;
    size_t bytes;
};

static size_t a256(size_t x) { return (x + 255) & ~size_t(255); }

static int mace_quads(int C) { return (int)ceil_div(C, 4); }

static MaceWs mace_ws(void* base, int64_t N, int64_t E, int C, bool backward) {
    char* p = static_cast<char*>(base);
    size_t o = 0;
    MaceWs w{};
    auto take = [&](size_t bytes) {
        void* r = p ? static_cast<void*>(p + o) : nullptr;
        o = a256(o + bytes);
        return r;
    };
    const size_t e = (size_t)std::max<int64_t>(E, 1);
    w.deg = static_cast<int64_t*>(take(sizeof(int64_t) * (size_t)std::max<int64_t>(N, 1)));
    w.pos0 = static_cast<int64_t*>(take(sizeof(int64_t) * (size_t)(N + 1)));
    w.perm = static_cast<int64_t*>(take(sizeof(int64_t) * e));
    w.wstart = static_cast<int64_t*>(take(sizeof(int64_t) * (kMaceMaxWorkers + 1)));
    w.u4 = static_cast<float4*>(take(sizeof(float4) * e));
    w.srcp = static_cast<int*>(take(sizeof(int) * e));
    w.dstp = static_cast<int*>(take(sizeof(int) * e));
    w.h = static_cast<v4u*>(take(sizeof(v4u) * kHRow * e));
    if (backward) {
        w.sg = static_cast<v4u*>(take(sizeof(v4u) * kHRow * e));
        w.rl = static_cast<float*>(take(sizeof(float) * e));
        w.gv_part = static_cast<float*>(take(sizeof(float) * 3 * e * (size_t)mace_quads(C)));
        w.gv = static_cast<float*>(take(sizeof(float) * 3 * e));
    }
    w.bytes = o;
    return w;
}

static int gemm_launch(const float* A, const float* B, float* Cm, int64_t M, int N, int K, bool tb,
                       hipStream_t s) {
    if (M <= 0 || N <= 0 || K <= 0) return BM_OK;
    const bool narrow = N <= 64;  // 128 x 64 tiles for narrow outputs, else 128 x 128
    const int bn = narrow ? 64 : 128;
    dim3 grid((unsigned)ceil_div(N, bn), (unsigned)ceil_div(M, 128));
    if (grid.y > 65535) return BM_ERR_ARG;
    if (tb) {
        if (narrow) gemm_f32_kernel<true, 64><<<grid, 256, 0, s>>>(A, B, Cm, (int)M, N, K);
        else gemm_f32_kernel<true, 128><<<grid, 256, 0, s>>>(A, B, Cm, (int)M, N, K);
    } else {
        if (narrow) gemm_f32_kernel<false, 64><<<grid, 256, 0, s>>>(A, B, Cm, (int)M, N, K);
        else gemm_f32_kernel<false, 128><<<grid, 256, 0, s>>>(A, B, Cm, (int)M, N, K);
    }
    return (int)hipGetLastError();
}

// Compute units of the current device.
static int mace_cu_count() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        n = 256;
    return n;
}

// Launch shape of a fused kernel: every quad of a position range on one XCD.  The
// workgroups of an XCD, ranges x quads, run in rounds of its resident ones (occupancy
// from the runtime for this kernel).  A round fills the workgroup's W2 fragments, which
// takes about as long as a tile of each wave (7 to 8 us), and then the wave's share of the
// tiles, so the time goes as rounds (1 + tiles / waves).  The ranges are the fewest that
// bring it within 5% of the least over the first eight counts from one full round on.
// C = 80 (20 quads on 32 slots): one range leaves 12 slots idle, three fill 60 of 64, from
// 7,600 edges on.  C = 112 (28 quads): eight ranges fill seven rounds; by rounds / ranges
// alone they were taken at any size, us forward with them / now at 60, 1,000 and 4,000
// atoms of 30 edges: 92 / 48, 170 / 139, 425 / 401.
struct MaceShape {
    int n_quads, ranges_per_xcd, n_workers;
    unsigned grid;
};

template <typename K>
static int mace_shape(K kernel, int waves, int C, int64_t n_edges, MaceShape* sh) {
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, 64 * waves, 0) != hipSuccess ||
        occ < 1)
        occ = 1;
    const int per_xcd = std::max(1, mace_cu_count() / 8);
    sh->n_quads = mace_quads(C);
    const int slots = per_xcd * occ, first = std::max(1, slots / sh->n_quads);
    const int last = std::min(first + 7, kMaceMaxWorkers / (8 * waves));
    const double tiles = (double)ceil_div(n_edges, 16);
    auto cost = [&](int r) {
        return ceil_div((int64_t)r * sh->n_quads, slots) * (1.0 + tiles / (8.0 * r * waves));
    };
    int best = first;
    for (int r = first + 1; r <= last; ++r)
        if (cost(r) < 0.95 * cost(best)) best = r;
    sh->ranges_per_xcd = best;
    sh->n_workers = 8 * sh->ranges_per_xcd * waves;
    if (sh->n_workers > kMaceMaxWorkers) return BM_ERR_ARG;
    sh->grid = (unsigned)(8 * sh->ranges_per_xcd * sh->n_quads);
    return BM_OK;
}

// Positions (destinations in `order`, each destination's edges ascending), the
// workers' ranges, and the per-position operands.
static int mace_prepare(const float* positions, const MaceBox& bx, const float* w1,
                        const float* b1, const int64_t* src, const int64_t* dst,
                        const int64_t* row_ptr, const int64_t* order, int64_t N, int64_t E,
                        float cutoff, const MaceShape& sh, const MaceWs& w, bool backward,
                        hipStream_t stream) {
    const unsigned nb = (unsigned)ceil_div(N, 256);
    mace_order_degrees_kernel<<<nb, 256, 0, stream>>>(row_ptr, order, N, w.deg);
    int rc = batteries_exclusive_scan_i64(w.deg, w.pos0, N, stream);
    if (rc != BM_OK) return rc;
    mace_positions_kernel<<<nb, 256, 0, stream>>>(row_ptr, order, w.pos0, N, E, w.perm);
    mace_worker_starts_kernel<<<(unsigned)ceil_div(sh.n_workers + 1, 256), 256, 0, stream>>>(
        w.pos0, N, E, sh.n_workers, w.wstart);
    mace_prep_kernel<<<(unsigned)ceil_div(E, kPrepPositions), 256, 0, stream>>>(
        positions, bx, src, dst, w.perm, w1, b1, cutoff, E, w.u4, w.srcp, w.dstp, w.h,
        backward ? w.sg : nullptr, backward ? w.rl : nullptr);
    return (int)hipGetLastError();
}

}  // namespace bmhip

using namespace bmhip;

extern "C" int batteries_gemm_f32(const float* A, const float* B, float* C, int64_t M, int N, int K,
                                  int trans_b, hipStream_t stream) {
    if (M < 0 || N < 0 || K < 0 || M > INT32_MAX) return BM_ERR_ARG;
    return gemm_launch(A, B, C, M, N, K, trans_b != 0, stream);
}

extern "C" size_t batteries_mace_workspace_bytes(int64_t N, int64_t N_edges, int C, int backward) {
    if (N < 0 || N_edges < 0 || C <= 0) return 0;
    return mace_ws(nullptr, N, N_edges, C, backward != 0).bytes;
}

extern "C" int batteries_mace_reverse_edges(const int64_t* row_ptr, const int64_t* src,
                                            int64_t* rev, int* d_missing, int64_t N,
                                            int64_t N_edges, hipStream_t stream) {
    if (N < 0 || N_edges < 0 || !d_missing) return BM_ERR_ARG;
    mace_zero_int_kernel<<<1, 1, 0, stream>>>(d_missing);
    if (N_edges == 0) return (int)hipGetLastError();
    mace_reverse_edges_kernel<<<(unsigned)ceil_div(N_edges, 256), 256, 0, stream>>>(
        row_ptr, src, rev, d_missing, N, N_edges);
    return (int)hipGetLastError();
}

static bool mace_args_ok(const float* box, int64_t N, int64_t E, int C, float cutoff) {
    if (!box || N < 0 || E < 0 || C <= 0 || C > 256 || !(cutoff > 0.0f)) return false;
    if (N > INT32_MAX || E > INT32_MAX) return false;  // int32 indices per position
    for (int k = 0; k < 3; ++k)
        if (!(box[k] > 0.0f)) return false;
    return true;
}

static MaceBox mace_box(const float* box) {
    MaceBox b;
    for (int k = 0; k < 3; ++k) {
        b.box[k] = box[k];
        b.inv[k] = 1.0f / box[k];
    }
    return b;
}

extern "C" int batteries_mace_forward(const float* positions, const float* box,
                                      const float* node_features, const float* w1,
                                      const float* b1, const float* w2, const int64_t* src,
                                      const int64_t* dst, const int64_t* row_ptr,
                                      const int64_t* order, float* out, int64_t N,
                                      int64_t N_edges, int C, float cutoff, void* workspace,
                                      size_t workspace_bytes, hipStream_t stream) {
    if (!mace_args_ok(box, N, N_edges, C, cutoff)) return BM_ERR_ARG;
    if (N == 0) return BM_OK;
    if ((reinterpret_cast<uintptr_t>(node_features) | reinterpret_cast<uintptr_t>(out)) & 15)
        return BM_ERR_ARG;
    const MaceWs w = mace_ws(workspace, N, N_edges, C, false);
    if (!workspace || workspace_bytes < w.bytes) return BM_ERR_WORKSPACE;
    const int64_t n4 = N * (int64_t)C * 4;
    mace_zero_empty_rows_kernel<<<(unsigned)ceil_div(n4, 256), 256, 0, stream>>>(
        row_ptr, N, C, reinterpret_cast<float4*>(out));
    if (N_edges == 0) return (int)hipGetLastError();
    MaceShape sh;
    int rc = mace_shape(mace_fused_forward_kernel, kMaceFwdWaves, C, N_edges, &sh);
    if (rc != BM_OK) return rc;
    rc = mace_prepare(positions, mace_box(box), w1, b1, src, dst, row_ptr, order, N, N_edges,
                      cutoff, sh, w, false, stream);
    if (rc != BM_OK) return rc;
    mace_fused_forward_kernel<<<sh.grid, 64 * kMaceFwdWaves, 0, stream>>>(w.u4, w.srcp, w.dstp, w.h, w2,
                                                            node_features, w.wstart, out, C,
                                                            sh.n_quads, sh.ranges_per_xcd);
    return (int)hipGetLastError();
}

extern "C" int batteries_mace_backward(const float* positions, const float* box,
                                       const float* node_features, const float* w1,
                                       const float* b1, const float* w2, const int64_t* src,
                                       const int64_t* dst, const int64_t* row_ptr,
                                       const int64_t* order, const int64_t* rev,
                                       const float* grad_out, float* grad_pos, int64_t N,
                                       int64_t N_edges, int C, float cutoff, void* workspace,
                                       size_t workspace_bytes, hipStream_t stream) {
    if (!mace_args_ok(box, N, N_edges, C, cutoff)) return BM_ERR_ARG;
    if (N == 0) return BM_OK;
    if ((reinterpret_cast<uintptr_t>(node_features) | reinterpret_cast<uintptr_t>(grad_out)) & 15)
        return BM_ERR_ARG;
    const MaceWs w = mace_ws(workspace, N, N_edges, C, true);
    if (!workspace || workspace_bytes < w.bytes) return BM_ERR_WORKSPACE;
    if (N_edges == 0) {
        mace_fill_zero_kernel<<<(unsigned)ceil_div(N * 3, 256), 256, 0, stream>>>(grad_pos, N * 3);
        return (int)hipGetLastError();
    }
    MaceShape sh;
    int rc = mace_shape(mace_fused_backward_kernel, kMaceBwdWaves, C, N_edges, &sh);
    if (rc != BM_OK) return rc;
    rc = mace_prepare(positions, mace_box(box), w1, b1, src, dst, row_ptr, order, N, N_edges,
                      cutoff, sh, w, true, stream);
    if (rc != BM_OK) return rc;
    mace_fused_backward_kernel<<<sh.grid, 64 * kMaceBwdWaves, 0, stream>>>(
        w.u4, w.srcp, w.dstp, w.h, w.sg, w.rl, w2, node_features, grad_out, w.wstart, w.gv_part,
        N_edges, C, sh.n_quads, sh.ranges_per_xcd);
    mace_gv_reduce_kernel<<<(unsigned)ceil_div(N_edges, 256), 256, 0, stream>>>(
        w.gv_part, w.perm, N_edges, sh.n_quads, w.gv);
    mace_forces_kernel<<<(unsigned)ceil_div(N, 256), 256, 0, stream>>>(w.gv, row_ptr, rev, grad_pos,
                                                                        N);
    return (int)hipGetLastError();
}
