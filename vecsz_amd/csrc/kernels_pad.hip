// Pad values of the padding modes (src/utils/padding.hh; src/dualquant.hh:36-46,
// :226-246, :553-573; src/vecsz_interface.hh:70-90, :287-298).
//
//   k_pad_blocks     the blocks of the reference's block grid ((d + B + 1) / B
//                    blocks per dimension, src/dimensions.hh:31):
//                    find_pad_value over the block (block mode) or over its
//                    first row / column / planes (edge mode), in the
//                    reference's loop order, then the block_pad / edge_pad
//                    prequantization; 1D keeps the raw value
//   k_pad_global_mm  max / min of the field ignoring NaN, and the first index
//                    holding a zero (the sign of a zero extreme)
//   k_pad_global_sum find_avg's float running sum: one wavefront adds the
//                    field in index order, since float addition is not
//                    associative and the reference's sum is sequential
//   k_pad_global_fin the global pad constant, stored and used values
//   k_pad_halo       decompress: halo values from an archive's pad section
//
// Elements outside the field read as +0.0 (the reference reads its
// uninitialised block buffer there).
#include "common.hpp"
#include "kernels.hpp"

namespace vsz {

namespace {

// find_max / find_min / find_avg (src/utils/padding.hh:65-119) as a running
// fold in the reference's order: max / min keep the first value and replace
// it by a strictly larger / smaller one; avg sums in float.  add(): the next
// n values, `stride` apart.
struct Find {
    int type;
    float m;
    bool first;
    __device__ explicit Find(int t) : type(t), m(0.f), first(true) {}
    __device__ __forceinline__ void add(const float* v, uint32_t n, uint32_t stride) {
        if (first && type != kPadAvg) m = v[0];
        first = false;
        if (type == kPadMax) {
#pragma unroll 8
            for (uint32_t s = 0; s < n; s++) m = (v[s * stride] > m) ? v[s * stride] : m;
        } else if (type == kPadMin) {
#pragma unroll 8
            for (uint32_t s = 0; s < n; s++) m = (v[s * stride] < m) ? v[s * stride] : m;
        } else {
#pragma unroll 32
            for (uint32_t s = 0; s < n; s++) m = m + v[s * stride];
        }
    }
    __device__ __forceinline__ float result(uint64_t count, float constant) const {
        return type == kPadConst ? constant : type == kPadAvg ? m / (float)count : m;
    }
};

// block_pad / edge_pad prequantization (src/utils/padding.hh:219-220,
// :236-237, :259-263): scaled in double, stored to float, rounded half away.
__device__ __forceinline__ float pad_q_block(float p, double r_d) {
    const float t = (float)((double)p * r_d);
    return (float)__builtin_round((double)t);
}

__device__ __forceinline__ double pad_rd(const PadArgs& a) { return a.ebd ? a.ebd->r_d : a.r_d; }

}  // namespace

// One pad value is a fold over a sequence of L = B, B^2 or B^3 elements (a
// power of two): the block's elements in block mode, and in edge mode
// blockIdx.y picks one of
//   2D (find_edge_pad_value, src/utils/padding.hh:145-206): the first row, the
//      first column; halo (i == 0) ? row value : column value
//   3D: the z = 0 plane (x fastest), the x = 0 plane (y fastest), the y = 0
//      plane (x fastest); halo (k == 0) ? p0 : (j == 0) ? p1 : p2
// avg adds in float, so a sequence's order is fixed and its fold is one
// lane's chain.  What can be spread is the reading: a workgroup takes
// kPadTile / S blocks and stages S = min(L, 256) elements of each per round
// (x fastest: whole row pieces of B floats per load), the next round's loads
// in flight while one lane per block folds this round's out of LDS.  A thread
// that read its own block's elements waited for memory on each
// (201 x 333 x 413, B 16, block avg: 1033 -> 74 us).
constexpr uint32_t kPadTile = 4096;
constexpr uint32_t kPadPer = kPadTile / 256;  // loads per thread and round
constexpr uint32_t kPadLgMaxS = 8, kPadMaxS = 1u << kPadLgMaxS;

__global__ void __launch_bounds__(256) k_pad_blocks(PadArgs a, uint32_t lb, uint32_t lS, uint64_t L, uint32_t nseq,
                                                    float* __restrict__ pad_out, float* __restrict__ halo) {
    __shared__ float tile[kPadTile + kPadMaxS];  // element s of block g at s * (G + 1) + g
    const uint32_t B = 1u << lb, S = 1u << lS, G = kPadTile >> lS, t = threadIdx.x, face = blockIdx.y;
    const uint64_t nb = a.hb0 * a.hb1 * a.hb2, id0 = (uint64_t)blockIdx.x * G;
    const uint64_t sy = a.d0, sz = a.d0 * a.d1;
    // Element s of a sequence is (p0, p1, p2) in base B; a round's first s is a
    // multiple of S, so its part of p1 and p2 is one for the workgroup and a
    // thread's loads keep their own: an offset, and how many rows and planes
    // from there the field has (0: a block that starts past the field).
    // (A thread's loads are 256 apart and S divides 256, so they share s.)
    const uint32_t s = t & (S - 1), p0 = s & (B - 1), p1 = s >> lb & (B - 1), p2 = s >> (2 * lb);
    const bool edge = nseq > 1, yz = edge && face > 0;  // yz: p1 counts planes
    uint64_t off[kPadPer];
    uint32_t ny[kPadPer], nz[kPadPer];
#pragma unroll
    for (uint32_t m = 0; m < kPadPer; m++) {
        uint32_t i = p0, j = p1, k = p2;
        if (edge && face == 1) i = 0, j = p0, k = p1;
        if (edge && face == 2) j = 0, k = p1;
        const uint64_t id = id0 + ((t + 256 * m) >> lS);
        const uint64_t x = id % a.hb0 * B + i, y = id / a.hb0 % a.hb1 * B + j, z = id / (a.hb0 * a.hb1) * B + k;
        off[m] = x + y * sy + z * sz;
        const bool in = id < nb && x < a.d0 && y < a.d1 && z < a.d2;
        ny[m] = in ? (uint32_t)min<uint64_t>(a.d1 - y, B) : 0u;
        nz[m] = in ? (uint32_t)min<uint64_t>(a.d2 - z, B) : 0u;
    }
    float v[kPadPer];
    auto fetch = [&](uint64_t s0) {
        const uint32_t r1 = (uint32_t)(s0 >> lb) & (B - 1), r2 = (uint32_t)(s0 >> (2 * lb));
        const uint32_t yr = yz ? 0 : r1, zr = yz ? r1 : r2;
        const float* src = a.x + yr * sy + zr * sz;
#pragma unroll
        for (uint32_t m = 0; m < kPadPer; m++) {
            v[m] = 0.f;
            if (yr < ny[m] && zr < nz[m]) v[m] = src[off[m]];
        }
    };
    // a thread folds block t, and block t + 256 where there are as many
    Find f0(a.type), f1(a.type);
    if (a.type != kPadConst) {
        fetch(0);
        for (uint64_t s0 = 0; s0 < L; s0 += S) {
            lds_sync();
#pragma unroll
            for (uint32_t m = 0; m < kPadPer; m++) {
                tile[s * (G + 1) + ((t + 256 * m) >> lS)] = v[m];
            }
            lds_sync();
            if (s0 + S < L) fetch(s0 + S);
            if (t < G) f0.add(tile + t, S, G + 1);
            if (t + 256 < G) f1.add(tile + t + 256, S, G + 1);
        }
    }
    const double rd = pad_rd(a);
    for (uint32_t g = t; g < G; g += 256) {
        const uint64_t id = id0 + g;
        if (id >= nb) break;
        float p = (g == t ? f0 : f1).result(L, a.constant);
        if (a.ndim > 1) p = pad_q_block(p, rd);  // (1D keeps the raw value, src/dualquant.hh:37-42)
        pad_out[nseq * id + face] = p;
        if (nseq == 1) {
            halo[3 * id] = halo[3 * id + 1] = halo[3 * id + 2] = p;
        } else if (nseq == 2) {
            halo[3 * id + (face == 0 ? 2 : 1)] = p;
            if (face == 0) halo[3 * id] = 0.f;
        } else {
            halo[3 * id + face] = p;
        }
    }
}

// scratch: [0] ordered max, [1] ordered min (u32), [2..3] first zero index (u64)
__device__ __forceinline__ uint32_t f2ord_p(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f_p(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

__global__ void k_pad_global_init(uint32_t* s) {
    if (threadIdx.x == 0) {
        s[0] = 0u;
        s[1] = 0xFFFFFFFFu;
        reinterpret_cast<unsigned long long*>(s)[1] = ~0ull;
        reinterpret_cast<float*>(s)[4] = 0.f;
    }
}

__global__ void __launch_bounds__(256) k_pad_global_mm(const float* __restrict__ x, uint64_t n, uint32_t* s) {
    uint32_t mx = 0u, mn = 0xFFFFFFFFu;
    unsigned long long z = ~0ull;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += stride) {
        const float v = x[i];
        if (v == v) {
            const uint32_t o = f2ord_p(v);
            mx = o > mx ? o : mx;
            mn = o < mn ? o : mn;
        }
        if (v == 0.f && i < z) z = i;
    }
    for (int d = 32; d > 0; d >>= 1) {
        const uint32_t a = __shfl_xor(mx, d), b = __shfl_xor(mn, d);
        const unsigned long long c = __shfl_xor(z, d);
        mx = a > mx ? a : mx;
        mn = b < mn ? b : mn;
        z = c < z ? c : z;
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(&s[0], mx);
        atomicMin(&s[1], mn);
        atomicMin(reinterpret_cast<unsigned long long*>(s) + 1, z);
    }
}

// find_avg over the whole field (src/utils/padding.hh:101-119): the float
// running sum in index order, on one wavefront.  Lanes load 64 consecutive
// values at a time; every lane then adds them in order (the same scalar
// chain in each lane), the next batch's loads already in flight.
__global__ void __launch_bounds__(64) k_pad_global_sum(const float* __restrict__ x, uint64_t n, uint32_t* s) {
    constexpr int U = 16;
    const uint32_t lane = threadIdx.x;
    float sum = 0.f;
    float cur[U], nxt[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint64_t i = (uint64_t)u * 64 + lane;
        cur[u] = i < n ? x[i] : 0.f;
    }
    for (uint64_t base = 0; base < n; base += 64 * U) {
        const uint64_t nb = base + 64 * U;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint64_t i = nb + (uint64_t)u * 64 + lane;
            nxt[u] = i < n ? x[i] : 0.f;
        }
        const uint64_t left = n - base;
        if (left >= 64 * U) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int k = 0; k < 64; k++)
                    sum = sum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cur[u]), k));
        } else {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int k = 0; k < 64; k++) {
                    const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cur[u]), k));
                    if ((uint64_t)u * 64 + k < left) sum = sum + v;
                }
        }
#pragma unroll
        for (int u = 0; u < U; u++) cur[u] = nxt[u];
    }
    if (lane == 0) reinterpret_cast<float*>(s)[4] = sum;
}

// The global constant (src/vecsz_interface.hh:73-80): find_pad_value over the
// field; stored as round(c * ebx2_r) in double, and used by the 2D/3D blocks
// through block_pad with CONST_VAL, by 1D as the stored value
// (src/dualquant.hh:43-46).
__global__ void k_pad_global_fin(PadArgs a, const uint32_t* s, float* pad_out, float* halo) {
    if (threadIdx.x != 0) return;
    float c;
    if (a.type == kPadConst) {
        c = a.constant;
    } else if (a.type == kPadAvg) {
        c = reinterpret_cast<const float*>(s)[4] / (float)a.n;
    } else {
        const float x0 = a.x[0];
        if (x0 != x0) {
            c = x0;  // nothing compares greater or smaller than a leading NaN
        } else {
            c = ord2f_p(a.type == kPadMax ? s[0] : s[1]);
            // equal values keep the first one: only zeros differ in bits
            if (c == 0.f) c = a.x[reinterpret_cast<const unsigned long long*>(s)[1]];
        }
    }
    const double rd = pad_rd(a);
    const float stored = (float)__builtin_round((double)c * rd);
    const float used = a.ndim == 1 ? stored : pad_q_block(c, rd);
    pad_out[0] = stored;
    halo[0] = halo[1] = halo[2] = used;
}

// Halo values from an archive's pad section (x_block_pad / x_edge_pad,
// src/utils/padding.hh:302-372; src/dualquant.hh:918-927, :951-964,
// :1003-1016; mode from the count, src/vecsz_interface.hh:287-298).
__global__ void __launch_bounds__(256) k_pad_halo(int ndim, int mode, const float* __restrict__ pad, uint64_t pad_len,
                                                  uint64_t nblocks, float* __restrict__ halo) {
    const uint64_t b = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    float hz = 0.f, hy = 0.f, hx = 0.f;
    if (mode == kPadGlobal) {
        hz = hy = hx = pad[0];
    } else if (mode == kPadBlock) {
        hz = hy = hx = pad[b];
    } else if (mode == kPadEdge) {
        if (ndim == 2) {
            hx = pad[2 * b];
            hy = pad[2 * b + 1];
        } else {
            hz = pad[3 * b];
            hy = pad[3 * b + 1];
            hx = pad[3 * b + 2];
        }
    } else if (ndim == 1 && pad_len > 0) {
        hz = hy = hx = pad[0];  // x_lorenzo_1d1l's pad_vals[0] without a mode
    }
    halo[3 * b] = hz;
    halo[3 * b + 1] = hy;
    halo[3 * b + 2] = hx;
}

void launch_pad_blocks(const PadArgs& a, float* pad_out, float* halo, hipStream_t st) {
    const uint64_t nb = a.hb0 * a.hb1 * a.hb2;
    const uint32_t nseq = a.mode == kPadEdge && a.ndim > 1 ? (uint32_t)a.ndim : 1u;
    const uint32_t lb = (uint32_t)__builtin_ctz((unsigned)a.B);
    // block mode: B^ndim elements; edge mode: B^(ndim - 1) (1D: as block mode)
    const uint32_t lL = lb * (uint32_t)(nseq == 1 ? a.ndim : a.ndim - 1);
    const uint32_t lS = std::min(lL, kPadLgMaxS);
    const uint64_t G = kPadTile >> lS;
    hipLaunchKernelGGL(k_pad_blocks, dim3((unsigned)((nb + G - 1) / G), nseq), dim3(256), 0, st, a, lb, lS, 1ull << lL,
                       nseq, pad_out, halo);
}

void launch_pad_global(const PadArgs& a, void* scratch, float* pad_out, float* halo, hipStream_t st) {
    uint32_t* s = static_cast<uint32_t*>(scratch);
    hipLaunchKernelGGL(k_pad_global_init, dim3(1), dim3(64), 0, st, s);
    if (a.type == kPadMax || a.type == kPadMin) {
        const unsigned g = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((a.n + 1023) / 1024, 2048));
        hipLaunchKernelGGL(k_pad_global_mm, dim3(g), dim3(256), 0, st, a.x, a.n, s);
    } else if (a.type == kPadAvg) {
        hipLaunchKernelGGL(k_pad_global_sum, dim3(1), dim3(64), 0, st, a.x, a.n, s);
    }
    hipLaunchKernelGGL(k_pad_global_fin, dim3(1), dim3(64), 0, st, a, s, pad_out, halo);
}

void launch_pad_halo(int ndim, int mode, const float* pad, uint64_t pad_len, uint64_t nblocks, float* halo,
                     hipStream_t st) {
    hipLaunchKernelGGL(k_pad_halo, dim3((unsigned)((nblocks + 255) / 256)), dim3(256), 0, st, ndim, mode, pad,
                       pad_len, nblocks, halo);
}

}  // namespace vsz
