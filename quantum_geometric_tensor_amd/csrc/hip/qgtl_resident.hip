// Derivative states of small circuits (4 <= n <= 13) in one launch: every
// state lives in the LDS of one workgroup from |0..0> to the end of the
// circuit.
//
// A workgroup evolves the primal state through all blocks (the U-layer's 2x2
// matrices, then the M-stage's index permutation); after the block that holds
// its parameter it replaces the state by the parameter's derivative
// (injection, with the FP64 sums <d|psi>, |d|^2, |psi|^2) and carries that
// through the remaining blocks.  One more workgroup's state is never replaced:
// the primal state itself.  Nothing but the final states is written to memory
// and no state is read, where the pass kernels of the wider circuits write and
// read every state once per block and need two or three launches per block.
//
// Repeating the primal evolution in every workgroup costs less than the chain
// it replaces: all workgroups run at once (P + 1 <= 256 CUs for up to nine
// layers at n = 13), so the call takes one circuit's latency instead of 2 L
// dependent launches.  Kernel time of one call, before (passes, injections and
// their reductions) and now: n = 13, L = 6 (P = 156) 579 -> 44 us; n = 10,
// L = 4 (P = 80) 99 -> 18 us; n = 6, L = 3 (P = 36) 50 -> 11 us; the whole
// Plan.set_angles + execute 701 -> 117, 184 -> 65 and 126 -> 45 us (with what else changed around it).
//
// Work split: 16 amplitudes per thread (four tile bits in registers, 2^(n-4)
// threads), so a block is ceil(n / 4) LDS round trips of four gates each.
// Below n = 10 one wave holds 2^(10-n) states.  What bounds it: the latency of
// one wave's dependent steps (LDS round trips) at n <= 10,
// LDS traffic (2 x 64 KB per round trip) and the gates' multiply-adds at n = 13.
//
// QGTL counterpart: the shifted-circuit evaluations of
// src/quantum_geometric/core/quantum_geometric_gradient.c:2356-2366, one
// circuit run per parameter.
#include "qgtl_hip_common.h"

namespace {

// LDS word of tile element j (complex64 words): bits 0..3 XORed with bits 4..7,
// 8..11 and 12.  Linear over GF(2); with four contiguous register bits every
// access of 16 lanes hits 16 distinct 8-byte banks.
__device__ __forceinline__ uint32_t rpad(uint32_t j) { return j ^ (((j >> 4) ^ (j >> 8) ^ (j >> 12)) & 15u); }

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x));
}

__device__ __forceinline__ float2 cmadd(float2 acc, float2 a, float2 b) {
    acc.x = fmaf(a.x, b.x, acc.x);
    acc.x = fmaf(-a.y, b.y, acc.x);
    acc.y = fmaf(a.x, b.y, acc.y);
    acc.y = fmaf(a.y, b.x, acc.y);
    return acc;
}

// a value every lane holds, as a scalar
__device__ __forceinline__ float uni(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// z with the sign (-1)^n
__device__ __forceinline__ float2 flip_sign(float2 z, uint32_t n) {
    const uint32_t m = n << 31;
    return make_float2(__uint_as_float(__float_as_uint(z.x) ^ m), __uint_as_float(__float_as_uint(z.y) ^ m));
}

// A rotation [[c, -s], [s, c]] on register bit I with its larger entry taken
// out (the block's phase table carries it): |t| <= 1, one multiply-add per
// component and no copies in either branch.
template <int I>
__device__ __forceinline__ void rotate(float2 (&v)[16], float t, int swapped) {
    if (swapped) {          // s [[t, -1], [1, t]]
#pragma unroll
        for (int r = 0; r < 16; r++) {
            if ((r >> I) & 1) continue;
            const float2 a = v[r], b = v[r | (1 << I)];
            v[r] = make_float2(fmaf(t, a.x, -b.x), fmaf(t, a.y, -b.y));
            v[r | (1 << I)] = make_float2(fmaf(t, b.x, a.x), fmaf(t, b.y, a.y));
        }
    } else {                // c [[1, -t], [t, 1]]
#pragma unroll
        for (int r = 0; r < 16; r++) {
            if ((r >> I) & 1) continue;
            const float2 a = v[r], b = v[r | (1 << I)];
            v[r] = make_float2(fmaf(-t, b.x, a.x), fmaf(-t, b.y, a.y));
            v[r | (1 << I)] = make_float2(fmaf(t, a.x, b.x), fmaf(t, a.y, b.y));
        }
    }
}

// Tile index of register 0 of thread t when the register bits are base .. base + 3.
template <int BASE>
__device__ __forceinline__ uint32_t deposit(uint32_t t) {
    return (t & ((1u << BASE) - 1u)) | ((t >> BASE) << (BASE + 4));
}

__device__ __forceinline__ double lane_sum(double v, int width) {
    for (int o = width >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int NQ>
struct Shape {
    static constexpr int kM = NQ < 10 ? 10 : NQ;           // tile bits of a workgroup
    static constexpr int kThreads = 1 << (kM - 4);
    static constexpr int kStates = 1 << (kM - NQ);         // states of a workgroup
    static constexpr int kGroups = (NQ + 3) / 4;
    static constexpr int base(int g) { return 4 * g < NQ - 4 ? 4 * g : NQ - 4; }
};

// Gates of group G (bits max(base, 4 G) .. base + 3), and on.
template <int NQ, int G, bool SIGN>
__device__ __forceinline__ void groups(const qgtl_res_block_t &b, float2 *tile, uint32_t t, float2 pre, float2 post) {
    typedef Shape<NQ> S;
    if constexpr (G < S::kGroups) {
        constexpr int B = S::base(G), first = 4 * G - B;     // register bits below `first` had their gate
        const uint32_t j0 = deposit<B>(t);
        const uint32_t l0 = rpad(j0);
        float2 v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = tile[l0 ^ rpad((uint32_t)r << B)];
        if (G == 0 && qgtl::uniform(b.has_pre)) {
#pragma unroll
            for (int r = 0; r < 16; r++) v[r] = cmul(v[r], cmul(pre, make_float2(uni(b.reg_pre[r].re), uni(b.reg_pre[r].im))));
        }
        if constexpr (first <= 0) rotate<0>(v, uni(b.tan[B]), qgtl::uniform(b.swapped[B]));
        if constexpr (first <= 1) rotate<1>(v, uni(b.tan[B + 1]), qgtl::uniform(b.swapped[B + 1]));
        if constexpr (first <= 2) rotate<2>(v, uni(b.tan[B + 2]), qgtl::uniform(b.swapped[B + 2]));
        rotate<3>(v, uni(b.tan[B + 3]), qgtl::uniform(b.swapped[B + 3]));
        if constexpr (G + 1 == S::kGroups) {
#pragma unroll
            for (int r = 0; r < 16; r++) v[r] = cmul(v[r], cmul(post, make_float2(uni(b.reg_post[r].re), uni(b.reg_post[r].im))));
            if (SIGN && qgtl::uniform(b.has_sign)) {
                // (-1)^{q(j)}: q(j0 + r) = q(j0) + q(r) + the polar form of both
                uint32_t acc = 0;
#pragma unroll
                for (int i = 0; i < NQ; i++) acc ^= (0u - ((j0 >> i) & 1u)) & b.sgn[i];
                constexpr uint32_t kBit[4] = {0xaaaau, 0xccccu, 0xf0f0u, 0xff00u};
                uint32_t neg = b.sgn_reg ^ (0u - ((uint32_t)__popc(acc & j0) & 1u));
#pragma unroll
                for (int i = 0; i < 4; i++) neg ^= (0u - ((uint32_t)__popc(b.sgn_bil[i] & j0) & 1u)) & kBit[i];
#pragma unroll
                for (int r = 0; r < 16; r++) v[r] = flip_sign(v[r], neg >> r);
            }
            if (qgtl::uniform(b.has_perm)) {
                // element j goes to pi(j), the XOR of the images of its bits
                uint32_t p = j0 & ~((1u << NQ) - 1u);        // the state's number in the tile
#pragma unroll
                for (int i = 0; i < NQ; i++)
                    if (i < B || i >= B + 4) p ^= (0u - ((j0 >> i) & 1u)) & qgtl::uniform(b.img[i]);
                const uint32_t lp = rpad(p);
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    uint32_t u = 0;
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if ((r >> i) & 1) u ^= qgtl::uniform(b.img[B + i]);
                    tile[lp ^ rpad(u)] = v[r];
                }
                __syncthreads();
                return;
            }
        }
#pragma unroll
        for (int r = 0; r < 16; r++) tile[l0 ^ rpad((uint32_t)r << B)] = v[r];
        __syncthreads();
        groups<NQ, G + 1, SIGN>(b, tile, t, pre, post);
    }
}

// States blockIdx.x * kStates .. of the P derivative states (slot order) and
// the primal state (number P): D receives the former, psi the latter, sums
// (4 doubles per slot) the FP64 injection sums.  SIGN: some block's M-stage has
// CZ gates (a variant of its own: it costs 16 registers, and n = 13 has 12 left).
template <int NQ, bool SIGN>
__global__ __launch_bounds__(Shape<NQ>::kThreads) void resident_states_kernel(
    const qgtl_res_block_t *__restrict__ blocks, int nblocks, const float2 *__restrict__ tabs,
    const qgtl_res_slot_t *__restrict__ slots, int P, float2 *__restrict__ D, float2 *__restrict__ psi,
    double *__restrict__ sums) {
    typedef Shape<NQ> S;
    __shared__ float2 tile[1 << S::kM];
    __shared__ double red[16][4];
    // NQ < 13: the descriptors of this block and the next, fetched a block ahead (a wave alone on its
    // SIMD waits several times a block for scalar loads: n = 10, L = 4 68 -> 65 us a call, n = 12, L = 6
    // 105 -> 101; at n = 13, with two waves a SIMD and LDS the bound, 122 -> 124)
    constexpr bool kAhead = NQ < 13;
    __shared__ qgtl_res_block_t sb[2];
    constexpr int kWords = sizeof(qgtl_res_block_t) / 4, kPer = (kWords + S::kThreads - 1) / S::kThreads;
    const uint32_t t = threadIdx.x;
    uint32_t ahead[kPer];
    auto fetch = [&](int bi) {
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int w = (int)t + k * S::kThreads;
            ahead[k] = (bi < nblocks && w < kWords) ? reinterpret_cast<const uint32_t *>(blocks + bi)[w] : 0u;
        }
    };
    auto put = [&](int bi) {
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int w = (int)t + k * S::kThreads;
            if (w < kWords) reinterpret_cast<uint32_t *>(&sb[bi & 1])[w] = ahead[k];
        }
    };
    if constexpr (kAhead) {
        fetch(0);
        put(0);
        fetch(1);
    }
    auto block = [&](int bi) -> const qgtl_res_block_t & {
        if constexpr (kAhead) return sb[bi & 1];
        else return blocks[bi];
    };
    const int s_first = (int)blockIdx.x * S::kStates;
    const uint32_t Nm = (1u << NQ) - 1u;
    // in the layout of group 0 (register bits 0..3) a thread's amplitudes are of one state
    const uint32_t j0 = t << 4, l0 = rpad(j0), y0 = j0 & Nm;
    const int slot = s_first + (int)(j0 >> NQ);
    const qgtl_res_slot_t q = slots[slot < P ? slot : P];    // entry P: no injection
    const int blk_first = slots[s_first < P ? s_first : P].block;
    const int last = s_first + S::kStates - 1;
    const int blk_last = slots[last < P ? last : P].block;

#pragma unroll
    for (int r = 0; r < 16; r++) tile[l0 ^ (uint32_t)r] = make_float2(y0 == 0 && r == 0 ? 1.f : 0.f, 0.f);
    __syncthreads();

    const uint32_t yl = deposit<S::base(S::kGroups - 1)>(t) & Nm;   // register 0 of the last group
    for (int bi = 0; bi < nblocks; bi++) {
        if constexpr (kAhead) {
            put(bi + 1);                                      // block bi - 1's buffer; read after this block's barriers
            fetch(bi + 2);
        }
        const qgtl_res_block_t &b = block(bi);
        const float2 *tb = tabs + (size_t)bi * QGTL_RES_TAB * 2;
        // thread parts of the phase layers (from the caches, ahead of their use)
        const float2 post = cmul(tb[yl & 127u], tb[128u + (yl >> 7)]);
        float2 pre = make_float2(1.f, 0.f);
        if (qgtl::uniform(b.has_pre)) pre = cmul(tb[QGTL_RES_TAB + (y0 & 127u)], tb[QGTL_RES_TAB + 128u + (y0 >> 7)]);
        groups<NQ, 0, SIGN>(b, tile, t, pre, post);
        if (bi < blk_first || bi > blk_last) continue;        // uniform: slots are in block order
        // d[y] = M[s][s] psi[y] + (-1)^parity(y & z) M[s][1 - s] psi[y ^ v], s = parity(y & w)
        const bool mine = q.block == bi;
        double sr = 0.0, si = 0.0, sd = 0.0, sp = 0.0;
        float2 o[16];
#pragma unroll
        for (int r = 0; r < 16; r++) o[r] = tile[l0 ^ (uint32_t)r];
        if (mine) {
            const float2 m00 = make_float2(q.M[0].re, q.M[0].im), m01 = make_float2(q.M[1].re, q.M[1].im);
            const float2 m10 = make_float2(q.M[2].re, q.M[2].im), m11 = make_float2(q.M[3].re, q.M[3].im);
            const uint32_t lv = l0 ^ rpad(q.v);
            const uint32_t s0 = (uint32_t)__popc(y0 & q.w), z0 = (uint32_t)__popc(y0 & q.z);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const bool sg = ((s0 + (uint32_t)__popc((uint32_t)r & q.w)) & 1u) != 0;
                const float2 a = o[r];
                float2 p = tile[lv ^ (uint32_t)r];
                if constexpr (SIGN) p = flip_sign(p, z0 + (uint32_t)__popc((uint32_t)r & q.z));
                const float2 d = cmadd(cmadd(make_float2(0.f, 0.f), sg ? m11 : m00, a), sg ? m10 : m01, p);
                const double dr = d.x, di = d.y, pr = a.x, pi = a.y;
                sr += dr * pr + di * pi;
                si += dr * pi - di * pr;
                sd += dr * dr + di * di;
                sp += pr * pr + pi * pi;
                o[r] = d;
            }
        }
        constexpr int width = NQ < 10 ? 1 << (NQ - 4) : 64;   // lanes of one state within a wave
        sr = lane_sum(sr, width); si = lane_sum(si, width); sd = lane_sum(sd, width); sp = lane_sum(sp, width);
        if constexpr (NQ <= 10) {
            if (mine && (t & (width - 1)) == 0) {
                double *out = sums + 4 * (size_t)slot;
                out[0] = sr; out[1] = si; out[2] = sd; out[3] = sp;
            }
        } else if ((t & 63) == 0) {
            red[t >> 6][0] = sr; red[t >> 6][1] = si; red[t >> 6][2] = sd; red[t >> 6][3] = sp;
        }
        __syncthreads();                                      // every partner is read
        if (mine)
#pragma unroll
            for (int r = 0; r < 16; r++) tile[l0 ^ (uint32_t)r] = o[r];
        if constexpr (NQ > 10) {
            if (t < 4) {
                double s = 0.0;
                for (int w = 0; w < S::kThreads / 64; w++) s += red[w][t];
                sums[4 * (size_t)slot + t] = s;               // one state per workgroup: slot < P here
            }
        }
        __syncthreads();
    }
    // two adjacent amplitudes per store
    constexpr uint32_t N = 1u << NQ;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t j = 2u * ((uint32_t)i * S::kThreads + t);
        const int s = s_first + (int)(j >> NQ);
        if (s > P) continue;
        const float2 a = tile[rpad(j)], c = tile[rpad(j) ^ 1u];
        float2 *dst = (s < P ? D + (size_t)s * N : psi) + (j & Nm);
        *reinterpret_cast<float4 *>(dst) = make_float4(a.x, a.y, c.x, c.y);
    }
}

template <int NQ, bool SIGN>
int launch(const void *blocks, int nblocks, const void *tabs, const void *slots, int P, void *D, void *psi,
           double *sums) {
    typedef Shape<NQ> S;
    const unsigned grid = (unsigned)((P + 1 + S::kStates - 1) / S::kStates);
    hipLaunchKernelGGL((resident_states_kernel<NQ, SIGN>), dim3(grid), dim3(S::kThreads), 0, qgtl::stream(),
                       (const qgtl_res_block_t *)blocks, nblocks, (const float2 *)tabs,
                       (const qgtl_res_slot_t *)slots, P, (float2 *)D, (float2 *)psi, sums);
    QGTL_LAUNCH_CHECK("resident_states");
    return 0;
}

}  // namespace

extern "C" {

int qgtl_hip_resident_states(int n, const void *blocks, int nblocks, const void *tabs, const void *slots, int P,
                             int signs, void *D, void *psi, double *sums) {
    if (!blocks || !tabs || !slots || !D || !psi || !sums || nblocks < 1 || P < 1)
        return qgtl::set_error_msg(-118, "qgtl_hip_resident_states: bad arguments");
#define QGTL_RES_CASE(N)                                                                                     \
    case N:                                                                                                  \
        return signs ? launch<N, true>(blocks, nblocks, tabs, slots, P, D, psi, sums)                        \
                     : launch<N, false>(blocks, nblocks, tabs, slots, P, D, psi, sums)
    switch (n) {
    QGTL_RES_CASE(4);
    QGTL_RES_CASE(5);
    QGTL_RES_CASE(6);
    QGTL_RES_CASE(7);
    QGTL_RES_CASE(8);
    QGTL_RES_CASE(9);
    QGTL_RES_CASE(10);
    QGTL_RES_CASE(11);
    QGTL_RES_CASE(12);
    QGTL_RES_CASE(13);
    default: return qgtl::set_error_msg(-118, "qgtl_hip_resident_states: needs 4 <= n <= 13");
    }
#undef QGTL_RES_CASE
}

}  // extern "C"
