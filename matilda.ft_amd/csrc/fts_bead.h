// One propagation step of a discrete chain as one kernel per bead.
//
// A bead is q_s = e^{-W_b(s)} D q_{s-1} with the diffusion D = Dx Dy Dz, one
// real symmetric circulant matrix per axis (g(k) = exp(-k^2/(Nr-1)) factorises
// and depends on k^2 only).  The axes commute, so the launch that finishes bead
// s along its last axis `a` already holds whole (x, a) planes of q_s and starts
// bead s + 1 on them:
//   t (bead s without axis a) -> D_a -> times E = e^{-W} -> store q_s
//                             -> D_a -> D_x -> t (bead s + 1 without the other
//                                              axis), in place
// and `a` alternates between z and y from bead to bead.  One launch per bead
// instead of two, and per bead a slice of t read and written, E read and q_s
// written (the two-pass form read q, wrote and read the intermediate, and read
// E and wrote q: five slices).  Per bead of two chains, against the plane and z
// kernels before: 32^3 5.5 + 4.6 -> 3.7 us (a dependent launch alone takes 2.7),
// 64^3 9.0 + 5.1 -> 7.9 us, 96^3 22.2 + 18.9 -> 18.8 us; for three 64^3 replicas
// 13.1 + 7.7 -> 12.2 us, of which 10.9 are the four slices (4.6 TB/s).
//
// Along an axis of N points D is applied as a matrix product, not through the
// transform: a symmetric circulant commutes with the reflection j -> N-1-j and
// the shift by N/2, which send each row index to an orbit of F = 4 (N >= 40, a
// multiple of 4) or 2 rows.  Sums and differences over the orbits split D into F
// real blocks of S = N / F rows, S <= 32, applied with the 16x16x4 matrix
// instructions.  The 16 columns of an operand are 8 grid columns' real and
// imaginary parts (neighbouring lanes), so a wavefront owns 8 columns, 64 points
// take 8 wavefronts, and a plane has twice the wavefronts to hide its latency
// with than whole complex columns per lane would give.  An orbit's rows sit in
// one lane, so the sums need no exchange, and a product's output registers are
// the next product's input when its reduction index is numbered the same way:
// D_a, E and D_a again chain in registers.  LDS carries the plane once, between
// the a and the x direction.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_core.h"

namespace mft {

// src: the intermediate of bead s (or q_0 where E is null: then only D_a D_x of
// bead 1 is started); dst: the intermediate of the next bead (null at the
// chain's last bead); q: where q_s goes.
struct BeadDesc {
    const float2* src;
    float2* dst;
    const float2* E;
    float2* q;
    const float *ta, *tx; // bead_table() of axis a and of x
};

// Blocks of an axis of N points: F rows per orbit, S orbits in RT tiles of 16
// operand rows.  Lane group q (of 16 lanes) holds four orbits of every full tile
// and R of the last, J in all, so a last tile of S % 16 orbits costs only R
// steps of the reduction.
template <int N>
struct BeadAxis {
    static constexpr int F = N % 4 == 0 && N >= 40 ? 4 : (N > 16 ? 2 : 1);
    static constexpr int S = N / F;
    static constexpr int RT = (S + 15) / 16;
    static constexpr int R = (S - 16 * (RT - 1) + 3) / 4;
    static constexpr int J = 4 * (RT - 1) + R;
    static constexpr int BLOCK = RT * J * 64; // operands of one block
    static constexpr int TABLE = F * BLOCK;   // floats of bead_table()
    // the last lane group has orbits past S: they read other rows of the grid,
    // their products meet zero columns of the table, and they are not stored
    static constexpr bool ragged = 4 * J != S;
    // orbit j of lane group q
    __host__ __device__ static constexpr int orbit(int j, int q)
    {
        return j < 4 * (RT - 1) ? 16 * (j / 4) + 4 * q + j % 4 : 16 * (RT - 1) + R * q + j - 4 * (RT - 1);
    }
    // orbits per lane in tile o
    __host__ __device__ static constexpr int in_tile(int o) { return o == RT - 1 ? R : 4; }
};

// row of orbit i's member f: i, N-1-i, i + N/2, N/2-1-i
template <int N>
__host__ __device__ constexpr int bead_row(int f, int i)
{
    return f == 0 ? i : f == 1 ? N - 1 - i : f == 2 ? i + N / 2 : N / 2 - 1 - i;
}

// Row of (member f, orbit j of lane group q) as uniform part + lane part, the
// lane part 0 .. 3 steps of the rows a lane group holds: one byte offset per
// lane and direction serves every access, the rest of the address is scalar.
template <int N>
struct BeadRow {
    using A = BeadAxis<N>;
    __device__ __forceinline__ static constexpr int step(int j) { return j < 4 * (A::RT - 1) ? 4 : A::R; }
    __device__ __forceinline__ static constexpr int uniform(int f, int j)
    {
        return f & 1 ? bead_row<N>(f, A::orbit(j, 3)) : bead_row<N>(f, A::orbit(j, 0));
    }
    __device__ __forceinline__ static int lane(int f, int j, int q) { return (f & 1 ? 3 - q : q) * step(j); }
};


typedef float bead_f4 __attribute__((ext_vector_type(4)));

// Pointers out of a descriptor are global memory, which the compiler cannot see:
// as generic pointers they would be flat accesses, with 64-bit lane addresses
// and waits shared with LDS.
#define BeadGlobal __attribute__((address_space(1)))
__device__ __forceinline__ BeadGlobal char* bead_global(const void* p)
{
    return (BeadGlobal char*)(const_cast<void*>(p));
}
__device__ __forceinline__ float bead_load(const BeadGlobal char* p) { return *(const BeadGlobal float*)p; }
__device__ __forceinline__ void bead_store(float2* p, float4 v)
{
    *(BeadGlobal bead_f4*)bead_global(p) = bead_f4{v.x, v.y, v.z, v.w};
}

__device__ __forceinline__ void bead_stage(float4* to, const float* tab, int i)
{
    const bead_f4 v = *(const BeadGlobal bead_f4*)(bead_global(tab) + 16u * (unsigned)i);
    to[i] = make_float4(v.x, v.y, v.z, v.w);
}

// the neighbouring lane's value (lanes 2 k and 2 k + 1 swap): a column's other
// component
__device__ __forceinline__ float bead_swap(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}

// Operands of an axis: in registers, loaded with the slices (one tile), or
// staged in LDS (two tiles: 16 KB, too much for registers beside the data).
template <int N>
struct BeadOps {
    using A = BeadAxis<N>;
    static constexpr bool in_regs = A::F * A::RT * A::J <= 48;
    static constexpr int K = in_regs ? A::RT * A::J : 1, FF = in_regs ? A::F : 1;
    float m[FF][K];
    const float* lds;
    __device__ __forceinline__ void load(const float* tab)
    {
#pragma unroll
        for (int f = 0; f < FF; ++f)
#pragma unroll
            for (int k = 0; k < K; ++k) m[f][k] = bead_load(bead_global(tab + f * A::BLOCK + k * 64) + 4 * (threadIdx.x & 63));
    }
    __device__ __forceinline__ float op(int f, int k) const
    {
        if constexpr (in_regs) return m[f][k];
        else return lds[f * A::BLOCK + k * 64 + (threadIdx.x & 63)];
    }
};

// sums and differences over the orbits
template <int F, int J>
__device__ __forceinline__ void bead_orbits(float (&d)[F][J])
{
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int h = 1; h < F; h <<= 1)
#pragma unroll
            for (int f = 0; f < F; ++f)
                if (!(f & h)) {
                    const float a = d[f][j], b = d[f | h][j];
                    d[f][j] = a + b;
                    d[f | h][j] = a - b;
                }
    }
}

// d <- D d along an axis: a lane holds, of its column and component, the orbits
// BeadAxis::orbit(j, lane / 16).
//
// Block 0 (the orbit sums) carries the mean of a slice, and the slices of weak
// fields are close to constant: float products then err the same way at every
// point of every bead (log Q of a 100-bead 64^3 chain was off by 1.1e-6, against
// 2e-8 with the transforms).  D leaves a constant alone, so the block is applied
// to the distance from one of its own values, `ref`, which is added back last,
// with one rounding; its table rows sum to 1/F to better than 1e-11.
template <int N>
__device__ __forceinline__ void bead_diffuse(float (&d)[BeadAxis<N>::F][BeadAxis<N>::J], const BeadOps<N>& ops)
{
    using A = BeadAxis<N>;
    constexpr int F = A::F, RT = A::RT, J = A::J;
    bead_orbits<F, J>(d);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d[0][0]), 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d[0][0]), 1));
    float ref = threadIdx.x & 1 ? r1 : r0;
#pragma unroll
    for (int j = 0; j < J; ++j) d[0][j] -= ref;
    bead_f4 v[F][RT];
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int o = 0; o < RT; ++o) v[f][o] = bead_f4{0.f, 0.f, 0.f, 0.f};
    // F RT independent sums side by side
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int o = 0; o < RT; ++o)
                v[f][o] = __builtin_amdgcn_mfma_f32_16x16x4f32(ops.op(f, o * J + j), d[f][j], v[f][o], 0, 0, 0);
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int j = 0; j < J; ++j) d[f][j] = v[f][j / 4][j % 4];
    bead_orbits<F, J>(d);
    ref *= 1.0f / F;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int f = 0; f < F; ++f) d[f][j] += ref;
}

template <int NX, int NA>
struct BeadShape {
    static constexpr int CW = (NX + 7) / 8;     // wavefronts of the a direction
    static constexpr int MW = (NA + 7) / 8;     // wavefronts of the x direction
    static constexpr int W = CW > MW ? CW : MW;
    // LDS: real and imaginary parts as planes of floats with a row pitch of an
    // odd multiple of four and 32 banks between the planes: the x direction's
    // 16-byte reads of 8 rows' two components fall on 16 different bank groups
    static constexpr int P = (NX / 4) % 2 ? NX : NX + 4;
    static constexpr int CP = (NA * P + 31) / 64 * 64 + 32;
    static constexpr size_t PLANES = sizeof(float) * 2 * CP;
    // staged operands, one axis at a time
    static constexpr size_t TA = BeadOps<NA>::in_regs ? 0 : sizeof(float) * BeadAxis<NA>::TABLE;
    static constexpr size_t TX = BeadOps<NX>::in_regs ? 0 : sizeof(float) * BeadAxis<NX>::TABLE;
    static constexpr size_t LDS = PLANES + (TA > TX ? TA : TX);
};

// Up to kBeadInline chains travel as kernel arguments: a single system's bead
// then waits for one memory latency less before its first load.
constexpr int kBeadInline = 8;
struct BeadArgs {
    BeadDesc d[kBeadInline];
};

template <int NX, int NA>
__global__ void __launch_bounds__((64 * BeadShape<NX, NA>::W))
    k_fts_bead(const BeadArgs args, const BeadDesc* __restrict__ descs, long plane_stride, long row_stride)
{
    using SH = BeadShape<NX, NA>;
    using AA = BeadAxis<NA>;
    using AX = BeadAxis<NX>;
    constexpr int P = SH::P, NT = 64 * SH::W;
    extern __shared__ float4 bead_lds[];
    float* planes = reinterpret_cast<float*>(bead_lds);
    float4* staged = bead_lds + SH::PLANES / sizeof(float4);
    // both sources are constant memory: scalar loads, and scalar pointers
    using DescPtr = const __attribute__((address_space(4))) BeadDesc*;
    const DescPtr dd = (DescPtr)(descs ? descs : args.d) + blockIdx.y;
    const BeadDesc D = {dd->src, dd->dst, dd->E, dd->q, dd->ta, dd->tx};
    const long base = (long)blockIdx.x * plane_stride;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 1;
    const int line = 8 * w + (lane & 15) / 2; // the lane's column, later its row
    BeadOps<NA> oa;
    BeadOps<NX> ox;
    oa.lds = ox.lds = reinterpret_cast<const float*>(staged);
    const bool incol = SH::CW == SH::W || w < SH::CW;
    const bool cok = NX % 8 == 0 || line < NX;
    float d[AA::F][AA::J], e[AA::F][AA::J];
    using Row = BeadRow<NA>;
    const unsigned rs8 = 8u * (unsigned)row_stride, c8 = 8u * (unsigned)(line < NX ? line : NX - 1) + 4u * c;
    // the lane's component of (member, orbit) in a slice
    auto at = [&](const float2* slice, int f, int j) {
        return bead_global(slice + base + (long)Row::uniform(f, j) * row_stride) +
               (c8 + (unsigned)Row::lane(f, j, q) * rs8);
    };
    if (incol) {
#pragma unroll
        for (int j = 0; j < AA::J; ++j)
#pragma unroll
            for (int f = 0; f < AA::F; ++f) d[f][j] = bead_load(at(D.src, f, j));
        if (AA::RT == 1 && D.E) {
#pragma unroll
            for (int j = 0; j < AA::J; ++j)
#pragma unroll
                for (int f = 0; f < AA::F; ++f) e[f][j] = bead_load(at(D.E, f, j));
        }
    }
    if constexpr (BeadOps<NA>::in_regs) {
        oa.load(D.ta);
    } else {
        for (int i = threadIdx.x; i < (int)(SH::TA / 16); i += NT) bead_stage(staged, D.ta, i);
        __syncthreads();
    }
    if constexpr (BeadOps<NX>::in_regs && AX::RT == 1) ox.load(D.tx);
    if (incol) {
        if (D.E) {
            bead_diffuse<NA>(d, oa);
            if (AA::RT > 1) {
#pragma unroll
                for (int j = 0; j < AA::J; ++j)
#pragma unroll
                    for (int f = 0; f < AA::F; ++f) e[f][j] = bead_load(at(D.E, f, j));
            }
#pragma unroll
            for (int j = 0; j < AA::J; ++j) {
                const bool ok = cok && (!AA::ragged || AA::orbit(j, q) < AA::S);
#pragma unroll
                for (int f = 0; f < AA::F; ++f) {
                    // (re, im) times e: re e.re - im e.im and im e.re + re e.im
                    const float o = bead_swap(d[f][j]), g = bead_swap(e[f][j]);
                    d[f][j] = fmaf(d[f][j], c ? g : e[f][j], o * (c ? e[f][j] : -g));
                    // read again only by the density pass: not kept in the caches
                    // beside t and E (two 64^3 chains 3 to 4 % faster)
                    if (ok) __builtin_nontemporal_store(d[f][j], (BeadGlobal float*)at(D.q, f, j));
                }
            }
        }
        if (D.dst) {
            bead_diffuse<NA>(d, oa);
#pragma unroll
            for (int j = 0; j < AA::J; ++j) {
                const int i = AA::orbit(j, q);
                const bool ok = cok && (!AA::ragged || i < AA::S);
#pragma unroll
                for (int f = 0; f < AA::F; ++f)
                    if (ok) planes[c * SH::CP + bead_row<NA>(f, i) * P + line] = d[f][j];
            }
        }
    }
    if (!D.dst) return;
    if constexpr (BeadOps<NX>::in_regs && AX::RT > 1) ox.load(D.tx);
    __syncthreads();
    if constexpr (!BeadOps<NX>::in_regs) {
        for (int i = threadIdx.x; i < (int)(SH::TX / 16); i += NT) bead_stage(staged, D.tx, i);
        __syncthreads();
    }
    if (SH::MW < SH::W && w >= SH::MW) return;
    const bool rok = NA % 8 == 0 || line < NA;
    const float* rp = planes + c * SH::CP + (rok ? line : NA - 1) * P;
    float v[AX::F][AX::J];
    // consecutive orbits of a member are consecutive values, ascending (members
    // 0 and 2) or descending (1 and 3); orbits past the last one read other
    // values of the row
#pragma unroll
    for (int o = 0; o < AX::RT; ++o)
#pragma unroll
        for (int f = 0; f < AX::F; ++f) {
            const int x0 = bead_row<NX>(f, AX::orbit(4 * o, q));
            if (AX::in_tile(o) == 4) {
                const float4 a = *reinterpret_cast<const float4*>(rp + (f & 1 ? x0 - 3 : x0));
                const float t[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int r = 0; r < 4; ++r) v[f][4 * o + r] = t[f & 1 ? 3 - r : r];
            } else {
#pragma unroll
                for (int r = 0; r < AX::in_tile(o); ++r) v[f][4 * o + r] = rp[f & 1 ? x0 - r : x0 + r];
            }
        }
    bead_diffuse<NX>(v, ox);
    if constexpr (AX::RT == 1 && AX::R == 4) {
        // a lane's values are four of one component: the two lanes of a row
        // swap halves and store two complex values each
        if (!rok) return;
        float2* dp = D.dst + base + line * row_stride + 2 * c;
#pragma unroll
        for (int f = 0; f < AX::F; ++f) {
            const int x0 = bead_row<NX>(f, AX::orbit(0, q));
            float t[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = v[f][f & 1 ? 3 - r : r];
            const float s0 = bead_swap(c ? t[0] : t[2]), s1 = bead_swap(c ? t[1] : t[3]);
            bead_store(dp + (f & 1 ? x0 - 3 : x0),
                       c ? make_float4(s0, t[2], s1, t[3]) : make_float4(t[0], s0, t[1], s1));
        }
    } else {
        // back to the wavefront's own rows in LDS, then out in row order
        float* wp = planes + c * SH::CP + line * P;
        if (rok) {
#pragma unroll
            for (int j = 0; j < AX::J; ++j)
#pragma unroll
                for (int f = 0; f < AX::F; ++f)
                    if (!AX::ragged || AX::orbit(j, q) < AX::S) wp[bead_row<NX>(f, AX::orbit(j, q))] = v[f][j];
        }
        exchange_barrier<true>();
        const float* lp = planes + 8 * w * P;
        float2* dp = D.dst + base + 8 * w * row_stride;
#pragma unroll
        for (int k = 0; k < (4 * NX + 63) / 64; ++k) {
            const int i = 64 * k + lane, row = i / (NX / 2), x = 2 * (i - row * (NX / 2));
            if (row >= 8 || (NA % 8 != 0 && 8 * w + row >= NA)) continue;
            const float2 re = *reinterpret_cast<const float2*>(lp + row * P + x);
            const float2 im = *reinterpret_cast<const float2*>(lp + SH::CP + row * P + x);
            bead_store(dp + row * row_stride + x, make_float4(re.x, im.x, re.y, im.y));
        }
    }
}

} // namespace mft
