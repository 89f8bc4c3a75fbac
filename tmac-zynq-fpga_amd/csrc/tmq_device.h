// tmq_device.h -- device helpers shared by the kernel sources.
#pragma once
#include <hip/hip_runtime.h>

#include "tmq_internal.h"

// The kernel's arguments into the scalar cache in one round trip: one
// s_load_dword per 64-byte line of the argument struct (in one asm statement
// so that nothing is scheduled between them), then one wait.  The compiler
// otherwise loads them where each is first needed, behind the branches that
// depend on earlier ones: a round trip (~0.3 us) each.  The loaded values are
// not used: the destinations are scratch registers the compiler picks (dead
// after the statement), so the kernel's SGPR count, which bounds how many
// waves a SIMD holds, does not grow.
template <int BYTES>
static __device__ __forceinline__ void tmq_warm_kernargs() {
    constexpr int N = (BYTES + 63) / 64;
    static_assert(N >= 1 && N <= 16, "one to sixteen lines");
    const auto p = __builtin_amdgcn_kernarg_segment_ptr();
    int d[16];
    if constexpr (N == 1)
        asm volatile("s_load_dword %0, %1, 0x0\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]) : "s"(p) : "memory");
    else if constexpr (N == 2)
        asm volatile("s_load_dword %0, %2, 0x0\n" "s_load_dword %1, %2, 0x40\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]) : "s"(p) : "memory");
    else if constexpr (N == 3)
        asm volatile("s_load_dword %0, %3, 0x0\n" "s_load_dword %1, %3, 0x40\n" "s_load_dword %2, %3, 0x80\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]) : "s"(p) : "memory");
    else if constexpr (N == 4)
        asm volatile("s_load_dword %0, %4, 0x0\n" "s_load_dword %1, %4, 0x40\n" "s_load_dword %2, %4, 0x80\n" "s_load_dword %3, %4, 0xc0\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]) : "s"(p) : "memory");
    else if constexpr (N == 5)
        asm volatile("s_load_dword %0, %5, 0x0\n" "s_load_dword %1, %5, 0x40\n" "s_load_dword %2, %5, 0x80\n" "s_load_dword %3, %5, 0xc0\n" "s_load_dword %4, %5, 0x100\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]) : "s"(p) : "memory");
    else if constexpr (N == 6)
        asm volatile("s_load_dword %0, %6, 0x0\n" "s_load_dword %1, %6, 0x40\n" "s_load_dword %2, %6, 0x80\n" "s_load_dword %3, %6, 0xc0\n" "s_load_dword %4, %6, 0x100\n" "s_load_dword %5, %6, 0x140\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]) : "s"(p) : "memory");
    else if constexpr (N == 7)
        asm volatile("s_load_dword %0, %7, 0x0\n" "s_load_dword %1, %7, 0x40\n" "s_load_dword %2, %7, 0x80\n" "s_load_dword %3, %7, 0xc0\n" "s_load_dword %4, %7, 0x100\n" "s_load_dword %5, %7, 0x140\n" "s_load_dword %6, %7, 0x180\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]) : "s"(p) : "memory");
    else if constexpr (N == 8)
        asm volatile("s_load_dword %0, %8, 0x0\n" "s_load_dword %1, %8, 0x40\n" "s_load_dword %2, %8, 0x80\n" "s_load_dword %3, %8, 0xc0\n" "s_load_dword %4, %8, 0x100\n" "s_load_dword %5, %8, 0x140\n" "s_load_dword %6, %8, 0x180\n" "s_load_dword %7, %8, 0x1c0\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]) : "s"(p) : "memory");
    else if constexpr (N == 9)
        asm volatile("s_load_dword %0, %9, 0x0\n" "s_load_dword %1, %9, 0x40\n" "s_load_dword %2, %9, 0x80\n" "s_load_dword %3, %9, 0xc0\n" "s_load_dword %4, %9, 0x100\n" "s_load_dword %5, %9, 0x140\n" "s_load_dword %6, %9, 0x180\n" "s_load_dword %7, %9, 0x1c0\n" "s_load_dword %8, %9, 0x200\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]) : "s"(p) : "memory");
    else if constexpr (N == 10)
        asm volatile("s_load_dword %0, %10, 0x0\n" "s_load_dword %1, %10, 0x40\n" "s_load_dword %2, %10, 0x80\n" "s_load_dword %3, %10, 0xc0\n" "s_load_dword %4, %10, 0x100\n" "s_load_dword %5, %10, 0x140\n" "s_load_dword %6, %10, 0x180\n" "s_load_dword %7, %10, 0x1c0\n" "s_load_dword %8, %10, 0x200\n" "s_load_dword %9, %10, 0x240\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]) : "s"(p) : "memory");
    else if constexpr (N == 11)
        asm volatile("s_load_dword %0, %11, 0x0\n" "s_load_dword %1, %11, 0x40\n" "s_load_dword %2, %11, 0x80\n" "s_load_dword %3, %11, 0xc0\n" "s_load_dword %4, %11, 0x100\n" "s_load_dword %5, %11, 0x140\n" "s_load_dword %6, %11, 0x180\n" "s_load_dword %7, %11, 0x1c0\n" "s_load_dword %8, %11, 0x200\n" "s_load_dword %9, %11, 0x240\n" "s_load_dword %10, %11, 0x280\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]) : "s"(p) : "memory");
    else if constexpr (N == 12)
        asm volatile("s_load_dword %0, %12, 0x0\n" "s_load_dword %1, %12, 0x40\n" "s_load_dword %2, %12, 0x80\n" "s_load_dword %3, %12, 0xc0\n" "s_load_dword %4, %12, 0x100\n" "s_load_dword %5, %12, 0x140\n" "s_load_dword %6, %12, 0x180\n" "s_load_dword %7, %12, 0x1c0\n" "s_load_dword %8, %12, 0x200\n" "s_load_dword %9, %12, 0x240\n" "s_load_dword %10, %12, 0x280\n" "s_load_dword %11, %12, 0x2c0\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]), "=&s"(d[11]) : "s"(p) : "memory");
    else if constexpr (N == 13)
        asm volatile("s_load_dword %0, %13, 0x0\n" "s_load_dword %1, %13, 0x40\n" "s_load_dword %2, %13, 0x80\n" "s_load_dword %3, %13, 0xc0\n" "s_load_dword %4, %13, 0x100\n" "s_load_dword %5, %13, 0x140\n" "s_load_dword %6, %13, 0x180\n" "s_load_dword %7, %13, 0x1c0\n" "s_load_dword %8, %13, 0x200\n" "s_load_dword %9, %13, 0x240\n" "s_load_dword %10, %13, 0x280\n" "s_load_dword %11, %13, 0x2c0\n" "s_load_dword %12, %13, 0x300\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]), "=&s"(d[11]), "=&s"(d[12]) : "s"(p) : "memory");
    else if constexpr (N == 14)
        asm volatile("s_load_dword %0, %14, 0x0\n" "s_load_dword %1, %14, 0x40\n" "s_load_dword %2, %14, 0x80\n" "s_load_dword %3, %14, 0xc0\n" "s_load_dword %4, %14, 0x100\n" "s_load_dword %5, %14, 0x140\n" "s_load_dword %6, %14, 0x180\n" "s_load_dword %7, %14, 0x1c0\n" "s_load_dword %8, %14, 0x200\n" "s_load_dword %9, %14, 0x240\n" "s_load_dword %10, %14, 0x280\n" "s_load_dword %11, %14, 0x2c0\n" "s_load_dword %12, %14, 0x300\n" "s_load_dword %13, %14, 0x340\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]), "=&s"(d[11]), "=&s"(d[12]), "=&s"(d[13]) : "s"(p) : "memory");
    else if constexpr (N == 15)
        asm volatile("s_load_dword %0, %15, 0x0\n" "s_load_dword %1, %15, 0x40\n" "s_load_dword %2, %15, 0x80\n" "s_load_dword %3, %15, 0xc0\n" "s_load_dword %4, %15, 0x100\n" "s_load_dword %5, %15, 0x140\n" "s_load_dword %6, %15, 0x180\n" "s_load_dword %7, %15, 0x1c0\n" "s_load_dword %8, %15, 0x200\n" "s_load_dword %9, %15, 0x240\n" "s_load_dword %10, %15, 0x280\n" "s_load_dword %11, %15, 0x2c0\n" "s_load_dword %12, %15, 0x300\n" "s_load_dword %13, %15, 0x340\n" "s_load_dword %14, %15, 0x380\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]), "=&s"(d[11]), "=&s"(d[12]), "=&s"(d[13]), "=&s"(d[14]) : "s"(p) : "memory");
    else if constexpr (N == 16)
        asm volatile("s_load_dword %0, %16, 0x0\n" "s_load_dword %1, %16, 0x40\n" "s_load_dword %2, %16, 0x80\n" "s_load_dword %3, %16, 0xc0\n" "s_load_dword %4, %16, 0x100\n" "s_load_dword %5, %16, 0x140\n" "s_load_dword %6, %16, 0x180\n" "s_load_dword %7, %16, 0x1c0\n" "s_load_dword %8, %16, 0x200\n" "s_load_dword %9, %16, 0x240\n" "s_load_dword %10, %16, 0x280\n" "s_load_dword %11, %16, 0x2c0\n" "s_load_dword %12, %16, 0x300\n" "s_load_dword %13, %16, 0x340\n" "s_load_dword %14, %16, 0x380\n" "s_load_dword %15, %16, 0x3c0\n" "s_waitcnt lgkmcnt(0)" : "=&s"(d[0]), "=&s"(d[1]), "=&s"(d[2]), "=&s"(d[3]), "=&s"(d[4]), "=&s"(d[5]), "=&s"(d[6]), "=&s"(d[7]), "=&s"(d[8]), "=&s"(d[9]), "=&s"(d[10]), "=&s"(d[11]), "=&s"(d[12]), "=&s"(d[13]), "=&s"(d[14]), "=&s"(d[15]) : "s"(p) : "memory");
    (void)d;
}

// Wave reductions by DPP lane moves (VALU only; __shfl_xor is a chain of six
// LDS round trips): pairs and quads (quad permutations), rows of 8 and 16
// (half-row and row mirrors), row 0 into row 1 and row 2 into row 3
// (row_bcast15), rows 0-1 into rows 2-3 (row_bcast31); lane 63 then holds
// the whole wave's value.  `old` is what a lane that a move leaves without a
// source reads: the identity of the operation.
template <int CTRL, int ROW_MASK = 0xf>
static __device__ __forceinline__ int tmq_dpp_i32(int v, int old) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROW_MASK, 0xf, false);
}
// fmaxf over the wave, the same value in every lane (a quiet NaN is fmaxf's
// identity; fmaxf picks the same value in any order for the inputs used
// here, which hold no -0)
static __device__ __forceinline__ float tmq_wave_max(float x) {
    const int q = 0x7fc00000;
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0xb1>(__float_as_int(x), q)));
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0x4e>(__float_as_int(x), q)));
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0x141>(__float_as_int(x), q)));
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0x140>(__float_as_int(x), q)));
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0x142, 0xa>(__float_as_int(x), q)));
    x = fmaxf(x, __int_as_float(tmq_dpp_i32<0x143, 0xc>(__float_as_int(x), q)));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
// integer sum over each 16-lane row, in every lane of the row
static __device__ __forceinline__ int tmq_row_sum(int x) {
    x += tmq_dpp_i32<0xb1>(x, 0);
    x += tmq_dpp_i32<0x4e>(x, 0);
    x += tmq_dpp_i32<0x141>(x, 0);
    x += tmq_dpp_i32<0x140>(x, 0);
    return x;
}
// integer sum over the wave, the same value in every lane
static __device__ __forceinline__ int tmq_wave_sum(int x) {
    x = tmq_row_sum(x);
    x += tmq_dpp_i32<0x142, 0xa>(x, 0);
    x += tmq_dpp_i32<0x143, 0xc>(x, 0);
    return __builtin_amdgcn_readlane(x, 63);
}

// int64 row sums of a K-split GEMV live at the device coherence point
// (device-scope atomics); reads go there too.
static __device__ __forceinline__ int64_t tmq_ld_acc(const int64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Row i of a K-split GEMV, finalised (TmqDeferred).
static __device__ float tmq_fin(const TmqDeferred& D, int i) {
    const double xs = (double)*D.xs;
    float v;
    if (D.val) {
        v = __hip_atomic_load(D.val + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (D.ntiles == 0) {
        v = (float)(((double)tmq_ld_acc(D.acc + i) * xs) / (double)D.row_inv[i]);
    } else {
        const double rs = (double)D.row_scale[i];
        float y = 0.0f;
        for (int t = 0; t < D.ntiles; t++)
            y = (float)((double)y + ((double)tmq_ld_acc(D.acc + (size_t)i * D.ntiles + t) * xs) * rs);
        v = y;
    }
    if (D.bias) v = v + D.bias[i];
    return v;
}

// tmq_fin split in two, so that a kernel can issue the loads of several
// deferred values before it waits for any of them: fin_load takes the raw
// terms of row i (no branch on the data; Q8 selects the tiled form, up to
// TMQ_FIN_MAXT tiles), fin_finish forms the value as tmq_fin does.
#define TMQ_FIN_MAXT 16
template <bool Q8>
struct TmqFinRaw {
    int64_t p[Q8 ? TMQ_FIN_MAXT : 1];
    float r, b;
};
template <bool Q8>
static __device__ __forceinline__ TmqFinRaw<Q8> fin_load(const TmqDeferred& D, int i) {
    TmqFinRaw<Q8> f;
    if (D.val) {
        // FP32 path: the value itself (its bits in p[0])
#pragma unroll
        for (int t = 0; t < (Q8 ? TMQ_FIN_MAXT : 1); t++) f.p[t] = 0;
        f.p[0] = (int64_t)__float_as_uint(__hip_atomic_load(D.val + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        f.r = 1.0f;
    } else if constexpr (Q8) {
        const int nt = D.ntiles;
#pragma unroll
        for (int t = 0; t < TMQ_FIN_MAXT; t++) f.p[t] = tmq_ld_acc(D.acc + (size_t)i * nt + min(t, nt - 1));
        f.r = D.row_scale[i];
    } else {
        f.p[0] = tmq_ld_acc(D.acc + i);
        f.r = D.row_inv[i];
    }
    // no bias: any valid row vector stands in (the value is not used)
    const float* bp = D.bias ? D.bias : D.val ? D.val : Q8 ? D.row_scale : D.row_inv;
    f.b = bp[i];
    return f;
}
template <bool Q8>
static __device__ __forceinline__ float fin_finish(const TmqDeferred& D, const TmqFinRaw<Q8>& f, double xs) {
    float v;
    if (D.val) {
        v = __uint_as_float((uint32_t)f.p[0]);
    } else if constexpr (Q8) {
        const double rs = (double)f.r;
        float y = 0.0f;
#pragma unroll
        for (int t = 0; t < TMQ_FIN_MAXT; t++)
            if (t < D.ntiles) y = (float)((double)y + ((double)f.p[t] * xs) * rs);
        v = y;
    } else {
        v = (float)(((double)f.p[0] * xs) / (double)f.r);
    }
    if (D.bias) v = v + f.b;
    return v;
}

// sum += the 64 values of a group, in order, in every lane: each lane of a
// 16-lane row holds four of them (lane i: values 4i .. 4i+3, the same in the
// four rows), and v_add_f32_dpp row_newbcast:i adds lane i's value of the
// lane's own row as src0 (src0 + src1 = v + sum, the same rounded value as
// sum + v).  No LDS traffic inside the chain; a dependent DPP add issues
// about every 7 cycles.  s_nop 1: the two wait states a DPP read of a VGPR
// needs after a VALU write of it.
static __device__ __forceinline__ float add64_rowbcast(float4 x, float sum) {
#define TMQ_RB4(N)                                                                 \
    "v_add_f32_dpp %0, %1, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t" \
    "v_add_f32_dpp %0, %2, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t" \
    "v_add_f32_dpp %0, %3, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t" \
    "v_add_f32_dpp %0, %4, %0 row_newbcast:" #N " row_mask:0xf bank_mask:0xf\n\t"
    asm volatile("s_nop 1\n\t" TMQ_RB4(0) TMQ_RB4(1) TMQ_RB4(2) TMQ_RB4(3) TMQ_RB4(4) TMQ_RB4(5) TMQ_RB4(6)
                     TMQ_RB4(7) TMQ_RB4(8) TMQ_RB4(9) TMQ_RB4(10) TMQ_RB4(11) TMQ_RB4(12) TMQ_RB4(13)
                         TMQ_RB4(14) TMQ_RB4(15)
                 : "+v"(sum)
                 : "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w));
#undef TMQ_RB4
    return sum;
}
// Lane i's four values of group g of [i0, i1) (v[i0 + 64g + 4i ..]), +0.0
// past i1.
static __device__ __forceinline__ float4 seq_group(const float* v, int i0, int i1, int g, int i) {
    const int b = i0 + 64 * g + 4 * i;
    if (b + 4 <= i1) return *(const float4*)(v + b);
    float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (b + 0 < i1) r.x = v[b + 0];
    if (b + 1 < i1) r.y = v[b + 1];
    if (b + 2 < i1) r.z = v[b + 2];
    return r;
}
// Sequential fp32 sum of v[i0..i1) in index order from each lane's `sum`
// (the reference's loops), by a whole wave (the same i0, i1 in every lane;
// i0 a multiple of 4), from LDS, in groups of 64 (add64_rowbcast), the next
// group's values read during the current one's adds.  The values past i1 in
// the last group are +0.0: adding +0.0 leaves any sum whose sign bit is
// clear unchanged, which the callers guarantee (v >= 0, starts of
// non-negative bits).
static __device__ __forceinline__ float seq_chain_lds(const float* v, int i0, int i1, float sum) {
    const int i = threadIdx.x & 15, ng = (i1 - i0 + 63) >> 6;
    float4 x = ng > 0 ? seq_group(v, i0, i1, 0, i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int g = 0; g < ng; g++) {
        const float4 cur = x;
        if (g + 1 < ng) x = seq_group(v, i0, i1, g + 1, i);
        sum = add64_rowbcast(cur, sum);
    }
    return sum;
}

// One DPP move of a double across lanes (lanes the control leaves without a
// source, or outside ROW_MASK, read 0.0).
template <int CTRL, int ROW_MASK = 0xf>
static __device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROW_MASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROW_MASK, 0xf, false);
    return __hiloint2double(hi, lo);
}
// Sum of x over the wave's 64 lanes, complete in lane 63: pairs and quads
// (quad permutations), rows of 8 and 16 (half-row and row mirrors), then
// row 0 into row 1 and row 2 into row 3 (row_bcast15), rows 0-1 into row 3
// (row_bcast31).  VALU lane moves only, no LDS round trips.
static __device__ __forceinline__ double wave_sum_f64(double x) {
    x += dpp_f64<0xb1>(x);       // quad_perm [1,0,3,2]
    x += dpp_f64<0x4e>(x);       // quad_perm [2,3,0,1]
    x += dpp_f64<0x141>(x);      // row_half_mirror
    x += dpp_f64<0x140>(x);      // row_mirror
    x += dpp_f64<0x142, 0xa>(x);  // row_bcast15
    x += dpp_f64<0x143, 0xc>(x);  // row_bcast31
    return x;
}

// The same sequential sum of v[0..n) (0 + v[0] + v[1] + ..., each add
// rounded; n a multiple of 4), by S waves of the workgroup at once (S at
// most the workgroup's waves); every thread calls it, and the result is
// returned to the lanes of wave 0.  The range is cut into S segments of L
// values (whole batches of 64); wave j runs segment j from 64 starting
// values, lane l from the float whose bits are those of c_j plus l - 32, c_j
// being the fp64 sum of v[0 .. jL) rounded to float (wave 0 from the exact
// start, 0).  Wave 0 then walks the segments in order: the exact start of
// segment j is the result of segment j-1, and the lane that started from
// those very bits performed exactly the sequential adds of that segment, so
// its result is taken.  When no lane did (the fp32 chain drifted more than
// 32 ulps from the fp64 sum, as over long runs of equal values), wave 0 runs
// the segment again from the exact start.  For v >= 0 the float bits order
// the values, so the 64 starts are 64 consecutive floats; lane l started
// from max(0, c_j + l - 32), which for the index l = b - c_j + 32 in
// [0, 64) of an exact start with bits b is b itself whenever b >= 0 as an
// integer (a float without its sign bit).  miss != 0 moves every window
// away (each segment then runs again: a test of that path).  scr: S*64
// words of LDS, scr_c: S words.
template <int S>
static __device__ __forceinline__ float seq_sum_spec(const float* v, int n, float* scr, int* scr_c, int miss) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int L = ((n + S - 1) / S + 63) & ~63;
    if (wave < S) {
        const int j0 = min(n, wave * L), j1 = min(n, j0 + L);
        // centre: lane l adds the runs of 16 values at 16 l + 1024 i
        double p = 0.0;
        for (int base = 16 * lane; base < j0; base += 1024) {
            float4 q4[4];
#pragma unroll
            for (int e = 0; e < 4; e++) q4[e] = *(const float4*)(v + min(base + 4 * e, n - 4));
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x[4] = {q4[e].x, q4[e].y, q4[e].z, q4[e].w};
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (base + 4 * e + u < j0) p += (double)x[u];
            }
        }
        const int cb = min(__builtin_amdgcn_readlane((int)__float_as_uint((float)wave_sum_f64(p)), 63), 0x7f800000) +
                       (miss ? (1 << 20) : 0);
        const float s0 = __uint_as_float((uint32_t)(wave == 0 ? 0 : max(0, cb + lane - 32)));
        scr[wave * 64 + lane] = seq_chain_lds(v, j0, j1, s0);
        if (lane == 0) scr_c[wave] = cb;
    }
    __syncthreads();
    float sum = 0.0f;
    if (wave == 0) {
        // the segments' results (lane l holds lane l's) and centres into
        // registers, all read at once (the empty asm keeps the compiler from
        // moving each read down to its step), then the walk reads them across
        // lanes with uniform indices
        float o[S];
        int c[S];
#pragma unroll
        for (int j = 0; j < S; j++) {
            o[j] = scr[j * 64 + lane];
            c[j] = scr_c[j];
        }
#pragma unroll
        for (int j = 0; j < S; j++) {
            c[j] = __builtin_amdgcn_readfirstlane(c[j]);
            asm volatile("" : "+v"(o[j]), "+s"(c[j]));
        }
        // the exact running sum as bits in a scalar register: a step is a
        // few scalar instructions and one lane read
        int sb = __builtin_amdgcn_readfirstlane(__float_as_int(o[0]));  // segment 0: exact in every lane
#pragma unroll
        for (int j = 1; j < S; j++) {
            const int j0 = min(n, j * L), j1 = min(n, j0 + L);
            if (j0 >= j1) break;
            // idx = sb - c_j + 32; a hit when idx is in [0, 64) and sb >= 0
            int nsb, miss, idx;
            asm volatile(
                "s_sub_i32 %[i], %[sb], %[c]\n\t"
                "s_add_i32 %[i], %[i], 32\n\t"
                "s_cmp_lt_u32 %[i], 64\n\t"
                "s_cselect_b32 %[m], 0, 1\n\t"
                "s_cmp_lt_i32 %[sb], 0\n\t"
                "s_cselect_b32 %[m], 1, %[m]\n\t"
                "s_and_b32 %[i], %[i], 63\n\t"
                "v_readlane_b32 %[r], %[o], %[i]"
                : [r] "=s"(nsb), [m] "=&s"(miss), [i] "=&s"(idx)
                : [sb] "s"(sb), [c] "s"(c[j]), [o] "v"(o[j])
                : "scc");
            sb = __builtin_expect(miss, 0)
                     ? __builtin_amdgcn_readfirstlane(__float_as_int(seq_chain_lds(v, j0, j1, __int_as_float(sb))))
                     : nsb;
        }
        sum = __int_as_float(sb);
    }
    return sum;
}

// tmq_expf_tab's 2^(i/32) and tmq_logf_tab's tables kept in LDS: read from
// constant memory with an index a lane, each call waits for a global load
// (and for whatever loads the wave has in flight before it).
struct Exp2TabLds {
    const uint64_t* p;
    __device__ uint64_t operator()(int i) const { return p[i]; }
};
struct LogfTabLds {
    const double* p;
    __device__ double operator()(int j) const { return p[j]; }
};
