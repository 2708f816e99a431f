// mi355_quant_dot: argument checking, kernel selection, and the any-stride
// kernel that serves what no matrix-core kernel takes (transposed A, uint8,
// unaligned e5m2, K below 16 and the like) and short unaligned K.
#include "common.h"
#include <atomic>
#include <mutex>

bool mi355_mfma_gemm_supported(const mi355_quant_dot_desc*, const void*, const void*, const void*);
int mi355_mfma_gemm_launch(const mi355_quant_dot_desc*,
                           const void*,
                           const void*,
                           void*,
                           const float*,
                           const float*,
                           const int32_t*,
                           const int32_t*,
                           const float*,
                           hipStream_t);
bool mi355_ragged_gemm_supported(const mi355_quant_dot_desc*);
bool mi355_ragged_gemm_one_slab(const mi355_quant_dot_desc*);
int mi355_ragged_gemm_launch(const mi355_quant_dot_desc*,
                             const void*,
                             const void*,
                             void*,
                             const float*,
                             const float*,
                             const int32_t*,
                             const int32_t*,
                             const float*,
                             bool,
                             hipStream_t);
bool mi355_dma_gemm_supported(const mi355_quant_dot_desc*, const void*, const void*);
int mi355_dma_gemm_launch(const mi355_quant_dot_desc*,
                          const void*,
                          const void*,
                          void*,
                          const float*,
                          const float*,
                          const int32_t*,
                          const int32_t*,
                          const float*,
                          void*,
                          size_t,
                          int,
                          hipStream_t);
size_t mi355_dma_gemm_workspace(const mi355_quant_dot_desc*);
int mi355_dma_gemm_shares(const mi355_quant_dot_desc*, const void*, const void*, size_t, bool*);
int mi355_dma_gemm_shares_with_room(const mi355_quant_dot_desc*);

namespace {

struct generic_params
{
    const uint8_t* a;
    const uint8_t* b;
    void* c;
    int64_t m, n, k;
    int64_t a_sm, a_sk, b_sk, b_sn, ldc;
    int64_t stride_a, stride_b, stride_c;
    const float* scale_a;
    const float* scale_b;
    const int32_t* colsum_b;
    const int32_t* rowsum_a;
    const float* bias;
    int scale_a_mode, scale_b_mode, zp_a, zp_b;
    int fp8, dequant, out_type; // fp8: 0 integers, 1 e4m3fn, 2 e5m2
    int is_unsigned; // uint8 operands (bare quant_dot only)
};

MI355_DEVINL float decode_operand(uint8_t raw, const generic_params& p)
{
    if(p.fp8 == 1)
        return fp8_to_f32(raw);
    if(p.fp8 == 2)
        return bf8_to_f32(raw);
    return p.is_unsigned ? (float)raw : (float)(int8_t)raw;
}

// 16 x 16 outputs per workgroup, K walked in steps of 16 through LDS.  int8
// accumulates in int32 (exact); fp8 accumulates in double, which holds the
// sum exactly for any K this path sees, as the ref target's double
// accumulator does.
__global__ __launch_bounds__(256) void quant_dot_generic_kernel(generic_params p)
{
    __shared__ float as[16][17];
    __shared__ float bs[16][17];
    const int tx = threadIdx.x & 15;
    const int ty = threadIdx.x >> 4;
    const int64_t row = (int64_t)blockIdx.y * 16 + ty;
    const int64_t col = (int64_t)blockIdx.x * 16 + tx;
    const uint8_t* a  = p.a + (int64_t)blockIdx.z * p.stride_a;
    const uint8_t* b  = p.b + (int64_t)blockIdx.z * p.stride_b;
    int32_t iacc = 0;
    double facc  = 0.0;
    for(int64_t k0 = 0; k0 < p.k; k0 += 16)
    {
        // as[ty][tx] = A[row, k0 + tx];  bs[ty][tx] = B[k0 + ty, col]
        float av = 0.f, bv = 0.f;
        if(row < p.m && k0 + tx < p.k)
        {
            uint8_t raw = a[row * p.a_sm + (k0 + tx) * p.a_sk];
            av          = decode_operand(raw, p);
        }
        if(col < p.n && k0 + ty < p.k)
        {
            uint8_t raw = b[(k0 + ty) * p.b_sk + col * p.b_sn];
            bv          = decode_operand(raw, p);
        }
        as[ty][tx] = av;
        bs[ty][tx] = bv;
        __syncthreads();
        if(p.fp8)
        {
#pragma unroll
            for(int kk = 0; kk < 16; kk++)
                facc += (double)as[ty][kk] * (double)bs[kk][tx];
        }
        else
        {
#pragma unroll
            for(int kk = 0; kk < 16; kk++)
                iacc += (int32_t)as[ty][kk] * (int32_t)bs[kk][tx];
        }
        __syncthreads();
    }
    if(row >= p.m || col >= p.n)
        return;
    const int64_t idx = (int64_t)blockIdx.z * p.stride_c + row * p.ldc + col;
    if(!p.dequant)
    {
        if(p.fp8)
            static_cast<float*>(p.c)[idx] = (float)facc;
        else
            static_cast<int32_t*>(p.c)[idx] = iacc;
        return;
    }
    float sa = 1.f, sb = 1.f;
    if(p.scale_a_mode == MI355_QP_PER_TENSOR)
        sa = p.scale_a[0];
    else if(p.scale_a_mode == MI355_QP_PER_ROW)
        sa = p.scale_a[row];
    if(p.scale_b_mode == MI355_QP_PER_TENSOR)
        sb = p.scale_b[0];
    else if(p.scale_b_mode == MI355_QP_PER_COL)
        sb = p.scale_b[col];
    const float s = sa * sb;
    double d;
    if(p.fp8)
    {
        // the ref target rounds the accumulator to float (quant_dot's output
        // type) before dequantizelinear reads it
        d = (double)(float)facc;
    }
    else
    {
        int64_t zp = 0;
        if(p.zp_a != 0)
            zp += (int64_t)p.zp_a * p.colsum_b[col];
        if(p.zp_b != 0)
            zp += (int64_t)p.zp_b * p.rowsum_a[row];
        if(p.zp_a != 0 && p.zp_b != 0)
            zp -= p.k * (int64_t)p.zp_a * p.zp_b;
        d = (double)iacc - (double)(int32_t)zp;
    }
    float v = (float)(d * (double)s);
    if(p.bias != nullptr)
        v = add_bias(v, p.bias[col]);
    switch(p.out_type)
    {
    case MI355_F32: static_cast<float*>(p.c)[idx] = v; break;
    case MI355_F16: static_cast<uint16_t*>(p.c)[idx] = convert_f32_to_half(v); break;
    case MI355_BF16: static_cast<uint16_t*>(p.c)[idx] = convert_f32_to_bf16(v); break;
    default: break;
    }
}

// out[i] = sum over `len` int8 elements, element j of vector i at
// base + i*stride_i + j*stride_j.  One wave per output.
__global__ __launch_bounds__(256) void sum_i8_kernel(
    const int8_t* base, int64_t count, int64_t len, int64_t stride_i, int64_t stride_j, int32_t* out)
{
    const int lane    = threadIdx.x & 63;
    const int64_t vec = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if(vec >= count)
        return;
    const int8_t* p = base + vec * stride_i;
    int32_t s       = 0;
    for(int64_t j = lane; j < len; j += 64)
        s += p[j * stride_j];
#pragma unroll
    for(int off = 32; off > 0; off >>= 1)
        s += __shfl_xor(s, off, 64);
    if(lane == 0)
        out[vec] = s;
}

// column sums of row-major [K, N]: consecutive threads take consecutive
// columns so every row read is coalesced; K is split over blockIdx.y slices
// that combine with integer atomics (exact, order independent).
__global__ __launch_bounds__(256) void colsum_rowmajor_kernel(
    const int8_t* b, int64_t k, int64_t n, int64_t ldb, int64_t k_per_slice, int32_t* out)
{
    const int64_t col = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if(col >= n)
        return;
    const int64_t k0 = (int64_t)blockIdx.y * k_per_slice;
    const int64_t k1 = min(k, k0 + k_per_slice);
    int32_t s        = 0;
    for(int64_t kk = k0; kk < k1; kk++)
        s += b[kk * ldb + col];
    atomicAdd(out + col, s);
}

// What a product takes (us) in the kernels that compete for it, fitted to 11800 products on one MI355X: M
// of 1 to 4096, N of 16 to 28672, K of 16 to 28672 over weights that no cache holds, and 2 to 384
// batches that one may hold; both types, both orders of B, with and without epilogue and workspace.
// Nine products in ten take 0.9 to 1.15 times their fit (shares added into C: 0.8 to 1.3).
//   fixed       launch, and the first loads' way
//   wave        a round of workgroups over the chip: a tile's prologue and epilogue, and `rows` for the part
//               of the epilogue that a tile's rows and columns fill
//   k_wave      per step of K in every round; k_fill: and in proportion to the workgroups, not the rounds
//   b_mb, out_m per MB of B from memory, per million outputs
struct fit
{
    double fixed, wave, rows, k_wave, k_fill, b_mb, out_m;
};

double fitted_us(const fit& f, const mi355_quant_dot_desc* d, double fill, double rows, double k)
{
    const double waves = __builtin_ceil(fill);
    return f.fixed + waves * (f.wave + rows * f.rows + k * f.k_wave) + fill * k * f.k_fill +
           (double)d->batch * (double)d->n * (double)d->k * 1e-6 * f.b_mb +
           (double)d->batch * (double)d->m * (double)d->n * 1e-6 * f.out_m;
}

// tiles of a product; the share of a tile's or wave's `side` that a dimension fills
double tiles_of(const mi355_quant_dot_desc* d, int64_t side)
{
    return (double)d->batch * (double)((d->m + side - 1) / side) * (double)((d->n + side - 1) / side);
}

double part(int64_t dim, double side) { return __builtin_fmin((double)dim, side) / side; }

// The register-staged kernel (qgemm_ragged.hip), tiles of 64 x 64, or 128 x 128 where those fill the chip.  A
// workgroup of it starts sooner and several share a CU, so it wins wherever the 256 x 256 tiles of
// the other two leave CUs idle or are mostly padding, and where K is short:
//   96 batches of 197 x 197 x 64 int8 -> float   23.7 -> 11.3 us     384 of 64 x 64 x 64   19.7 -> 8.2
//   1024 x 1024 x 1024 int8 -> bfloat16          23.5 -> 6.5         512 x 4096 x 4096 (split)   30.9 -> 21.3
//   48 x 1024 x 1024 x 128                       49.8 against 53.7 (stays)
// It never splits K: few tiles of a long K stay with shares (5 x 192 x 25472 int8: 79.9 against 16.4 us).
double two_slab_us(const mi355_quant_dot_desc* d)
{
    const int deq = d->dequant != 0, tb = d->trans_b != 0;
    const double k = (double)d->k;
    // (the kernel's own choice of the tile; two of the large ones share a CU)
    if(const double big = tiles_of(d, 128); big >= 256)
    {
        // [epilogue][B as [N, K]]
        static const fit large[2][2] = {
            {{3.8, 0.15, 1.4, 0.0099, 0.0030, 0.120, 0.61}, {3.8, 0.25, 1.3, 0.0082, 0.0027, 0.110, 0.62}},
            {{3.4, 2.1, 1.8, 0.0080, 0.0052, 0.130, 0.29}, {3.5, 2.2, 1.8, 0.0083, 0.0028, 0.083, 0.33}}};
        return fitted_us(large[deq][tb], d, big / 512.0, part(d->m, 128.0), k);
    }
    // A second workgroup on a CU costs less of K than the first.  Rows of a row-major B that lie a
    // multiple of 1 KiB apart meet in few of the memory's channels: 16 x 2048 x 8192 34.8 us, where other
    // N of that size take 29.
    static const fit small[2][2] = {{{3.4, 0.1, 0.2, 0, 0, 0, 1.04}, {3.4, 0.2, 0.2, 0, 0, 0, 0.90}},
                                    {{3.95, 0.2, 0.6, 0, 0, 0, 0.63}, {3.95, 0.3, 0.45, 0, 0, 0, 0.68}}};
    const bool pitched = !tb && d->ldb % 1024 == 0;
    const double fill  = tiles_of(d, 64) / 256.0;
    fit f              = small[deq][tb];
    f.k_wave           = tb ? 0.0016 : pitched ? 0.0018 : 0.0026;
    f.b_mb             = tb ? 0.080 : fill > 1.0 ? 0.170 : 0.100;
    const double first = tb ? 0.0020 : pitched ? 0.0036 : 0.0030;
    return fitted_us(f, d, fill, part(d->m, 64.0), k) + (first - f.k_wave) * k;
}

// The same kernel with K in one slab where it has one: a start, the tiles, the results, and what of those no cache
// takes; many tiles of bare results take longer (1300 random products of up to 128 of K: nine in ten take 0.85 to 1.25
// times that).  It is hardly ever the slower one, so what two slabs would win stays won.
double ragged_us(const mi355_quant_dot_desc* d)
{
    const double two = two_slab_us(d);
    if(!mi355_ragged_gemm_one_slab(d))
        return two;
    const double tiles = tiles_of(d, 64);
    const double out   = (double)d->batch * (double)d->m * (double)d->n * 1e-6;
    const double mb    = out * (d->dequant && d->out_type != MI355_F32 ? 2.0 : 4.0);
    double one = (d->dequant ? 3.8 : 3.0) + 0.0016 * tiles + 0.25 * out + (mb > 200.0 ? 0.17 * (mb - 200.0) : 0.0);
    if(!d->dequant && tiles > 4096.0)
        one = __builtin_fmax(one, 4.6 + tiles * (d->k <= 64 ? 0.0029 : 0.0037));
    return __builtin_fmin(two, one);
}

// direct-to-LDS kernels; `shares` of K through a workspace, or added into C
double dma_us(const mi355_quant_dot_desc* d, int shares, bool atomic)
{
    // [epilogue]: one pass with eight waves, and with four from K = 3072 on
    static const fit i8[2]   = {{2.0, 3.5, 0.6, 0.0113, 0.0010, 0.060, 0.49}, {3.2, 2.5, 6.7, 0.0106, 0, 0.120, 0.48}};
    static const fit i8_4[2] = {{3.8, 0, 11.8, 0.0089, 0.0025, 0.030, 0}, {4.1, 13.2, 2.0, 0.0081, 0.0040, 0.020, 0.05}};
    static const fit f8[2]   = {{3.9, 0, 2.0, 0.0100, 0, 0.090, 0.92}, {2.7, 3.2, 2.6, 0.0098, 0.0017, 0.070, 0.41}};
    static const fit f8_4[2] = {{4.7, 8.2, 7.0, 0.0071, 0.0038, 0.073, 0}, {2.0, 11.8, 6.5, 0.0074, 0.0030, 0.073, 0}};
    static const fit i8_shares = {0, 8.0, 2.7, 0.0098, 0, 0.074, 0.7}, f8_shares = {0, 7.5, 3.1, 0.0087, 0, 0.095, 1.1};
    const bool fp8     = d->in_type == MI355_FP8;
    const double fill  = tiles_of(d, 256) * shares / 256.0;
    const double rows  = part(d->m, 128.0);
    const double k     = (double)d->k / shares;
    const double sums  = (double)shares * (double)d->batch * (double)d->m * (double)d->n * 1e-6;
    if(atomic) // at most two rounds; clearing C, then the slower of the shares and of B's way through so few CUs
        return __builtin_fmax((double)d->batch * (double)d->n * (double)d->k * 1e-6 * 0.37,
                              5.3 + 11.3 * rows + k * (0.0129 + 0.003 * fill) + 0.76 * sums + 5.7 * fill);
    if(shares > 1)
        return fitted_us(fp8 ? f8_shares : i8_shares, d, fill, rows, k) + (fp8 ? 1.75 : 1.51) * sums;
    const fit* one = d->k >= 3072 && d->n % 4 == 0 ? (fp8 ? f8_4 : i8_4) : (fp8 ? f8 : i8);
    return fitted_us(one[d->dequant != 0], d, fill, rows * part(d->n, 64.0), k);
}

// the matrix-core kernel for K that is no multiple of 64
double mfma_us(const mi355_quant_dot_desc* d)
{
    static const fit i8[2] = {{3.2, 1.6, 2.7, 0.0152, 0.0023, 0.080, 0.41}, {3.2, 2.0, 8.7, 0.0153, 0.0015, 0.090, 0.37}};
    static const fit f8[2] = {{2.1, 2.2, 1.0, 0.0145, 0.0022, 0.120, 0.55}, {3.4, 1.7, 6.7, 0.0149, 0.0010, 0.120, 0.36}};
    return fitted_us((d->in_type == MI355_FP8 ? f8 : i8)[d->dequant != 0], d, tiles_of(d, 256) / 256.0,
                     part(d->m, 128.0), (double)d->k);
}

// A vector of column scales per batch entry exists in the direct-to-LDS kernels only.  `left` of the time is
// left to the fits' errors, a fourteenth, against shares of K a tenth: so 28 of the 11800 products take
// over 1.05 times what the other kernel does (1.27 at most), and 141 miss a tenth and more.
bool ragged_is_faster(const mi355_quant_dot_desc* d, double other_us, double left)
{
    return d->k > 0 && mi355_ragged_gemm_supported(d) &&
           !(d->dequant && d->scale_b_mode == MI355_QP_PER_COL_BATCH) && ragged_us(d) < (1.0 - left) * other_us;
}

// Matrices aligned to nothing: the any-stride kernel, whose blocks of 16 x 16 outputs start at once, against
// the register-staged one, whose first barrier stands behind a slab that a short K hardly fills (fitted
// to 500 products of K below 128; the results are the same bits).  44 x 87 x 16 fp8 with the epilogue 5.7
// against 3.5 us, 74 x 7 x 31 int8 6.0 against 4.0; from K = 80 on the register-staged kernel is the faster
// one at any size.
bool short_k_is_faster(const mi355_quant_dot_desc* d)
{
    if(d->k >= 128 || (d->m + 15) / 16 > 65535)
        return false;
    const bool fp8   = d->in_type == MI355_FP8;
    const double k   = (double)d->k;
    const double out = (double)d->batch * (double)d->m * (double)d->n * 1e-6;
    const double any = 3.0 + 0.036 * k + tiles_of(d, 16) / 2048.0 * (1.8 + 0.06 * k);
    const double staged =
        fp8 ? (d->dequant ? 5.7 : 5.0) + 0.0015 * k + tiles_of(d, 64) / 256.0 * (0.7 + 0.013 * k) + 1.4 * out
            : (d->dequant ? 5.3 : 4.25) + 0.0007 * k + 1.9 * out;
    return any < staged;
}

size_t small_tile_bytes(const mi355_quant_dot_desc* d, int shares)
{
    return (size_t)shares * (size_t)d->m * (size_t)((d->n + 3) / 4 * 4) * 4;
}

// Shares of K in 128 x 128 tiles (qgemm_shares.h), 1 where another kernel is the faster one: what a slab of 128
// costs a workgroup alone on its CU, the partial sums' way, and a start that grows with the workgroups, fitted to 40
// products of 20 to 1000 rows (within 10 %), against the fits above.  Not beyond one workgroup a CU, whose partial
// sums are 16 MiB at most; from 65 tiles on two or three shares gain nothing (512 x 4096 x 4096 28.0 us in one pass of
// 64 x 64 tiles).  Any count that leaves every share a slab, the last one fewer than the others; fp8 sums, whose bits
// depend on the slices, keep equal ones as the 256 x 256 kernels cut them (a count that divides K / 64), or none,
// unless that takes a third longer: 344 x 400 x 6016 in 2 16.4 us, in 8 13.1; 8 x 32 x 9664 (151 halves of a slab)
// unsplit 30.5, in shares 7.0.
// A function of the shape, B's order and the operands' types alone (the fits look at dense matrices, whatever the
// distance of the rows), so that the size asked for ahead of a call is that of the call.
int small_tile_shares(const mi355_quant_dot_desc* d0)
{
    if((d0->in_type != MI355_I8 && d0->in_type != MI355_FP8) || d0->batch != 1 || d0->trans_a || d0->m <= 0 ||
       d0->n <= 0 || d0->k < 1024 || d0->k % 64 != 0 || d0->m > (1 << 30) || d0->n > (1 << 30) || d0->k > (1 << 30) ||
       (!d0->trans_b && d0->n % 16 != 0) || (d0->dequant && d0->scale_b_mode == MI355_QP_PER_COL_BATCH))
        return 1;
    mi355_quant_dot_desc d = *d0;
    d.dequant              = 0;
    d.lda                  = d.k;
    d.ldb                  = d.trans_b ? d.k : d.n;
    d.ldc                  = d.n;
    const double tiles     = tiles_of(&d, 128);
    if(tiles > 64)
        return 1;
    const int slabs = (int)((d.k + 127) / 128);
    const double mb = (double)d.m * (double)d.n * 4e-6;
    double any_us = 0, equal_us = 0;
    int any = 1, equal = 1;
    for(int s = 2; s * tiles <= 256 && s <= slabs / 2; s++)
    {
        const int per = (slabs + s - 1) / s;
        if((slabs + per - 1) / per != s)
            continue;
        const double us = 5.6 + 0.011 * s * tiles + per * (0.6 + 0.0004 * s * tiles) + 0.38 * s * mb;
        if(any == 1 || us < any_us)
        {
            any_us = us;
            any    = s;
        }
        if(d.k / 64 % s == 0 && (equal == 1 || us < equal_us))
        {
            equal_us = us;
            equal    = s;
        }
    }
    if(any == 1)
        return 1;
    double other = dma_us(&d, mi355_dma_gemm_shares_with_room(&d), false);
    if(mi355_ragged_gemm_supported(&d))
        other = __builtin_fmin(other, ragged_us(&d));
    if(d.in_type == MI355_FP8 && any_us >= 0.75 * (equal > 1 ? __builtin_fmin(equal_us, other) : other))
    {
        any    = equal;
        any_us = equal_us;
    }
    return any > 1 && any_us < 0.9 * other ? any : 1;
}

// the same for a call, whose workspace has to hold them
int small_tile_shares(const mi355_quant_dot_desc* d, const void* workspace, size_t workspace_bytes)
{
    if(workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
        return 1;
    const int shares = small_tile_shares(d);
    return shares > 1 && small_tile_bytes(d, shares) <= workspace_bytes ? shares : 1;
}

__global__ void zero_i32_kernel(int32_t* p, int64_t n)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n)
        p[i] = 0;
}

} // namespace

extern "C" int mi355_quant_dot(const mi355_quant_dot_desc* d,
                               const void* a,
                               const void* b,
                               void* c,
                               const float* scale_a,
                               const float* scale_b,
                               const int32_t* colsum_b,
                               const int32_t* rowsum_a,
                               void* stream)
{
    return mi355_quant_dot_bias(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, nullptr, stream);
}

extern "C" int mi355_quant_dot_bias(const mi355_quant_dot_desc* d,
                                    const void* a,
                                    const void* b,
                                    void* c,
                                    const float* scale_a,
                                    const float* scale_b,
                                    const int32_t* colsum_b,
                                    const int32_t* rowsum_a,
                                    const float* bias,
                                    void* stream)
{
    return mi355_quant_dot_ws(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, nullptr, 0, stream);
}

extern "C" size_t mi355_quant_dot_workspace_size(const mi355_quant_dot_desc* d)
{
    if(d == nullptr)
        return 0;
    const int shares = small_tile_shares(d);
    return shares > 1 ? small_tile_bytes(d, shares) : mi355_dma_gemm_workspace(d);
}

namespace {

// which kernel a call runs
enum class kernel_id : int
{
    none         = 0, // nothing to compute
    generic      = 1,
    ragged       = 2, // register-staged; fp8 sums in float
    ragged_exact = 3, // fp8 sums exact
    mfma         = 4,
    dma          = 5, // direct-to-LDS, one pass over K
    dma_shares   = 6, // K in shares through the workspace
    dma_atomic   = 7  // K in shares added into C
};

bool dma_takes(const mi355_quant_dot_desc* d, const void* a, const void* b, const float* bias)
{
    // int8 with N % 4 != 0 would take the DMA path's 32 x 32 kernel, which applies no bias
    const bool fp8 = d->in_type == MI355_FP8;
    return (fp8 || d->in_type == MI355_I8) && d->k > 0 && (bias == nullptr || fp8 || d->n % 4 == 0) &&
           mi355_dma_gemm_supported(d, a, b);
}

bool mfma_takes(const mi355_quant_dot_desc* d, const void* a, const void* b, const void* c)
{
    return d->in_type != MI355_U8 && d->k > 0 && !(d->dequant && d->scale_b_mode == MI355_QP_PER_COL_BATCH) &&
           mi355_mfma_gemm_supported(d, a, b, c);
}

// argument checks and the choice of the kernel, and for dma_shares of the tiles: *small shares in those of 128 x 128
// (1: 256 x 256); the pointers are looked at, not through
int choose_kernel(const mi355_quant_dot_desc* d,
                  const void* a,
                  const void* b,
                  const void* c,
                  const float* scale_a,
                  const float* scale_b,
                  const int32_t* colsum_b,
                  const int32_t* rowsum_a,
                  const float* bias,
                  const void* workspace,
                  size_t workspace_bytes,
                  kernel_id* kernel,
                  int* small)
{
    if(d == nullptr)
        return MI355_ERR_BAD_ARG;
    if(d->m < 0 || d->n < 0 || d->k < 0 || d->batch < 0)
        return MI355_ERR_BAD_ARG;
    const bool empty = d->m == 0 || d->n == 0 || d->batch == 0;
    if(!empty && (a == nullptr || b == nullptr || c == nullptr))
        return MI355_ERR_BAD_ARG;
    if(d->in_type != MI355_I8 && d->in_type != MI355_FP8 && d->in_type != MI355_U8 &&
       d->in_type != MI355_BF8)
        return MI355_ERR_UNSUPPORTED;
    // e5m2 x e5m2 -> float (op/quant_dot.hpp:62-66 takes every fp8 type): the 16x16x128 MFMA
    // kernel or the generic one
    const bool bf8 = d->in_type == MI355_BF8;
    const bool fp8 = d->in_type == MI355_FP8 || bf8;
    // uint8 x uint8 -> int32 (op/quant_dot.hpp:62-64 lists it): bare result only, correctness path
    const bool u8 = d->in_type == MI355_U8;
    if(u8 && d->dequant)
        return MI355_ERR_UNSUPPORTED;
    if(bias != nullptr && !d->dequant)
        return MI355_ERR_BAD_ARG; // the bias is a float added to the dequantized value
    if(d->dequant)
    {
        if(d->out_type != MI355_F32 && d->out_type != MI355_F16 && d->out_type != MI355_BF16)
            return MI355_ERR_BAD_ARG;
        if(d->scale_a_mode != MI355_QP_NONE && d->scale_a_mode != MI355_QP_PER_TENSOR &&
           d->scale_a_mode != MI355_QP_PER_ROW)
            return MI355_ERR_BAD_ARG;
        if(d->scale_b_mode != MI355_QP_NONE && d->scale_b_mode != MI355_QP_PER_TENSOR &&
           d->scale_b_mode != MI355_QP_PER_COL && d->scale_b_mode != MI355_QP_PER_COL_BATCH)
            return MI355_ERR_BAD_ARG;
        if(d->scale_a_mode != MI355_QP_NONE && scale_a == nullptr)
            return MI355_ERR_BAD_ARG;
        if(d->scale_b_mode != MI355_QP_NONE && scale_b == nullptr)
            return MI355_ERR_BAD_ARG;
        if(fp8 && (d->zp_a != 0 || d->zp_b != 0))
            return MI355_ERR_UNSUPPORTED;
        if(d->zp_a != 0 && colsum_b == nullptr)
            return MI355_ERR_BAD_ARG;
        if(d->zp_b != 0 && rowsum_a == nullptr)
            return MI355_ERR_BAD_ARG;
        if(d->zp_a < -128 || d->zp_a > 127 || d->zp_b < -128 || d->zp_b > 127)
            return MI355_ERR_BAD_ARG;
        if((d->zp_a != 0 || d->zp_b != 0) && d->batch > 1)
            return MI355_ERR_UNSUPPORTED; // sums are given for one matrix
    }
    else
    {
        if(d->out_type != (fp8 ? MI355_F32 : MI355_I32))
            return MI355_ERR_BAD_ARG;
    }
    *kernel = kernel_id::none;
    *small  = 1;
    if(empty)
        return MI355_OK;
    if(d->ldc < d->n)
        return MI355_ERR_BAD_ARG;
    if((d->trans_a ? d->lda < d->m : d->lda < d->k) || (d->trans_b ? d->ldb < d->k : d->ldb < d->n))
        return MI355_ERR_BAD_ARG;
    if(d->batch > 65535)
        return MI355_ERR_UNSUPPORTED;

    if(dma_takes(d, a, b, bias))
    {
        // fp8: the sums of all are float
        *small = small_tile_shares(d, workspace, workspace_bytes);
        if(*small > 1)
        {
            *kernel = kernel_id::dma_shares;
            return MI355_OK;
        }
        bool atomic      = false;
        const int shares = mi355_dma_gemm_shares(d, c, workspace, workspace_bytes, &atomic);
        // results of a short K whose rows are no whole groups of 4 leave these kernels element by element: 2 to 5 times
        // the register-staged kernel's time (7187 x 24363 x 64 int8 519 us against 254, 14 x 882 x 882 x 64 fp8 46 against 12)
        const bool broken_rows = d->trans_b && d->k <= 128 && d->n % 4 != 0;
        if(ragged_is_faster(d, broken_rows ? HUGE_VAL : dma_us(d, shares, atomic), shares > 1 ? 0.1 : 0.07))
            *kernel = kernel_id::ragged;
        else
            *kernel = shares == 1 ? kernel_id::dma : atomic ? kernel_id::dma_atomic : kernel_id::dma_shares;
        return MI355_OK;
    }
    // a vector of column scales per batch entry exists in the kernels above only
    if(d->dequant && d->scale_b_mode == MI355_QP_PER_COL_BATCH)
        return MI355_ERR_UNSUPPORTED;
    if(mfma_takes(d, a, b, c))
    {
        *kernel = !bf8 && ragged_is_faster(d, mfma_us(d), 0.07) ? kernel_id::ragged : kernel_id::mfma;
        return MI355_OK;
    }
    // rows aligned to nothing; fp8 sums stay exact there, as in the generic kernel
    if(mi355_ragged_gemm_supported(d) && !short_k_is_faster(d))
    {
        *kernel = kernel_id::ragged_exact;
        return MI355_OK;
    }
    *kernel = kernel_id::generic;
    return (d->m + 15) / 16 > 65535 ? MI355_ERR_UNSUPPORTED : MI355_OK;
}

} // namespace

namespace {

int launch_kernel(kernel_id kernel,
                  int small, // as choose_kernel gives it
                  const mi355_quant_dot_desc* d,
                  const void* a,
                  const void* b,
                  void* c,
                  const float* scale_a,
                  const float* scale_b,
                  const int32_t* colsum_b,
                  const int32_t* rowsum_a,
                  const float* bias,
                  void* workspace,
                  size_t workspace_bytes,
                  hipStream_t s)
{
    switch(kernel)
    {
    case kernel_id::none: return MI355_OK;
    case kernel_id::ragged:
    case kernel_id::ragged_exact:
        return mi355_ragged_gemm_launch(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias,
                                        kernel == kernel_id::ragged, s);
    case kernel_id::mfma:
        return mi355_mfma_gemm_launch(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, s);
    case kernel_id::dma:
    case kernel_id::dma_shares:
    case kernel_id::dma_atomic:
        return mi355_dma_gemm_launch(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, workspace,
                                     workspace_bytes, small, s);
    case kernel_id::generic: break;
    }

    generic_params p;
    p.a            = static_cast<const uint8_t*>(a);
    p.b            = static_cast<const uint8_t*>(b);
    p.c            = c;
    p.m            = d->m;
    p.n            = d->n;
    p.k            = d->k;
    p.a_sm         = d->trans_a ? 1 : d->lda;
    p.a_sk         = d->trans_a ? d->lda : 1;
    p.b_sk         = d->trans_b ? 1 : d->ldb;
    p.b_sn         = d->trans_b ? d->ldb : 1;
    p.ldc          = d->ldc;
    p.stride_a     = d->stride_a;
    p.stride_b     = d->stride_b;
    p.stride_c     = d->stride_c;
    p.scale_a      = scale_a;
    p.scale_b      = scale_b;
    p.colsum_b     = colsum_b;
    p.rowsum_a     = rowsum_a;
    p.bias         = bias;
    p.scale_a_mode = d->scale_a_mode;
    p.scale_b_mode = d->scale_b_mode;
    p.zp_a         = d->zp_a;
    p.zp_b         = d->zp_b;
    p.fp8          = d->in_type == MI355_BF8 ? 2 : d->in_type == MI355_FP8 ? 1 : 0;
    p.is_unsigned  = d->in_type == MI355_U8;
    p.dequant      = d->dequant;
    p.out_type     = d->out_type;
    const int64_t gx = (d->n + 15) / 16, gy = (d->m + 15) / 16;
    dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)d->batch);
    hipLaunchKernelGGL(quant_dot_generic_kernel, grid, dim3(256), 0, s, p);
    return mi355_launch_status();
}

} // namespace

extern "C" int mi355_quant_dot_ws(const mi355_quant_dot_desc* d,
                                  const void* a,
                                  const void* b,
                                  void* c,
                                  const float* scale_a,
                                  const float* scale_b,
                                  const int32_t* colsum_b,
                                  const int32_t* rowsum_a,
                                  const float* bias,
                                  void* workspace,
                                  size_t workspace_bytes,
                                  void* stream)
{
    kernel_id kernel = kernel_id::none;
    int small        = 1;
    const int status = choose_kernel(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, workspace,
                                     workspace_bytes, &kernel, &small);
    return status != MI355_OK ? status
                              : launch_kernel(kernel, small, d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias,
                                              workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

// The four below are not part of the public interface.  Tests ask the first, without a GPU, which kernel their
// shapes reach (the kernel_id, or the call's negative status), the second how many shares a workspace of those bytes
// has in 128 x 128 tiles (1: none), the third what 256 x 256 tiles would ask for, and with the fourth run the edges of
// a kernel at sizes that the rules leave to another (the product, or MI355_ERR_UNSUPPORTED where the
// kernel does not take it).
extern "C" int mi355_internal_quant_dot_kernel(const mi355_quant_dot_desc* d,
                                               const void* a,
                                               const void* b,
                                               const void* c,
                                               const float* scale_a,
                                               const float* scale_b,
                                               const int32_t* colsum_b,
                                               const int32_t* rowsum_a,
                                               const float* bias,
                                               const void* workspace,
                                               size_t workspace_bytes)
{
    kernel_id kernel = kernel_id::none;
    int small        = 1;
    const int status = choose_kernel(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, workspace,
                                     workspace_bytes, &kernel, &small);
    return status == MI355_OK ? (int)kernel : status;
}

extern "C" int mi355_internal_quant_dot_small_shares(const mi355_quant_dot_desc* d, size_t workspace_bytes)
{
    const int shares = small_tile_shares(d);
    return shares > 1 && small_tile_bytes(d, shares) <= workspace_bytes ? shares : 1;
}

extern "C" size_t mi355_internal_quant_dot_large_workspace(const mi355_quant_dot_desc* d)
{
    return mi355_dma_gemm_workspace(d);
}

extern "C" int mi355_internal_quant_dot_run(int32_t which,
                                            const mi355_quant_dot_desc* d,
                                            const void* a,
                                            const void* b,
                                            void* c,
                                            const float* scale_a,
                                            const float* scale_b,
                                            const int32_t* colsum_b,
                                            const int32_t* rowsum_a,
                                            const float* bias,
                                            void* workspace,
                                            size_t workspace_bytes,
                                            void* stream)
{
    kernel_id kernel = kernel_id::none;
    int small        = 1;
    const int status = choose_kernel(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, workspace,
                                     workspace_bytes, &kernel, &small);
    if(status != MI355_OK || kernel == kernel_id::none)
        return status;
    bool takes = false;
    switch(static_cast<kernel_id>(which))
    {
    case kernel_id::dma: takes = dma_takes(d, a, b, bias); break;
    case kernel_id::mfma: takes = mfma_takes(d, a, b, c); break;
    case kernel_id::ragged:
    case kernel_id::ragged_exact:
        takes = mi355_ragged_gemm_supported(d) && !(d->dequant && d->scale_b_mode == MI355_QP_PER_COL_BATCH);
        break;
    default: break;
    }
    return !takes ? MI355_ERR_UNSUPPORTED
                  : launch_kernel(static_cast<kernel_id>(which), 1, d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a,
                                  bias, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

// ---- quant_dot that allocates nothing and takes no workspace -------------------------------
// The split-K partial sums of mi355_quant_dot_ws go to a device array that is part of the
// library's code object: every GPU the library runs on holds its own copy from the moment the
// module is loaded there until the process ends.  In host code the array's name only stands for
// the symbol; the memory is reached through the address hipGetSymbolAddress reports on the
// device that is current, looked up once per device and kept.
static __device__ __align__(256) unsigned char scratch[MI355_QUANT_DOT_STATIC_SCRATCH_BYTES];

namespace {
constexpr int max_devices = 64;
std::atomic<void*> scratch_of_device[max_devices];
std::mutex scratch_lookup;

// address of this device's copy of `scratch`; null with *status set when HIP reports an error
void* device_scratch(int* status)
{
    int dev = -1;
    if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= max_devices)
    {
        *status = MI355_ERR_LAUNCH;
        return nullptr;
    }
    void* ptr = scratch_of_device[dev].load(std::memory_order_acquire);
    if(ptr != nullptr)
        return ptr;
    std::lock_guard<std::mutex> guard(scratch_lookup);
    ptr = scratch_of_device[dev].load(std::memory_order_acquire);
    if(ptr != nullptr)
        return ptr;
    if(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr)
    {
        (void)hipGetLastError();
        *status = MI355_ERR_LAUNCH;
        return nullptr;
    }
    scratch_of_device[dev].store(ptr, std::memory_order_release);
    return ptr;
}
} // namespace

extern "C" int mi355_quant_dot_static(const mi355_quant_dot_desc* d,
                                      const void* a,
                                      const void* b,
                                      void* c,
                                      const float* scale_a,
                                      const float* scale_b,
                                      const int32_t* colsum_b,
                                      const int32_t* rowsum_a,
                                      const float* bias,
                                      void* stream)
{
    if(d == nullptr)
        return MI355_ERR_BAD_ARG;
    // By the need of the 256 x 256 tiles, whatever the smaller ones ask for: callers rely on what is refused, and on
    // what shares nothing with a call on another stream, and neither follows the choice of a tile.
    const size_t large = mi355_dma_gemm_workspace(d);
    if(large > MI355_QUANT_DOT_STATIC_SCRATCH_BYTES)
        return MI355_ERR_SCRATCH_TOO_SMALL;
    const size_t need = mi355_quant_dot_workspace_size(d);
    if(large == 0) // no split for this description: the one-pass kernels use no scratch memory
        return mi355_quant_dot_ws(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, nullptr, 0, stream);
    int status = MI355_OK;
    void* ptr  = device_scratch(&status);
    if(ptr == nullptr)
        return status;
    // every element of the partial sums that the second kernel reads is stored by the first one in
    // the same call, so nothing has to be cleared between calls
    return mi355_quant_dot_ws(d, a, b, c, scale_a, scale_b, colsum_b, rowsum_a, bias, ptr, need, stream);
}

extern "C" int mi355_colsum_i8(const void* b,
                               int64_t k,
                               int64_t n,
                               int64_t ldb,
                               int32_t trans_b,
                               int32_t* out,
                               void* stream)
{
    if(b == nullptr || out == nullptr || k < 0 || n < 0)
        return MI355_ERR_BAD_ARG;
    if(n == 0)
        return MI355_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if(trans_b)
    {
        // [N, K] storage: each column is a contiguous K run
        hipLaunchKernelGGL(sum_i8_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s,
                           static_cast<const int8_t*>(b), n, k, ldb, (int64_t)1, out);
        return mi355_launch_status();
    }
    hipLaunchKernelGGL(zero_i32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, out, n);
    if(k == 0)
        return mi355_launch_status();
    int64_t slices      = (k + 255) / 256;
    if(slices > 64)
        slices = 64;
    int64_t k_per_slice = (k + slices - 1) / slices;
    slices              = (k + k_per_slice - 1) / k_per_slice;
    hipLaunchKernelGGL(colsum_rowmajor_kernel, dim3((unsigned)((n + 255) / 256), (unsigned)slices),
                       dim3(256), 0, s, static_cast<const int8_t*>(b), k, n, ldb, k_per_slice, out);
    return mi355_launch_status();
}

extern "C" int mi355_rowsum_i8(const void* a,
                               int64_t m,
                               int64_t k,
                               int64_t lda,
                               int32_t trans_a,
                               int32_t* out,
                               void* stream)
{
    if(a == nullptr || out == nullptr || k < 0 || m < 0)
        return MI355_ERR_BAD_ARG;
    if(m == 0)
        return MI355_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if(trans_a)
    {
        // [K, M] storage: identical to column sums of a row-major matrix
        return mi355_colsum_i8(a, k, m, lda, 0, out, stream);
    }
    hipLaunchKernelGGL(sum_i8_kernel, dim3((unsigned)((m + 3) / 4)), dim3(256), 0, s,
                       static_cast<const int8_t*>(a), m, k, lda, (int64_t)1, out);
    return mi355_launch_status();
}

extern "C" const char* mi355_status_string(int status)
{
    switch(status)
    {
    case MI355_OK: return "ok";
    case MI355_ERR_BAD_ARG: return "bad argument";
    case MI355_ERR_UNSUPPORTED: return "unsupported configuration";
    case MI355_ERR_LAUNCH: return "HIP launch error";
    case MI355_ERR_SCRATCH_TOO_SMALL: return "the problem needs more scratch memory than the library's static buffer holds";
    default: return "unknown status";
    }
}

extern "C" int mi355_version(void) { return 100; }
