// HBM-bound elementwise operators of the quantized path: quantizelinear,
// dequantizelinear, unpack_int4, pack_int4, convert.  Each thread handles a
// short run of consecutive elements so loads and stores are wide and
// coalesced; the arithmetic follows the ref target step by step.
#include "common.h"

namespace {

constexpr int PW_THREADS = 256;

template <int XT>
MI355_DEVINL float load_x(const void* x, int64_t i)
{
    if constexpr(XT == MI355_F32)
        return static_cast<const float*>(x)[i];
    else if constexpr(XT == MI355_F16)
        return half_to_f32(static_cast<const uint16_t*>(x)[i]);
    else
        return bf16_to_f32(static_cast<const uint16_t*>(x)[i]);
}

// a quotient in x's own type (generic_float's operator/ converts the float
// quotient back to the narrow type, generic_float.hpp:318-326)
template <int XT>
MI355_DEVINL float in_type(float d)
{
    if constexpr(XT == MI355_F16)
        d = half_to_f32(f32_to_half_rtz(d));
    else if constexpr(XT == MI355_BF16)
        d = bf16_to_f32(f32_to_bf16_rtz(d));
    return d;
}

template <int XT>
MI355_DEVINL float div_in_type(float x, float s)
{
    return in_type<XT>(x / s);
}

struct qparams
{
    const void* scale;
    int64_t s_sr, s_sc;
    const void* zp;
    int64_t z_sr, z_sc;
};

template <int XT, int OT>
__global__ __launch_bounds__(PW_THREADS) void quantizelinear_kernel(
    const void* x, qparams q, void* out, int64_t rows, int64_t cols)
{
    // 4 consecutive elements of one row per thread (cols is padded up per row)
    const int64_t cols4  = (cols + 3) / 4;
    const int64_t gid    = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x;
    if(gid >= rows * cols4)
        return;
    const int64_t r  = gid / cols4;
    const int64_t c0 = (gid - r * cols4) * 4;
    uint8_t res[4];
    const int cnt = (int)min((int64_t)4, cols - c0);
    for(int e = 0; e < cnt; e++)
    {
        const int64_t c = c0 + e;
        const float xv  = load_x<XT>(x, r * cols + c);
        const float sv  = load_x<XT>(q.scale, r * q.s_sr + c * q.s_sc);
        if constexpr(OT == MI355_FP8)
        {
            double z = 0.0;
            if(q.zp != nullptr)
                z = (double)fp8_to_f32(static_cast<const uint8_t*>(q.zp)[r * q.z_sr + c * q.z_sc]);
            double v = clamp_like_ref((double)xv / (double)sv + z, -448.0, 448.0);
            res[e]   = f32_to_fp8_rne((float)v);
        }
        else if constexpr(OT == MI355_BF8)
        {
            double z = 0.0;
            if(q.zp != nullptr)
                z = (double)bf8_to_f32(static_cast<const uint8_t*>(q.zp)[r * q.z_sr + c * q.z_sc]);
            double v = clamp_like_ref((double)xv / (double)sv + z, -57344.0, 57344.0);
            res[e]   = f32_to_bf8_rne((float)v);
        }
        else
        {
            double z = 0.0;
            if(q.zp != nullptr)
            {
                if constexpr(OT == MI355_I8)
                    z = (double)static_cast<const int8_t*>(q.zp)[r * q.z_sr + c * q.z_sc];
                else
                    z = (double)static_cast<const uint8_t*>(q.zp)[r * q.z_sr + c * q.z_sc];
            }
            double qv = (double)rintf(div_in_type<XT>(xv, sv)) + z;
            if constexpr(OT == MI355_I8)
                res[e] = (uint8_t)(int8_t)(int)clamp_like_ref(qv, -128.0, 127.0);
            else
                res[e] = (uint8_t)(int)clamp_like_ref(qv, 0.0, 255.0);
        }
    }
    uint8_t* o = static_cast<uint8_t*>(out) + r * cols + c0;
    if(cnt == 4 && ((reinterpret_cast<uintptr_t>(o) & 3) == 0))
        *reinterpret_cast<uint32_t*>(o) =
            res[0] | ((uint32_t)res[1] << 8) | ((uint32_t)res[2] << 16) | ((uint32_t)res[3] << 24);
    else
        for(int e = 0; e < cnt; e++)
            o[e] = res[e];
}

// ---- runs of elements ----------------------------------------------------------------------------
// What bounds both operators is memory: the kernels below move 16 or 4 consecutive elements of one row
// per thread, up to 16 bytes a load or store, at whatever address the row has (a global load takes
// any).  Everything an element used to pay for by itself is gone:
// the 64-bit division that finds its row (a multiplication by the reciprocal here, once per run), the
// loads of scale and zero point (once per run where they don't vary along the row, else as a vector),
// and arithmetic in double where float provably gives the same bits:
//   x / s       rounding the double quotient of two floats to float is the float quotient (53 bits are
//               more than twice 24 and two), and what overflows saturates on both ways;
//   rint + zp   whole numbers below 2^24, or saturated;
//   (x - zp) s  the difference of two 8-bit values, fp8 e4m3fn's 2^-9 ... 896 included, is exact in
//               float, so is the double product: one rounding to float either way.
// The last run of a row ends where the row ends: it does again what the run before it did of it, and
// writes the same values (one element at a time, what is left of a row was a chain of up to 15 loads and
// divisions: [3, 1023] half with a scale per row to int8 3.1 us before the runs, 9.5 with the chain).
// Left to the kernels of any strides: strides along the row other than 0 and 1, e5m2 (whose zero
// points cost more than 24 bits), fp8 quantization with a zero point (the sum is rounded as a
// double there), int32 and float32 inputs of dequantizelinear, a single element, 2^31 runs and beyond.
// Measured, [8192, 1024] bfloat16 with a scale per row: to uint8 14.3 -> 7.5 us, back
// from uint8 with zero points 28 -> 7.0 us; [2048, 8192] bfloat16 to fp8
// 30 -> 13 us (50 MB).

struct run_params
{
    const void* x;
    void* out;
    qparams q;
    int64_t cols;
    int run;           // elements
    uint32_t runs;     // in all
    uint32_t per_row;  // runs of a row, the last of which may overlap the one before it
    uint32_t magic;    // run / per_row = (run * magic) >> shift for run < 2^31
    uint32_t shift;
};

// consecutive elements at any address
template <class T, int N>
struct __attribute__((packed, aligned(1))) run_of
{
    T v[N];
};

template <int N, class T>
MI355_DEVINL run_of<T, N> load_run(const T* p)
{
    return *reinterpret_cast<const run_of<T, N>*>(p);
}

template <class T, int N>
MI355_DEVINL void store_run(T* p, const run_of<T, N>& r)
{
    *reinterpret_cast<run_of<T, N>*>(p) = r;
}

// N float32 / float16 / bfloat16 values, or 8-bit codes, as floats
template <int T, int N>
MI355_DEVINL void load_f32(float (&f)[N], const void* p, int64_t i)
{
    if constexpr(T == MI355_F32)
    {
        const auto r = load_run<N>(static_cast<const float*>(p) + i);
#pragma unroll
        for(int e = 0; e < N; e++)
            f[e] = r.v[e];
    }
    else if constexpr(T == MI355_F16 || T == MI355_BF16)
    {
        const auto r = load_run<N>(static_cast<const uint16_t*>(p) + i);
#pragma unroll
        for(int e = 0; e < N; e++)
            f[e] = T == MI355_F16 ? half_to_f32(r.v[e]) : bf16_to_f32(r.v[e]);
    }
    else
    {
        const auto r = load_run<N>(static_cast<const uint8_t*>(p) + i);
#pragma unroll
        for(int e = 0; e < N; e++)
            f[e] = T == MI355_I8 ? (float)(int8_t)r.v[e] : T == MI355_U8 ? (float)r.v[e] : fp8_to_f32(r.v[e]);
    }
}

// the scales (or zero points) of N elements: one for all of them, or their own
template <int T, int N>
MI355_DEVINL void load_param(float (&f)[N], const void* p, int64_t i, int64_t stride)
{
    if(stride == 0)
    {
        float one[1];
        load_f32<T>(one, p, i);
#pragma unroll
        for(int e = 0; e < N; e++)
            f[e] = one[0];
    }
    else
        load_f32<T>(f, p, i);
}

MI355_DEVINL float clamp_like_ref_f32(float q, float lo, float hi)
{
    const float v = (q < hi) ? q : hi;
    return (lo < v) ? v : lo;
}

// The correctly rounded quotient of x by one s from its correctly rounded reciprocal: each of the
// two steps adds what the exact remainder says is missing, the first leaves a quotient within one
// unit of its last place, the second the nearest (P. Markstein, "Computation of elementary functions
// on the IBM RISC System/6000 processor", 1990).  Five instructions in place of a division's eleven.
// No step overflows for 2^-60 <= |s| <= 2^60 and |x| <= 2^60.  Bits lost below the normal range
// belong to quotients under 2^-40: the 8-bit code is zero with or without them, with the quotient's
// sign (of x = 0 alone the sign may be lost).
MI355_DEVINL bool reciprocal_serves(float s)
{
    return __builtin_fabsf(s) >= 0x1p-60f && __builtin_fabsf(s) <= 0x1p60f;
}

MI355_DEVINL float div_by_reciprocal(float x, float s, float rs)
{
    float q = x * rs;
    q       = __builtin_fmaf(__builtin_fmaf(-q, s, x), rs, q);
    return __builtin_fmaf(__builtin_fmaf(-q, s, x), rs, q);
}

template <int XT, int OT, int N>
MI355_DEVINL void quantize_elements(const run_params& p, int64_t r, int64_t c)
{
    float x[N], s[N], z[N] = {};
    load_param<XT>(s, p.q.scale, r * p.q.s_sr + c * p.q.s_sc, p.q.s_sc);
    if constexpr(OT != MI355_FP8)
        if(p.q.zp != nullptr)
            load_param<OT>(z, p.q.zp, r * p.q.z_sr + c * p.q.z_sc, p.q.z_sc);
    load_f32<XT>(x, p.x, r * p.cols + c);
    // the quotients: where one scale serves all, so does its reciprocal
    float q[N];
    uint32_t most = 0; // of the magnitudes' bits, which order like the magnitudes, NaN on top
#pragma unroll
    for(int e = 0; e < N; e++)
        most = max(most, __builtin_bit_cast(uint32_t, x[e]) & 0x7fffffffu);
    const bool serves = p.q.s_sc == 0 && reciprocal_serves(s[0]) && most <= 0x5d800000u; // 2^60
    if(N > 1 && serves)
    {
        const float rs = 1.f / s[0];
#pragma unroll
        for(int e = 0; e < N; e++)
            q[e] = div_by_reciprocal(x[e], s[0], rs);
    }
    else
    {
#pragma unroll
        for(int e = 0; e < N; e++)
            q[e] = x[e] / s[e];
    }
#pragma unroll
    for(int e = 0; e < N; e++)
    {
        if constexpr(OT == MI355_FP8)
        {
            // the double sum with no zero point turns an exact -0 into +0, but no tiny negative quotient
            const float zero = x[e] == 0.f || __builtin_isinf(s[e]) ? 0.f : -0.f;
            q[e]             = clamp_like_ref_f32(q[e] + zero, -448.f, 448.f);
        }
        else
        {
            const float lo = OT == MI355_I8 ? -128.f : 0.f;
            q[e]           = clamp_like_ref_f32(rintf(in_type<XT>(q[e])) + z[e], lo, lo + 255.f);
        }
    }
    uint8_t* out = static_cast<uint8_t*>(p.out) + r * p.cols + c;
    if constexpr(N % 4 == 0)
    {
        uint32_t w[N / 4];
#pragma unroll
        for(int h = 0; h < N / 4; h++)
        {
            if constexpr(OT == MI355_FP8)
            {
                w[h] = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * h], q[4 * h + 1], 0, false);
                w[h] = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * h + 2], q[4 * h + 3], w[h], true);
            }
            else
            {
                // an int8 code is its value + 128 with the top bit flipped
                w[h] = 0;
#pragma unroll
                for(int e = 0; e < 4; e++)
                    w[h] = __builtin_amdgcn_cvt_pk_u8_f32(OT == MI355_I8 ? q[4 * h + e] + 128.f : q[4 * h + e], e, w[h]);
                if constexpr(OT == MI355_I8)
                    w[h] ^= 0x80808080u;
            }
        }
        store_run(out, __builtin_bit_cast(run_of<uint8_t, N>, w));
    }
    else
    {
#pragma unroll
        for(int e = 0; e < N; e++)
            out[e] = OT == MI355_FP8 ? f32_to_fp8_rne(q[e]) : (uint8_t)(int)q[e];
    }
}

template <int XT, int ST, int N>
MI355_DEVINL void dequantize_elements(const run_params& p, int64_t r, int64_t c)
{
    float x[N], s[N], z[N] = {};
    load_param<ST>(s, p.q.scale, r * p.q.s_sr + c * p.q.s_sc, p.q.s_sc);
    if(p.q.zp != nullptr)
        load_param<XT>(z, p.q.zp, r * p.q.z_sr + c * p.q.z_sc, p.q.z_sc);
    const int64_t i = r * p.cols + c;
    load_f32<XT>(x, p.x, i);
#pragma unroll
    for(int e = 0; e < N; e++)
        x[e] = (x[e] - z[e]) * s[e];
    if constexpr(ST == MI355_F32)
        store_run(static_cast<float*>(p.out) + i, __builtin_bit_cast(run_of<float, N>, x));
    else
    {
        run_of<uint16_t, N> res;
#pragma unroll
        for(int e = 0; e < N; e++)
            res.v[e] = ST == MI355_F16 ? f32_to_half_rtz(x[e]) : f32_to_bf16_rtz(x[e]);
        store_run(static_cast<uint16_t*>(p.out) + i, res);
    }
}

// QUANTIZE: IN a float type, OUT a code's; else the other way
template <bool QUANTIZE, int IN, int OUT, int N>
__global__ __launch_bounds__(PW_THREADS) void run_kernel(run_params p)
{
    const uint32_t run = blockIdx.x * PW_THREADS + threadIdx.x;
    if(run >= p.runs)
        return;
    const uint32_t r = (uint32_t)(((uint64_t)run * p.magic) >> p.shift);
    const int64_t c  = min((int64_t)(run - r * p.per_row) * N, p.cols - N);
    if constexpr(QUANTIZE)
        quantize_elements<IN, OUT, N>(p, r, c);
    else
        dequantize_elements<IN, OUT, N>(p, r, c);
}

// Strides along the row of 0 and 1 only; rows that are one vector for the parameters as well become
// one long row.  `wide`: runs of 16 may pay.  False where the kernels of any strides have to take the call.
bool run_plan(run_params& p, const void* x, const qparams& q, void* out, int64_t rows, int64_t cols, bool wide)
{
    const bool has_zp = q.zp != nullptr;
    p.x   = x;
    p.out = out;
    p.q   = q;
    if(cols == 1) // rows of one element: the stride along the rows is the one along a single row
    {
        p.q.s_sc = q.s_sr;
        p.q.z_sc = q.z_sr;
    }
    if(p.q.s_sc < 0 || p.q.s_sc > 1 || (has_zp && (p.q.z_sc < 0 || p.q.z_sc > 1)))
        return false;
    // element i of the tensor has parameter i (a full tensor of them), or the one there is
    auto flat = [&](int64_t sr, int64_t sc) { return sr == sc * cols; };
    if(flat(p.q.s_sr, p.q.s_sc) && (!has_zp || flat(p.q.z_sr, p.q.z_sc)))
    {
        cols *= rows;
        rows = 1;
    }
    if(cols < 2)
        return false;
    // 16 elements a thread pay for their latency where there are many and one parameter serves them all, 4
    // otherwise.  Over 2500 tensors, 4 against 16: below 2^21 elements 0.8 to 0.95 of the time, above
    // 1.0 to 1.25; with parameters of their own 0.75 to 1.0 at any size; to float32 (64 bytes a
    // thread side by side) 0.6 to 0.8.
    const bool one = p.q.s_sc == 0 && (!has_zp || p.q.z_sc == 0);
    p.run          = wide && one && cols >= 16 && rows * cols >= 1 << 21 ? 16 : cols >= 4 ? 4 : 2;
    const int64_t per_row = (cols + p.run - 1) / p.run;
    if(per_row > 0x7fffffff || rows > 0x7fffffff / per_row)
        return false;
    p.cols    = cols;
    p.per_row = (uint32_t)per_row;
    p.runs    = (uint32_t)(rows * per_row);
    // ceil(2^(31 + l) / d) with 2^l >= d is exact for every numerator below 2^31; it fits 32 bits
    uint32_t l = 0;
    while(((uint64_t)1 << l) < p.per_row)
        l++;
    p.shift = 31 + l;
    p.magic = (uint32_t)((((uint64_t)1 << p.shift) + p.per_row - 1) / p.per_row);
    return true;
}

template <bool QUANTIZE, int IN, int OUT>
int launch_runs(const run_params& p, hipStream_t s)
{
    const dim3 grid((p.runs + PW_THREADS - 1) / PW_THREADS), block(PW_THREADS);
    if constexpr(QUANTIZE || OUT != MI355_F32)
        if(p.run == 16)
        {
            hipLaunchKernelGGL((run_kernel<QUANTIZE, IN, OUT, 16>), grid, block, 0, s, p);
            return mi355_launch_status();
        }
    if(p.run == 4)
        hipLaunchKernelGGL((run_kernel<QUANTIZE, IN, OUT, 4>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((run_kernel<QUANTIZE, IN, OUT, 2>), grid, block, 0, s, p);
    return mi355_launch_status();
}

__global__ __launch_bounds__(PW_THREADS) void dequantizelinear_kernel(const void* x,
                                                                      int x_type,
                                                                      qparams q,
                                                                      int s_type,
                                                                      void* out,
                                                                      int64_t rows,
                                                                      int64_t cols)
{
    const int64_t i = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x;
    if(i >= rows * cols)
        return;
    const int64_t r = i / cols;
    const int64_t c = i - r * cols;
    double z        = 0.0;
    if(q.zp != nullptr)
        z = load_as_f64(q.zp, x_type, r * q.z_sr + c * q.z_sc);
    const double s = load_as_f64(q.scale, s_type, r * q.s_sr + c * q.s_sc);
    const double v = (load_as_f64(x, x_type, i) - z) * s;
    // stored to the scale's type: double -> float (nearest even), then the
    // narrow type's own conversion from float (round toward zero)
    const float f = (float)v;
    if(s_type == MI355_F32)
        static_cast<float*>(out)[i] = f;
    else if(s_type == MI355_F16)
        static_cast<uint16_t*>(out)[i] = f32_to_half_rtz(f);
    else
        static_cast<uint16_t*>(out)[i] = f32_to_bf16_rtz(f);
}

// one packed byte -> two bytes: 8 packed bytes per thread, one load and one 16-byte store at any
// address, four codes a register ([8192, 512] packed: 10.9 -> 3.7 us)
__global__ __launch_bounds__(PW_THREADS) void unpack_int4_kernel(
    const uint8_t* in, uint8_t* out, int is_signed, int64_t total)
{
    const int64_t i0 = ((int64_t)blockIdx.x * PW_THREADS + threadIdx.x) * 8;
    if(i0 >= total)
        return;
    const int cnt = (int)min((int64_t)8, total - i0);
    uint64_t v = 0;
    if(cnt == 8)
        v = __builtin_bit_cast(uint64_t, load_run<8>(in + i0));
    else
        for(int e = 0; e < cnt; e++)
            v |= (uint64_t)in[i0 + e] << (8 * e);
    uint32_t w[4];
#pragma unroll
    for(int h = 0; h < 2; h++)
    {
        const uint32_t b = (uint32_t)(v >> (32 * h));
        uint32_t lo = b & 0x0f0f0f0fu, hi = (b >> 4) & 0x0f0f0f0fu;
        if(is_signed)
        {
            // bit 3 of a code into the four above it: 8 * 30 = 0xf0, no carry leaves its byte
            lo |= (lo & 0x08080808u) * 30u;
            hi |= (hi & 0x08080808u) * 30u;
        }
        // low nibble first: bytes 0 to 3 of a selector are lo's, 4 to 7 hi's
        w[2 * h]     = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
        w[2 * h + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
    }
    if(cnt == 8)
        store_run(out + 2 * i0, __builtin_bit_cast(run_of<uint8_t, 16>, w));
    else
    {
#pragma unroll
        for(int e = 0; e < 16; e++)
            if(e < 2 * cnt)
                out[2 * i0 + e] = (uint8_t)(w[e >> 2] >> (8 * (e & 3)));
    }
}

// fp4 (e2m1): sign, two exponent bits, one mantissa bit; magnitudes 0, .5, 1, 1.5, 2, 3, 4, 6.
// Their fp8 e4m3fn codes (exponent bias 7, three mantissa bits), indexed by the low three bits:
__constant__ const uint8_t fp4_as_fp8[8] = {0x00, 0x30, 0x38, 0x3c, 0x40, 0x44, 0x48, 0x4c};

// one packed byte -> two fp8 bytes, low nibble first; 8 packed bytes per thread
__global__ __launch_bounds__(PW_THREADS) void unpack_fp4_kernel(const uint8_t* in, uint8_t* out, int64_t total)
{
    const int64_t i0 = ((int64_t)blockIdx.x * PW_THREADS + threadIdx.x) * 8;
    if(i0 >= total)
        return;
    const int cnt = (int)min((int64_t)8, total - i0);
    for(int e = 0; e < cnt; e++)
    {
        const uint8_t v       = in[i0 + e];
        out[2 * (i0 + e)]     = fp4_as_fp8[v & 7] | ((v & 0x08) << 4);
        out[2 * (i0 + e) + 1] = fp4_as_fp8[(v >> 4) & 7] | (v & 0x80);
    }
}

// float -> fp4 code: nearest magnitude, a tie to the neighbour with the even code, beyond 5 -> 6
// (infinity included), NaN -> 0, sign kept (also for zero)
MI355_DEVINL uint8_t f32_to_fp4(float x)
{
    if(x != x)
        return 0;
    const uint8_t sign = (__builtin_bit_cast(uint32_t, x) >> 31) ? 8 : 0;
    const float a      = __builtin_fabsf(x);
    uint8_t i;
    if(a <= 0.25f)
        i = 0;
    else if(a < 0.75f)
        i = 1;
    else if(a <= 1.25f)
        i = 2;
    else if(a < 1.75f)
        i = 3;
    else if(a <= 2.5f)
        i = 4;
    else if(a < 3.5f)
        i = 5;
    else if(a <= 5.0f)
        i = 6;
    else
        i = 7;
    return i | sign;
}

__global__ __launch_bounds__(PW_THREADS) void pack_fp4_kernel(const float* in, uint8_t* out, int64_t total_out)
{
    const int64_t i = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x;
    if(i >= total_out)
        return;
    out[i] = (uint8_t)((f32_to_fp4(in[2 * i + 1]) << 4) | f32_to_fp4(in[2 * i]));
}

// two bytes -> one packed byte: 16 bytes per thread, one load and one 8-byte store at any address
// ([8192, 1024] bytes: 7.9 -> 3.4 us).  The last thread's 8 end where the tensor ends and are in part
// the ones before them again, with the same values; less than 8 are one a thread.
__global__ __launch_bounds__(PW_THREADS) void pack_int4_kernel(
    const uint8_t* in, uint8_t* out, int is_signed, int64_t total_out)
{
    const int64_t i = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x;
    auto packed = [&](uint32_t two) {
        int u1 = (int)(two & 0xff), u2 = (int)(two >> 8);
        if(is_signed)
        {
            u1 = max(-8, min(7, (int)(int8_t)u1));
            u2 = max(-8, min(7, (int)(int8_t)u2));
        }
        else
        {
            u1 = min(u1, 15);
            u2 = min(u2, 15);
        }
        return (uint8_t)((u2 << 4) | (u1 & 0xf));
    };
    if(total_out < 8)
    {
        if(i < total_out)
            out[i] = packed(in[2 * i] | ((uint32_t)in[2 * i + 1] << 8));
        return;
    }
    if(8 * i >= total_out)
        return;
    const int64_t i0 = min(8 * i, total_out - 8);
    const auto v     = load_run<8>(reinterpret_cast<const uint16_t*>(in) + i0);
    run_of<uint8_t, 8> res;
#pragma unroll
    for(int e = 0; e < 8; e++)
        res.v[e] = packed(v.v[e]);
    store_run(out + i0, res);
}

__global__ __launch_bounds__(PW_THREADS) void convert_kernel(
    const void* in, int in_type, void* out, int out_type, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x;
    if(i >= n)
        return;
    const double dx = load_as_f64(in, in_type, i);
    const float f   = (float)dx;
    switch(out_type)
    {
    case MI355_F32:
        static_cast<float*>(out)[i] = (dx != dx) ? __builtin_bit_cast(float, 0x7fc00000u) : f;
        break;
    case MI355_F16: static_cast<uint16_t*>(out)[i] = convert_f32_to_half(f); break;
    case MI355_BF16: static_cast<uint16_t*>(out)[i] = convert_f32_to_bf16(f); break;
    case MI355_FP8:
        if(dx != dx)
            static_cast<uint8_t*>(out)[i] = 0x7f;
        else
            static_cast<uint8_t*>(out)[i] =
                f32_to_fp8_rne((float)fmin(448.0, fmax(-448.0, dx)));
        break;
    case MI355_I8:
        // integral targets: NaN -> numeric_limits::quiet_NaN() = 0, saturate, then truncate toward zero
        static_cast<int8_t*>(out)[i] = dx != dx ? (int8_t)0 : (int8_t)(int)fmin(127.0, fmax(-128.0, dx));
        break;
    case MI355_U8:
        static_cast<uint8_t*>(out)[i] = dx != dx ? (uint8_t)0 : (uint8_t)(int)fmin(255.0, fmax(0.0, dx));
        break;
    case MI355_I32:
        static_cast<int32_t*>(out)[i] =
            dx != dx ? 0 : (int32_t)fmin(2147483647.0, fmax(-2147483648.0, dx));
        break;
    case MI355_BF8:
        // numeric_limits<fp8e5m2>::quiet_NaN() is 0xff (float8.hpp:364); infinities go through
        // the clipping constructor
        if(dx != dx)
            static_cast<uint8_t*>(out)[i] = 0xff;
        else
            static_cast<uint8_t*>(out)[i] =
                f32_to_bf8_rne((float)fmin(57344.0, fmax(-57344.0, dx)));
        break;
    default: break;
    }
}

inline unsigned blocks_for(int64_t n) { return (unsigned)((n + PW_THREADS - 1) / PW_THREADS); }

template <int XT>
int launch_quantize(int out_type,
                    const void* x,
                    const qparams& q,
                    void* out,
                    int64_t rows,
                    int64_t cols,
                    hipStream_t s)
{
    run_params p;
    if((out_type == MI355_I8 || out_type == MI355_U8 || (out_type == MI355_FP8 && q.zp == nullptr)) &&
       run_plan(p, x, q, out, rows, cols, true))
    {
        if(out_type == MI355_I8)
            return launch_runs<true, XT, MI355_I8>(p, s);
        if(out_type == MI355_U8)
            return launch_runs<true, XT, MI355_U8>(p, s);
        return launch_runs<true, XT, MI355_FP8>(p, s);
    }
    const int64_t work = rows * ((cols + 3) / 4);
    switch(out_type)
    {
    case MI355_I8:
        hipLaunchKernelGGL((quantizelinear_kernel<XT, MI355_I8>), dim3(blocks_for(work)),
                           dim3(PW_THREADS), 0, s, x, q, out, rows, cols);
        break;
    case MI355_U8:
        hipLaunchKernelGGL((quantizelinear_kernel<XT, MI355_U8>), dim3(blocks_for(work)),
                           dim3(PW_THREADS), 0, s, x, q, out, rows, cols);
        break;
    case MI355_FP8:
        hipLaunchKernelGGL((quantizelinear_kernel<XT, MI355_FP8>), dim3(blocks_for(work)),
                           dim3(PW_THREADS), 0, s, x, q, out, rows, cols);
        break;
    case MI355_BF8:
        hipLaunchKernelGGL((quantizelinear_kernel<XT, MI355_BF8>), dim3(blocks_for(work)),
                           dim3(PW_THREADS), 0, s, x, q, out, rows, cols);
        break;
    default: return MI355_ERR_UNSUPPORTED;
    }
    return mi355_launch_status();
}

template <int XT>
int launch_dequantize_runs(int s_type, const run_params& p, hipStream_t s)
{
    if(s_type == MI355_F32)
        return launch_runs<false, XT, MI355_F32>(p, s);
    if(s_type == MI355_F16)
        return launch_runs<false, XT, MI355_F16>(p, s);
    return launch_runs<false, XT, MI355_BF16>(p, s);
}

} // namespace

extern "C" int mi355_quantizelinear(const void* x,
                                    int32_t x_type,
                                    const void* scale,
                                    int64_t scale_stride_r,
                                    int64_t scale_stride_c,
                                    const void* zp,
                                    int64_t zp_stride_r,
                                    int64_t zp_stride_c,
                                    void* out,
                                    int32_t out_type,
                                    int64_t rows,
                                    int64_t cols,
                                    void* stream)
{
    if(x == nullptr || scale == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    if(rows == 0 || cols == 0)
        return MI355_OK;
    if(rows * ((cols + 3) / 4) > (int64_t)0x7fffffff * PW_THREADS)
        return MI355_ERR_UNSUPPORTED;
    qparams q{scale, scale_stride_r, scale_stride_c, zp, zp_stride_r, zp_stride_c};
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch(x_type)
    {
    case MI355_F32: return launch_quantize<MI355_F32>(out_type, x, q, out, rows, cols, s);
    case MI355_F16: return launch_quantize<MI355_F16>(out_type, x, q, out, rows, cols, s);
    case MI355_BF16: return launch_quantize<MI355_BF16>(out_type, x, q, out, rows, cols, s);
    default: return MI355_ERR_UNSUPPORTED;
    }
}

extern "C" int mi355_dequantizelinear(const void* x,
                                      int32_t x_type,
                                      const void* scale,
                                      int32_t scale_type,
                                      int64_t scale_stride_r,
                                      int64_t scale_stride_c,
                                      const void* zp,
                                      int64_t zp_stride_r,
                                      int64_t zp_stride_c,
                                      void* out,
                                      int64_t rows,
                                      int64_t cols,
                                      void* stream)
{
    if(x == nullptr || scale == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    if(x_type != MI355_I8 && x_type != MI355_U8 && x_type != MI355_I32 && x_type != MI355_F32 &&
       x_type != MI355_FP8 && x_type != MI355_BF8)
        return MI355_ERR_UNSUPPORTED;
    if(scale_type != MI355_F32 && scale_type != MI355_F16 && scale_type != MI355_BF16)
        return MI355_ERR_UNSUPPORTED;
    if(rows == 0 || cols == 0)
        return MI355_OK;
    qparams q{scale, scale_stride_r, scale_stride_c, zp, zp_stride_r, zp_stride_c};
    run_params p;
    if((x_type == MI355_I8 || x_type == MI355_U8 || x_type == MI355_FP8) && run_plan(p, x, q, out, rows, cols, scale_type != MI355_F32))
    {
        hipStream_t s = static_cast<hipStream_t>(stream);
        if(x_type == MI355_I8)
            return launch_dequantize_runs<MI355_I8>(scale_type, p, s);
        if(x_type == MI355_U8)
            return launch_dequantize_runs<MI355_U8>(scale_type, p, s);
        return launch_dequantize_runs<MI355_FP8>(scale_type, p, s);
    }
    hipLaunchKernelGGL(dequantizelinear_kernel, dim3(blocks_for(rows * cols)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), x, x_type, q, scale_type, out, rows, cols);
    return mi355_launch_status();
}

extern "C" int mi355_unpack_int4(
    const void* in, void* out, int32_t is_signed, int64_t rows, int64_t cols, void* stream)
{
    if(in == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    const int64_t total = rows * cols;
    if(total == 0)
        return MI355_OK;
    hipLaunchKernelGGL(unpack_int4_kernel, dim3(blocks_for((total + 7) / 8)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(in),
                       static_cast<uint8_t*>(out), is_signed, total);
    return mi355_launch_status();
}

extern "C" int mi355_pack_int4(
    const void* in, void* out, int32_t is_signed, int64_t rows, int64_t cols, void* stream)
{
    if(in == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    if(cols % 2 != 0)
        return MI355_ERR_BAD_ARG; // PACK_INT4: can not pack an axis of odd length
    const int64_t total_out = rows * (cols / 2);
    if(total_out == 0)
        return MI355_OK;
    hipLaunchKernelGGL(pack_int4_kernel, dim3(blocks_for((total_out + 7) / 8)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(in),
                       static_cast<uint8_t*>(out), is_signed, total_out);
    return mi355_launch_status();
}

// ---- int4 pack / unpack along any axis of a strided view ------------------------------------
// One thread per packed byte.  `lens` are the lengths of the packed tensor (unpack: the input,
// pack: the output); the byte with multi-index idx pairs with the elements idx[axis] * 2 and
// idx[axis] * 2 + 1 of the unpacked tensor.  The strided side (the input) is addressed through
// element strides, zero for a broadcast dimension; the output is dense row-major.
struct int4_nd_params
{
    const uint8_t* in;
    uint8_t* out;
    int64_t lens[MI355_MAX_DIMS];
    int64_t in_strides[MI355_MAX_DIMS];
    int64_t out_strides[MI355_MAX_DIMS];
    int64_t total;
    int ndim, axis, is_signed;
};

template <bool PACK>
__global__ __launch_bounds__(PW_THREADS) void int4_nd_kernel(int4_nd_params p)
{
    for(int64_t i = (int64_t)blockIdx.x * PW_THREADS + threadIdx.x; i < p.total;
        i += (int64_t)gridDim.x * PW_THREADS)
    {
        int64_t rest = i, in_off = 0, out_off = 0;
        for(int d = p.ndim - 1; d >= 0; d--)
        {
            const int64_t idx = rest % p.lens[d];
            rest /= p.lens[d];
            // along the axis the unpacked side holds two elements per packed byte
            in_off += idx * p.in_strides[d] * ((PACK && d == p.axis) ? 2 : 1);
            out_off += idx * p.out_strides[d] * ((!PACK && d == p.axis) ? 2 : 1);
        }
        if constexpr(PACK)
        {
            const uint8_t r1 = p.in[in_off], r2 = p.in[in_off + p.in_strides[p.axis]];
            uint8_t u1, u2;
            if(p.is_signed)
            {
                u1 = (uint8_t)max(-8, min(7, (int)(int8_t)r1));
                u2 = (uint8_t)max(-8, min(7, (int)(int8_t)r2));
            }
            else
            {
                u1 = (uint8_t)min((int)r1, 15);
                u2 = (uint8_t)min((int)r2, 15);
            }
            p.out[out_off] = (uint8_t)((u2 << 4) | (u1 & 0xf));
        }
        else
        {
            const uint8_t v = p.in[in_off];
            uint8_t lo, hi;
            if(p.is_signed)
            {
                lo = (uint8_t)((int8_t)(uint8_t)(v << 4) >> 4);
                hi = (uint8_t)((int8_t)v >> 4);
            }
            else
            {
                lo = v & 0xf;
                hi = v >> 4;
            }
            p.out[out_off]                         = lo;
            p.out[out_off + p.out_strides[p.axis]] = hi;
        }
    }
}

template <bool PACK>
static int launch_int4_nd(const void* in, void* out, int32_t is_signed, int32_t ndim, const int64_t* lens,
                          const int64_t* in_strides, int32_t axis, void* stream)
{
    if(ndim < 1 || ndim > MI355_MAX_DIMS || lens == nullptr || in_strides == nullptr)
        return MI355_ERR_BAD_ARG;
    if(axis < 0)
        axis += ndim;
    if(axis < 0 || axis >= ndim)
        return MI355_ERR_BAD_ARG;
    int4_nd_params p{};
    p.total = 1;
    for(int d = 0; d < ndim; d++)
    {
        if(lens[d] < 0 || in_strides[d] < 0)
            return MI355_ERR_BAD_ARG;
        p.lens[d]       = lens[d]; // lengths of the INPUT
        p.in_strides[d] = in_strides[d];
    }
    if(PACK)
    {
        if(lens[axis] % 2 != 0)
            return MI355_ERR_BAD_ARG; // PACK_INT4: can not pack an axis of odd length
        p.lens[axis] = lens[axis] / 2; // the kernel walks the packed tensor
    }
    // dense strides of the output
    int64_t run = 1;
    for(int d = ndim - 1; d >= 0; d--)
    {
        p.out_strides[d] = run;
        run *= (!PACK && d == axis) ? p.lens[d] * 2 : p.lens[d];
        p.total *= p.lens[d];
    }
    if(p.total == 0)
        return MI355_OK;
    if(in == nullptr || out == nullptr)
        return MI355_ERR_BAD_ARG;
    p.in        = static_cast<const uint8_t*>(in);
    p.out       = static_cast<uint8_t*>(out);
    p.ndim      = ndim;
    p.axis      = axis;
    p.is_signed = is_signed;
    int64_t blocks = (p.total + PW_THREADS - 1) / PW_THREADS;
    if(blocks > 256 * 16)
        blocks = 256 * 16;
    hipLaunchKernelGGL(int4_nd_kernel<PACK>, dim3((unsigned)blocks), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), p);
    return mi355_launch_status();
}

extern "C" int mi355_unpack_int4_nd(const void* in, void* out, int32_t is_signed, int32_t ndim,
                                    const int64_t* lens, const int64_t* in_strides, int32_t axis, void* stream)
{
    return launch_int4_nd<false>(in, out, is_signed, ndim, lens, in_strides, axis, stream);
}

extern "C" int mi355_pack_int4_nd(const void* in, void* out, int32_t is_signed, int32_t ndim,
                                  const int64_t* lens, const int64_t* in_strides, int32_t axis, void* stream)
{
    return launch_int4_nd<true>(in, out, is_signed, ndim, lens, in_strides, axis, stream);
}

extern "C" int mi355_unpack_fp4(const void* in, void* out, int64_t rows, int64_t cols, void* stream)
{
    if(in == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    const int64_t total = rows * cols;
    if(total == 0)
        return MI355_OK;
    hipLaunchKernelGGL(unpack_fp4_kernel, dim3(blocks_for((total + 7) / 8)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), static_cast<const uint8_t*>(in),
                       static_cast<uint8_t*>(out), total);
    return mi355_launch_status();
}

extern "C" int mi355_pack_fp4(const float* in, void* out, int64_t rows, int64_t cols, void* stream)
{
    if(in == nullptr || out == nullptr || rows < 0 || cols < 0)
        return MI355_ERR_BAD_ARG;
    if(cols % 2 != 0)
        return MI355_ERR_BAD_ARG; // PACK_FP4: can not pack along an axis of odd length
    const int64_t total_out = rows * (cols / 2);
    if(total_out == 0)
        return MI355_OK;
    hipLaunchKernelGGL(pack_fp4_kernel, dim3(blocks_for(total_out)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), in, static_cast<uint8_t*>(out), total_out);
    return mi355_launch_status();
}

extern "C" int mi355_convert(
    const void* in, int32_t in_type, void* out, int32_t out_type, int64_t n, void* stream)
{
    if(in == nullptr || out == nullptr || n < 0)
        return MI355_ERR_BAD_ARG;
    if(mi355_dtype_size(in_type) == 0 || mi355_dtype_size(out_type) == 0)
        return MI355_ERR_BAD_ARG;
    if(out_type != MI355_F32 && out_type != MI355_F16 && out_type != MI355_BF16 &&
       out_type != MI355_FP8 && out_type != MI355_BF8 && out_type != MI355_I8 && out_type != MI355_U8 &&
       out_type != MI355_I32)
        return MI355_ERR_UNSUPPORTED;
    if(n == 0)
        return MI355_OK;
    hipLaunchKernelGGL(convert_kernel, dim3(blocks_for(n)), dim3(PW_THREADS), 0,
                       static_cast<hipStream_t>(stream), in, in_type, out, out_type, n);
    return mi355_launch_status();
}
