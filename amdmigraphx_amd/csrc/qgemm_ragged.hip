// quant_dot of matrices whose rows start anywhere: K, N and the leading dimensions are multiples of
// nothing (an attention layer over 197 patches, a vocabulary of 30522), where neither a 16-byte
// direct-to-LDS load nor a group of 4 aligned outputs exists.  Same results, bit for bit, as the
// scalar kernel that still serves a transposed A, e5m2 and the tiniest shapes.
//
// Data path: global memory -> registers -> LDS -> v_mfma_i32_16x16x64_i8, two LDS stages, one barrier
// per slab of K; the loads of the next slab are in flight while the current one is multiplied.
//   K-contiguous operand: 16 bytes a lane wherever they start (global loads of this card need no
//     alignment); the piece that crosses the end of a row is the row's last 16 bytes, shifted down, so
//     nothing outside the matrix is read and what lies behind K is zero.
//   row-major B: 4 columns of 16 (fp8: 4) rows a lane, transposed with v_perm_b32; a group that crosses
//     N is the row's last 4 columns, shifted.  Rows behind K repeat row K - 1: A is zero there.
// In the LDS the rows of B are permuted (row j*16 + i of a wave's part holds column TJ*i + j), so that a
// lane owns TJ adjacent outputs of a row and 16 lanes store 16 * TJ adjacent ones.
//
// fp8 (e4m3fn): the operator's sum is exact in double, and float accumulation would lose that.  Every
// code is a whole multiple of 2^-9 below 2^18 of them, so it is three signed bytes d0 + 256 d1 + 65536 d2,
// and the product is nine int8 products whose int32 sums, by weight, are put together in double at the
// end: exact, at 5/9 of the int8 rate per product against the 1/64 of it that double FMAs reach.  A NaN
// code has no digits: rows of A and columns of B that hold one are noted while they are loaded.
//
// What bounds it: 500 x 30522 x 768 int8 -> float is 1810 us in the scalar kernel and 38 us here, of which
// the 61 MB of C are 12 us at this card's copy rate: matrix cores are busy 15 % of it, a quarter of the waves' time
// is vector work (the transposition of B, for every 128 rows of A again), a quarter waits.  A tile's 128 columns
// of an unaligned row lie in two lines; while the four tiles that share them ran on different XCDs (956 tiles, no
// multiple of 8, dealt in turn) B came in eight times from behind the L2s and the call took 46 us.
// fp8 of that size: 150 us, bound by the making of digits (tiles of 128 x 128 with eight waves, which make half as
// many, take the same 1750 us for 1615 x 12800 x 7825).  96 batches of 197 x 197 x 64 (B as [N, K]) 23.7 us in the
// scalar kernel, 11.3 in two-slab tiles, 9.3 in one slab (16 KiB of loads a workgroup and nothing to hide
// them behind but seven workgroups on a CU); of 197 x 64 x 197 7.7 us.
// Loads without branches and a barrier that leaves them in flight took 128 x 4096 x 4096 from 18.5 to 12.5.
#include "common.h"

namespace {

constexpr int THREADS = 256;

struct ragged_params
{
    const uint8_t* a;
    const uint8_t* b;
    void* c;
    int m, n, k;
    uint32_t lda, ldb;
    int64_t ldc, stride_a, stride_b, stride_c;
    int tiles_m, tiles_n;
    const float* scale_a;
    const float* scale_b;
    const int32_t* colsum_b;
    const int32_t* rowsum_a;
    const float* bias;
    int scale_a_mode, scale_b_mode, zp_a, zp_b;
};

MI355_DEVINL uint4 load16(const uint8_t* p)
{
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

MI355_DEVINL uint32_t load4(const uint8_t* p)
{
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

// the LDS accesses of all waves done; __syncthreads() would also wait for the loads that are meant to
// stay in flight
MI355_DEVINL void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// v moved down by `bytes` bytes, zeros from above; 16 and more: all zero
MI355_DEVINL uint4 shift_down(uint4 v, int bytes)
{
    uint64_t lo = v.x | ((uint64_t)v.y << 32), hi = v.z | ((uint64_t)v.w << 32);
    const int s = 8 * (bytes & 7);
    if(bytes & 8)
    {
        lo = hi;
        hi = 0;
    }
    if(s != 0)
    {
        lo = (lo >> s) | (hi << (64 - s));
        hi >>= s;
    }
    if(bytes >= 16)
        lo = hi = 0;
    return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

// rows r0..r3 hold bytes [n0 n1 n2 n3] of four consecutive k; c[j]: the four k bytes of column j
MI355_DEVINL void transpose4(const uint32_t* r, uint32_t c[4])
{
    const uint32_t t01l = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);
    const uint32_t t01h = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
    const uint32_t t23l = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
    const uint32_t t23h = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    c[0]                = __builtin_amdgcn_perm(t23l, t01l, 0x05040100u);
    c[1]                = __builtin_amdgcn_perm(t23l, t01l, 0x07060302u);
    c[2]                = __builtin_amdgcn_perm(t23h, t01h, 0x05040100u);
    c[3]                = __builtin_amdgcn_perm(t23h, t01h, 0x07060302u);
}

// bit 7 of every byte that is an e4m3fn NaN (0x7f, 0xff)
MI355_DEVINL uint32_t nan_bytes(uint32_t w) { return ((w & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u; }

// The three digit bytes of four e4m3fn codes.  512 v + 0x8080 + 2^22 + 2^23 in float: its mantissa is
// 2^22 + 512 v + 0x8080, whose bytes are d0 + 128, d1 + 128 and d2 + 64 with d0, d1 in [-128, 127] and
// d2 in [-4, 4].
MI355_DEVINL void fp8_digits(uint32_t w, uint32_t d[3])
{
    const auto lo    = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    const auto hi    = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    const float base = 8388608.f + 4194304.f + 32896.f;
    const uint32_t x0 = __builtin_bit_cast(uint32_t, __builtin_fmaf(lo[0], 512.f, base));
    const uint32_t x1 = __builtin_bit_cast(uint32_t, __builtin_fmaf(lo[1], 512.f, base));
    const uint32_t x2 = __builtin_bit_cast(uint32_t, __builtin_fmaf(hi[0], 512.f, base));
    const uint32_t x3 = __builtin_bit_cast(uint32_t, __builtin_fmaf(hi[1], 512.f, base));
    const uint32_t a01 = __builtin_amdgcn_perm(x1, x0, 0x05010400u); // bytes 0 and 1 of both
    const uint32_t a23 = __builtin_amdgcn_perm(x3, x2, 0x05010400u);
    const uint32_t b01 = __builtin_amdgcn_perm(x1, x0, 0x0c0c0602u); // byte 2 of both
    const uint32_t b23 = __builtin_amdgcn_perm(x3, x2, 0x0c0c0602u);
    d[0] = __builtin_amdgcn_perm(a23, a01, 0x05040100u) ^ 0x80808080u;
    d[1] = __builtin_amdgcn_perm(a23, a01, 0x07060302u) ^ 0x80808080u;
    d[2] = (__builtin_amdgcn_perm(b23, b01, 0x05040100u) + 0x40404040u) ^ 0x80808080u;
}

template <int OUT, int N>
MI355_DEVINL void store_n(void* c, int64_t idx, const float* v, int cnt)
{
    if constexpr(OUT == MI355_F32)
    {
        float* o = static_cast<float*>(c) + idx;
        if(cnt >= N)
            __builtin_memcpy(o, v, 4 * N);
        else
        {
#pragma unroll
            for(int e = 0; e < N; e++)
                if(e < cnt)
                    o[e] = v[e];
        }
    }
    else
    {
        uint16_t h[N];
#pragma unroll
        for(int e = 0; e < N; e++)
            h[e] = OUT == MI355_F16 ? convert_f32_to_half(v[e]) : convert_f32_to_bf16(v[e]);
        uint16_t* o = static_cast<uint16_t*>(c) + idx;
        if(cnt >= N)
            __builtin_memcpy(o, h, 2 * N);
        else
        {
#pragma unroll
            for(int e = 0; e < N; e++)
                if(e < cnt)
                    o[e] = h[e];
        }
    }
}

enum operand_form { INT8, FP8_DIGITS, FP8_FLOAT };

template <int FORM>
struct sum_of
{
    using type = v4i;
};
template <>
struct sum_of<FP8_FLOAT>
{
    using type = v4f;
};

// FORM: int8, or e4m3fn summed exactly (digits) or in float; TRANS_B: B is [N, K]; OUT: element type of
// the result, -1 for the bare sums.  BIG: a 128 x 128 tile in slabs of 128 (a wave owns 64 x 64), else
// 64 x 64 in slabs of 256 (digits: 64), a wave 32 x 32.  ONE: 64 x 64, all of K in one slab of ONE bytes (B as
// [N, K]): nothing is fetched ahead, and with a quarter of the LDS and of the registers several workgroups
// share a CU and hide each other's loads and stores.
template <int FORM, bool TRANS_B, int OUT, bool BIG, int ONE = 0>
__global__ __launch_bounds__(THREADS) void qgemm_ragged_kernel(ragged_params p)
{
    constexpr bool DIGITS = FORM == FP8_DIGITS;
    static_assert(!(DIGITS && BIG) && (ONE == 0 || (TRANS_B && !BIG && !DIGITS)));
    using sum_t          = typename sum_of<FORM>::type;
    constexpr int BT     = BIG ? 128 : 64; // rows and columns of the tile
    constexpr int BK     = ONE != 0 ? ONE : DIGITS ? 64 : BIG ? 128 : 256;
    constexpr int STAGES = ONE != 0 ? 1 : 2;
    constexpr int T      = BT / 32; // 16 x 16 tiles of a wave along either side
    constexpr int PLANES = DIGITS ? 3 : 1;
    constexpr int SUMS   = DIGITS ? 5 : 1;
    constexpr int PITCH  = BK + 16; // 16 lanes read 16 bytes of 16 rows: all banks, once
    constexpr int OPERAND = PLANES * BT * PITCH;
    constexpr int CHUNKS  = BT * BK / 16 / THREADS; // 16-byte pieces of an operand a thread moves
    constexpr int KR      = DIGITS ? 4 : 16;          // rows of row-major B a thread moves, 4 columns each
    static_assert(TRANS_B || (BK / KR) * (BT / 4) == THREADS);
    __shared__ __attribute__((aligned(16))) uint8_t lds[STAGES][2][OPERAND];
    __shared__ uint8_t nan_of[2][BT];

    const int tid    = threadIdx.x;
    const int lane   = tid & 63;
    const int wave   = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1;

    // a contiguous run of tiles per XCD (workgroups are dealt to the 8 of them in turn), rows first: the
    // tiles that share a panel of B follow each other in one L2
    const int total = p.tiles_m * p.tiles_n;
    // (one slab: runs everywhere; in turn 1.01 of their time over 350 products, up to 1.14)
    const int v     = ONE != 0 ? xcd_run(blockIdx.x, total) : xcd_place(blockIdx.x, total, p.tiles_m, p.tiles_n, p.k, total);
    const int m0 = (v % p.tiles_m) * BT;
    const int n0 = (v / p.tiles_m) * BT;

    const uint8_t* __restrict__ ga = p.a + (int64_t)blockIdx.y * p.stride_a;
    const uint8_t* __restrict__ gb = p.b + (int64_t)blockIdx.y * p.stride_b;

    // LDS row of column c of the tile
    auto b_row = [](int c) { return c / (16 * T) * (16 * T) + (c % T) * 16 + c % (16 * T) / T; };

    constexpr int KC = BK / 16; // chunks of a row
    const int ld_kc  = (tid % KC) * 16;
    uint32_t a_off[CHUNKS], b_off[TRANS_B ? CHUNKS : 1];
#pragma unroll
    for(int s = 0; s < CHUNKS; s++)
    {
        const int r = (tid + THREADS * s) / KC;
        a_off[s]    = (uint32_t)min(m0 + r, p.m - 1) * p.lda;
        if constexpr(TRANS_B)
            b_off[s] = (uint32_t)min(n0 + r, p.n - 1) * p.ldb;
    }
    // row-major B
    const int bc = (tid % (BT / 4)) * 4, bk = tid / (BT / 4) * KR;
    const int first = min(n0 + bc, p.n - 4);
    const int shift = min(8 * (n0 + bc - first), 31); // all four behind N: never stored

    // slabs on their way: a small one is multiplied in far less time than a load takes; the registers of
    // two big ones would leave room for one wave on a SIMD instead of two
    constexpr int AHEAD = BIG ? 1 : 2;
    uint4 ra[AHEAD][CHUNKS], rb4[AHEAD][TRANS_B ? CHUNKS : 1];
    uint32_t rb[AHEAD][TRANS_B ? 1 : KR];

    // no branch around a load: what lies behind K is put right on the way to the LDS, and slabs behind the
    // last are loads of its end again
    auto load_slab = [&](int k0, int u) {
        const int at = min(k0 + ld_kc, p.k - 16);
#pragma unroll
        for(int s = 0; s < CHUNKS; s++)
            ra[u][s] = load16(ga + a_off[s] + at);
        if constexpr(TRANS_B)
        {
#pragma unroll
            for(int s = 0; s < CHUNKS; s++)
                rb4[u][s] = load16(gb + b_off[s] + at);
        }
        else
        {
#pragma unroll
            for(int i = 0; i < KR; i++)
                rb[u][i] = load4(gb + (uint32_t)min(k0 + bk + i, p.k - 1) * p.ldb + first);
        }
    };

    uint32_t nan_a[CHUNKS] = {}, nan_b[CHUNKS] = {}; // row-major B: one, a byte for each of the four columns
    auto put16 = [&](uint8_t* at, uint4 w, uint32_t& nan) {
        if constexpr(DIGITS)
        {
            nan |= nan_bytes(w.x) | nan_bytes(w.y) | nan_bytes(w.z) | nan_bytes(w.w);
            uint32_t d[4][3];
            fp8_digits(w.x, d[0]);
            fp8_digits(w.y, d[1]);
            fp8_digits(w.z, d[2]);
            fp8_digits(w.w, d[3]);
#pragma unroll
            for(int q = 0; q < 3; q++)
                *reinterpret_cast<uint4*>(at + q * BT * PITCH) = make_uint4(d[0][q], d[1][q], d[2][q], d[3][q]);
        }
        else
            *reinterpret_cast<uint4*>(at) = w;
    };
    auto store_slab = [&](int kt, int stage, int u) {
        uint8_t* as = lds[stage][0];
        uint8_t* bs = lds[stage][1];
        if((kt + 1) * BK > p.k)
        {
            const int kk = kt * BK + ld_kc, past = kk - min(kk, p.k - 16);
#pragma unroll
            for(int s = 0; s < CHUNKS; s++)
            {
                ra[u][s] = shift_down(ra[u][s], past);
                if constexpr(TRANS_B)
                    rb4[u][s] = shift_down(rb4[u][s], past);
            }
        }
#pragma unroll
        for(int s = 0; s < CHUNKS; s++)
            put16(as + (tid + THREADS * s) / KC * PITCH + ld_kc, ra[u][s], nan_a[s]);
        if constexpr(TRANS_B)
        {
#pragma unroll
            for(int s = 0; s < CHUNKS; s++)
                put16(bs + b_row((tid + THREADS * s) / KC) * PITCH + ld_kc, rb4[u][s], nan_b[s]);
        }
        else
        {
            uint32_t w[KR];
#pragma unroll
            for(int i = 0; i < KR; i++)
                w[i] = rb[u][i] >> shift;
            if constexpr(DIGITS)
            {
                uint32_t c[4], d[3];
#pragma unroll
                for(int i = 0; i < 4; i++)
                    nan_b[0] |= nan_bytes(w[i]);
                transpose4(w, c);
#pragma unroll
                for(int j = 0; j < 4; j++)
                {
                    fp8_digits(c[j], d);
#pragma unroll
                    for(int q = 0; q < 3; q++)
                        *reinterpret_cast<uint32_t*>(bs + (q * BT + b_row(bc + j)) * PITCH + bk) = d[q];
                }
            }
            else
            {
                uint32_t c[4][4];
#pragma unroll
                for(int q = 0; q < 4; q++)
                    transpose4(w + 4 * q, c[q]);
#pragma unroll
                for(int j = 0; j < 4; j++)
                    *reinterpret_cast<uint4*>(bs + b_row(bc + j) * PITCH + bk) =
                        make_uint4(c[0][j], c[1][j], c[2][j], c[3][j]);
            }
        }
    };

    sum_t acc[SUMS][T][T];
#pragma unroll
    for(int w = 0; w < SUMS; w++)
#pragma unroll
        for(int i = 0; i < T; i++)
#pragma unroll
            for(int j = 0; j < T; j++)
                acc[w][i][j] = sum_t{0, 0, 0, 0};

    // lane l supplies row l % 16 of an operand tile and K bytes 16 * (l / 16) .. + 15 of 64 (float sums:
    // 32 * (l / 16) .. + 31 of 128)
    constexpr int PIECE = FORM == FP8_FLOAT ? 32 : 16;
    const int frag_off  = (lane & 15) * PITCH + (lane >> 4) * PIECE;
    auto multiply = [&](int stage) {
        const uint8_t* as = lds[stage][0] + frag_off + wave_m * 16 * T * PITCH;
        const uint8_t* bs = lds[stage][1] + frag_off + wave_n * 16 * T * PITCH;
#pragma unroll
        for(int h = 0; h < BK; h += 4 * PIECE)
        {
            if constexpr(FORM == FP8_FLOAT)
            {
                v8i fa[T], fb[T];
#pragma unroll
                for(int i = 0; i < T; i++)
                {
                    __builtin_memcpy(&fa[i], __builtin_assume_aligned(as + 16 * i * PITCH + h, 16), 32);
                    __builtin_memcpy(&fb[i], __builtin_assume_aligned(bs + 16 * i * PITCH + h, 16), 32);
                }
#pragma unroll
                for(int i = 0; i < T; i++)
#pragma unroll
                    for(int j = 0; j < T; j++) // scales of zero select the unscaled instruction
                        acc[0][i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[i], fb[j], acc[0][i][j], 0, 0,
                                                                                        0, 0, 0, 0);
            }
            else
            {
                v4i fa[PLANES][T], fb[PLANES][T];
#pragma unroll
                for(int q = 0; q < PLANES; q++)
#pragma unroll
                    for(int i = 0; i < T; i++)
                    {
                        fa[q][i] = *reinterpret_cast<const v4i*>(as + (q * BT + 16 * i) * PITCH + h);
                        fb[q][i] = *reinterpret_cast<const v4i*>(bs + (q * BT + 16 * i) * PITCH + h);
                    }
#pragma unroll
                for(int qa = 0; qa < PLANES; qa++)
#pragma unroll
                    for(int qb = 0; qb < PLANES; qb++)
#pragma unroll
                        for(int i = 0; i < T; i++)
#pragma unroll
                            for(int j = 0; j < T; j++)
                                acc[qa + qb][i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[qa][i], fb[qb][j],
                                                                                           acc[qa + qb][i][j], 0, 0, 0);
            }
        }
    };
    if constexpr(DIGITS)
    {
        if(tid < 2 * BT)
            nan_of[tid / BT][tid % BT] = 0;
    }
    // slab kt sits in stage kt & 1; while it is multiplied, the next ones are loaded
    const int nk = (p.k + BK - 1) / BK;
    load_slab(0, 0);
    if constexpr(AHEAD == 2 && ONE == 0)
        load_slab(BK, 1);
    store_slab(0, 0, 0);
    __syncthreads();
    [[maybe_unused]] auto step = [&](int kt, int u) {
        load_slab((kt + AHEAD) * BK, AHEAD == 2 ? u : 0);
        multiply(u);
        // the other stage was last read before the barrier that ended the step before
        if(kt + 1 < nk)
            store_slab(kt + 1, u ^ 1, AHEAD == 2 ? u ^ 1 : 0);
        lds_barrier();
    };
    int kt = 0;
    if constexpr(ONE == 0)
    {
        for(; kt + 1 < nk; kt += 2)
        {
            step(kt, 0);
            step(kt + 1, 1);
        }
    }
    if(kt < nk)
        multiply(0);
    if constexpr(DIGITS)
    {
        static_assert(CHUNKS == 1);
        if(nan_a[0] != 0)
            nan_of[0][tid / KC] = 1;
        if constexpr(TRANS_B)
        {
            if(nan_b[0] != 0)
                nan_of[1][tid / KC] = 1;
        }
        else
        {
#pragma unroll
            for(int j = 0; j < 4; j++)
                if(nan_b[0] >> (8 * j) & 0x80u)
                    nan_of[1][bc + j] = 1;
        }
        __syncthreads();
    }

    // acc[.][i][j][r]: row 16 i + 4 (lane / 16) + r, column T (lane % 16) + j of the wave's part
    const int col = n0 + wave_n * 16 * T + T * (lane & 15);
    const int cnt = p.n - col;
    if(cnt <= 0)
        return;
    float sa[T][4], sb[T], bias[T];
    int32_t cs[T];
    if constexpr(OUT >= 0)
    {
#pragma unroll
        for(int i = 0; i < T; i++)
#pragma unroll
            for(int r = 0; r < 4; r++)
                sa[i][r] = 1.f;
        // one branch for a group of loads, all ahead of the stores
        const int last = p.n - 1 - col;
#pragma unroll
        for(int j = 0; j < T; j++)
        {
            sb[j]   = 1.f;
            bias[j] = -0.0f;
            cs[j]   = 0;
        }
        if(p.scale_a_mode != MI355_QP_NONE)
        {
            const int each = p.scale_a_mode == MI355_QP_PER_ROW ? 1 : 0;
#pragma unroll
            for(int i = 0; i < T; i++)
#pragma unroll
                for(int r = 0; r < 4; r++)
                    sa[i][r] = p.scale_a[each * min(m0 + wave_m * 16 * T + 16 * i + 4 * (lane >> 4) + r, p.m - 1)];
        }
        if(p.scale_b_mode != MI355_QP_NONE)
        {
            const int each = p.scale_b_mode == MI355_QP_PER_COL ? 1 : 0;
#pragma unroll
            for(int j = 0; j < T; j++)
                sb[j] = p.scale_b[each * (col + min(j, last))];
        }
        if(p.bias != nullptr)
        {
#pragma unroll
            for(int j = 0; j < T; j++)
                bias[j] = p.bias[col + min(j, last)];
        }
        if(p.zp_a != 0)
        {
#pragma unroll
            for(int j = 0; j < T; j++)
                cs[j] = p.colsum_b[col + min(j, last)];
        }
    }
#pragma unroll
    for(int i = 0; i < T; i++)
#pragma unroll
        for(int r = 0; r < 4; r++)
        {
            const int in_tile = wave_m * 16 * T + 16 * i + 4 * (lane >> 4) + r;
            const int row     = m0 + in_tile;
            if(row >= p.m)
                continue;
            const int64_t idx = (int64_t)blockIdx.y * p.stride_c + (int64_t)row * p.ldc + col;
            double sum[T]; // digits, put together
            if constexpr(DIGITS)
            {
#pragma unroll
                for(int j = 0; j < T; j++)
                {
                    double t = acc[SUMS - 1][i][j][r];
#pragma unroll
                    for(int w = SUMS - 2; w >= 0; w--)
                        t = t * 256.0 + (double)acc[w][i][j][r];
                    // a whole number below 2^51 in units of 2^-18, rounded once (quant_dot's own type)
                    sum[j] = (double)(float)(t * 0x1p-18);
                    if(nan_of[0][in_tile] | nan_of[1][wave_n * 16 * T + T * (lane & 15) + j])
                        sum[j] = __builtin_nan("");
                }
            }
            float out[T];
            if constexpr(OUT < 0)
            {
#pragma unroll
                for(int j = 0; j < T; j++)
                    if constexpr(DIGITS)
                        out[j] = (float)sum[j];
                    else if constexpr(FORM == INT8)
                        out[j] = __builtin_bit_cast(float, (int)acc[0][i][j][r]);
                    else
                        out[j] = acc[0][i][j][r];
                store_n<MI355_F32, T>(p.c, idx, out, cnt);
            }
            else
            {
                int64_t zrow = 0;
                if(FORM == INT8 && p.zp_b != 0)
                    zrow = (int64_t)p.zp_b * p.rowsum_a[row] - (int64_t)p.k * p.zp_a * p.zp_b;
#pragma unroll
                for(int j = 0; j < T; j++)
                {
                    const float s = sa[i][r] * sb[j];
                    double d;
                    if constexpr(DIGITS)
                        d = sum[j];
                    else if constexpr(FORM == FP8_FLOAT)
                        d = (double)acc[0][i][j][r];
                    else
                        d = (double)acc[0][i][j][r] - (double)(int32_t)(zrow + (int64_t)p.zp_a * cs[j]);
                    out[j] = add_bias((float)(d * (double)s), bias[j]);
                }
                store_n<OUT, T>(p.c, idx, out, cnt);
            }
        }
}

// B as [N, K], K in one slab of 128 at most, in 64 x 64 tiles; a grid holds less than 2^32 threads along x.  The slab is
// the faster one while the result stays within 1.4 times the last-level cache (1360 random products of both types:
// 0.80 of the two-slab tiles' time): 96 x 197 x 197 x 64 int8 11.3 -> 9.3 us, 104 x 475 x 475 x 64 36.4 -> 27.4, 64 x 1000 x
// 1000 x 64 67 -> 48 (all to float32).  Larger ones leave at the memory's rate, which rows that end inside a line of
// 128 bytes hold up, less so from tiles of 128 x 128: 11707 x 16424 x 128 fp8 bare 241 us against 278, 10874 x 13531 x 32
// int8 230 against 266.  The slab stays where those would be padding for a third and more (1910 x 828 x 64 x 114
// 243 -> 139), and for scaled results of many matrices (312 x 975 x 975 x 64 fp8 to half 359 -> 302).
bool one_slab(bool trans_b, int64_t batch, int64_t m, int64_t n, int64_t k, int64_t elem_bytes, bool scaled)
{
    const int64_t tiles = ((m + 63) / 64) * ((n + 63) / 64), big = ((m + 127) / 128) * ((n + 127) / 128);
    return trans_b && k <= 128 && tiles < ((int64_t)1 << 32) / THREADS &&
           (batch * m * n * elem_bytes <= 350000000 || n * elem_bytes % 128 == 0 || 8 * big >= 3 * tiles ||
            (scaled && batch > 1));
}

template <int FORM, bool TRANS_B, int OUT, bool BIG, int ONE = 0>
int launch_tile(ragged_params& p, int batch, hipStream_t s)
{
    constexpr int BT = BIG ? 128 : 64;
    p.tiles_m        = (p.m + BT - 1) / BT;
    p.tiles_n        = (p.n + BT - 1) / BT;
    hipLaunchKernelGGL((qgemm_ragged_kernel<FORM, TRANS_B, OUT, BIG, ONE>), dim3((unsigned)(p.tiles_m * p.tiles_n), batch),
                       dim3(THREADS), 0, s, p);
    return mi355_launch_status();
}

template <int FORM, bool TRANS_B, int OUT>
int launch_out(ragged_params& p, int batch, hipStream_t s)
{
    if constexpr(TRANS_B && FORM != FP8_DIGITS)
    {
        if(one_slab(TRANS_B, batch, p.m, p.n, p.k, OUT == MI355_F16 || OUT == MI355_BF16 ? 2 : 4, OUT != -1))
        {
            if constexpr(FORM == INT8)
            {
                if(p.k <= 64)
                    return launch_tile<FORM, TRANS_B, OUT, false, 64>(p, batch, s);
            }
            return launch_tile<FORM, TRANS_B, OUT, false, 128>(p, batch, s);
        }
    }
    // the larger tile re-reads half as much and multiplies twice as often per LDS read, once it gives every
    // CU a workgroup (digits: its five sums would not fit the registers)
    if constexpr(FORM != FP8_DIGITS)
    {
        const int64_t big = (int64_t)batch * ((p.m + 127) / 128) * ((p.n + 127) / 128);
        if(big >= 256)
            return launch_tile<FORM, TRANS_B, OUT, true>(p, batch, s);
    }
    return launch_tile<FORM, TRANS_B, OUT, false>(p, batch, s);
}

template <int FORM, bool TRANS_B>
int launch_type(ragged_params& p, bool deq, int out, int batch, hipStream_t s)
{
    if(!deq)
        return launch_out<FORM, TRANS_B, -1>(p, batch, s);
    switch(out)
    {
    case MI355_F32: return launch_out<FORM, TRANS_B, MI355_F32>(p, batch, s);
    case MI355_F16: return launch_out<FORM, TRANS_B, MI355_F16>(p, batch, s);
    case MI355_BF16: return launch_out<FORM, TRANS_B, MI355_BF16>(p, batch, s);
    default: return MI355_ERR_UNSUPPORTED;
    }
}

template <int FORM>
int launch_form(ragged_params& p, bool trans_b, bool deq, int out, int batch, hipStream_t s)
{
    return trans_b ? launch_type<FORM, true>(p, deq, out, batch, s) : launch_type<FORM, false>(p, deq, out, batch, s);
}

} // namespace

// Any alignment and leading dimension, A row-major; what the loads need is a whole 16-byte piece in a
// row along K and a whole group of 4 in a row of row-major B, and offsets that fit 32 bits.  fp8: the
// digit sums (up to three products of 2^14 per k) stay in int32 up to K = 43690.
bool mi355_ragged_gemm_supported(const mi355_quant_dot_desc* d)
{
    if(d->in_type != MI355_I8 && d->in_type != MI355_FP8)
        return false;
    if(d->trans_a || d->k < 16 || (!d->trans_b && d->n < 4))
        return false;
    if(d->in_type == MI355_FP8 && d->k > 32768)
        return false;
    const int64_t lim = (int64_t)1 << 31;
    // positions along K are ints and run up to two slabs of 256 and a row of pieces past the end
    if(d->m >= lim / 256 || d->n >= lim / 256 || d->lda >= lim || d->ldb >= lim || d->k >= lim - 1024)
        return false;
    // a grid holds less than 2^32 threads along x; int8 results that large take tiles of 128 x 128
    const int64_t side  = d->in_type == MI355_I8 ? 128 : 64;
    const int64_t tiles = ((d->m + side - 1) / side) * ((d->n + side - 1) / side);
    return d->m * d->lda < lim && (d->trans_b ? d->n * d->ldb : d->k * d->ldb) < lim &&
           tiles < ((int64_t)1 << 32) / THREADS;
}

// not for the exact sums of e4m3fn
bool mi355_ragged_gemm_one_slab(const mi355_quant_dot_desc* d)
{
    return one_slab(d->trans_b, d->batch, d->m, d->n, d->k, d->dequant ? (int64_t)mi355_dtype_size(d->out_type) : 4,
                    d->dequant != 0);
}

int mi355_ragged_gemm_launch(const mi355_quant_dot_desc* d,
                             const void* a,
                             const void* b,
                             void* c,
                             const float* scale_a,
                             const float* scale_b,
                             const int32_t* colsum_b,
                             const int32_t* rowsum_a,
                             const float* bias,
                             bool float_sums,
                             hipStream_t stream)
{
    ragged_params p{};
    p.a            = static_cast<const uint8_t*>(a);
    p.b            = static_cast<const uint8_t*>(b);
    p.c            = c;
    p.m            = (int)d->m;
    p.n            = (int)d->n;
    p.k            = (int)d->k;
    p.lda          = (uint32_t)d->lda;
    p.ldb          = (uint32_t)d->ldb;
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
    const bool deq = d->dequant != 0;
    const int batch = (int)d->batch;
    if(d->in_type == MI355_I8)
        return launch_form<INT8>(p, d->trans_b, deq, d->out_type, batch, stream);
    return float_sums ? launch_form<FP8_FLOAT>(p, d->trans_b, deq, d->out_type, batch, stream)
                      : launch_form<FP8_DIGITS>(p, d->trans_b, deq, d->out_type, batch, stream);
}
