// Split K for results of few 128 x 128 tiles (included by qgemm_dma.hip inside its anonymous namespace): float or
// int32 sums of a share each in a workspace, added by reduce_partials_kernel.
//
// The 256 x 256 kernels spend half of their loads and products on rows that 128 rows of A do not have, and
// need eight shares of K to give every CU a tile: 32 MiB of partial sums for 128 x 8192 results.  Here a
// workgroup of 8 waves (2 x 4, 64 x 32 each) walks its share of K in slabs of 128 bytes; A and B go straight into an
// LDS ring of four slabs, three of them in flight.  What bounds it is the rate at which a CU that owns one workgroup
// takes lines in (0.7 us for the 32 KiB of a slab, 15 bytes a busy clock; matrix cores busy 23 %, LDS reads in conflict
// 40 % of their cycles), then the partial sums' way out and back (0.38 us a MB).
// Both launches, B as [K, N] from memory, before -> now: 128 x 8192 x 8192 fp8 33.2 -> 25.9 us, 256 x 4096 x 8192
// 32.9 -> 24.6, 1000 x 1024 x 8192 31.5 -> 24.8, 32 x 4096 x 4096 16.0 -> 11.7, 20 x 512 x 4096 9.8 -> 6.9,
// 100 x 4096 x 14336 29.9 -> 22.7; int8 the same within 4 %.
//
// LDS: a row of 128 bytes is 8 chunks of 16; chunk c of row r of a K-contiguous operand sits at position
// c ^ (r / 2 % 8), so that 16 rows of one chunk are 16 different bank groups; chunk c (16 columns) of row k of a
// row-major B at c ^ (k / 2 % 4 + 4 * (k / 32 % 2)), which keeps the 8 x 16 blocks of two lane groups apart.
// Lane group g multiplies K bytes 32 g .. 32 g + 31 of a slab, int8 in two products of 16 each.
// What lies behind K (half a slab, K being whole runs of 64) is zero in A's registers; B repeats rows of its own
// there, which brings no NaN into a column that has none.
constexpr int SH_T      = 128; // rows and columns of the tile
constexpr int SH_SLAB   = 128; // bytes of K
constexpr int SH_RING   = 4;
constexpr int SH_OPER   = SH_T * SH_SLAB;
constexpr int SH_STAGE  = 2 * SH_OPER;
constexpr int SH_LDS    = SH_RING * SH_STAGE;
constexpr int SH_LOADS  = SH_STAGE / 1024 / 8; // a wave's loads of a slab

template <bool FP8, bool TRANS_B>
__global__ __launch_bounds__(512) void qgemm_shares_kernel(dma_params p, int per)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    using sum_t      = std::conditional_t<FP8, v4f, v4i>;
    const int tid    = threadIdx.x;
    const int lane   = tid & 63;
    const int wave   = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 2, wave_n = wave & 3;
    const int i = lane & 15, g = lane >> 4;

    // A contiguous run of (share, column) pairs per XCD, the row tiles that share a panel of B one after the other, where
    // the workgroups are a multiple of 8; any other number is dealt in turn.  (xcd_run for those too: 70 products 0.83 to
    // 1.06 of the time, 1.006 in the mean: these few workgroups share less than its divisions cost.)
    const int total = (int)gridDim.x;
    int v           = blockIdx.x;
    if(total % 8 == 0)
        v = (v % 8) * (total / 8) + v / 8;
    const int m0    = (v % p.tiles_m) * SH_T;
    const int n0    = (v / p.tiles_m % p.tiles_n) * SH_T;
    const int share = v / (p.tiles_m * p.tiles_n);
    const int first = share * per; // slab
    const int nk    = min(per, (p.k + SH_SLAB - 1) / SH_SLAB - first);

    // ---- global -> LDS: a load is 8 rows of 128 bytes ---------------------------------------------------
    const int lr = lane >> 3, pos = lane & 7;
    uint32_t off[SH_LOADS];
    int k_of[SH_LOADS]; // K of the lane's piece within a slab
#pragma unroll
    for(int s = 0; s < SH_LOADS; s++)
    {
        const int r = (wave + 8 * (s & 1)) * 8 + lr; // s = 0, 1: A; 2, 3: B
        if(s >= 2 && !TRANS_B)
        {
            const int c = pos ^ ((r >> 1 & 3) | (r >> 5 & 1) << 2);
            k_of[s]     = r;
            off[s]      = (uint32_t)min(n0 + 16 * c, p.n - 16);
        }
        else
        {
            const int c = pos ^ (r >> 1 & 7);
            k_of[s]     = 16 * c;
            off[s]      = s < 2 ? (uint32_t)min(m0 + r, p.m - 1) * (uint32_t)p.lda
                                : (uint32_t)min(n0 + r, p.n - 1) * (uint32_t)p.ldb;
        }
    }
    auto issue = [&](int kt) {
        uint8_t* stage = lds + (kt & (SH_RING - 1)) * SH_STAGE + wave * 1024;
        const int k0   = (first + kt) * SH_SLAB;
#pragma unroll
        for(int s = 0; s < SH_LOADS; s++)
        {
            int k = k0 + k_of[s];
            k     = k < p.k ? k : k - 64; // behind K: the half in front of it
            const uint32_t at = s >= 2 && !TRANS_B ? off[s] + (uint32_t)k * (uint32_t)p.ldb : off[s] + (uint32_t)k;
            load_to_lds((s < 2 ? p.a : p.b) + at, stage + (s >= 2 ? SH_OPER : 0) + (s & 1) * 8192);
        }
    };

    // ---- LDS -> fragments; every read is waited for in the statement that issues it -------------------------
    const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) uint8_t*)lds);
    const int a_row     = wave_m * 64 + i; // tiles of 16 rows follow each other: the same swizzle in each
    uint32_t a_at[2], b_at[2];
#pragma unroll
    for(int h = 0; h < 2; h++)
    {
        a_at[h] = (uint32_t)(a_row * SH_SLAB + ((2 * g + h) ^ (a_row >> 1 & 7)) * 16);
        if constexpr(TRANS_B)
        {
            const int r = wave_n * 32 + i;
            b_at[h]     = (uint32_t)(SH_OPER + r * SH_SLAB + ((2 * g + h) ^ (r >> 1 & 7)) * 16);
        }
        else
        {
            // h: the column tile.  Lane i of a group supplies half i % 2 of row i / 2 of an 8 x 16 block and
            // receives column i; blocks of 8 rows of K follow each other
            const int k = 32 * g + (i >> 1), c = wave_n * 2 + h;
            b_at[h] = (uint32_t)(SH_OPER + k * SH_SLAB + (c ^ ((k >> 1 & 3) | (k >> 5 & 1) << 2)) * 16 + 8 * (i & 1));
        }
    }
    auto join = [](v4i lo, v4i hi) { return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w}; };

    sum_t acc[4][2];
#pragma unroll
    for(int a = 0; a < 4; a++)
#pragma unroll
        for(int b = 0; b < 2; b++)
            acc[a][b] = sum_t{0, 0, 0, 0};
    // B first: a lane owns 4 consecutive columns of one row
    auto product = [&](const v8i& fa, const v8i& fb, sum_t c) -> sum_t {
        if constexpr(FP8) // scales of zero select the unscaled instruction
            return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, c, 0, 0, 0, 0, 0, 0);
        else
        {
            c = __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{fb[0], fb[1], fb[2], fb[3]}, v4i{fa[0], fa[1], fa[2], fa[3]}, c,
                                                      0, 0, 0);
            return __builtin_amdgcn_mfma_i32_16x16x64_i8(v4i{fb[4], fb[5], fb[6], fb[7]}, v4i{fa[4], fa[5], fa[6], fa[7]},
                                                         c, 0, 0, 0);
        }
    };
    auto multiply = [&](int kt) {
        const uint32_t base = lds0 + (uint32_t)((kt & (SH_RING - 1)) * SH_STAGE);
        const uint32_t a0 = base + a_at[0], a1 = base + a_at[1], b0 = base + b_at[0], b1 = base + b_at[1];
        v8i fb[2];
        v4i l0, h0, l1, h1;
        if constexpr(TRANS_B)
        {
            v4i p0, q0, p1, q1;
            asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %8 offset:2048\n\t"
                         "ds_read_b128 %3, %9 offset:2048\n\tds_read_b128 %4, %10\n\tds_read_b128 %5, %11\n\t"
                         "ds_read_b128 %6, %10 offset:2048\n\tds_read_b128 %7, %11 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(p0), "=&v"(q0), "=&v"(p1), "=&v"(q1), "=&v"(l0), "=&v"(h0), "=&v"(l1), "=&v"(h1)
                         : "v"(b0), "v"(b1), "v"(a0), "v"(a1)
                         : "memory");
            fb[0] = join(p0, q0);
            fb[1] = join(p1, q1);
        }
        else
        {
            v2i p0, p1, p2, p3, q0, q1, q2, q3;
            asm volatile("ds_read_b64_tr_b8 %0, %12\n\tds_read_b64_tr_b8 %1, %12 offset:1024\n\t"
                         "ds_read_b64_tr_b8 %2, %12 offset:2048\n\tds_read_b64_tr_b8 %3, %12 offset:3072\n\t"
                         "ds_read_b64_tr_b8 %4, %13\n\tds_read_b64_tr_b8 %5, %13 offset:1024\n\t"
                         "ds_read_b64_tr_b8 %6, %13 offset:2048\n\tds_read_b64_tr_b8 %7, %13 offset:3072\n\t"
                         "ds_read_b128 %8, %14\n\tds_read_b128 %9, %15\n\t"
                         "ds_read_b128 %10, %14 offset:2048\n\tds_read_b128 %11, %15 offset:2048\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(p0), "=&v"(p1), "=&v"(p2), "=&v"(p3), "=&v"(q0), "=&v"(q1), "=&v"(q2), "=&v"(q3),
                           "=&v"(l0), "=&v"(h0), "=&v"(l1), "=&v"(h1)
                         : "v"(b0), "v"(b1), "v"(a0), "v"(a1)
                         : "memory");
            fb[0] = v8i{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
            fb[1] = v8i{q0.x, q0.y, q1.x, q1.y, q2.x, q2.y, q3.x, q3.y};
        }
        v8i fa0 = join(l0, h0), fa1 = join(l1, h1);
        const bool half = (first + kt) * SH_SLAB + 64 >= p.k;
        const v8i zero  = {0, 0, 0, 0, 0, 0, 0, 0};
        if(half && g >= 2)
            fa0 = fa1 = zero;
#pragma unroll
        for(int b = 0; b < 2; b++)
        {
            acc[0][b] = product(fa0, fb[b], acc[0][b]);
            acc[1][b] = product(fa1, fb[b], acc[1][b]);
        }
        asm volatile("ds_read_b128 %0, %4 offset:4096\n\tds_read_b128 %1, %5 offset:4096\n\t"
                     "ds_read_b128 %2, %4 offset:6144\n\tds_read_b128 %3, %5 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(l0), "=&v"(h0), "=&v"(l1), "=&v"(h1)
                     : "v"(a0), "v"(a1)
                     : "memory");
        fa0 = join(l0, h0);
        fa1 = join(l1, h1);
        if(half && g >= 2)
            fa0 = fa1 = zero;
#pragma unroll
        for(int b = 0; b < 2; b++)
        {
            acc[2][b] = product(fa0, fb[b], acc[2][b]);
            acc[3][b] = product(fa1, fb[b], acc[3][b]);
        }
    };

    // ---- main loop: behind barrier kt slab kt has landed for every wave, and every wave has read slab kt - 1, whose
    // stage the loads of slab kt + 3 overwrite.  A wave's loads land in order.
#pragma unroll
    for(int s = 0; s < SH_RING - 1; s++)
        if(s < nk)
            issue(s);
    for(int kt = 0; kt < nk; kt++)
    {
        if(kt + 2 < nk)
            wait_vmcnt<2 * SH_LOADS>();
        else if(kt + 1 < nk)
            wait_vmcnt<SH_LOADS>();
        else
            wait_vmcnt<0>();
        block_barrier();
        if(kt + SH_RING - 1 < nk)
            issue(kt + SH_RING - 1);
        multiply(kt);
    }

    // element r of lane (i, g) of tile (a, b): row 16 a + i, column 16 b + 4 g + r of the wave's part
    int32_t* out = p.partial + (int64_t)share * p.m * p.partial_ld;
#pragma unroll
    for(int a = 0; a < 4; a++)
    {
        const int row = m0 + wave_m * 64 + 16 * a + i;
        if(row >= p.m)
            continue;
#pragma unroll
        for(int b = 0; b < 2; b++)
        {
            const int col = n0 + wave_n * 32 + 16 * b + 4 * g;
            if(col < p.n)
                *reinterpret_cast<v4i*>(out + (int64_t)row * p.partial_ld + col) = __builtin_bit_cast(v4i, acc[a][b]);
        }
    }
}

template <bool FP8, bool TRANS_B>
int launch_shares(dma_params p, int shares, hipStream_t s)
{
    auto kern = qgemm_shares_kernel<FP8, TRANS_B>;
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, SH_LDS);
    if(attr != hipSuccess)
        return MI355_ERR_LAUNCH;
    p.tiles_m     = (p.m + SH_T - 1) / SH_T;
    p.tiles_n     = (p.n + SH_T - 1) / SH_T;
    const int nk  = (p.k + SH_SLAB - 1) / SH_SLAB;
    const int per = (nk + shares - 1) / shares;
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n * shares)), dim3(512), SH_LDS, s, p, per);
    return mi355_launch_status();
}
