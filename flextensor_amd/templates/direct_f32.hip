// fp32 GEMM and convolution without LDS tiles, for gfx950 (CDNA4), compiled with hiprtc.
//
//   C[M][N] = A[M][K] * B[K][N]           fp32 in, fp32 out, fp32 sums
//
// The same operators, addressing modes and group index as igemm_f32.hip (MODE 0: B [K][N], MODE 2: B stored
// [N][K], MODE 1: conv2d NCHW with B gathered from the image and A the weight; CG groups or batch entries). Operands
// go from memory straight to the registers of the lane that feeds them to the matrix core, without LDS and without a
// barrier in the main loop: a lane's eight k of a row are 32 consecutive bytes, four lanes read a whole line, and for
// B [K][N] a lane takes REP_N neighbouring columns with one load per k (so its REP_N blocks of 16 columns are
// interleaved). The wavefronts of a workgroup divide K rather than the tile (WAVES_K groups, summed through LDS at
// the end), so none of them waits for another, and few tiles still fill the chip.
//
// What bounds it: matrix clocks where tiles are many, the loads' latency where they are few; PD steps of 32 k are on
// their way at a time. igemm_f32.hip shares every operand between the wavefronts of a tile through LDS and pays a
// barrier and an LDS round trip per K tile for it; this is the better split where tiles are small or few (few rows,
// few output channels), or where the LDS kernels compute channel, tap and predicate anew for every gathered element (here
// they come from a table in LDS, made once per workgroup). Measured, LDS kernel and this one: 4x54x24x24 -> 27 3x3 5.8 and
// 4.2 us, 13x77x8x8 -> 130 3x3 8.2 and 7.2, 74x3120x1200 22.7 and 14.4 (matrix cores busy 18 and 42 % of the time),
// 16x119x24x23 -> 74 5x5 90.9 and 68.7; the other way round 112x4096x4096 36.6 and 50.4, 16x128x57x57 -> 256 3x3 stride 2 77.7
// and 142.

#ifndef FT_SPLIT
#define MODE FT_MODE
#define M FT_M
#define N FT_N
#define K FT_K
#define WAVES_M FT_WAVES_M
#define WAVES_N FT_WAVES_N
#define REP_M FT_REP_M
#define REP_N FT_REP_N
#define WAVES_K FT_WAVES_K      /* wavefront groups that divide K, summed through LDS */
#define GROUP_M FT_GROUP_M
#define XCD_REMAP FT_XCD_REMAP
#define PD FT_PD                /* k steps in registers or on their way to them */
#ifdef FT_HAS_BIAS
#define HAS_BIAS FT_HAS_BIAS
#else
#define HAS_BIAS 0
#endif
#ifdef FT_COLOUT
#define COLOUT FT_COLOUT
#else
#define COLOUT 0
#endif
#ifdef FT_CG
#define CG FT_CG
#else
#define CG 1
#endif

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

#define BM (WAVES_M * REP_M * 16)
#define BN (WAVES_N * REP_N * 16)
#define NW (WAVES_M * WAVES_N)          /* wavefronts of one k group */
#define NTW (NW * WAVES_K * 64)
#define TILES_M ((M + BM - 1) / BM)
#define TILES_N ((N + BN - 1) / BN)
#define STEPS ((K + 31) / 32)
#define GSTEPS ((STEPS + WAVES_K - 1) / WAVES_K)        /* k steps of a group; the last groups may have fewer */
#define NBLK (REP_M * REP_N)
#define NOUT ((NBLK + WAVES_K - 1) / WAVES_K)           /* blocks a wavefront sums and stores */
#if K < 32
#error "rows of a k step and more"
#endif

#define OOB 0x80000000u
#if MODE == 1
#define CB FT_CB
#define CC FT_CC
#define CH FT_CH
#define CW FT_CW
#define CR FT_CR
#define CS FT_CS
#define CSTRH FT_CSTRH
#define CSTRW FT_CSTRW
#define CPADH FT_CPADH
#define CPADW FT_CPADW
#define CDILH FT_CDILH
#define CDILW FT_CDILW
#define CP FT_CP
#define CQ FT_CQ
#define OHW (CP * CQ)
#define B_BYTES (CB * CC * CH * CW * 4)
#define PADDED (CPADH > 0 || CPADW > 0)
#if CR * CS > 31
#error "a pixel's valid taps are bits of a word"
#endif
#define TABLE (STEPS * 32)              /* entries (byte offset, tap) of the gathered operand's k */
#else
#define TABLE 0
#if MODE == 0
/* B ends where its rows end: rows at and behind K are beyond the buffer and read as zero */
#define B_BYTES ((gi + 1) * K * N * 4)
#else
#define B_BYTES (CG * K * N * 4)
#endif
#endif
#define A_BYTES (CG * M * K * 4)
#if MODE == 0
#define COLUMN(j) (REP_N * li + (j))    /* column inside the wavefront's tile */
#if REP_N != 1 && REP_N != 2 && REP_N != 4
#error "a lane's columns are one load"
#endif
#else
#define COLUMN(j) (16 * (j) + li)
#endif

#ifdef FT_CLKPROBE          /* as in igemm_f32.hip */
#define CLK_PARAM , unsigned long long* __restrict__ ft_clk
#if FT_CLKPROBE == 2
#define CLK_BEGIN const unsigned long long ft_r0 = wall_clock64();
#define CLK_END do { __builtin_amdgcn_s_waitcnt(0x0F70); \
        if (threadIdx.x == 0) { ft_clk[2 * blockIdx.x] = ft_r0; ft_clk[2 * blockIdx.x + 1] = wall_clock64(); } } while (0)
#else
#define CLK_BEGIN const unsigned long long ft_t0 = __builtin_readcyclecounter(), ft_r0 = wall_clock64();
#define CLK_END do { __builtin_amdgcn_s_waitcnt(0x0F70); \
        if (threadIdx.x == 0) { ft_clk[2 * blockIdx.x] = __builtin_readcyclecounter() - ft_t0; \
                                ft_clk[2 * blockIdx.x + 1] = wall_clock64() - ft_r0; } } while (0)
#endif
#else
#define CLK_PARAM
#define CLK_BEGIN
#define CLK_END do { } while (0)
#endif

static __device__ __forceinline__ float ld1(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, so, 0));
}
static __device__ __forceinline__ f32x4 ld4(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, so, 0));
}
static __device__ __forceinline__ f32x2 ld2(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)vo, so, 0));
}

extern "C" __global__ __launch_bounds__(NTW, 2)         /* two wavefronts a SIMD */
void igemm_f32(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C
#if HAS_BIAS
               , const float* __restrict__ bias
#endif
               CLK_PARAM)
{
    CLK_BEGIN
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int kg = wave / NW, wm = wave % NW / WAVES_N, wn = wave % WAVES_N;
    const int li = lane & 15, lg = lane >> 4;

    /* ---- workgroup -> (group, tile): with XCD_REMAP consecutive logical tiles stay on one XCD, whatever their number
     * (the first nblk % 8 XCDs have one more) --------------------------------------------------------------- */
    int bid = blockIdx.x;
#if XCD_REMAP
    const int nblk = TILES_M * TILES_N * CG;
    bid = (bid % 8) * (nblk / 8) + (nblk % 8 == 0 ? 0 : bid % 8 < nblk % 8 ? bid % 8 : nblk % 8) + bid / 8;
#endif
    const int gi = bid / (TILES_M * TILES_N);
    int m0, n0;                         /* of the wavefront's tile */
    {
        const int r = bid % (TILES_M * TILES_N);
        const int first_m = r / (GROUP_M * TILES_N) * GROUP_M;
        const int gsz = (TILES_M - first_m) < GROUP_M ? (TILES_M - first_m) : GROUP_M;
        const int rr = r % (GROUP_M * TILES_N);
        m0 = (first_m + rr % gsz) * BM + wm * REP_M * 16;
        n0 = (rr / gsz) * BN + wn * REP_N * 16;
    }

    /* ---- operands: raw buffer loads, an offset beyond the buffer reads as zero. Offsets are selects of two values,
     * never branches. ------------------------------------------------------------------------------------------- */
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, A_BYTES, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, B_BYTES, 0x00020000);
    unsigned a_off[REP_M];
#pragma unroll
    for (int i = 0; i < REP_M; ++i) {
        const int m = m0 + 16 * i + li;
        const unsigned off = (unsigned)((gi * M + m) * K + 8 * lg) * 4u;
        a_off[i] = m < M ? off : OOB;
    }
#if MODE == 0
    unsigned b_off;
    {
        const int n = n0 + COLUMN(0);   /* columns behind N belong to the next row and feed results that are not stored */
        const unsigned off = (unsigned)((gi * K + 8 * lg) * N + n) * 4u;
        b_off = n < N ? off : OOB;
    }
#else
    unsigned b_off[REP_N];
#if MODE == 1
    unsigned b_bad[REP_N];              /* bit 31 - t: tap t of this pixel is padding */
#endif
#pragma unroll
    for (int j = 0; j < REP_N; ++j) {
        const int n = n0 + COLUMN(j);
#if MODE == 2
        const unsigned off = (unsigned)((gi * N + n) * K + 8 * lg) * 4u;
        b_off[j] = n < N ? off : OOB;
#else
        const int nn = n < N ? n : 0, ib = nn / OHW, p = nn % OHW;
        const int h = p / CQ * CSTRH - CPADH, w = p % CQ * CSTRW - CPADW;
        b_off[j] = (unsigned)(((ib * CC + gi * (CC / CG)) * CH + h) * CW + w) * 4u;     /* of tap (0, 0), inside or not */
        unsigned cols = 0, bad = 0;     /* rows and columns of the window apart, as in igemm_f32.hip */
#pragma unroll
        for (int t = 0; t < CS; ++t) cols = cols << 1 | ((unsigned)(w + t * CDILW) < (unsigned)CW ? 0u : 1u);
#pragma unroll
        for (int t = 0; t < CR; ++t) bad = bad << CS | ((unsigned)(h + t * CDILH) < (unsigned)CH ? cols : (1u << CS) - 1u);
        bad <<= 32 - CR * CS;
        b_bad[j] = n < N ? bad : ~0u;
#endif
    }
#endif
#define SUM_CHUNKS (WAVES_K > 1 ? NW * WAVES_K * NBLK * 64 : 0)
#define TABLE_CHUNKS (TABLE / 2)
    __shared__ u32x4 smem[(SUM_CHUNKS > TABLE_CHUNKS ? SUM_CHUNKS : TABLE_CHUNKS) + 1];
#if MODE == 1
    /* k -> offset of its element from tap (0, 0) of channel 0, and its tap (k behind K: the bit that is always bad) */
    u32x2* const table = reinterpret_cast<u32x2*>(smem);
    for (int k = threadIdx.x; k < TABLE; k += NTW) {
        const int c = k / (CR * CS), t = k % (CR * CS);
        const unsigned off = (unsigned)(c * (CH * CW) + t / CS * CDILH * CW + t % CS * CDILW) * 4u;
        const u32x2 entry = {k < K ? off : 0u, k < K ? (unsigned)t : 31u};
        table[k] = entry;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < REP_N; ++j) b_bad[j] |= 1u;
#endif

    /* ---- one k step of 32: a lane holds k = 8 * lg .. 8 * lg + 7 of each of its rows and columns ---------------- */
    float ax[PD][REP_M][8], bx[PD][REP_N][8];
    auto load_row = [&](const __amdgpu_buffer_rsrc_t& rsrc, unsigned off, int k0, float (&x)[8]) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const f32x4 y = ld4(rsrc, off + 16u * v, k0 * 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[4 * v + i] = y[i];
        }
    };
    auto load = [&](int s, int set) {
        const int k0 = s * 32;
#pragma unroll
        for (int i = 0; i < REP_M; ++i) load_row(rsrc_a, a_off[i], k0, ax[set][i]);
#if MODE == 2
#pragma unroll
        for (int j = 0; j < REP_N; ++j) load_row(rsrc_b, b_off[j], k0, bx[set][j]);
#elif MODE == 0
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#if REP_N == 4
            const f32x4 y = ld4(rsrc_b, b_off + (unsigned)(i * N * 4), k0 * (N * 4));
#elif REP_N == 2
            const f32x2 y = ld2(rsrc_b, b_off + (unsigned)(i * N * 4), k0 * (N * 4));
#else
            const float y[1] = {ld1(rsrc_b, b_off + (unsigned)(i * N * 4), k0 * (N * 4))};
#endif
#pragma unroll
            for (int j = 0; j < REP_N; ++j) bx[set][j][i] = y[j];
        }
#else
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u32x2 entry = table[k0 + 8 * lg + i];
#pragma unroll
            for (int j = 0; j < REP_N; ++j) {
#if PADDED || STEPS * 32 != K || N % BN != 0
                bx[set][j][i] = ld1(rsrc_b, (b_off[j] + entry[0]) | ((b_bad[j] << entry[1]) & OOB), 0);
#else
                bx[set][j][i] = ld1(rsrc_b, b_off[j] + entry[0], 0);
#endif
            }
        }
#endif
    };
    /* what a row's loads took from behind K */
    auto cut = [&](int k0, float (&x)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = k0 + 8 * lg + i < K ? x[i] : 0.0f;
    };

    f32x4 acc[REP_M][REP_N];
#pragma unroll
    for (int i = 0; i < REP_M; ++i)
#pragma unroll
        for (int j = 0; j < REP_N; ++j) acc[i][j] = (f32x4)(0.0f);

    /* ---- main loop: PD steps are in registers or on their way to them; a set of registers is loaded anew as soon as
     * its step is done with. Behind the last step the last one is loaded once more rather than none: a load in a
     * branch would end in copies. ------------------------------------------------------------------------------- */
    const int first = kg * GSTEPS, end = first + GSTEPS < STEPS ? first + GSTEPS : STEPS;
    if (first < end) {
#pragma unroll
        for (int u = 0; u < PD; ++u) load(first + u < end ? first + u : end - 1, u);
    }
    for (int s0 = first; s0 < end; s0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            const int s = s0 + u;
            if (u > 0 && s >= end) break;
            if (K % 32 != 0 && s == STEPS - 1) {
#pragma unroll
                for (int i = 0; i < REP_M; ++i) cut(s * 32, ax[u][i]);
#if MODE == 2
#pragma unroll
                for (int j = 0; j < REP_N; ++j) cut(s * 32, bx[u][j]);
#endif
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int i = 0; i < REP_M; ++i)
#pragma unroll
                    for (int j = 0; j < REP_N; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ax[u][i][q], bx[u][j][q], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            load(s + PD < end ? s + PD : end - 1, u);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    /* the distance an MFMA's result registers need, made explicit (see igemm_f32.hip) */
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    /* ---- sum over the k groups: every group sums and stores NOUT of the tile's blocks ------------------------- */
    f32x4 out[NOUT];
#if WAVES_K > 1
    __syncthreads();                    /* the table's last readers */
    {
        f32x4* const sums = reinterpret_cast<f32x4*>(smem) + (wave % NW) * (WAVES_K * NBLK * 64);
#pragma unroll
        for (int i = 0; i < REP_M; ++i)
#pragma unroll
            for (int j = 0; j < REP_N; ++j) sums[(kg * NBLK + i * REP_N + j) * 64 + lane] = acc[i][j];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NOUT; ++b) {
            if (NBLK % WAVES_K != 0 && kg * NOUT + b >= NBLK) continue;
            out[b] = sums[(kg * NOUT + b) * 64 + lane];
#pragma unroll
            for (int g = 1; g < WAVES_K; ++g) out[b] += sums[(g * NBLK + kg * NOUT + b) * 64 + lane];
        }
    }
#else
#pragma unroll
    for (int b = 0; b < NOUT; ++b) out[b] = acc[b / REP_N][b % REP_N];
#endif

    /* ---- stores ---------------------------------------------------------------------------------------------- */
#pragma unroll
    for (int b = 0; b < NOUT; ++b) {
        if (NBLK % WAVES_K != 0 && kg * NOUT + b >= NBLK) continue;
        const int i = (kg * NOUT + b) / REP_N, j = (kg * NOUT + b) % REP_N;
        const int n = n0 + COLUMN(j);
#if MODE == 1 && !COLOUT
        float* const col = C + ((size_t)(n / OHW) * (CG * M) + (size_t)gi * M) * OHW + n % OHW;
        const size_t row = OHW;
#else
        float* const col = C + (size_t)gi * M * N + n;
        const size_t row = N;
#endif
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = m0 + i * 16 + 4 * lg + v;
            float val = out[b][v];
            if ((M % BM == 0 || m < M) & (N % BN == 0 || n < N)) {
#if HAS_BIAS
                val += bias[gi * M + m];
#endif
                col[m * row] = val;
            }
        }
    }
    CLK_END;
}

#else  /* FT_SPLIT */
/* ============ the same operators on the bf16 matrix cores: FT_SPLIT ================================================
 *
 * Numbers (2^23 times each) in three bf16 parts, six products, the sums looked at, as the second kernel of igemm_f32.hip explains them; here
 * a wavefront works alone: it multiplies REP_M x REP_N blocks of 32 x 32 over its share of K, splits what it needs itself
 * and waits for no barrier before the sum over the groups. Rows of A (and B^T) go through LDS, which is the wavefront's
 * own, because eight lanes a row load at three times the rate of four (44 and 15 bytes a clock and unit) and the loads
 * need no registers on their way; B [K][N] and gathered elements are loaded by the lane that multiplies them, whole lines
 * already. Two steps of A are in LDS or on their way, of B one.
 *
 * What bounds it: thirteen vector instructions for two numbers, 1 664 clocks a step of 64 x 64 x 32 where the MFMAs are
 * 1 536, and the operands of a 64 x 64 tile, 1 900 clocks from L2. Of GEMM 1024^3 (two wavefronts a SIMD) vector
 * instructions and MFMAs are 16.7 k and 12.3 k clocks, the whole life of a workgroup, first loads and sums included, 29.0 k:
 * they overlap by little. LDS tiles of several wavefronts (igemm_f32.hip) split and gather every element once, this kernel
 * once for each wavefront's tile, but a gathered tile of theirs waits for its slowest wavefront at every barrier: us a
 * call, best tile there and here, and the default's kernel of fp32 products, 3x3 8x256x14x14 -> 512 44.9, 32.1 and 47.0 (the
 * shipped one, with K streaming, 34.9), 1x289x63x63 -> 90 48.6, 25.4 and 32.6; but stride 2 16x128x57x57 -> 256 56.0, 74.4 and
 * 77.8.
 *
 * Up to two blocks a wavefront have accumulators of their own for the five small products; with four there are no registers
 * for them and every product rounds the sum, so K has to be divided by four or more: error against float64 of
 * 8x256x14x14 -> 512 2.5e-7, with fp32 MFMAs 4.6e-7. */
#define MODE FT_MODE
#define M FT_M
#define N FT_N
#define K FT_K
#define WAVES_M FT_WAVES_M
#define WAVES_N FT_WAVES_N
#define REP_M FT_REP_M
#define REP_N FT_REP_N
#define WAVES_K FT_WAVES_K      /* wavefront groups that divide K, summed through LDS */
#define GROUP_M FT_GROUP_M
#define XCD_REMAP FT_XCD_REMAP
#ifdef FT_HAS_BIAS
#define HAS_BIAS FT_HAS_BIAS
#else
#define HAS_BIAS 0
#endif
#ifdef FT_COLOUT
#define COLOUT FT_COLOUT
#else
#define COLOUT 0
#endif
#ifdef FT_IMAGES
#define IMAGES FT_IMAGES
#define CG FT_IMAGES
#define AGROUP(g) 0               /* one weight and bias for every image */
#else
#define IMAGES 0
#define AGROUP(g) (g)
#ifdef FT_CG
#define CG FT_CG
#else
#define CG 1
#endif
#endif

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

#define BM (WAVES_M * REP_M * 32)
#define BN (WAVES_N * REP_N * 32)
#define NW (WAVES_M * WAVES_N)          /* wavefronts of one k group */
#define NTW (NW * WAVES_K * 64)
#define TILES_M ((M + BM - 1) / BM)
#define TILES_N ((N + BN - 1) / BN)
#define STEPS ((K + 31) / 32)
#define GSTEPS ((STEPS + WAVES_K - 1) / WAVES_K)        /* k steps of a group; the last groups may have fewer */
#define NBLK (REP_M * REP_N)
#define LOW (NBLK <= 2)                 /* the small products have accumulators of their own */
#if !LOW && WAVES_K < 4
#error "one set of accumulators only where K is divided"
#endif

#define OOB 0x80000000u
#if MODE == 1
#define CB FT_CB
#define CC FT_CC
#define CH FT_CH
#define CW FT_CW
#define CR FT_CR
#define CS FT_CS
#define CSTRH FT_CSTRH
#define CSTRW FT_CSTRW
#define CPADH FT_CPADH
#define CPADW FT_CPADW
#define CDILH FT_CDILH
#define CDILW FT_CDILW
#define CP FT_CP
#define CQ FT_CQ
#define OHW (CP * CQ)
#define B_BYTES (CB * CC * CH * CW * 4)
#define PADDED (CPADH > 0 || CPADW > 0)
#if CR * CS > 31
#error "a pixel's valid taps are bits of a word"
#endif
#define TABLE_BYTES (STEPS * 256)       /* entries (byte offset, tap) of the gathered operand's k */
#else
#define TABLE_BYTES 0
#if MODE == 0
/* B ends where its rows end: rows at and behind K are beyond the buffer and read as zero */
#define B_BYTES ((gi + 1) * K * N * 4)
#else
#define B_BYTES (CG * K * N * 4)
#endif
#endif
#define A_BYTES ((IMAGES ? 1 : CG) * M * K * 4)
#if MODE == 0
#define COLUMN(j) (REP_N * li + (j))    /* column inside the wavefront's tile */
#else
#define COLUMN(j) (32 * (j) + li)
#endif

/* LDS: two buffers per wavefront of rows of 32 k; then the table */
#define ROWS (REP_M * 32 + (MODE == 2 ? REP_N * 32 : 0))
#define BUF_BYTES (ROWS * 128)
#define TILE_BYTES (NW * WAVES_K * 2 * BUF_BYTES)
#define SUM_BYTES (WAVES_K > 1 ? WAVES_K * BM * BN * 4 : 0)
#define SMEM_BYTES (TILE_BYTES + TABLE_BYTES > SUM_BYTES ? TILE_BYTES + TABLE_BYTES : SUM_BYTES)
#define B_LOADS (MODE == 2 ? 0 : MODE == 0 ? 16 : 16 * REP_N)   /* a step's loads into registers */
#if B_LOADS > 63
#error "loads in flight are counted to 63"
#endif

#ifdef FT_CLKPROBE          /* as above */
#define CLK_PARAM , unsigned long long* __restrict__ ft_clk
#if FT_CLKPROBE == 2
#define CLK_BEGIN const unsigned long long ft_r0 = wall_clock64();
#define CLK_END do { __builtin_amdgcn_s_waitcnt(0x0F70); \
        if (threadIdx.x == 0) { ft_clk[2 * blockIdx.x] = ft_r0; ft_clk[2 * blockIdx.x + 1] = wall_clock64(); } } while (0)
#else
#define CLK_BEGIN const unsigned long long ft_t0 = __builtin_readcyclecounter(), ft_r0 = wall_clock64();
#define CLK_END do { __builtin_amdgcn_s_waitcnt(0x0F70); \
        if (threadIdx.x == 0) { ft_clk[2 * blockIdx.x] = __builtin_readcyclecounter() - ft_t0; \
                                ft_clk[2 * blockIdx.x + 1] = wall_clock64() - ft_r0; } } while (0)
#endif
#else
#define CLK_PARAM
#define CLK_BEGIN
#define CLK_END do { } while (0)
#endif

static __device__ __forceinline__ float ld1(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)vo, so, 0));
}
static __device__ __forceinline__ f32x2 ld2(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)vo, so, 0));
}
static __device__ __forceinline__ f32x4 ld4(__amdgpu_buffer_rsrc_t r, unsigned vo, int so) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)vo, so, 0));
}
struct parts { static constexpr bool exact = false; };
struct whole { static constexpr bool exact = true; };

extern "C" __global__ __launch_bounds__(NTW, 2)         /* two wavefronts a SIMD */
void igemm_f32(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C
#if HAS_BIAS
               , const float* __restrict__ bias
#endif
               CLK_PARAM)
{
    CLK_BEGIN
    __shared__ __attribute__((aligned(128))) unsigned char smem[SMEM_BYTES];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int kg = wave / NW, wm = wave % NW / WAVES_N, wn = wave % WAVES_N;
    const int li = lane & 31, lg = lane >> 5;

    int bid = blockIdx.x;
    if (XCD_REMAP) {                    /* neighbouring tiles share an XCD; the first count % 8 XCDs have one more */
        const int count = TILES_M * TILES_N * CG;
        bid = (bid % 8) * (count / 8) + (bid % 8 < count % 8 ? bid % 8 : count % 8) + bid / 8;
    }
    const int gi = bid / (TILES_M * TILES_N);
    int m0, n0;                         /* of the wavefront's tile */
    {
        const int r = bid % (TILES_M * TILES_N);
        const int first_m = r / (GROUP_M * TILES_N) * GROUP_M;
        const int gsz = (TILES_M - first_m) < GROUP_M ? (TILES_M - first_m) : GROUP_M;
        const int rr = r % (GROUP_M * TILES_N);
        m0 = (first_m + rr % gsz) * BM + wm * REP_M * 32;
        n0 = (rr / gsz) * BN + wn * REP_N * 32;
    }
    /* The wait for rows in LDS counts the loads behind them, so none may go missing (see load_b as well): where one tile
     * holds all columns the compiler would know blocks that lie behind the last, make one load of two that both miss the
     * buffer and drop those nothing is stored from (5 columns in three blocks: 32 loads a step instead of 48, and products
     * of what the LDS held before the rows arrived). */
    asm volatile("" : "+s"(n0));

    auto descriptor = [](const float* base, unsigned bytes) {
        const unsigned long long p = (unsigned long long)base;
        i32x4 d;                             /* raw buffer: base, stride 0, bytes, untyped dwords */
        d[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)p);
        d[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(p >> 32) & 0xffffu));
        d[2] = (int)bytes;
        d[3] = 0x00020000;
        return d;
    };
    const i32x4 desc_a = descriptor(A, (unsigned)A_BYTES);
#if MODE == 2
    const i32x4 desc_b = descriptor(B, (unsigned)B_BYTES);
#else
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, B_BYTES, 0x00020000);
#endif
    /* ---- rows of 32 k that go through LDS: eight lanes a row, eight rows an instruction. Row r's vector v lies at
     * v ^ (r >> 1 & 7), for which the fragments' reads are free of bank conflicts ------------------------------ */
    unsigned char* const lds = smem + wave * (2 * BUF_BYTES);
    unsigned row_off[ROWS / 8];
#pragma unroll
    for (int e = 0; e < ROWS / 8; ++e) {
        const int r = 8 * e + lane / 8, v = (lane & 7) ^ (r >> 1 & 7);
        if (e < REP_M * 4) {
            const int m = m0 + r;
            const unsigned off = (unsigned)((AGROUP(gi) * M + m) * K + 4 * v) * 4u;
            row_off[e] = m < M ? off : OOB;
        } else {
            const int n = n0 + r - REP_M * 32;
            const unsigned off = (unsigned)((gi * N + n) * K + 4 * v) * 4u;
            row_off[e] = n < N ? off : OOB;
        }
    }
    const unsigned lds_at = __builtin_amdgcn_readfirstlane((int)(unsigned)(__UINTPTR_TYPE__)(lds_void*)lds);
    auto load_rows = [&](int s, int buf) {
#pragma unroll
        for (int e = 0; e < ROWS / 8; ++e) {
#if MODE == 2
            const i32x4 d = e < REP_M * 4 ? desc_a : desc_b;
#else
            const i32x4 d = desc_a;
#endif
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(lds_at + buf * BUF_BYTES + e * 1024), "v"(row_off[e]), "s"(d), "s"(s * 128) : "memory", "m0");
        }
    };
    /* eight k of row block i (behind A's: columns of B^T) */
    auto read_row = [&](int buf, int i, int t, float (&x)[8]) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const f32x4 y = *reinterpret_cast<const f32x4*>(lds + buf * BUF_BYTES + (32 * i + li) * 128
                                                            + ((4 * t + 2 * lg + v) ^ (li >> 1 & 7)) * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q) x[4 * v + q] = y[q];
        }
    };
    auto cut = [&](int s, int t, float (&x)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = s * 32 + 16 * t + 8 * lg + i < K ? x[i] : 0.0f;
    };

#if MODE == 0
    unsigned b_off;
    {
        const int n = n0 + COLUMN(0);   /* columns behind N belong to the next row and feed results that are not stored */
        const unsigned off = (unsigned)((gi * K + 8 * lg) * N + n) * 4u;
        b_off = n < N ? off : OOB;
    }
#elif MODE == 1
    unsigned b_off[REP_N], b_bad[REP_N];
#pragma unroll
    for (int j = 0; j < REP_N; ++j) {
        const int n = n0 + COLUMN(j);
        const int nn = n < N ? n : 0, ib = nn / OHW, p = nn % OHW;
        const int h = p / CQ * CSTRH - CPADH, w = p % CQ * CSTRW - CPADW;
        b_off[j] = (unsigned)(((ib * CC + gi * (CC / CG)) * CH + h) * CW + w) * 4u;     /* of tap (0, 0), inside or not */
        unsigned cols = 0, bad = 0;
#pragma unroll
        for (int t = 0; t < CS; ++t) cols = cols << 1 | ((unsigned)(w + t * CDILW) < (unsigned)CW ? 0u : 1u);
#pragma unroll
        for (int t = 0; t < CR; ++t) bad = bad << CS | ((unsigned)(h + t * CDILH) < (unsigned)CH ? cols : (1u << CS) - 1u);
        bad = bad << (32 - CR * CS) | 1u;
        b_bad[j] = n < N ? bad : ~0u;
    }
    u32x2* const table = reinterpret_cast<u32x2*>(smem + TILE_BYTES);
    for (int k = threadIdx.x; k < STEPS * 32; k += NTW) {
        const int c = k / (CR * CS), t = k % (CR * CS);
        const unsigned off = (unsigned)(c * (CH * CW) + t / CS * CDILH * CW + t % CS * CDILW) * 4u;
        const u32x2 entry = {k < K ? off : 0u, k < K ? (unsigned)t : 31u};
        table[k] = entry;
    }
    __syncthreads();
#endif

    float bx[2][REP_N][8];
    auto load_b = [&](int s, int t) {
        const int k0 = s * 32;
#if MODE == 0
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#if K % 32 == 0
            unsigned vo = b_off;
            const int so = (k0 + 16 * t + i) * (N * 4);
#else
            unsigned vo = b_off + (unsigned)((16 * t + i) * N * 4);
            const int so = k0 * (N * 4);
#endif
            /* as many columns as a load takes: the loads of two rows are neighbours, which the compiler would make one */
            if (N == REP_N) asm volatile("" : "+v"(vo));
#if REP_N == 4
            const f32x4 y = ld4(rsrc_b, vo, so);
#elif REP_N == 2
            const f32x2 y = ld2(rsrc_b, vo, so);
#else
            const float y[1] = {ld1(rsrc_b, vo, so)};
#endif
#pragma unroll
            for (int j = 0; j < REP_N; ++j) bx[t][j][i] = y[j];
        }
#elif MODE == 1
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u32x2 entry = table[k0 + 16 * t + 8 * lg + i];
#pragma unroll
            for (int j = 0; j < REP_N; ++j) {
#if PADDED || STEPS * 32 != K || N % BN != 0
                bx[t][j][i] = ld1(rsrc_b, (b_off[j] + entry[0]) | ((b_bad[j] << entry[1]) & OOB), 0);
#else
                bx[t][j][i] = ld1(rsrc_b, b_off[j] + entry[0], 0);
#endif
            }
        }
#endif
    };

    auto split = [&](const float (&x)[8], bf16x8 (&p)[3]) {         /* of 2^23 x */
        u32x4 q[3];
        float y[8];
#pragma unroll
        for (int h = 0; h < 8; ++h) y[h] = x[h] * 0x1p23f;
#pragma unroll
        for (int part = 0; part < 3; ++part) {
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const f32x2 t = {y[2 * h], y[2 * h + 1]};
                const bf16x2 r = __builtin_convertvector(t, bf16x2);
                q[part][h] = __builtin_bit_cast(unsigned, r);
                if (part < 2) {
                    y[2 * h] -= __builtin_bit_cast(float, q[part][h] << 16);
                    y[2 * h + 1] -= __builtin_bit_cast(float, q[part][h] & 0xffff0000u);
                }
            }
        }
#pragma unroll
        for (int part = 0; part < 3; ++part) p[part] = __builtin_bit_cast(bf16x8, q[part]);
    };

    f32x16 acc[REP_M][REP_N];
#if LOW
    f32x16 low[REP_M][REP_N];
#else
    auto& low = acc;
#endif
    const int first = kg * GSTEPS, end = first + GSTEPS < STEPS ? first + GSTEPS : STEPS;
    auto run = [&](auto how) {
#pragma unroll
        for (int i = 0; i < REP_M; ++i)
#pragma unroll
            for (int j = 0; j < REP_N; ++j) acc[i][j] = low[i][j] = (f32x16)(0.0f);
        if (first >= end) return;
        load_b(first, 0);
        load_rows(first, 0);
        load_b(first, 1);
        for (int s = first; s < end; ++s) {
            const int buf = (s - first) & 1, next = s + 1 < end ? s + 1 : s;
            /* this step's rows are in LDS when only loads behind them are left: the second half of B's */
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x0F70 | (B_LOADS / 2 & 15) | ((B_LOADS / 2 >> 4) << 14));
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                float ax[REP_M][8];
#pragma unroll
                for (int i = 0; i < REP_M; ++i) read_row(buf, i, t, ax[i]);
#if MODE == 2
#pragma unroll
                for (int j = 0; j < REP_N; ++j) read_row(buf, REP_M + j, t, bx[t][j]);
#endif
                if (K % 32 != 0 && s == STEPS - 1) {
#pragma unroll
                    for (int i = 0; i < REP_M; ++i) cut(s, t, ax[i]);
#if MODE == 2
#pragma unroll
                    for (int j = 0; j < REP_N; ++j) cut(s, t, bx[t][j]);
#endif
                }
                if constexpr (decltype(how)::exact) {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
#pragma unroll
                        for (int i = 0; i < REP_M; ++i)
#pragma unroll
                            for (int j = 0; j < REP_N; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(ax[i][q], bx[t][j][q], acc[i][j], 0, 0, 0);
                    if (t == 1) load_rows(next, buf ^ 1);
                    load_b(next, t);
                } else {
                    bf16x8 a[REP_M][3], b[REP_N][3];
#pragma unroll
                    for (int j = 0; j < REP_N; ++j) split(bx[t][j], b[j]);
                    if (t == 1) load_rows(next, buf ^ 1);
                    load_b(next, t);
#pragma unroll
                    for (int i = 0; i < REP_M; ++i) split(ax[i], a[i]);
                    const int pa[5] = {2, 0, 1, 1, 0}, pb[5] = {0, 2, 1, 0, 1};
#pragma unroll
                    for (int q = 0; q < 5; ++q)
#pragma unroll
                        for (int i = 0; i < REP_M; ++i)
#pragma unroll
                            for (int j = 0; j < REP_N; ++j)
                                low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][pa[q]], b[j][pb[q]], low[i][j], 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < REP_M; ++i)
#pragma unroll
                        for (int j = 0; j < REP_N; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][0], b[j][0], acc[i][j], 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);         /* rows behind the last step's: the LDS is for the sums now */
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    run(parts());
    {
        float nan = 0.0f;
#pragma unroll
        for (int i = 0; i < REP_M; ++i)
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
#if LOW
                    acc[i][j][v] += low[i][j][v];
#endif
                    acc[i][j][v] *= 0x1p-46f;
                    nan = __builtin_fmaf(acc[i][j][v], 0.0f, nan);
                }
        if (__any(!(nan == 0.0f))) run(whole());
    }

    /* ---- sum over the k groups and stores: a group takes every WAVES_K-th set of four rows a lane ------------- */
#define UNITS (REP_M * 4)
#define SHARE ((UNITS + WAVES_K - 1) / WAVES_K)
#if WAVES_K > 1
    f32x4* const sums = reinterpret_cast<f32x4*>(smem) + (wave % NW) * (WAVES_K * NBLK * 256) + lane;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int j = 0; j < REP_N; ++j) {
            const f32x16& x = acc[u / 4][j];
            const f32x4 y = {x[u % 4 * 4], x[u % 4 * 4 + 1], x[u % 4 * 4 + 2], x[u % 4 * 4 + 3]};
            sums[((kg * UNITS + u) * REP_N + j) * 64] = y;
        }
    __syncthreads();
#endif
#pragma unroll
    for (int b = 0; b < SHARE; ++b) {
        f32x4 out[REP_N];
#if WAVES_K > 1
        const int u = kg + b * WAVES_K;
        if (UNITS % WAVES_K != 0 && u >= UNITS) continue;
#pragma unroll
        for (int j = 0; j < REP_N; ++j) {
            out[j] = sums[(u * REP_N + j) * 64];
#pragma unroll
            for (int g = 1; g < WAVES_K; ++g) out[j] += sums[((g * UNITS + u) * REP_N + j) * 64];
        }
#else
        const int u = b;
#pragma unroll
        for (int j = 0; j < REP_N; ++j) {
            const f32x16& x = acc[u / 4][j];
            const f32x4 y = {x[u % 4 * 4], x[u % 4 * 4 + 1], x[u % 4 * 4 + 2], x[u % 4 * 4 + 3]};
            out[j] = y;
        }
#endif
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = m0 + u / 4 * 32 + u % 4 * 8 + 4 * lg + v;
            if (M % BM != 0 && m >= M) continue;
#if HAS_BIAS
#pragma unroll
            for (int j = 0; j < REP_N; ++j) out[j][v] += bias[AGROUP(gi) * M + m];
#endif
#if MODE == 0 && REP_N > 1
            const int n = n0 + COLUMN(0);
            float* const dst = C + (size_t)(gi * M + m) * N + n;
            if (N % BN == 0 || n + REP_N <= N) {
#if REP_N == 2
                const f32x2u y = {out[0][v], out[1][v]};
                *reinterpret_cast<f32x2u*>(dst) = y;
#else
                const f32x4u y = {out[0][v], out[1][v], out[2][v], out[3][v]};
                *reinterpret_cast<f32x4u*>(dst) = y;
#endif
            } else {
#pragma unroll
                for (int j = 0; j < REP_N; ++j)
                    if (n + j < N) dst[j] = out[j][v];
            }
#else
#pragma unroll
            for (int j = 0; j < REP_N; ++j) {
                const int n = n0 + COLUMN(j);
                if (N % BN != 0 && n >= N) continue;
#if MODE == 1 && !COLOUT
                C[((size_t)(n / OHW) * (CG * M) + (size_t)gi * M + m) * OHW + n % OHW] = out[j][v];
#else
                C[(size_t)(gi * M + m) * N + n] = out[j][v];
#endif
            }
#endif
        }
    }
    CLK_END;
}
#endif  /* FT_SPLIT */
