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
