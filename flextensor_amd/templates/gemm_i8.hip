// int8 x int8 -> int32 GEMM kernel template for gfx950 (CDNA4), hiprtc-compiled.
//
//   C[M][N] = sum_k int32(A[m][k]) * int32(B[n][k])
//
// A is [M][K] and B is [N][K], both K-contiguous ("B in K-major layout"), C is
// row-major int32 — the compute of
// flextensor/test/test_tvm/legacy/gemm_int8.py:15-21.
//
// Knobs (-D constants set by the scheduler from a Config):
//   MFMA        32 -> v_mfma_i32_32x32x32_i8, 16 -> v_mfma_i32_16x16x64_i8
//   WAVES_M/N   wavefronts per workgroup along M / N
//   REP_M/N     MFMA tiles per wavefront along M / N
//   BK          bytes of K per LDS tile (multiple of the MFMA K)
//   STAGES      1 or 2 LDS buffers, with DTL 1 also 3
//   PD          prefetch distance: global loads of tile t+PD are in flight
//               (in PD register sets) while tile t is multiplied
//   FRAGPF      1: fragment-prefetch pipeline. Tile t+1 is written to LDS at
//               the *start* of iteration t (its global loads were issued one
//               iteration earlier), the operand fragments of the next k-step
//               are read from LDS while the MFMAs of the current one run, and
//               the first fragments of tile t+1 are read right after the one
//               barrier of the iteration, so that the matrix cores have work
//               immediately after every barrier (needs STAGES 2, PD 1)
//   GROUP_M     tile-traversal group height (L2 locality)
//   XCD_REMAP   1: consecutive logical tiles stay on one XCD
//   PAD         LDS row padding in bytes (multiple of 16); -1 selects
//               unpadded rows whose 16-byte chunks are XOR-swizzled by row
//   DTL         1: tiles travel global -> LDS directly (buffer loads with the
//               lds modifier, 16 bytes per lane): no staging registers, no
//               LDS store instructions; the row swizzle is applied on the
//               global side, since a wavefront's 64 chunks land contiguously.
//               With three buffers two tiles are under way while one is
//               multiplied, and a step waits for loads that are two steps old.
//               What bounds a long K on few tiles is that wait: a strip of K is
//               new to the XCD's L2 in every step, so a step with one tile ahead
//               lasts as long as a load from behind it (64x64 tiles: 430 ns a
//               step of 128 with two buffers, 260 with three; 207 tiles at
//               K = 1900 7.8 -> 5.6 us)
//               DTL 3: the same data path with the instruction order of the
//               main loop written out and pinned: the LDS fragment reads of
//               the next k-step and the direct-to-LDS loads of the tile after
//               next are issued one at a time between the MFMAs of the current
//               k-step, and the one barrier of a tile sits a quarter into its
//               last k-step, so that the matrix cores always have queued work
//               (left to itself the compiler issues the fragment reads right
//               before their first use and waits for them)
//   NT_STORE    1: non-temporal stores for C
//   EARLYST     1 (with DTL 2 and two k-steps per tile): the last tile is multiplied
//               block by block instead of k-step by k-step, and every accumulator
//               block is stored as soon as its last MFMA has been issued and the
//               next group's MFMAs cover the distance to the read: the stores of C
//               start a tile's time before the workgroup's last MFMA instead of
//               behind it
//   SPLITK      grid-level split of K: SPLITK workgroups per tile, each over a
//               contiguous range of K; the partial sums meet in C (zero-filled by a
//               kernel in front) through integer atomic adds, which are exact and
//               order-independent, so the result stays bit-exact and repeatable
//   WAVES_K     split of K inside the workgroup: WAVES_K groups of WAVES_M x WAVES_N
//               wavefronts, each with its own LDS tiles and its own range of K; the
//               groups' accumulators are summed through LDS and group 0 stores
//   CVEC        1: the MFMA operands are swapped (the core computes the
//               transposed tile), so a lane holds four consecutive columns of
//               one row of C and writes them with one 128-bit store
//
// Both operands live in LDS as [rows][BK+PAD] bytes and are read as one
// 128-bit load per lane per MFMA: lane (i, g) takes the 16 bytes at
// k = kstep + 16*g of row i, identically for A and B, so whatever order the
// matrix core assigns to those 16 values inside its K dimension, A and B
// agree and the integer sum is exact.

/* Constants arrive as -DFT_<NAME>=value: single-letter macros on the command line
 * would be visible to (and break) the runtime-compilation built-in headers. */
#define M FT_M
#define N FT_N
#define K FT_K
#define KP FT_KP
#define MFMA FT_MFMA
#define WAVES_M FT_WAVES_M
#define WAVES_N FT_WAVES_N
#define REP_M FT_REP_M
#define REP_N FT_REP_N
#define BK FT_BK
#define STAGES FT_STAGES
#define PD FT_PD
#define FRAGPF FT_FRAGPF
#define GROUP_M FT_GROUP_M
#define XCD_REMAP FT_XCD_REMAP
#define PAD FT_PAD
#define NT_STORE FT_NT_STORE
#ifdef FT_DTL
#define DTL FT_DTL
#else
#define DTL 0
#endif
#ifdef FT_CVEC
#define CVEC FT_CVEC
#else
#define CVEC 0
#endif
#ifdef FT_EARLYST
#define EARLYST FT_EARLYST
#else
#define EARLYST 0
#endif
#ifdef FT_SPLITK
#define SPLITK FT_SPLITK
#else
#define SPLITK 1
#endif
#ifdef FT_WAVES_K
#define WAVES_K FT_WAVES_K
#else
#define WAVES_K 1
#endif

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

#if MFMA == 32
typedef i32x16 acc_t;
#define NACC 16
#define MFMA_K 32
#define MFMA_RAW(a, b, c) __builtin_amdgcn_mfma_i32_32x32x32_i8((a), (b), (c), 0, 0, 0)
#elif MFMA == 16
typedef i32x4 acc_t;
#define NACC 4
#define MFMA_K 64
#define MFMA_RAW(a, b, c) __builtin_amdgcn_mfma_i32_16x16x64_i8((a), (b), (c), 0, 0, 0)
#else
#error "MFMA must be 16 or 32"
#endif
#if CVEC
#define MFMA_OP(a, b, c) MFMA_RAW((b), (a), (c))   /* rows of the result follow B's rows (n) */
#else
#define MFMA_OP(a, b, c) MFMA_RAW((a), (b), (c))
#endif

#define BM (WAVES_M * REP_M * MFMA)
#define BN (WAVES_N * REP_N * MFMA)
#define NT (WAVES_M * WAVES_N * 64)      /* threads of one k-group */
#define NTW (NT * WAVES_K)               /* threads of the workgroup */
#define CRW (BK / 16)             /* 16-byte chunks per LDS row */
#if PAD < 0
#define SROW (BK)                 /* LDS row stride in bytes */
#if CRW >= 16
#define SWZ(row) ((row) & 15)
#else
#define SWZ(row) (((row) / (16 / CRW)) & (CRW - 1))
#endif
#else
#define SROW (BK + PAD)
#define SWZ(row) 0
#endif
/* byte column c (multiple of 16) of `row` -> physical byte column */
#define PCOL(row, c) (((((c) >> 4) ^ SWZ(row)) << 4))
#define OOB 0x80000000u
#define TILES_M ((M + BM - 1) / BM)
#define TILES_N ((N + BN - 1) / BN)
/* KP = SPLITK * WAVES_K * (K tiles of a group) * BK, which covers K; chunks
 * beyond K are zero-filled by the load predicate. When K is no multiple of 16
 * the rows of A and B are not 16-byte aligned: a buffer load of 16 bytes needs
 * dword alignment only, which is enough for K % 4 == 0; otherwise a chunk is cut
 * out of the five dwords it lies in (one 128-bit and one 32-bit load, four
 * byte-aligning shifts). The last chunk of a row is partly beyond it (those
 * bytes are the next row's): they are zeroed in A on the way into LDS, or, with three
 * direct-to-LDS buffers (K % 4 == 0), in the fragments of the last tile: 3269x1388x381 7.17 ->
 * 6.17 us, 408x552x3249 5.16 -> 4.64 against register staging. Rows that begin inside a dword stay
 * register-staged: with the fragments cut out of five dwords behind LDS, 1000x1531x777 was 7.08
 * us against 6.24 (every fragment reads LDS twice, and a row's last dword is a load of its own). */
#define KT (KP / BK / (SPLITK * WAVES_K))      /* tiles of one k-group (host checks divisibility) */
/* K offset of a tile that goes into the scalar offset of its loads. The range check of a buffer load compares
 * the lane's offset with (bytes - scalar offset): a scalar offset beyond the buffer would wrap that difference
 * and let every lane pass. A tile wholly behind K (its lanes are all out of range) therefore takes 0. */
#if KP - K >= BK
#define K_AT(k0) ((k0) < K ? (k0) : 0)
#else
#define K_AT(k0) (k0)
#endif
#if EARLYST && (SPLITK > 1 || WAVES_K > 1)
#error "early stores write finished sums: no K division"
#endif

#if BK % MFMA_K != 0
#error "BK must be a multiple of the MFMA K extent"
#endif
#if PAD >= 0 && PAD % 16 != 0
#error "PAD must be a multiple of 16 bytes"
#endif

#define CHUNKS_ROW (BK / 16)
#define A_CHUNKS (BM * CHUNKS_ROW)
#define B_CHUNKS (BN * CHUNKS_ROW)
#define EA ((A_CHUNKS + NT - 1) / NT)
#define EB ((B_CHUNKS + NT - 1) / NT)
#if DTL
#if PAD > 0 || STAGES < 2 || (STAGES > 2 && DTL != 1) || A_CHUNKS % NT != 0 || B_CHUNKS % NT != 0 || (K % 16 != 0 && (STAGES == 2 || K % 4 != 0))
#error "direct-to-LDS tiles need unpadded rows, two buffers and K % 16 == 0 or three and K % 4 == 0, and whole rounds of chunks"
#endif
#if DTL == 3 && ((BK / MFMA_K) % 2 != 0 || REP_M * REP_N / 4 + REP_M + REP_N > REP_M * REP_N || REP_M * REP_N / 4 + EA + EB > REP_M * REP_N)
#error "the pinned schedule needs an even number of k-steps per tile and enough MFMAs per k-step to interleave with"
#endif
typedef __attribute__((address_space(3))) void lds_void;
#endif

/* FT_CLKPROBE: an instrumented build that measures the shader clock the kernel runs at. Every
 * workgroup writes, through one more argument, how many shader clocks (s_memtime) and how many ticks
 * of the constant 100 MHz counter (s_memrealtime) passed between its first instruction and the
 * completion of its first wavefront's last store. */
#ifdef FT_CLKPROBE
#define CLK_PARAM , unsigned long long* __restrict__ ft_clk
#if FT_CLKPROBE == 2
/* the two stamps of the 100 MHz counter themselves (it is common to the device): when the workgroup began and
 * when its first wavefront's stores had completed, to lay the workgroups of consecutive launches on one time axis */
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

#define A_TILE_BYTES (BM * SROW)
#define B_TILE_BYTES (BN * SROW)
#define TILE_BYTES (WAVES_K * STAGES * (A_TILE_BYTES + B_TILE_BYTES))
#define RED_BYTES ((WAVES_K - 1) * NT * REP_M * REP_N * NACC * 4)
#define SMEM_BYTES (TILE_BYTES > RED_BYTES ? TILE_BYTES : RED_BYTES)

extern "C" __global__ __launch_bounds__(NTW)
void gemm_i8(const signed char* __restrict__ A, const signed char* __restrict__ B,
             int* __restrict__ C CLK_PARAM)
{
    CLK_BEGIN
#if WAVES_K > 1
    /* every k-group has its own tiles; the memory is reused for the sum of the groups */
    __shared__ __attribute__((aligned(16))) signed char smem[SMEM_BYTES];
    const int kg = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / NT));
    const int tid = threadIdx.x - kg * NT;          /* thread index inside the k-group */
    signed char (*As)[A_TILE_BYTES] = reinterpret_cast<signed char (*)[A_TILE_BYTES]>(smem + kg * STAGES * A_TILE_BYTES);
    signed char (*Bs)[B_TILE_BYTES] = reinterpret_cast<signed char (*)[B_TILE_BYTES]>(
        smem + WAVES_K * STAGES * A_TILE_BYTES + kg * STAGES * B_TILE_BYTES);
#else
    __shared__ __attribute__((aligned(16))) signed char As[STAGES][BM * SROW];
    __shared__ __attribute__((aligned(16))) signed char Bs[STAGES][BN * SROW];
    const int kg = 0;
    const int tid = threadIdx.x;
#endif
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WAVES_N;
    const int wn = wave % WAVES_N;
    const int li = lane % MFMA;
    const int lg = lane / MFMA;

    const int nblk = TILES_M * TILES_N * SPLITK;
    int bid = blockIdx.x;
#if XCD_REMAP
    /* as in igemm_f32.hip: 2752x1120x80, 172 tiles, 4.43 -> 3.77 us for renumbering counts that 8 does not divide too */
    bid = (bid % 8) * (nblk / 8) + (nblk % 8 == 0 ? 0 : bid % 8 < nblk % 8 ? bid % 8 : nblk % 8) + bid / 8;
#endif
#if SPLITK > 1
    const int kz = bid / (TILES_M * TILES_N);       /* which part of K */
    bid = bid % (TILES_M * TILES_N);
#else
    const int kz = 0;
#endif
    const int kbase = (kz * WAVES_K + kg) * (KT * BK);     /* first k of this group's range */
    const int grp = bid / (GROUP_M * TILES_N);
    const int first_m = grp * GROUP_M;
    const int gsz = (TILES_M - first_m) < GROUP_M ? (TILES_M - first_m) : GROUP_M;
    const int rr = bid % (GROUP_M * TILES_N);
    const int tile_m = first_m + rr % gsz;
    const int tile_n = rr / gsz;
    const int m0 = tile_m * BM;
    const int n0 = tile_n * BN;

    int a_row[EA], a_col[EA], b_row[EB], b_col[EB];
#pragma unroll
    for (int e = 0; e < EA; ++e) {
        const int q = tid + e * NT;
        a_row[e] = q / CHUNKS_ROW;
#if DTL
        /* chunk q lands at byte 16*q of the tile = physical chunk q % CHUNKS_ROW
         * of its row: fetch the logical chunk that belongs there */
        a_col[e] = ((q % CHUNKS_ROW) ^ SWZ(a_row[e])) * 16;
#else
        a_col[e] = (q % CHUNKS_ROW) * 16;
#endif
    }
#pragma unroll
    for (int e = 0; e < EB; ++e) {
        const int q = tid + e * NT;
        b_row[e] = q / CHUNKS_ROW;
#if DTL
        b_col[e] = ((q % CHUNKS_ROW) ^ SWZ(b_row[e])) * 16;
#else
        b_col[e] = (q % CHUNKS_ROW) * 16;
#endif
    }

    /* raw buffer loads: an element that must read as zero (edge tile, idle
     * lane, K tail) gets an offset beyond the buffer and loads 0 */
#if K % 4 == 0
#define SHIFTED(p) (p)
#define A_SPAN (M * K)
#define B_SPAN (N * K)
#else
    /* Rows begin at any byte. The descriptors start at the dword the operand begins in, a chunk is
     * loaded from the dword its first byte lies in, and the byte inside that dword (the same for every
     * k tile, BK being a multiple of 4) becomes the shift. The spans are whole dwords: the last
     * one may hold bytes behind the operand, which share its page and are never used. */
#define SHIFTED(p) (const_cast<signed char*>(p) - ((unsigned long long)(p) & 3))
#define A_SPAN ((int)(((unsigned)(M * K) + (unsigned)a_lsb + 3u) & ~3u))
#define B_SPAN ((int)(((unsigned)(N * K) + (unsigned)b_lsb + 3u) & ~3u))
    const int a_lsb = __builtin_amdgcn_readfirstlane((int)((unsigned long long)A & 3));
    const int b_lsb = __builtin_amdgcn_readfirstlane((int)((unsigned long long)B & 3));
#endif
    const __amdgpu_buffer_rsrc_t rsrc_a =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<signed char*>(SHIFTED(A)), 0, A_SPAN, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<signed char*>(SHIFTED(B)), 0, B_SPAN, 0x00020000);
    unsigned a_voff[EA], b_voff[EB];
#if K % 4 == 0
#define A_SHIFT(e) 0
#define B_SHIFT(e) 0
#else
    int a_sh[EA], b_sh[EB];
#define A_SHIFT(e) a_sh[e]
#define B_SHIFT(e) b_sh[e]
#endif
#pragma unroll
    for (int e = 0; e < EA; ++e) {
        const int m = m0 + a_row[e];
        bool ok = (A_CHUNKS % NT == 0) || (tid + e * NT < A_CHUNKS);
        if (M % BM != 0) ok = ok && (m < M);
#if K % 4 == 0
        const unsigned off = (unsigned)(m * K + a_col[e]);
#else
        const unsigned byte = (unsigned)(m * K + a_col[e] + a_lsb), off = byte & ~3u;
        a_sh[e] = (int)(byte & 3u);
#endif
        a_voff[e] = ok ? off : OOB;
    }
#pragma unroll
    for (int e = 0; e < EB; ++e) {
        const int n = n0 + b_row[e];
        bool ok = (B_CHUNKS % NT == 0) || (tid + e * NT < B_CHUNKS);
        if (N % BN != 0) ok = ok && (n < N);
#if K % 4 == 0
        const unsigned off = (unsigned)(n * K + b_col[e]);
#else
        const unsigned byte = (unsigned)(n * K + b_col[e] + b_lsb), off = byte & ~3u;
        b_sh[e] = (int)(byte & 3u);
#endif
        b_voff[e] = ok ? off : OOB;
    }

    /* what a lane holds of a chunk between its load and its store to LDS */
#if K % 4 == 0
    typedef i32x4 chunk_t;
#else
    struct chunk_t { i32x4 lo; int hi; };     /* the five dwords its 16 bytes lie in */
#endif
    chunk_t areg[PD][EA], breg[PD][EB];

    auto load_chunk = [&](__amdgpu_buffer_rsrc_t rsrc, unsigned vo, int k0) -> chunk_t {
        const i32x4 lo = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)vo, K_AT(k0), 0));
#if K % 4 == 0
        return lo;
#else
        return {lo, (int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(vo + 16u), K_AT(k0), 0)};
#endif
    };
    /* the chunk's 16 bytes; sh = byte the chunk begins at inside its first dword */
    auto chunk_bytes = [&](const chunk_t& c, int sh) -> i32x4 {
#if K % 4 == 0
        (void)sh;
        return c;
#else
        i32x4 v;
        v[0] = (int)__builtin_amdgcn_alignbyte((unsigned)c.lo[1], (unsigned)c.lo[0], (unsigned)sh);
        v[1] = (int)__builtin_amdgcn_alignbyte((unsigned)c.lo[2], (unsigned)c.lo[1], (unsigned)sh);
        v[2] = (int)__builtin_amdgcn_alignbyte((unsigned)c.lo[3], (unsigned)c.lo[2], (unsigned)sh);
        v[3] = (int)__builtin_amdgcn_alignbyte((unsigned)c.hi, (unsigned)c.lo[3], (unsigned)sh);
        return v;
#endif
    };

    auto load_global = [&](int kt, int set) {
        const int k0 = kbase + kt * BK;
#pragma unroll
        for (int e = 0; e < EA; ++e) {
            unsigned vo = a_voff[e];
            if (KP != K) vo = (k0 + a_col[e] < K) ? vo : OOB;
            areg[set][e] = load_chunk(rsrc_a, vo, k0);
        }
#pragma unroll
        for (int e = 0; e < EB; ++e) {
            unsigned vo = b_voff[e];
            if (KP != K) vo = (k0 + b_col[e] < K) ? vo : OOB;
            breg[set][e] = load_chunk(rsrc_b, vo, k0);
        }
    };

    /* tile kt, which register set `set` holds, to LDS buffer buf */
    auto store_lds = [&](int kt, int buf, int set) {
        const int k0 = kbase + kt * BK;
#pragma unroll
        for (int e = 0; e < EA; ++e)
            if ((A_CHUNKS % NT == 0) || (tid + e * NT < A_CHUNKS)) {
                i32x4 v = chunk_bytes(areg[set][e], A_SHIFT(e));
#if K % 16 != 0
                /* the last chunk of a row runs into the next row: those bytes of A become zeros, and
                 * whatever B holds there does not count */
                if (k0 + BK > K) {
                    const int valid = K - k0 - a_col[e];         /* bytes of the chunk inside the row */
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int nb = valid - 4 * d;
                        v[d] = nb >= 4 ? v[d] : (nb <= 0 ? 0 : v[d] & ((1 << (8 * nb)) - 1));
                    }
                }
#endif
                *reinterpret_cast<i32x4*>(&As[buf][a_row[e] * SROW + PCOL(a_row[e], a_col[e])]) = v;
            }
#pragma unroll
        for (int e = 0; e < EB; ++e)
            if ((B_CHUNKS % NT == 0) || (tid + e * NT < B_CHUNKS))
                *reinterpret_cast<i32x4*>(&Bs[buf][b_row[e] * SROW + PCOL(b_row[e], b_col[e])]) =
                    chunk_bytes(breg[set][e], B_SHIFT(e));
    };

    acc_t acc[REP_M][REP_N];
#pragma unroll
    for (int i = 0; i < REP_M; ++i)
#pragma unroll
        for (int j = 0; j < REP_N; ++j)
            acc[i][j] = (acc_t)(0);

    /* accumulator block (i, j) -> C */
    auto store_block = [&](int i, int j) {
#if CVEC
        /* swapped operands: lane (li, lg) holds C[m = li][n = 4*lg + 0..3] (16x16),
         * or C[m = li][n = 8*q + 4*lg + 0..3] in registers 4q..4q+3 (32x32) */
        const int m = m0 + (wm * REP_M + i) * MFMA + li;
#pragma unroll
        for (int q = 0; q < NACC / 4; ++q) {
#if MFMA == 32
            const int n = n0 + (wn * REP_N + j) * MFMA + 8 * q + 4 * lg;
#else
            const int n = n0 + (wn * REP_N + j) * MFMA + 4 * lg;
#endif
            bool ok = true;
            if (M % BM != 0) ok = ok && (m < M);
            if (N % BN != 0) ok = ok && (n < N);      /* N % 4 == 0: whole vectors */
            if (ok) {
                i32x4 v4;
                v4[0] = acc[i][j][4 * q + 0]; v4[1] = acc[i][j][4 * q + 1];
                v4[2] = acc[i][j][4 * q + 2]; v4[3] = acc[i][j][4 * q + 3];
#if SPLITK > 1
#pragma unroll
                for (int x = 0; x < 4; ++x) atomicAdd(C + (size_t)m * N + n + x, v4[x]);
#else
                i32x4* dst = reinterpret_cast<i32x4*>(C + (size_t)m * N + n);
#if NT_STORE
                __builtin_nontemporal_store(v4, dst);
#else
                *dst = v4;
#endif
#endif
            }
        }
#else
        const int n = n0 + (wn * REP_N + j) * MFMA + li;
#pragma unroll
        for (int v = 0; v < NACC; ++v) {
#if MFMA == 32
            const int row = 8 * (v / 4) + 4 * lg + (v % 4);
#else
            const int row = 4 * lg + v;
#endif
            const int m = m0 + (wm * REP_M + i) * MFMA + row;
            bool ok = true;
            if (M % BM != 0) ok = ok && (m < M);
            if (N % BN != 0) ok = ok && (n < N);
            if (ok) {
#if SPLITK > 1
                atomicAdd(C + (size_t)m * N + n, acc[i][j][v]);
#elif NT_STORE
                __builtin_nontemporal_store(acc[i][j][v], C + (size_t)m * N + n);
#else
                C[(size_t)m * N + n] = acc[i][j][v];
#endif
            }
        }
#endif
    };

    /* tile in buffer buf; ends: bytes of it inside the rows, where rows of A end in it and what lies behind them (the next
     * row's bytes) has come into LDS as it is and becomes zeros here */
    auto compute = [&](int buf, int ends = BK) {
        const int arow = wm * REP_M * MFMA + li;
        const int brow = wn * REP_N * MFMA + li;
        const signed char* as = &As[buf][arow * SROW];
        const signed char* bs = &Bs[buf][brow * SROW];
#pragma unroll
        for (int kk = 0; kk < BK; kk += MFMA_K) {
            i32x4 a[REP_M], b[REP_N];
#pragma unroll
            for (int i = 0; i < REP_M; ++i)
                a[i] = *reinterpret_cast<const i32x4*>(as + i * MFMA * SROW + PCOL(arow + i * MFMA, kk + 16 * lg));
#if DTL && K % 16 != 0
            if (ends < BK) {
#pragma unroll
                for (int i = 0; i < REP_M; ++i)
#pragma unroll
                    for (int d = 0; d < 4; ++d)                  /* K % 4 == 0: whole dwords */
                        a[i][d] = kk + 16 * lg + 4 * d < ends ? a[i][d] : 0;
            }
#endif
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
                b[j] = *reinterpret_cast<const i32x4*>(bs + j * MFMA * SROW + PCOL(brow + j * MFMA, kk + 16 * lg));
#pragma unroll
            for (int i = 0; i < REP_M; ++i)
#pragma unroll
                for (int j = 0; j < REP_N; ++j)
                    acc[i][j] = MFMA_OP(a[i], b[j], acc[i][j]);
        }
    };

#if DTL
    {
        const int wv = __builtin_amdgcn_readfirstlane(wave);
        /* The load is written as an instruction, not through the builtin: the
         * compiler makes every later LDS read wait for a direct-to-LDS load it
         * knows of (it cannot tell the buffers apart), which would undo the
         * overlap. Completion is tracked by hand. Two buffers: vmcnt(0) and a
         * barrier at the end of every iteration. Three: a count of the loads
         * of the tile behind and a barrier at its start, and none behind the
         * last tile, so whatever uses the LDS next needs a barrier of its own. */
        auto descriptor = [](const signed char* base, unsigned bytes) {
            const unsigned long long p = (unsigned long long)base;
            i32x4 d;                         /* raw buffer: base, stride 0, size in bytes, untyped dwords */
            d[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)p);
            d[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(p >> 32) & 0xffffu));
            d[2] = __builtin_amdgcn_readfirstlane((int)bytes);
            d[3] = 0x00020000;
            return d;
        };
        const i32x4 ra = descriptor(A, (unsigned)(M * K));
        const i32x4 rb = descriptor(B, (unsigned)(N * K));
        auto dma16 = [&](const i32x4& rsrc, const signed char* dst, unsigned vo, int so) {
            const unsigned lds_addr = (unsigned)(__UINTPTR_TYPE__)(lds_void*)dst;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         :: "s"(lds_addr), "v"(vo), "s"(rsrc), "s"(so) : "memory", "m0");
        };
        auto dma_tile = [&](int kt, int buf) {
            const int k0 = kbase + kt * BK;
#pragma unroll
            for (int e = 0; e < EA; ++e) {
                unsigned vo = a_voff[e];
                if (KP != K) vo = (k0 + a_col[e] < K) ? vo : OOB;
                dma16(ra, &As[buf][(e * NT + wv * 64) * 16], vo, K_AT(k0));
            }
#pragma unroll
            for (int e = 0; e < EB; ++e) {
                unsigned vo = b_voff[e];
                if (KP != K) vo = (k0 + b_col[e] < K) ? vo : OOB;
                dma16(rb, &Bs[buf][(e * NT + wv * 64) * 16], vo, K_AT(k0));
            }
        };
#if STAGES > 2
#define AHEAD (STAGES - 2)                     /* tiles under way while the wavefront waits for one */
        static_assert(AHEAD * (EA + EB) <= 63, "the count of loads under way has six bits");
#pragma unroll
        for (int t = 0; t <= AHEAD; ++t)
            if (t < KT) dma_tile(t, t);
#else
        dma_tile(0, 0);
#endif
#if DTL != 3 && STAGES == 2
        __builtin_amdgcn_s_waitcnt(0x0F70);     /* vmcnt(0): this wavefront's chunks are in LDS */
        __syncthreads();
#endif
#if DTL == 3
        /* Pinned schedule. Two fragment sets alternate by k-step parity (an even
         * number of k-steps per tile, so a tile ends on the set it began with and
         * nothing is copied). Slot m is what is issued before MFMA m of a k-step:
         *   not the last k-step:  fragment read m of the next k-step   (m < NR)
         *   last k-step:          at m == NB the wait for tile kt+1 and the barrier
         *                         (everybody has read the last fragments of tile kt
         *                         one k-step ago), then fragment read m - NB of tile
         *                         kt+1 and direct-to-LDS load m - NB of tile kt+2,
         *                         which goes into the buffer the barrier has freed
         *                         and has a whole tile period to land. */
#define NKS (BK / MFMA_K)
#define NM (REP_M * REP_N)
#define NR (REP_M + REP_N)
#define NB (NM / 4)
        const int arow = wm * REP_M * MFMA + li;
        const int brow = wn * REP_N * MFMA + li;
        i32x4 fA[2][REP_M], fB[2][REP_N];
        auto rd = [&](int buf, int kk, int set, int g) {
            if (g < REP_M)
                fA[set][g] = *reinterpret_cast<const i32x4*>(&As[buf][(arow + g * MFMA) * SROW + PCOL(arow + g * MFMA, kk + 16 * lg)]);
            else
                fB[set][g - REP_M] = *reinterpret_cast<const i32x4*>(&Bs[buf][(brow + (g - REP_M) * MFMA) * SROW + PCOL(brow + (g - REP_M) * MFMA, kk + 16 * lg)]);
        };
        auto dma_one = [&](int kt, int buf, int e) {
            const int k0 = kbase + kt * BK;
            if (e < EA) {
                unsigned vo = a_voff[e];
                if (KP != K) vo = (k0 + a_col[e] < K) ? vo : OOB;
                dma16(ra, &As[buf][(e * NT + wv * 64) * 16], vo, K_AT(k0));
            } else {
                unsigned vo = b_voff[e - EA];
                if (KP != K) vo = (k0 + b_col[e - EA] < K) ? vo : OOB;
                dma16(rb, &Bs[buf][((e - EA) * NT + wv * 64) * 16], vo, K_AT(k0));
            }
        };
        /* one tile; NEXT: tile kt+1 exists (its fragments are fetched), NEXT2: tile kt+2 exists */
#define I8_TILE(NEXT, NEXT2)                                                                          \
        _Pragma("unroll")                                                                             \
        for (int ks = 0; ks < NKS; ++ks) {                                                            \
            const int set = ks & 1;                                                                   \
            _Pragma("unroll")                                                                         \
            for (int m = 0; m < NM; ++m) {                                                            \
                if (ks + 1 < NKS) {                                                                   \
                    if (m < NR) rd(cur, (ks + 1) * MFMA_K, set ^ 1, m);                               \
                } else if (NEXT) {                                                                    \
                    if (m == NB) {                                                                    \
                        __builtin_amdgcn_s_waitcnt(0x0F70);                                           \
                        __syncthreads();                                                              \
                    }                                                                                 \
                    if (m >= NB && m - NB < NR) rd(cur ^ 1, 0, set ^ 1, m - NB);                      \
                    if ((NEXT2) && m >= NB && m - NB < EA + EB) dma_one(kt + 2, cur, m - NB);         \
                }                                                                                     \
                __builtin_amdgcn_sched_barrier(0);                                                    \
                acc[m / REP_N][m % REP_N] = MFMA_OP(fA[set][m / REP_N], fB[set][m % REP_N], acc[m / REP_N][m % REP_N]); \
                __builtin_amdgcn_sched_barrier(0);                                                    \
            }                                                                                         \
        }
        if (KT > 1) dma_tile(1, 1);
        /* tile 0 has landed when at most the loads of tile 1 are outstanding */
        if (KT > 1) __builtin_amdgcn_s_waitcnt(0x0F70 | ((EA + EB) & 15) | (((EA + EB) >> 4) << 14));
        else __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
#pragma unroll
        for (int g = 0; g < NR; ++g) rd(0, 0, 0, g);
        int kt = 0;
        for (; kt + 2 < KT; ++kt) {
            const int cur = kt & 1;
            I8_TILE(1, 1)
        }
        for (; kt + 1 < KT; ++kt) {
            const int cur = kt & 1;
            I8_TILE(1, 0)
        }
        {
            const int cur = kt & 1;
            I8_TILE(0, 0)
        }
#undef I8_TILE
#elif DTL == 2
        /* with fragment prefetch: the LDS reads of step t+1 are issued before
         * the MFMAs of step t, across the tile boundary as well */
        const int arow = wm * REP_M * MFMA + li;
        const int brow = wn * REP_N * MFMA + li;
        auto load_frags = [&](int buf, int kk, i32x4 (&fa)[REP_M], i32x4 (&fb)[REP_N]) {
            const signed char* as = &As[buf][arow * SROW];
            const signed char* bs = &Bs[buf][brow * SROW];
#pragma unroll
            for (int i = 0; i < REP_M; ++i)
                fa[i] = *reinterpret_cast<const i32x4*>(as + i * MFMA * SROW + PCOL(arow + i * MFMA, kk + 16 * lg));
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
                fb[j] = *reinterpret_cast<const i32x4*>(bs + j * MFMA * SROW + PCOL(brow + j * MFMA, kk + 16 * lg));
        };
        i32x4 fa[REP_M], fb[REP_N];
        load_frags(0, 0, fa, fb);
#if EARLYST
#if BK != 2 * MFMA_K
#error "early stores: two k-steps per tile"
#endif
#define KT_LOOP (KT - 1)
#else
#define KT_LOOP KT
#endif
        for (int kt = 0; kt < KT_LOOP; ++kt) {
            const int cur = kt & 1;
            if (kt + 1 < KT) dma_tile(kt + 1, cur ^ 1);
#pragma unroll
            for (int kk = 0; kk < BK; kk += MFMA_K) {
                i32x4 na[REP_M], nb[REP_N];
                if (kk + MFMA_K < BK) {
                    load_frags(cur, kk + MFMA_K, na, nb);
                } else {
                    /* tile kt has been read by everybody, tile kt+1 has landed */
                    __builtin_amdgcn_s_waitcnt(0x0F70);
                    __syncthreads();
                    if (kt + 1 < KT) load_frags(cur ^ 1, 0, na, nb);
                }
#pragma unroll
                for (int i = 0; i < REP_M; ++i)
#pragma unroll
                    for (int j = 0; j < REP_N; ++j)
                        acc[i][j] = MFMA_OP(fa[i], fb[j], acc[i][j]);
                if (kk + MFMA_K < BK || kt + 1 < KT) {
#pragma unroll
                    for (int i = 0; i < REP_M; ++i) fa[i] = na[i];
#pragma unroll
                    for (int j = 0; j < REP_N; ++j) fb[j] = nb[j];
                }
            }
        }
#if EARLYST
        {
            /* the last tile, block-major: fa/fb hold the fragments of its first k-step, na/nb get
             * those of its second; blocks go in groups of EG, and the stores of a group are issued
             * behind the MFMAs of the next group, which cover the distance from an MFMA to the
             * read of its result */
            i32x4 na[REP_M], nb[REP_N];
            load_frags((KT - 1) & 1, MFMA_K, na, nb);
#define EG 4
#define NBLK (REP_M * REP_N)
#pragma unroll
            for (int g = 0; g <= (NBLK + EG - 1) / EG; ++g) {
                if (g * EG < NBLK) {
#pragma unroll
                    for (int b = g * EG; b < g * EG + EG && b < NBLK; ++b)
                        acc[b / REP_N][b % REP_N] = MFMA_OP(fa[b / REP_N], fb[b % REP_N], acc[b / REP_N][b % REP_N]);
#pragma unroll
                    for (int b = g * EG; b < g * EG + EG && b < NBLK; ++b)
                        acc[b / REP_N][b % REP_N] = MFMA_OP(na[b / REP_N], nb[b % REP_N], acc[b / REP_N][b % REP_N]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (g > 0) {
#pragma unroll
                    for (int b = (g - 1) * EG; b < g * EG && b < NBLK; ++b)
                        store_block(b / REP_N, b % REP_N);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#endif
#elif STAGES > 2
        int cur = 0, to = STAGES - 1;
        for (int kt = 0; kt < KT; ++kt) {
            /* tile kt has landed once the loads of the AHEAD tiles behind it are all that is under way */
            if (kt + AHEAD < KT)
                __builtin_amdgcn_s_waitcnt(0x0F70 | ((AHEAD * (EA + EB)) & 15) | (((AHEAD * (EA + EB)) >> 4) << 14));
            else
                __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();                   /* for everybody, who also has read tile kt - 1: its buffer is free */
            if (kt + STAGES - 1 < KT) dma_tile(kt + STAGES - 1, to);
#if K % 16 != 0
            if (kbase + (kt + 1) * BK > K) compute(cur, K - kbase - kt * BK);
            else
#endif
            compute(cur);
            to = cur;
            cur = cur + 1 == STAGES ? 0 : cur + 1;
        }
#else
        for (int kt = 0; kt < KT; ++kt) {
            const int cur = kt & 1;
            if (kt + 1 < KT) dma_tile(kt + 1, cur ^ 1);   /* lands while tile kt is multiplied */
            compute(cur);
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __syncthreads();
        }
#endif
    }
#elif FRAGPF
    {
        const int arow = wm * REP_M * MFMA + li;
        const int brow = wn * REP_N * MFMA + li;
        auto load_frags = [&](int buf, int kk, i32x4 (&fa)[REP_M], i32x4 (&fb)[REP_N]) {
            const signed char* as = &As[buf][arow * SROW];
            const signed char* bs = &Bs[buf][brow * SROW];
#pragma unroll
            for (int i = 0; i < REP_M; ++i)
                fa[i] = *reinterpret_cast<const i32x4*>(as + i * MFMA * SROW + PCOL(arow + i * MFMA, kk + 16 * lg));
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
                fb[j] = *reinterpret_cast<const i32x4*>(bs + j * MFMA * SROW + PCOL(brow + j * MFMA, kk + 16 * lg));
        };
        i32x4 fa[REP_M], fb[REP_N];
        load_global(0, 0);
        store_lds(0, 0, 0);
        if (KT > 1) load_global(1, 0);
        __syncthreads();
        load_frags(0, 0, fa, fb);
        for (int kt = 0; kt < KT; ++kt) {
            const int cur = kt & 1;
            if (kt + 1 < KT) {
                store_lds(kt + 1, cur ^ 1, 0);         /* tile kt+1, loaded during iteration kt-1 */
                __builtin_amdgcn_sched_barrier(0);
                if (kt + 2 < KT) load_global(kt + 2, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int kk = 0; kk < BK; kk += MFMA_K) {
                i32x4 na[REP_M], nb[REP_N];
                if (kk + MFMA_K < BK) {
                    load_frags(cur, kk + MFMA_K, na, nb);
                } else {
                    /* every wavefront has read tile kt and written tile kt+1 */
                    __syncthreads();
                    if (kt + 1 < KT) load_frags(cur ^ 1, 0, na, nb);
                }
#pragma unroll
                for (int i = 0; i < REP_M; ++i)
#pragma unroll
                    for (int j = 0; j < REP_N; ++j)
                        acc[i][j] = MFMA_OP(fa[i], fb[j], acc[i][j]);
                if (kk + MFMA_K < BK || kt + 1 < KT) {
#pragma unroll
                    for (int i = 0; i < REP_M; ++i) fa[i] = na[i];
#pragma unroll
                    for (int j = 0; j < REP_N; ++j) fb[j] = nb[j];
                }
            }
        }
    }
#else
    /* tile t: global -> register set t % PD -> LDS buffer -> MFMA */
#pragma unroll
    for (int p = 0; p < PD; ++p)
        if (p < KT) load_global(p, p);
    store_lds(0, 0, 0);
    __syncthreads();
    for (int kt0 = 0; kt0 < KT; kt0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            const int kt = kt0 + u;
            if (kt < KT) {
                const int cur = (STAGES == 2) ? (kt & 1) : 0;
                if (kt + PD < KT) load_global(kt + PD, u);
                /* keep the prefetch at the top of the iteration: without this
                 * fence the scheduler sinks the loads down to their use */
                __builtin_amdgcn_sched_barrier(0);
                compute(cur);
                if (STAGES == 1) __syncthreads();
                if (kt + 1 < KT) store_lds(kt + 1, (STAGES == 2) ? (cur ^ 1) : 0, (u + 1) % PD);
                __syncthreads();
            }
        }
    }

#endif
    /* The last MFMA's result registers may not be read for 19 issue slots
     * (16 passes) and the hardware does not enforce it; the compiler's hazard
     * pass can lose a short path through branchy code, so the distance from
     * the main loop to the first accumulator read is explicit. */
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

#if WAVES_K > 1
    /* ---- sum the k-groups' partial tiles through LDS ---- */
    __syncthreads();             /* every group has read its last fragments: tile memory is free */
    if (kg > 0) {
        int* red = reinterpret_cast<int*>(smem) + (kg - 1) * (NT * REP_M * REP_N * NACC);
#pragma unroll
        for (int i = 0; i < REP_M; ++i)
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
#pragma unroll
                for (int v = 0; v < NACC; ++v)
                    red[((i * REP_N + j) * NACC + v) * NT + tid] = acc[i][j][v];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < WAVES_K; ++g) {
        const int* red = reinterpret_cast<const int*>(smem) + (g - 1) * (NT * REP_M * REP_N * NACC);
#pragma unroll
        for (int i = 0; i < REP_M; ++i)
#pragma unroll
            for (int j = 0; j < REP_N; ++j)
#pragma unroll
                for (int v = 0; v < NACC; ++v)
                    acc[i][j][v] += red[((i * REP_N + j) * NACC + v) * NT + tid];
    }
#endif
#if !EARLYST
#pragma unroll
    for (int i = 0; i < REP_M; ++i)
#pragma unroll
        for (int j = 0; j < REP_N; ++j)
            store_block(i, j);
#endif
    CLK_END;
}
