/*
 * g2_matmul.hip -- fp32-accurate GEMM on the bf16 matrix cores (included by
 * g2_kernels.hip, which provides the shared helpers and types).
 *
 * An fp32 value is the sum of three bf16 values: p1 = bf16(v), p2 = bf16(v -
 * p1), p3 = bf16(v - p1 - p2), 8 significant bits each, both differences
 * exact; an fp16 value is the sum of two.  A product of two fp32 values is
 * then six bf16 products, p1q1 + p1q2 + p2q1 + p2q2 + p1q3 + p3q1 (five with
 * an fp16 factor, whose q3 is zero); the ones left out, p2q3 and p3q2 first,
 * are about 2^-24 of it at most.  The products are exact in fp32 and summed in fp32 by
 * v_mfma_f32_16x16x32_bf16, which takes 32 k per instruction at 16 times the
 * rate of the fp32 instruction (4 k): a sixth of 32 k against 4 k leaves
 * 2.7 times the fp32 peak and fewer roundings of the running sum.
 *
 * The conversion and both matrix instructions keep subnormals, so the parts
 * carry every value whose last bit, 2^-23 of its power of two, is a multiple
 * of bf16's smallest, 2^-133.  A work-group that reads a smaller one computes
 * its tile, or its split's part of it, again on the fp32 matrix instruction
 * (again_tile()): a factor of 2^-120 can meet one of 2^80, and the sum shows
 * nothing of it.  The test is whether what is left for the third part is
 * subnormal in fp32, one operation per value beside the 5.5 of its parts: it
 * is for every value that the parts do not carry and never for one of 2^-103
 * or more.  (A running minimum of the values took 1.5: 333 x 6400 x 1600 fp16
 * 54.5 us against 49.9; a test for large factors and small sums, with a second
 * look at the operands where it says so, was slower still.)  Such a tile takes
 * about what the fp32 instruction alone takes: 1024 x 8192 x 1600 of nothing
 * but small values 0.54 ms (0.14).
 * Infinities, NaN and magnitudes that round past bf16's largest make a sum not
 * finite; the tile is then computed again in the same way, so they come out as
 * fp32 arithmetic has them.
 */
namespace xg {
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
/* vectors at any element's address */
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef _Float16 f16x2u __attribute__((ext_vector_type(2), aligned(2)));

/* Eight consecutive k as the fragments (8 bf16 per lane) of P parts, and of
 * three what is left for the third: look() sets `lossy` where that may not be
 * all of it.  Two are, of any fp16 value. */
template <int P>
__device__ __forceinline__ void parts8(const float (&v)[8], u32x4 (&o)[P], float (&rest)[8])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f32x2 r = {v[2 * e], v[2 * e + 1]};
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (P == 3 && p == 2) {
                rest[2 * e] = r.x;
                rest[2 * e + 1] = r.y;
            }
            const unsigned w = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
            o[p][e] = w;
            if (p + 1 < P) {
                r.x -= __builtin_bit_cast(float, w << 16);
                r.y -= __builtin_bit_cast(float, w & 0xffff0000u);
            }
        }
    }
}

__device__ __forceinline__ void look(bool &lossy, const float (&rest)[8])
{
#pragma unroll
    for (int e = 0; e < 8; e += 2) lossy |= __builtin_amdgcn_classf(rest[e], 0x90) | __builtin_amdgcn_classf(rest[e + 1], 0x90);
}

template <int P>
__device__ __forceinline__ void parts8(const float (&v)[8], u32x4 (&o)[P], bool &lossy)
{
    float rest[8];
    parts8<P>(v, o, rest);
    if constexpr (P == 3) look(lossy, rest);
}

__device__ __forceinline__ f32x4 mma(const u32x4 &a, const u32x4 &b, const f32x4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

/* acc[j] += a . b[j] over 32 k: the six (PB 3) or five (PB 2) products,
 * small ones first.  Successive instructions take different accumulators:
 * a chain of them on one accumulator waits for each result. */
template <int PB, int J>
__device__ __forceinline__ void mma_parts(f32x4 (&acc)[J], const u32x4 (&a)[3], const u32x4 (&b)[J][PB])
{
    constexpr int pa[6] = {2, 1, 0, 1, 0, 0}, pb[6] = {0, 0, 1, 1, 2, 0};
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (pb[p] < PB) acc[j] = mma(a[pa[p]], b[j][pb[p] < PB ? pb[p] : 0], acc[j]);
}

/* Adds a NaN to z (zeros at first) for a sum that is not finite, else zero. */
__device__ __forceinline__ void finite(f32x4 &z, const f32x4 &v)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) z[q] = fmaf(v[q], 0.f, z[q]);
}

/* Whether what a thread has seen calls for the fp32 instruction. */
__device__ __forceinline__ bool not_carried(bool lossy, const f32x4 &z)
{
    const float s = (z[0] + z[1]) + (z[2] + z[3]);
    return lossy || s != s;
}

/* Whether any thread of the work-group says so: one word of LDS per wave, a
 * barrier for all. */
template <int WAVES>
__device__ __forceinline__ bool any_thread(unsigned (&words)[WAVES], bool mine)
{
    const bool wave_has = __ballot(mine) != 0;
    if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = wave_has;
    __syncthreads();
    unsigned any = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) any |= words[w];
    return any != 0;
}

/* A wave's IB x JB blocks of 16 x 16, rows m + 16 i and column n[j] of the
 * lane, over k0 <= k < k1, added to acc by the fp32 matrix instruction: a lane
 * takes four consecutive k of 16, straight from memory. */
template <typename BT, bool BNK, int IB, int JB>
__device__ __forceinline__ void again_tile(const float *A, const BT *B, int M, int N, int K, int m, const int (&n)[JB],
                                           int k0, int k1, f32x4 (&acc)[IB][JB])
{
    const int lane = threadIdx.x & 63, fk = 4 * (lane >> 4);
#pragma unroll 1
    for (int k = k0 + fk; k - fk < k1; k += 16) {
        const bool whole = k - fk + 16 <= k1;
        float x[IB][4], y[JB][4];
        auto four = [&](float (&v)[4], const float *p) {
            if (whole) {
                *(f32x4 *)v = *(const f32x4u *)p;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = k + e < k1 ? p[e] : 0.f;
            }
        };
#pragma unroll
        for (int i = 0; i < IB; ++i) four(x[i], A + (size_t)min(m + 16 * i + (lane & 15), M - 1) * K + k);
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const size_t c = min(n[j], N - 1);
            if constexpr (BNK) {
                four(y[j], B + c * K + k);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) y[j][e] = whole || k + e < k1 ? ldw(B, (size_t)(k + e) * N + c) : 0.f;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int j = 0; j < JB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][e], y[j][e], acc[i][j], 0, 0, 0);
    }
}

/* The k, within a step of 32, of element e of octet o is 4 o + koff(e), for
 * both factors: the four lanes of a row then load 64 consecutive bytes. */
__device__ __forceinline__ constexpr int koff(int e) { return e < 4 ? e : 12 + e; }

/* Tile of work-group w of T tiles: XCD w % 8 (consecutive work-groups go to
 * consecutive XCDs) takes a contiguous run of tiles, row blocks first, so
 * the row blocks of a column block share one XCD's L2; the runs differ by
 * at most one tile. */
__device__ __forceinline__ int tile_of(int w, int T)
{
    const int x = w & 7, q = T >> 3, r = T & 7;
    return x * q + min(x, r) + (w >> 3);
}
} /* namespace xg */

/* LDS-tiled: BM x BN outputs per work-group of 2 x 2 waves, K in steps of 32,
 * the steps of a split (gridDim.y splits of whole steps, GEPI_PARTIAL) in
 * order.  A step's tiles are loaded to registers one step ahead, split into
 * their parts and stored to LDS as [part][k octet][row] 16-byte fragments, so
 * a fragment read takes 16 consecutive rows of an octet.  The octet planes of
 * A are padded by 64 bytes so that the four octets of four rows that 16 lanes
 * store fall on distinct banks; SQ_LDS_BANK_CONFLICT is a third of
 * SQ_LDS_IDX_ACTIVE all the same, 16 cycles to each of A's stores.  B
 * [K,N]: a lane loads a column pair (BN 128) or a column (BN 64) of eight k
 * rows, so the transposition is a choice of registers; column n of a 128-wide
 * tile sits at position n / 2 + 64 (n odd), which makes a lane's two column
 * blocks neighbours in memory.  N >= 2 for BN 128; nothing else is asked of
 * M, N, K or alignment.
 *
 * Measured on MI355X (N(0,1) by N(0,0.02)): 1024 x 50257 x 1600 in 0.84 to
 * 0.89 ms with fp32 B (1.11 to 1.17 PFLOP/s of bf16 products; a library bf16
 * product of 8192^3 reaches 1.14; the fp32-instruction kernel before: 3.35
 * ms), 0.67 to 0.69 ms with fp16 B (3.05); the matrix cores are busy 56 and
 * 65% of the CUs' busy cycles.  With one work-group per CU a step takes
 * 1.85 us, its conversions, LDS traffic and products one after the other
 * (xduo_impl is for that).  Taken back: two steps in flight, two LDS buffers,
 * all fragments read ahead, raised wave priority (each within 5%). */
template <typename BT, int EPI, int BM, int BN>
__device__ void xgemm_impl(const g2_gemm_args &a)
{
    using namespace xg;
    constexpr int PB = sizeof(BT) == 4 ? 3 : 2;
    constexpr int SA = BM * 16 + 64, SB = BN * 16; /* octet plane strides, bytes */
    constexpr int RA = BM / 64, RB = BN / 64;                       /* octets (A) or columns (B) a thread stages */
    constexpr int IB = BM / 32, JB = BN / 32;                       /* 16-blocks of a wave */
    constexpr int ST = 3 * 4 * SA + PB * 4 * SB;                    /* bytes of a step's tiles */
    __shared__ __attribute__((aligned(16))) unsigned char lds[ST];
    __shared__ unsigned words[4];
    bool lossy = false;
    constexpr bool LATE = PB == 3; /* operands tested beside the products (fp16 B: 10% slower, a wave per SIMD lost) */
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int M = a.M, N = a.N, K = a.K;
    const int nmb = (M + BM - 1) / BM;
    const int tile = tile_of(blockIdx.x, gridDim.x);
    const int m0 = (tile % nmb) * BM, n0 = (tile / nmb) * BN;
    const int nkt = (K + 31) >> 5, ks = gridDim.y;
    const int s0 = (int)(((long)nkt * blockIdx.y) / ks), s1 = (int)(((long)nkt * (blockIdx.y + 1)) / ks);
    const int sf = min(s1, K >> 5); /* steps s0 .. sf - 1 are whole */
    const BT *B = (const BT *)a.B;

    const int ar = tid >> 2, ao = (tid & 3) * 4; /* A: row (+ 64 i), k offset */
    const float *ap[RA];
#pragma unroll
    for (int i = 0; i < RA; ++i) ap[i] = a.A + (size_t)min(m0 + ar + 64 * i, M - 1) * K + ao;
    /* B: column (pair), octet; the pair that the last column
     * begins is loaded one column early */
    const int bc = tid & 63, bo = wave;
    const bool late = n0 + bc * RB + RB - 1 == N;
    const BT *bp = B + min(n0 + bc * RB, N - RB);

    float av[RA][8], bv[RB][8], ra[RA][8], rb[RB][8];
    /* whole step t (past the last one: that one again, unused) */
    auto load = [&](int t) {
        const int k = min(t, sf - 1) * 32;
#pragma unroll
        for (int i = 0; i < RA; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) *(f32x4 *)(av[i] + 4 * h) = *(const f32x4u *)(ap[i] + k + 16 * h);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const size_t o = (size_t)(k + 4 * bo + koff(e)) * N;
            if constexpr (RB == 1) {
                bv[0][e] = ldw(bp, o);
            } else if constexpr (sizeof(BT) == 4) {
                const f32x2 w = *(const f32x2u *)((const float *)bp + o);
                bv[0][e] = w.x;
                bv[RB - 1][e] = w.y;
            } else {
                const f16x2u w = *(const f16x2u *)((const _Float16 *)bp + o);
                bv[0][e] = (float)w.x;
                bv[RB - 1][e] = (float)w.y;
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            u32x4 p[3];
            if constexpr (LATE) parts8<3>(av[i], p, ra[i]);
            else parts8<3>(av[i], p, lossy);
#pragma unroll
            for (int q = 0; q < 3; ++q) *(u32x4 *)(lds + (4 * q + (tid & 3)) * SA + (ar + 64 * i) * 16) = p[q];
        }
        if constexpr (RB == 2) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bv[0][e] = late ? bv[1][e] : bv[0][e];
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            u32x4 p[PB];
            if constexpr (LATE) parts8<PB>(bv[i], p, rb[i]);
            else parts8<PB>(bv[i], p, lossy);
#pragma unroll
            for (int q = 0; q < PB; ++q)
                *(u32x4 *)(lds + 12 * SA + (4 * q + bo) * SB + (bc + 64 * i) * 16) = p[q];
        }
    };

    f32x4 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    /* column block j of the wave: positions 16 j of its half (BN 64), or
     * (JB 4) blocks 0, 1 of the even columns and 2, 3 of the odd ones */
    constexpr bool PAIR = RB == 2;
    const int arow = (lane >> 4) * SA + (wm * (BM / 2) + (lane & 15)) * 16;
    const int brow = 12 * SA + (lane >> 4) * SB + (wn * (PAIR ? BN / 4 : BN / 2) + (lane & 15)) * 16;
    auto bblk = [](int j) { return PAIR ? (j & (JB / 2 - 1)) * 256 + (j / (JB / 2)) * (BN / 2) * 16 : j * 256; };
    auto multiply = [&]() {
        u32x4 b[JB][PB];
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
            for (int q = 0; q < PB; ++q) b[j][q] = *(const u32x4 *)(lds + brow + 4 * q * SB + bblk(j));
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            u32x4 f[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] = *(const u32x4 *)(lds + arow + 4 * q * SA + i * 256);
            mma_parts<PB, JB>(acc[i], f, b);
            if (LATE && i == 0) {
#pragma unroll
                for (int x = 0; x < RA; ++x) look(lossy, ra[x]);
#pragma unroll
                for (int x = 0; x < RB; ++x) look(lossy, rb[x]);
            }
        }
    };

    if (sf > s0) {
        load(s0);
        for (int t = s0; t < sf; ++t) {
            __syncthreads(); /* the previous step has been read */
            store();
            load(t + 1);
            __syncthreads();
            multiply();
        }
    }
    if (sf < s1) { /* the last, partial step: zeros past K */
        const int k = sf * 32;
#pragma unroll
        for (int i = 0; i < RA; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) av[i][e] = k + ao + koff(e) < K ? ap[i][k + koff(e)] : 0.f;
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int kk = k + koff(e) + 4 * bo;
                bv[i][e] = kk < K ? ldw(bp, (size_t)kk * N + i) : 0.f;
            }
        __syncthreads();
        store();
        __syncthreads();
        multiply();
    }

    /* output (row, column) of accumulator value (i, j, q) */
    auto om = [&](int i, int q) { return m0 + wm * (BM / 2) + i * 16 + 4 * (lane >> 4) + q; };
    auto on = [&](int j) {
        return PAIR ? n0 + 2 * (wn * (BN / 4) + (j & (JB / 2 - 1)) * 16 + (lane & 15)) + j / (JB / 2)
                    : n0 + wn * (BN / 2) + j * 16 + (lane & 15);
    };
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) finite(z, acc[i][j]);
    if (__builtin_expect(any_thread(words, not_carried(lossy, z)), 0)) {
        int n[JB];
#pragma unroll
        for (int j = 0; j < JB; ++j) n[j] = on(j);
#pragma unroll
        for (int i = 0; i < IB; ++i)
#pragma unroll
            for (int j = 0; j < JB; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        again_tile<BT, false>(a.A, B, M, N, K, m0 + wm * (BM / 2), n, s0 * 32, min(s1 * 32, K), acc);
        __syncthreads(); /* before any wave writes: C may lie in A or B */
    }

    float *C = EPI == GEPI_PARTIAL ? a.part + (size_t)blockIdx.y * M * N : a.C;
    if constexpr (EPI != GEPI_PARTIAL) {
        if (a.bias) {
#pragma unroll
            for (int j = 0; j < JB; ++j) {
                const float b = a.bias[min(on(j), N - 1)];
#pragma unroll
                for (int i = 0; i < IB; ++i) acc[i][j] += b;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = om(i, q);
            if (m >= M) continue;
            if constexpr (PAIR) {
#pragma unroll
                for (int j = 0; j < JB / 2; ++j) {
                    const int n = on(j);
                    float *c = C + (size_t)m * N + n;
                    if (n + 1 < N) *(f32x2u *)c = (f32x2){acc[i][j][q], acc[i][j + JB / 2][q]};
                    else if (n < N) *c = acc[i][j][q];
                }
            } else {
#pragma unroll
                for (int j = 0; j < JB; ++j)
                    if (on(j) < N) C[(size_t)m * N + on(j)] = acc[i][j][q];
            }
        }
}

#define G2_XGEMM(name, BT, EPI, BM, BN, OCC) \
    extern "C" __global__ __launch_bounds__(256, OCC) void name(const g2_gemm_args a) { xgemm_impl<BT, EPI, BM, BN>(a); }
G2_XGEMM(g2k_xgemm128_f32, float, GEPI_STORE, 128, 128, 2)
G2_XGEMM(g2k_xgemm128_f16, _Float16, GEPI_STORE, 128, 128, 2)
G2_XGEMM(g2k_xgemm64_f32, float, GEPI_STORE, 64, 64, 3)
G2_XGEMM(g2k_xgemm64_f16, _Float16, GEPI_STORE, 64, 64, 3)
G2_XGEMM(g2k_xgemm64_part_f32, float, GEPI_PARTIAL, 64, 64, 3)
G2_XGEMM(g2k_xgemm64_part_f16, _Float16, GEPI_PARTIAL, 64, 64, 3)

/* C = (part[0] + ... + part[ks-1]) + bias, the splits in order; four
 * elements of the M x N matrix per thread, ks <= G2_XG_MAXKS. */
G2K void g2k_xgemm_sum(const g2_gemm_args a)
{
    const size_t MN = (size_t)a.M * a.N;
    for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4; i < MN; i += (size_t)gridDim.x * 1024) {
        if (i + 4 <= MN) {
            f32x4 p[G2_XG_MAXKS];
#pragma unroll
            for (int z = 0; z < G2_XG_MAXKS; ++z)
                if (z < a.ksplit) p[z] = *(const f32x4u *)(a.part + z * MN + i);
            f32x4 v = p[0];
#pragma unroll
            for (int z = 1; z < G2_XG_MAXKS; ++z)
                if (z < a.ksplit) v += p[z];
            if (a.bias) {
                unsigned n = MN >> 32 ? (unsigned)(i % (size_t)a.N) : (unsigned)i % (unsigned)a.N;
#pragma unroll
                for (int e = 0; e < 4; ++e, n = n + 1 < (unsigned)a.N ? n + 1 : 0) v[e] += a.bias[n];
            }
            *(f32x4u *)(a.C + i) = v;
        } else {
            for (size_t j = i; j < MN; ++j) {
                float v = a.part[j];
                for (int z = 1; z < a.ksplit; ++z) v += a.part[z * MN + j];
                a.C[j] = a.bias ? v + a.bias[j % (size_t)a.N] : v;
            }
        }
    }
}

/* One tile per CU: BM x 128 outputs per work-group of two groups of 2 x 2
 * waves, each with an LDS buffer and every other K step of 32.  The groups
 * alternate: while one multiplies, the other splits its next step's values
 * into their parts and stores them, so a SIMD holds one wave of each and its
 * matrix core works through the other's conversions; the groups' sums are
 * added at the end.  Staging as in xgemm_impl.  Epilogues as g2_gemm_args
 * describes them; GEPI_PARTIAL: gridDim.y splits of whole steps.  A step
 * takes 1.02 us (0.75 at BM 64; 1.85 in xgemm_impl at one work-group per CU),
 * of which the products alone 0.79 and the reads in front of them 0.2; the
 * matrix cores are busy 42% of the CUs' busy cycles (56% whole with fp16 B).
 * W [N,K] of n_embd 1280 by 256 rows: fc 27 us in three splits (the fp32
 * instruction, whole: 47), fc2 27 in twelve (34), qkv 22 in four (30). */
template <typename BT, bool BNK, int EPI, int BM>
__device__ void xduo_impl(const g2_gemm_args &a)
{
    using namespace xg;
    constexpr int BN = 128, RA = BM / 64, IB = BM / 32, HB = IB / 2;
    constexpr int PB = sizeof(BT) == 4 ? 3 : 2;
    constexpr int SA = BM * 16 + 64, SB = BN * 16 + (BNK ? 64 : 0); /* octet plane strides, bytes */
    constexpr int ST = 3 * 4 * SA + PB * 4 * SB;                    /* bytes of a step's tiles */
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * ST];
    __shared__ unsigned words[8];
    bool lossy = false;
    const int tid = threadIdx.x & 255, lane = tid & 63;
    const int w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = w8 >> 2, wave = w8 & 3, wm = wave >> 1, wn = wave & 1;
    const int M = a.M, N = a.N, K = a.K;
    const int nmb = (M + BM - 1) / BM;
    const int tile = tile_of(blockIdx.x, gridDim.x);
    const int m0 = (tile % nmb) * BM, n0 = (tile / nmb) * BN;
    const int nkt = (K + 31) >> 5, ks = gridDim.y;
    const int s0 = (int)(((long)nkt * blockIdx.y) / ks), s1 = (int)(((long)nkt * (blockIdx.y + 1)) / ks);
    const int sf = min(s1, K >> 5); /* steps s0 .. sf - 1 are whole */
    const BT *B = (const BT *)a.B;
    unsigned char *st = lds + g * ST;

    const int ar = tid >> 2, ao = (tid & 3) * 4;
    const float *ap[RA];
#pragma unroll
    for (int i = 0; i < RA; ++i) ap[i] = a.A + (size_t)min(m0 + ar + 64 * i, M - 1) * K + ao;
    const int bc = tid & 63, bo = wave;
    const bool late = !BNK && n0 + bc * 2 + 1 == N;
    const BT *bp[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
        bp[i] = BNK ? B + (size_t)min(n0 + ar + 64 * i, N - 1) * K + ao : B + min(n0 + bc * 2, N - 2) + i;

    float av[RA][8], bv[2][8];
    /* whole step t (past the last one: that one again, unused) */
    auto load = [&](int t) {
        const int k = min(t, sf - 1) * 32;
#pragma unroll
        for (int i = 0; i < RA; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) *(f32x4 *)(av[i] + 4 * h) = *(const f32x4u *)(ap[i] + k + 16 * h);
        if constexpr (BNK) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) *(f32x4 *)(bv[i] + 4 * h) = *(const f32x4u *)((const float *)bp[i] + k + 16 * h);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const size_t o = (size_t)(k + 4 * bo + koff(e)) * N;
                if constexpr (sizeof(BT) == 4) {
                    const f32x2 w = *(const f32x2u *)((const float *)bp[0] + o);
                    bv[0][e] = w.x;
                    bv[1][e] = w.y;
                } else { /* both columns' bits; widened in store() */
                    bv[0][e] = __builtin_bit_cast(float, *(const f16x2u *)((const _Float16 *)bp[0] + o));
                }
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            u32x4 p[3];
            parts8<3>(av[i], p, lossy);
#pragma unroll
            for (int q = 0; q < 3; ++q) *(u32x4 *)(st + (4 * q + (tid & 3)) * SA + (ar + 64 * i) * 16) = p[q];
        }
        float b[2][8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (!BNK && sizeof(BT) == 2) {
                const f16x2u w = __builtin_bit_cast(f16x2u, bv[0][e]);
                b[0][e] = (float)w.x;
                b[1][e] = (float)w.y;
            } else {
                b[0][e] = bv[0][e];
                b[1][e] = bv[1][e];
            }
            if constexpr (!BNK) b[0][e] = late ? b[1][e] : b[0][e];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            u32x4 p[PB];
            parts8<PB>(b[i], p, lossy);
#pragma unroll
            for (int q = 0; q < PB; ++q)
                *(u32x4 *)(st + 12 * SA + (4 * q + (BNK ? (tid & 3) : bo)) * SB + ((BNK ? ar : bc) + 64 * i) * 16) = p[q];
        }
    };

    f32x4 acc[IB][4];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    /* column block j of the wave: positions 16 j of its half (BNK), or blocks
     * 0, 1 of the even columns and 2, 3 of the odd ones */
    const unsigned char *arow = st + (lane >> 4) * SA + (wm * (BM / 2) + (lane & 15)) * 16;
    const unsigned char *brow = st + 12 * SA + (lane >> 4) * SB + (wn * (BNK ? 64 : 32) + (lane & 15)) * 16;
    auto multiply = [&]() {
        u32x4 f[IB][3], b[4][PB];
        auto read_a = [&](int q) {
#pragma unroll
            for (int i = 0; i < IB; ++i) f[i][q] = *(const u32x4 *)(arow + 4 * q * SA + i * 256);
        };
        auto read_b = [&](int q) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b[j][q] = *(const u32x4 *)(brow + 4 * q * SB + (BNK ? j * 256 : (j & 1) * 256 + (j >> 1) * 1024));
        };
        auto products = [&](int p, int q) {
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mma(f[i][p], b[j][q], acc[i][j]);
        };
        /* a part's reads are issued one or two products ahead of its use */
#define XG_KEEP_ORDER __builtin_amdgcn_sched_barrier(0)
        read_b(0);
        read_a(2);
        read_a(1);
        XG_KEEP_ORDER;
        __builtin_amdgcn_s_setprio(1);
        products(2, 0);
        XG_KEEP_ORDER;
        read_a(0);
        XG_KEEP_ORDER;
        products(1, 0);
        XG_KEEP_ORDER;
        read_b(1);
        XG_KEEP_ORDER;
        products(0, 0);
        XG_KEEP_ORDER;
        if constexpr (PB == 3) read_b(PB - 1);
        XG_KEEP_ORDER;
        products(1, 1);
        products(0, 1);
        if constexpr (PB == 3) {
            XG_KEEP_ORDER;
            products(0, PB - 1);
        }
        XG_KEEP_ORDER;
        __builtin_amdgcn_s_setprio(0);
#undef XG_KEEP_ORDER
    };

    /* group g takes whole steps s0 + g, s0 + g + 2, ...; both groups pass the
     * same number of barriers */
    if (sf > s0) {
        const int n = (sf - s0 + 1) >> 1;
        load(s0 + g);
        if (g) __syncthreads();
        for (int i = 0; i < n; ++i) {
            const int t = s0 + g + 2 * i;
            store();
            load(t + 2);
            __syncthreads();
            if (t < sf) multiply();
            __syncthreads();
        }
        if (!g) __syncthreads();
    }
    if (sf < s1 && !g) { /* the last, partial step: zeros past K */
        const int k = sf * 32;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
            for (int i = 0; i < RA; ++i) av[i][e] = k + ao + koff(e) < K ? ap[i][k + koff(e)] : 0.f;
            const int kk = k + koff(e) + (BNK ? ao : 4 * bo);
            const size_t o = BNK ? (size_t)(k + koff(e)) : (size_t)kk * N;
            if constexpr (BNK || sizeof(BT) == 4) {
#pragma unroll
                for (int i = 0; i < 2; ++i) bv[i][e] = kk < K ? ldw(bp[i], o) : 0.f;
            } else {
                bv[0][e] = kk < K ? __builtin_bit_cast(float, *(const f16x2u *)((const _Float16 *)bp[0] + o)) : 0.f;
            }
        }
        store();
    }
    __syncthreads();
    if (sf < s1 && !g) multiply();
    __syncthreads();

    /* each group hands half of its row blocks to the other and finishes the
     * other half: group 0 blocks 0 .. HB - 1, group 1 the rest */
    f32x4 sum[HB][4];
    {
        f32x4 *x = (f32x4 *)lds + (g * 4 + wave) * (HB * 256) + lane;
        const f32x4 *y = (const f32x4 *)lds + ((1 - g) * 4 + wave) * (HB * 256) + lane;
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 lo = acc[i][j], hi = acc[i + HB][j];
                f32x4 give;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    give[q] = g ? lo[q] : hi[q];
                    sum[i][j][q] = g ? hi[q] : lo[q];
                }
                x[(i * 4 + j) * 64] = give;
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[i][j] += y[(i * 4 + j) * 64];
    }

    /* output (row, column) of value (i, j, q) */
    auto om = [&](int i, int q) { return m0 + wm * (BM / 2) + (g * HB + i) * 16 + 4 * (lane >> 4) + q; };
    auto on = [&](int j) {
        return BNK ? n0 + wn * 64 + j * 16 + (lane & 15) : n0 + 2 * (wn * 32 + (j & 1) * 16 + (lane & 15)) + (j >> 1);
    };
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < HB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) finite(z, sum[i][j]);
    if (__builtin_expect(any_thread(words, not_carried(lossy, z)), 0)) {
        const int n[4] = {on(0), on(1), on(2), on(3)};
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        again_tile<BT, BNK>(a.A, B, M, N, K, m0 + wm * (BM / 2) + g * HB * 16, n, s0 * 32, min(s1 * 32, K), sum);
    }

    /* every load of the epilogue before its first store */
    if constexpr (EPI != GEPI_PARTIAL) {
        float bias[4], rv[HB][4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j) bias[j] = a.bias ? a.bias[min(on(j), N - 1)] : 0.f;
        if constexpr (EPI == GEPI_RESID) {
#pragma unroll
            for (int i = 0; i < HB; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        rv[i][j][q] = a.C[(size_t)min(om(i, q), M - 1) * N + min(on(j), N - 1)];
        }
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (a.bias) sum[i][j][q] += bias[j];
                    if constexpr (EPI == GEPI_RESID) sum[i][j][q] += rv[i][j][q];
                    if constexpr (EPI == GEPI_GELU) sum[i][j][q] = gelu_f(sum[i][j][q]);
                }
    }
    if constexpr (EPI == GEPI_QKV) {
        const qkv_dst d = qkv_of(a);
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (on(j) < N) qkv_store4(d, om(i, 0), M, on(j), sum[i][j]);
        return;
    }
    float *C = EPI == GEPI_PARTIAL ? a.part + (size_t)blockIdx.y * M * N : a.C;
#pragma unroll
    for (int i = 0; i < HB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int m = om(i, q);
            if (m >= M) continue;
            if constexpr (!BNK) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int n = on(j);
                    float *c = C + (size_t)m * N + n;
                    if (n + 1 < N) *(f32x2u *)c = (f32x2){sum[i][j][q], sum[i][j + 2][q]};
                    else if (n < N) *c = sum[i][j][q];
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (on(j) < N) C[(size_t)m * N + on(j)] = sum[i][j][q];
            }
        }
}

#define G2_XDUO(name, BT, BNK, EPI, BM) \
    extern "C" __global__ __launch_bounds__(512, 2) void name(const g2_gemm_args a) { xduo_impl<BT, BNK, EPI, BM>(a); }
G2_XDUO(g2k_xduo_nk_part, float, true, GEPI_PARTIAL, 128)
G2_XDUO(g2k_xduo_nk_part64, float, true, GEPI_PARTIAL, 64)
G2_XDUO(g2k_xduo_nk_gelu, float, true, GEPI_GELU, 128)
G2_XDUO(g2k_xduo_nk_resid, float, true, GEPI_RESID, 128)
G2_XDUO(g2k_xduo_nk_qkv, float, true, GEPI_QKV, 128)
G2_XDUO(g2k_xduo_f32, float, false, GEPI_STORE, 128)
G2_XDUO(g2k_xduo_f16, _Float16, false, GEPI_STORE, 128)
G2_XDUO(g2k_xduo_part_f32, float, false, GEPI_PARTIAL, 128)
G2_XDUO(g2k_xduo_part_f16, _Float16, false, GEPI_PARTIAL, 128)

/* Few tiles: a work-group of 8 waves takes one 16 RB x 32 tile, the K steps
 * dealt to the waves in turn, their sums added in wave order through LDS.  No
 * staging: a lane loads its own fragments (8 k of a row of A; 8 rows of a
 * column pair of B) straight from memory, and the loads of the next step are
 * issued before the products of this one.  Bounded by load latency, one wait
 * per step: 64 x 2304 x 768 takes 8 us (the fp32-instruction kernel before:
 * 57), 96 x 768 x 3072 14 us (218).  16 waves, and 64-row tiles, were no
 * faster.  N >= 2. */
template <typename BT, int RB>
__device__ void xskinny_impl(const g2_gemm_args &a)
{
    using namespace xg;
    constexpr int PB = sizeof(BT) == 4 ? 3 : 2, NW = 8;
    __shared__ float red[NW][RB * 2][256];
    bool lossy = false;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = a.M, N = a.N, K = a.K;
    const int nmb = (M + 16 * RB - 1) / (16 * RB);
    const int tile = tile_of(blockIdx.x, gridDim.x);
    const int m0 = (tile % nmb) * 16 * RB, n0 = (tile / nmb) * 32;
    const BT *B = (const BT *)a.B;
    const int fr = lane & 15, fk = 4 * (lane >> 4);
    /* column pair; the pair that the last column begins is loaded one
     * column early */
    const bool late = n0 + 2 * fr + 1 == N;
    const float *ap[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) ap[i] = a.A + (size_t)min(m0 + 16 * i + fr, M - 1) * K + fk;
    const BT *bp = B + min(n0 + 2 * fr, N - 2);
    const int nkt = (K + 31) >> 5;

    float av[RB][8], bv[2][8];
    auto load = [&](int t) {
        const int k = t * 32;
        if (k + 32 <= K) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const size_t o = (size_t)(k + fk + koff(e)) * N;
                if constexpr (sizeof(BT) == 4) {
                    const f32x2 w = *(const f32x2u *)((const float *)bp + o);
                    bv[0][e] = w.x;
                    bv[1][e] = w.y;
                } else {
                    const f16x2u w = *(const f16x2u *)((const _Float16 *)bp + o);
                    bv[0][e] = (float)w.x;
                    bv[1][e] = (float)w.y;
                }
            }
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) *(f32x4 *)(av[i] + 4 * h) = *(const f32x4u *)(ap[i] + k + 16 * h);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int kk = k + fk + koff(e);
                bv[0][e] = kk < K ? ldw(bp, (size_t)kk * N) : 0.f;
                bv[1][e] = kk < K ? ldw(bp, (size_t)kk * N + 1) : 0.f;
#pragma unroll
                for (int i = 0; i < RB; ++i) av[i][e] = kk < K ? ap[i][k + koff(e)] : 0.f;
            }
        }
    };
    f32x4 acc[RB][2];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (wave < nkt) load(wave);
    for (int t = wave; t < nkt; t += NW) {
        u32x4 b[2][PB], f[RB][3];
#pragma unroll
        for (int e = 0; e < 8; ++e) bv[0][e] = late ? bv[1][e] : bv[0][e];
#pragma unroll
        for (int j = 0; j < 2; ++j) parts8<PB>(bv[j], b[j], lossy);
#pragma unroll
        for (int i = 0; i < RB; ++i) parts8<3>(av[i], f[i], lossy);
        if (t + NW < nkt) load(t + NW);
#pragma unroll
        for (int i = 0; i < RB; ++i) mma_parts<PB, 2>(acc[i], f[i], b);
    }
    /* [block][row 4 (l/16) + q][column l % 16] */
    auto hand_in = [&]() {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) red[wave][2 * i + j][(4 * (lane >> 4) + q) * 16 + fr] = acc[i][j][q];
    };
    /* a wave with something that the parts do not carry hands in NaN, which
     * shows in every thread's sum; finite sums never add up to one */
    f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) finite(z, acc[i][j]);
    if (__builtin_expect(__ballot(not_carried(lossy, z)) != 0, 0))
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){NAN, NAN, NAN, NAN};
    hand_in();
    __syncthreads();
    /* output o of the tile: its sum over the waves, in order */
    auto total = [&](int o) {
        const int i = o >> 9, r = (o >> 5) & 15, c = o & 31;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float x = red[w][2 * i + (c & 1)][r * 16 + (c >> 1)];
            v = w ? v + x : x;
        }
        return v;
    };
    float v = total(tid);
    if (__builtin_expect(v != v, 0)) { /* of all threads or none */
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
        const int n[2] = {n0 + 2 * fr, n0 + 2 * fr + 1};
        for (int t = wave; t < nkt; t += NW) again_tile<BT, false>(a.A, B, M, N, K, m0, n, 32 * t, min(32 * t + 32, K), acc);
        hand_in();
        __syncthreads();
        v = total(tid);
    }
#pragma unroll
    for (int o = tid; o < RB * 512; o += NW * 64) {
        const int m = m0 + (o >> 5), n = n0 + (o & 31);
        if (o >= 512) v = total(o);
        if (m < M && n < N) a.C[(size_t)m * N + n] = a.bias ? v + a.bias[n] : v;
    }
}
#define G2_XSKINNY(name, BT, RB) \
    extern "C" __global__ __launch_bounds__(512) void name(const g2_gemm_args a) { xskinny_impl<BT, RB>(a); }
G2_XSKINNY(g2k_xskinny1_f32, float, 1)
G2_XSKINNY(g2k_xskinny1_f16, _Float16, 1)
G2_XSKINNY(g2k_xskinny2_f32, float, 2)
G2_XSKINNY(g2k_xskinny2_f16, _Float16, 2)
