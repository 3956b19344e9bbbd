// W8A8 int8 GEMM for few rows or few output tiles: the waves of a workgroup share its output tile and each takes
// every KW-th step of 128 k.
//
// Tiles are small (16 to 64 rows by 16 to 64 columns), so that a product of few rows has a workgroup for every CU
// where the 128 x 256 tiles of i8_gemm_dma.hip give 43 (32 x 11008 x 4096), and a CU is kept loading by four to
// eight waves that do not wait for one another: a wave owns a ring of R stages in LDS that only it fills and reads,
// so there is no barrier until the partial sums meet.  A stage is one 128-byte line of each of the tile's rows,
// brought by LDS-destination loads of eight lines each (operands read straight into the MFMA layout would touch
// sixteen lines per load, four lanes of each).  Integer sums are exact in any order: the results are those of the
// other kernels bit for bit.
// What bounds it: the operand bytes of the tiles on their way into a CU, 58 to 66 bytes per ns whatever the tile,
// then the weight's bytes at 5.4 to 5.8 TB/s from HBM, on top of 2.7 us of launch, first load and reduction.  Us, here /
// on the 128 x 256 tiles, with the weight in the last-level cache (one weight, call after call) and from HBM (a gigabyte
// of weights in turn): 32 x 11008 x 4096 9.7 / 21.7 and 12.5 / 27.6, 1 x 11008 x 4096 9.1 / 21.2 and 11.4 / 26.0,
// 64 x 4096 x 4096 6.0 / 21.0 and 7.7 / 27.4, 32 x 1024 x 14336 6.2 / 61.5 and 10.6 / 82.4, 256 x 4096 x 4096 10.5 / 21.7
// and 12.8 / 29.3, 512 x 4096 x 4096 16.9 / 22.3 and 19.2 / 28.7.
#include "common.h"

#include <cmath>

namespace mh {

// 16 bytes per lane, global -> LDS at m0 + lane * 16; records past the end of the resource arrive as zeros.
__device__ __forceinline__ void rows_load_to_lds(uint32_t lds_addr, int voffset, const int4_t& rsrc, int soffset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_addr), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory", "m0");
}

__device__ __forceinline__ int4_t rows_rsrc(const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    int4_t r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    r[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)((a >> 32) & 0xffffu));
    r[2] = __builtin_amdgcn_readfirstlane((int)bytes);
    r[3] = kBufferRsrcFlags;
    return r;
}

template <int MT, int NT, int KW, int R>
__global__ __launch_bounds__(KW * 64) void i8_gemm_rows_kernel(
    const int8_t* __restrict__ A, const int8_t* __restrict__ W, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, half_t* __restrict__ out, int32_t* __restrict__ acc_out, int M, int N, int K,
    int tiles_m) {
    constexpr int kStep = 128;                      // k of a step: one 128-byte line of every row
    constexpr int kRows = (MT + NT) * 16;           // rows of a stage: A's, then W's
    constexpr int kStage = kRows * kStep;
    constexpr int kLoads = kRows / 8;               // a wave load brings eight lines
    constexpr int kTiles = MT * NT;
    constexpr int kItems = (kTiles + KW - 1) / KW;  // groups of four outputs per thread
    static_assert(R * kLoads < 64, "vmcnt counts to 63");
    constexpr int kLds = KW * R * kStage > KW * kTiles * 1024 ? KW * R * kStage : KW * kTiles * 1024;
    __shared__ __attribute__((aligned(1024))) int8_t smem[kLds];  // the waves' rings, then their partial sums

    // Consecutive workgroups go to different XCDs: each gets a run of tiles, row tiles of a column tile side by
    // side, so that the weight's rows are fetched into one L2.
    const unsigned total = gridDim.x, id = blockIdx.x, xcd = id & 7, q8 = total >> 3, r8 = total & 7;
    const unsigned tile = xcd * q8 + min(xcd, r8) + (id >> 3);
    const int m0 = (int)(tile % (unsigned)tiles_m) * (MT * 16), n0 = (int)(tile / (unsigned)tiles_m) * (NT * 16);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;

    // the scales, requested ahead of the operands (without an fp16 output they may be absent: the loads read the
    // first words of A instead, no branch around them)
    const float* as = out ? a_scale : reinterpret_cast<const float*>(A);
    const float* ws = out ? w_scale : reinterpret_cast<const float*>(A);
    const int m_last = out ? M - 1 : 0, n_last = out ? N - 1 : 0;
    float sa[kItems];
    float4_t sw[kItems];
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int t = min(u * KW + wave, kTiles - 1);
        sa[u] = as[min(m0 + t / NT * 16 + l16, m_last)];
#pragma unroll
        for (int e = 0; e < 4; ++e) sw[u][e] = ws[min(n0 + t % NT * 16 + lg * 4 + e, n_last)];
    }

    const int4_t a_rsrc = rows_rsrc(A + (size_t)m0 * K, (uint32_t)(min(MT * 16, M - m0) * (size_t)K));
    const int4_t w_rsrc = rows_rsrc(W + (size_t)n0 * K, (uint32_t)(min(NT * 16, N - n0) * (size_t)K));
    // Load j fills LDS rows 8 j .. 8 j + 7 of a stage; the lane that fills chunk position c of row r fetches chunk
    // c ^ (r / 2 % 8) of the row's line, which makes the fragment reads conflict-free.  Rows past the last one are
    // records past the end of the resource: zeros, no traffic.
    auto row_of = [&](int j) { return j * 8 + (lane >> 3); };
    auto swizzled = [&](int j) { return ((lane & 7) ^ ((row_of(j) >> 1) & 7)) * 16; };
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(size_t)smem) + (uint32_t)wave * (R * kStage);
    const int whole = K / kStep, steps = (K + kStep - 1) / kStep;
    const int mine = steps > wave ? (steps - wave + KW - 1) / KW : 0;
    int voff[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
        const int row = row_of(j);
        voff[j] = (row < MT * 16 ? row : row - MT * 16) * K + swizzled(j);
    }
    auto load_stage = [&](int i) {
        const int step = wave + i * KW;
        const uint32_t base = lds0 + (uint32_t)(i % R) * kStage;
        if (step < whole || step >= steps) {
            // past this wave's last step: no records, so no traffic, but the waits can count on the loads
            int4_t ar = a_rsrc, wr = w_rsrc;
            ar[2] = __builtin_amdgcn_readfirstlane(step < whole ? a_rsrc[2] : 0);
            wr[2] = __builtin_amdgcn_readfirstlane(step < whole ? w_rsrc[2] : 0);
            const int k0 = step < whole ? step * kStep : 0;
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                rows_load_to_lds(base + (uint32_t)j * 1024u, voff[j], j < MT * 2 ? ar : wr, k0);
        } else {  // the last 64 k of a K that is no multiple of 128: half lines, zeros behind them
#pragma unroll
            for (int j = 0; j < kLoads; ++j)
                rows_load_to_lds(base + (uint32_t)j * 1024u, swizzled(j) < 64 ? voff[j] + step * kStep : -16,
                                 j < MT * 2 ? a_rsrc : w_rsrc, 0);
        }
    };

    int4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = int4_t{0, 0, 0, 0};

#pragma unroll
    for (int i = 0; i < R; ++i) load_stage(i);
    const int8_t* ring = smem + wave * (R * kStage);
    auto frag = [&](const int8_t* st, int row, int c) {
        return *reinterpret_cast<const int4_t*>(st + row * 128 + ((c ^ ((row >> 1) & 7)) << 4));
    };
    int slot = 0;
    for (int i = 0; i < mine; ++i) {
        // this wave's stage i is there; only this wave reads or writes its part of the LDS: no barrier
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * kLoads) : "memory");
        const int8_t* st = ring + slot * kStage;
        int4_t fa[2][MT], fb[2][NT];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int t = 0; t < MT; ++t) fa[h][t] = frag(st, t * 16 + l16, h * 4 + lg);
#pragma unroll
            for (int t = 0; t < NT; ++t) fb[h][t] = frag(st, MT * 16 + t * 16 + l16, h * 4 + lg);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the stage is refilled
        load_stage(i + R);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int b = 0; b < NT; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[h][b], fa[h][a], acc[a][b], 0, 0, 0);
        slot = slot == R - 1 ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the empty loads past the end write LDS too
    __syncthreads();

    // acc[a][b][e] is row a * 16 + l16, column b * 16 + lg * 4 + e
    int4_t* part = reinterpret_cast<int4_t*>(smem);
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b) part[(wave * kTiles + a * NT + b) * 64 + lane] = acc[a][b];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kItems; ++u) {
        const int t = u * KW + wave;
        if (t >= kTiles) break;
        int4_t sum = part[t * 64 + lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) sum += part[(w * kTiles + t) * 64 + lane];
        const int m = m0 + t / NT * 16 + l16, n = n0 + t % NT * 16 + lg * 4;
        if (m >= M || n >= N) continue;
        const size_t at = (size_t)m * N + n;
        const bool vec = N % 4 == 0;
        if (acc_out) {
            if (vec) {
                *reinterpret_cast<int4_t*>(acc_out + at) = sum;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) acc_out[at + e] = sum[e];
            }
        }
        if (out) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // the scale product and its product with the sum are each rounded to fp32 and only then to fp16;
                // the empty asm keeps the compiler from fusing the last two steps into one that rounds once
                float prod = (float)sum[e] * (sa[u] * sw[u][e]);
                asm volatile("" : "+v"(prod));
                h[e] = (half_t)prod;
            }
            if (vec) {
                *reinterpret_cast<half4_t*>(out + at) = h;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) out[at + e] = h[e];
            }
        }
    }
}

// ---- which tile, and whether to take this kernel at all ------------------------------------------------------

// A tile of mt x nt times 16 and the waves of its workgroup; the four numbers are rows_time()'s.
struct RowsTile {
    int mt, nt, waves;
    double fixed, larger, smaller, pass;
};
constexpr RowsTile kRowsTiles[] = {
    {1, 1, 8, 4.88, 0.155, 0.365, 0.44}, {2, 1, 4, 4.96, 0.254, 0.292, 0.29}, {2, 2, 4, 4.12, 0.422, 0.655, 0.45},
    {1, 4, 4, 4.28, 0.573, 0.570, 0.00}, {2, 4, 8, 2.48, 0.594, 0.517, 1.87}, {4, 4, 4, 3.13, 0.787, 0.401, 1.26},
};

static size_t rows_tiles(const RowsTile& t, int M, int N) {
    return (((size_t)M + t.mt * 16 - 1) / (t.mt * 16)) * (((size_t)N + t.nt * 16 - 1) / (t.nt * 16));
}

// Us that the operand bytes take: of the fullest CU at 62 bytes per ns, and of the weight at 5.5 TB/s.
struct RowsBytes {
    double cu, weight, passes;
};
static RowsBytes rows_bytes(const RowsTile& t, int M, int N, int K) {
    const double passes = ceil((double)rows_tiles(t, M, N) / compute_units()), rows = t.mt * 16;
    return {passes * ((M < rows ? M : rows) + t.nt * 16) * K / 62e3, (double)N * K / 5.5e6, passes};
}

// The tile: the larger of the two and a quarter of the smaller.  Over the shapes that were measured (1 to 1024 rows, 1024 to
// 28672 columns, K 1024 to 14336) that names the fastest tile or one within 8 % of it.
static const RowsTile& rows_best(int M, int N, int K) {
    const RowsTile* best = nullptr;
    double least = 0;
    for (const RowsTile& t : kRowsTiles) {
        const RowsBytes b = rows_bytes(t, M, N, K);
        const double cost = b.cu > b.weight ? b.cu + 0.25 * b.weight : b.weight + 0.25 * b.cu;
        if (best == nullptr || cost < least) {
            least = cost;
            best = &t;
        }
    }
    return *best;
}

// Expected time in us, operands in the last-level cache: a fit per tile over 4800 shapes (1 to 4096 rows, 256 to 28672
// columns, K 192 to 14336), four of five within 15 %.
static double rows_time(const RowsTile& t, int M, int N, int K) {
    const RowsBytes b = rows_bytes(t, M, N, K);
    return t.fixed + t.larger * (b.cu > b.weight ? b.cu : b.weight) + t.smaller * (b.cu > b.weight ? b.weight : b.cu) +
           t.pass * b.passes;
}

// The same for the 128 x 256 tiles of the other kernels, by the kernel that K picks there: 128-k stages loaded straight
// into LDS, the same by registers (K 128 and 256), and 64-k stages.  `passes` of a tile on every CU.
static double tiled_time(int M, int N, int K) {
    const double passes = ceil((double)((((size_t)M + 127) / 128) * (((size_t)N + 255) / 256)) / compute_units());
    const double k = passes * K / 1e3, weight = (double)N * K / 5.5e6;
    if (K % 128 != 0) return -4.39 + 7.43 * k + 7.57 * passes + 1.02 * weight;
    return K < 384 ? -1.41 + 1.86 * k + 7.27 * passes + 0.38 * weight : -5.06 + 4.02 * k + 9.68 * passes + 0.63 * weight;
}

// Taken where a tenth is to be won: of 4800 shapes that a plain comparison of the bytes sent here 170 were more than a tenth
// slower than on the 128 x 256 tiles, up to 1.8 times (many rows and a short K: 752 x 4032 x 256 9.7 us against 7.1, 2113 x
// 1352 x 1920 18.9 / 14.5).  With this line 10 of 12400 others are, and the geometric mean over all of them is 0.54 of the
// 128 x 256 tiles' time.  A resource covers the rows of one tile, up to 64 rows of K bytes below 2 GiB, and a launch 2^32
// threads.
bool i8_gemm_rows_preferred(int M, int N, int K) {
    if (K >= (1 << 24)) return false;
    const RowsTile& t = rows_best(M, N, K);
    return rows_tiles(t, M, N) * t.waves * 64 < ((size_t)1 << 32) && rows_time(t, M, N, K) < 0.9 * tiled_time(M, N, K);
}

int i8_gemm_rows_tile(int M, int N, int K) {
    const RowsTile& t = rows_best(M, N, K);
    return t.mt * 16 << 16 | t.nt * 16;
}

int i8_gemm_rows_launch(hipStream_t stream, const int8_t* a, const int8_t* w, const float* a_scale,
                        const float* w_scale, void* out_f16, int32_t* acc_i32, int M, int N, int K) {
    const RowsTile& t = rows_best(M, N, K);
    const int tiles_m = (int)(((size_t)M + t.mt * 16 - 1) / (t.mt * 16));
    const unsigned tiles = (unsigned)rows_tiles(t, M, N);
    // LDS per workgroup 64, 72, 64, 80, 96 and 64 KiB: two of all but the fifth share a CU
#define MH_I8_ROWS(MT, NT, KW, R)                                                                                     \
    hipLaunchKernelGGL((i8_gemm_rows_kernel<MT, NT, KW, R>), dim3(tiles), dim3(KW * 64), 0, stream, a, w, a_scale,     \
                       w_scale, (half_t*)out_f16, acc_i32, M, N, K, tiles_m)
    switch (t.mt * 8 + t.nt) {
        case 1 * 8 + 1: MH_I8_ROWS(1, 1, 8, 2); break;
        case 2 * 8 + 1: MH_I8_ROWS(2, 1, 4, 3); break;
        case 2 * 8 + 2: MH_I8_ROWS(2, 2, 4, 2); break;
        case 1 * 8 + 4: MH_I8_ROWS(1, 4, 4, 2); break;
        case 2 * 8 + 4: MH_I8_ROWS(2, 4, 8, 1); break;
        default: MH_I8_ROWS(4, 4, 4, 1); break;
    }
#undef MH_I8_ROWS
    MH_CHECK_LAUNCH();
    return MH_OK;
}

}  // namespace mh
