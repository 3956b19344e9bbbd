// Dense fp16 product out[M, N] = a[M, K] @ b[N, K]^T for any M, N and K >= 8 and any alignment, single or
// batched: the products of a prompt (q k^T with K = 128, p v with K = the prompt's length, a weight over many
// rows), minit/cuda/dispatch.py:59-101 and minit/cuda/kernel/cublas.py:68-111 of the reference.
//
// A workgroup of four waves owns BM x 128 outputs and walks K in rounds of 64.  A stage (BM + 128 rows of
// 128 bytes) travels global -> registers -> LDS: two rounds of loads are in flight in registers, two stages
// lie in LDS (64 KiB at BM = 128: two workgroups per CU), one barrier per round.  (STAGES = 1: one stage and two
// barriers, four workgroups per CU.)  Through registers and not by
// LDS-destination loads because a row starts on any 2-byte boundary when K is odd -- p v over a prompt of 1499
// tokens -- and those loads want dword addresses; a 16-byte vector load takes any.
// The K % 64 remainder is the first round: its chunks are loaded from inside the row and shifted down by
// whole elements, so that what lies past the end of a row is zero in both operands whatever memory holds.
// What bounds it: q k^T of a prompt its 144 MB of scores (32 x [1500, 1500, 128] 46 us: a tile is one
// chain of load, two rounds and store, four workgroups per CU overlap: 3.1 TB/s; without the streaming hint on the stores half as long again at 2048), p v the read of p
// (32 x [1500, 128, 1500] 47 us, with rows on 128-byte lines, K = 1536, 41), a product of many rows and columns the operands on their way into LDS
// (2048 x 4096 x 4096 87 us, 790 TFLOP/s).  K not a multiple of 32 took one thread per output before: 27.6 ms
// for that p v.
// The weight fragment is the first MFMA operand: a lane ends with four consecutive n of one row, the tile
// leaves through LDS as 16-byte row pieces.
#include "common.h"

#include <algorithm>

namespace mh {

constexpr int kTiledBN = 128, kTiledBK = 64, kTiledThreads = 256;
constexpr int kTiledPitch = kTiledBN * 2 + 16;  // bytes of an output row in LDS

__device__ __forceinline__ int tiled_swz(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }

__device__ __forceinline__ uint4_t load_unaligned(const half_t* p) { return *reinterpret_cast<const uint4_any_t*>(p); }

// v moved down by n elements (0..8), zeros above
__device__ __forceinline__ uint4_t drop_elements(uint4_t v, int n) {
    unsigned long long lo = (unsigned long long)v.y << 32 | v.x, hi = (unsigned long long)v.w << 32 | v.z;
    const int s = n * 16;
    const unsigned long long lo_small = s == 0 ? lo : (lo >> s) | (hi << ((64 - s) & 63));
    const unsigned long long lo_big = s >= 128 ? 0ull : hi >> ((s - 64) & 63);
    const unsigned long long new_lo = s >= 64 ? lo_big : lo_small, new_hi = s >= 64 ? 0ull : hi >> (s & 63);
    return uint4_t{(unsigned)new_lo, (unsigned)(new_lo >> 32), (unsigned)new_hi, (unsigned)(new_hi >> 32)};
}

template <int BM, int STAGES>
__global__ __launch_bounds__(kTiledThreads, STAGES == 1 ? 4 : 2) void f16_matmul_nk_tiled_kernel(
    const half_t* __restrict__ a, const half_t* __restrict__ b, half_t* __restrict__ out, int M, int N, int K,
    int tiles_m, int tiles_n) {
    constexpr int WN = BM > 64 ? 2 : 4;        // waves along n
    constexpr int MT = BM / 16 / (4 / WN);     // 16-row tiles of a per wave
    constexpr int NT = kTiledBN / WN / 16;     // 16-column tiles per wave
    constexpr int AC = BM / 32, BC = 4;        // 16-byte chunks of a stage per thread
    constexpr int kStage = (BM + kTiledBN) * 128;
    constexpr int kLds = STAGES * kStage > BM * kTiledPitch ? STAGES * kStage : BM * kTiledPitch;
    __shared__ __attribute__((aligned(1024))) char smem[kLds];

    // Consecutive workgroups go to different XCDs: give each a run of tiles in (matrix, row, column) order, so
    // that the operands of a matrix are fetched into one L2.
    const unsigned total = gridDim.x, id = blockIdx.x, xcd = id & 7, q8 = total >> 3, r8 = total & 7;
    const unsigned tile = xcd * q8 + min(xcd, r8) + (id >> 3);
    const int tn = tile % tiles_n, tm = tile / tiles_n % tiles_m;
    const size_t batch = tile / (unsigned)(tiles_n * tiles_m);
    a += batch * M * K;
    b += batch * N * K;
    out += batch * M * N;
    const int m0 = tm * BM, n0 = tn * kTiledBN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wn = (wave % WN) * (NT * 16), wm = (wave / WN) * (MT * 16);
    const int l16 = lane & 15, lg = lane >> 4;

    // chunk tid % 8 of rows tid / 8 + 32 i of either operand
    const int chunk = tid & 7, row0 = tid >> 3;
    const half_t* ap[AC];
    const half_t* bp[BC];
#pragma unroll
    for (int i = 0; i < AC; ++i) ap[i] = a + (size_t)min(m0 + row0 + 32 * i, M - 1) * K;
#pragma unroll
    for (int i = 0; i < BC; ++i) bp[i] = b + (size_t)min(n0 + row0 + 32 * i, N - 1) * K;

    uint4_t ra[2][AC], rb[2][BC];
    const int rounds = K / kTiledBK, rest = K % kTiledBK;
    auto load = [&](int slot, int r) {
        const int k = min(r, rounds - 1) * kTiledBK + chunk * 8;
#pragma unroll
        for (int i = 0; i < AC; ++i) ra[slot][i] = load_unaligned(ap[i] + k);
#pragma unroll
        for (int i = 0; i < BC; ++i) rb[slot][i] = load_unaligned(bp[i] + k);
    };
    auto store = [&](int slot, int buf) {
        char* st = smem + buf * kStage;
#pragma unroll
        for (int i = 0; i < AC; ++i) *reinterpret_cast<uint4_t*>(st + tiled_swz(row0 + 32 * i, chunk)) = ra[slot][i];
#pragma unroll
        for (int i = 0; i < BC; ++i)
            *reinterpret_cast<uint4_t*>(st + BM * 128 + tiled_swz(row0 + 32 * i, chunk)) = rb[slot][i];
    };

    float4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int buf) {
        const char* st = smem + buf * kStage;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            half8_t fa[MT], fb[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i)
                fa[i] = *reinterpret_cast<const half8_t*>(st + tiled_swz(wm + i * 16 + l16, ks * 4 + lg));
#pragma unroll
            for (int j = 0; j < NT; ++j)
                fb[j] = *reinterpret_cast<const half8_t*>(st + BM * 128 + tiled_swz(wn + j * 16 + l16, ks * 4 + lg));
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
    };

    if (rest) {
        // the remainder: a chunk that reaches past the end of the row is read where it ends and moved down
        const int k = rounds * kTiledBK + chunk * 8, at = min(k, K - 8), drop = min(k - at, 8);
#pragma unroll
        for (int i = 0; i < AC; ++i) ra[0][i] = load_unaligned(ap[i] + at);
#pragma unroll
        for (int i = 0; i < BC; ++i) rb[0][i] = load_unaligned(bp[i] + at);
#pragma unroll
        for (int i = 0; i < AC; ++i) ra[0][i] = drop_elements(ra[0][i], drop);
#pragma unroll
        for (int i = 0; i < BC; ++i) rb[0][i] = drop_elements(rb[0][i], drop);
        store(0, STAGES - 1);
    }
    if (rounds) {
        load(0, 0);
        load(1, 1);
    }
    if (rest) {
        __syncthreads();
        compute(STAGES - 1);
        if (STAGES == 1) __syncthreads();
    }
    if constexpr (STAGES == 1) {
        for (int r = 0; r < rounds; r += 2) {
            store(0, 0);
            load(0, r + 2);
            __syncthreads();
            compute(0);
            if (r + 1 >= rounds) break;
            __syncthreads();
            store(1, 0);
            load(1, r + 3);
            __syncthreads();
            compute(0);
            if (r + 2 >= rounds) break;
            __syncthreads();
        }
    } else if (rounds) {
        store(0, 0);
        load(0, 2);
        __syncthreads();
        // round r reads buffer r % 2 while stage r + 1 goes into the other one, which every wave left before
        // the barrier of round r - 1
        for (int r = 0; r < rounds; r += 2) {
            compute(0);
            if (r + 1 >= rounds) break;
            store(1, 1);
            load(1, r + 3);
            __syncthreads();
            compute(1);
            if (r + 2 >= rounds) break;
            store(0, 0);
            load(0, r + 4);
            __syncthreads();
        }
    }
    __syncthreads();

    // acc[i][j][e]: row wm + i * 16 + l16, column wn + j * 16 + lg * 4 + e of the tile
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = (half_t)acc[i][j][e];
            *reinterpret_cast<half4_t*>(smem + (wm + i * 16 + l16) * kTiledPitch + (wn + j * 16 + lg * 4) * 2) = h;
        }
    __syncthreads();
    const int c8 = (tid & 15) * 8, n = n0 + c8;
#pragma unroll
    for (int i = 0; i < BM / 16; ++i) {
        const int row = (tid >> 4) + i * 16, m = m0 + row;
        if (m >= M || n >= N) continue;
        const uint4_t v = *reinterpret_cast<const uint4_t*>(smem + row * kTiledPitch + c8 * 2);
        half_t* dst = out + (size_t)m * N + n;
        if (n + 8 <= N) {
            __builtin_nontemporal_store((uint4_any_t)v, reinterpret_cast<uint4_any_t*>(dst));
        } else {
            const half8_t h = __builtin_bit_cast(half8_t, v);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n + e < N) dst[e] = h[e];
        }
    }
}

bool f16_matmul_lds_supported(int M, int N, int K);  // f16_matmul_lds.hip

// A launch holds 2^32 threads: tiles beyond that go into further launches, a row of tiles into one.
constexpr size_t kTiledMostTiles = ((size_t)1 << 32) / kTiledThreads - 1;
static int tiled_columns(int N) { return (int)(((long long)N + kTiledBN - 1) / kTiledBN); }

bool f16_matmul_tiled_supported(int M, int N, int K) {
    return M > 0 && N > 0 && K >= 8 && (size_t)tiled_columns(N) <= kTiledMostTiles;
}

// Of the shapes with whole 16-byte pieces the other kernels serve too (K a multiple of 32), those of more than
// 16 rows that the LDS-streaming kernel does not take (K below 384 or no multiple of 64: 32 x [1500, 1500, 128]
// 454 us on the kernel with operands straight from global memory, 45-53 here), and of those it does take
//   * up to 256 columns with more than 64 rows and K up to 4096, the p v of a prompt, whose matrices come in
//     batches (32 x [1500, 128, 1504] 132 us against 36);
//   * two tiles per CU and more, where tiles of 128 rows halve the traffic of its 64-row blocks (2048 x 4096 x 4096
//     100 us against 87, 1024 x 8192 x 8192 192 / 168; with 336 tiles on 256 CUs it stays ahead, 71 / 77);
//   * one block of 65 to 128 rows whose column tiles fill three quarters of the CUs (96 x 32000 x 4096 80 / 55).
bool f16_matmul_tiled_preferred(int M, int N, int K) {
    if (M <= 16 || !f16_matmul_tiled_supported(M, N, K)) return false;
    if (!f16_matmul_lds_supported(M, N, K)) return true;
    if (M <= 64) return false;
    const size_t cus = compute_units(), tiles_n = tiled_columns(N);
    return (N <= 256 && K <= 4096) || tiles_n * (((size_t)M + 127) / 128) >= 2 * cus || (M <= 128 && tiles_n * 4 >= 3 * cus);
}

// Height of the tiles.  A CU takes about a microsecond for a stage of 256 rows whether one workgroup asks or two, so
// the time goes with the staged rows of the CU that has most: ceil(tiles / CUs) * (BM + 128).  Measured in
// us, 128 / 64 / 32 rows: 16 x [479, 128, 479] 11.2 / 8.4 / 6.7 (the rule's 32), 8 x [1245, 128, 1245] 22.8 / 16.5 / 20.5
// (64), 8 x [300, 128, 300] 6.6 / 5.1 / 4.4 (32), 16 x [2000, 128, 2000] 35.6 / 43.7 / 57.8 (128), 32 x [1500, 128, 1500]
// 53.3 / 54.0 / 78.5, with 96 rows 47.1 (96).
// Two rounds of K and less (q k^T) are all beginnings and ends: tiles of 64 rows with one stage in LDS, four
// workgroups per CU (32 x [1500, 1500, 128] 49.5 -> 45.8, 8 x [300, 300, 128] 6.0 -> 4.3).
struct TiledPlan {
    int bm, stages;
};
static TiledPlan plan_tiled(int batch, int M, int N, int K) {
    if (K <= 2 * kTiledBK && M > 32) return {64, 1};
    const size_t cus = compute_units(), columns = (size_t)batch * tiled_columns(N);
    TiledPlan best = {32, 2};
    size_t least = 0;
    for (int bm = M <= 32 ? 32 : M <= 64 ? 64 : M <= 96 ? 96 : 128; bm >= 32; bm -= 32) {
        const size_t cost = (columns * (((size_t)M + bm - 1) / bm) + cus - 1) / cus * (bm + 128);
        if (least == 0 || cost < least) {
            least = cost;
            best.bm = bm;
        }
    }
    return best;
}

int f16_matmul_tiled_tile(int batch, int M, int N, int K) {
    const TiledPlan p = plan_tiled(batch, M, N, K);
    return p.bm << 16 | p.stages;
}

static int tiled_launch_part(hipStream_t stream, const TiledPlan& p, const half_t* a, const half_t* b, half_t* out, int batch,
                             int M, int N, int K) {
    const int tiles_m = (int)(((long long)M + p.bm - 1) / p.bm), tiles_n = tiled_columns(N);
    const unsigned tiles = (unsigned)((size_t)tiles_m * tiles_n * batch);
#define MH_TILED(BM, STAGES)                                                                                          \
    hipLaunchKernelGGL((f16_matmul_nk_tiled_kernel<BM, STAGES>), dim3(tiles), dim3(kTiledThreads), 0, stream, a, b, out, M, \
                       N, K, tiles_m, tiles_n)
    if (p.stages == 1) {
        MH_TILED(64, 1);
    } else {
        switch (p.bm) {
            case 32: MH_TILED(32, 2); break;
            case 64: MH_TILED(64, 2); break;
            case 96: MH_TILED(96, 2); break;
            default: MH_TILED(128, 2); break;
        }
    }
#undef MH_TILED
    MH_CHECK_LAUNCH();
    return MH_OK;
}

int f16_matmul_tiled_launch(hipStream_t stream, const void* a, const void* b, void* out, int batch, int M, int N, int K) {
    const TiledPlan p = plan_tiled(batch, M, N, K);
    const size_t tiles_n = tiled_columns(N), tiles = (((size_t)M + p.bm - 1) / p.bm) * tiles_n;
    const half_t *pa = (const half_t*)a, *pb = (const half_t*)b;
    half_t* po = (half_t*)out;
    // whole matrices per launch, or row blocks of one matrix
    const int matrices = tiles <= kTiledMostTiles ? (int)std::min((size_t)batch, kTiledMostTiles / tiles) : 1;
    const int rows = tiles <= kTiledMostTiles ? M : (int)(kTiledMostTiles / tiles_n * p.bm);
    for (int i = 0; i < batch; i += matrices)
        for (long long r = 0; r < M; r += rows) {
            const int rc = tiled_launch_part(stream, p, pa + ((size_t)i * M + r) * K, pb + (size_t)i * N * K,
                                             po + ((size_t)i * M + r) * N, std::min(matrices, batch - i),
                                             (int)std::min((long long)rows, M - r), N, K);
            if (rc) return rc;
        }
    return MH_OK;
}

}  // namespace mh
