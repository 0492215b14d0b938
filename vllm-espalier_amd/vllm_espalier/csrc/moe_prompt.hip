// esp_grouped_prompt: the grouped expert GEMM over a whole prompt's (expert, member tile) list on gfx950, an expert's
// weights decoded once for up to 64 member rows, with the sums of esp_grouped at any K split.
//
// A program is (listed tile, 128-column block, matrix) over the whole K. esp_grouped at SK splits stores each split's
// scaled sums and its readers add them in split order; here the same sums are added in registers as the program passes
// each split's end (tot), so the launch writes one partial a row, whose bits are those of the splits' sum. One split is
// esp_grouped's SK = 1.
#include "../../../include/espalier.h"
#include "gemm.hpp"

namespace esp {

__device__ int g_moe_prompt_status;       // ESP_STATUS_* bits raised by the launches of this file

struct GroupedPromptArgs {
    const uint16_t* X[2];
    const int64_t* TP[2];
    const int* B[2];
    const int* C[2];
    const int* uids;
    const int* ucount;
    const int* members;
    const int* tiles;              // esp_group_tiles' list for tiles of TR members
    float* Z;                      // [mats][P][N]
    int K, N, P, maxm, slots;
    int split_steps;               // 32-k steps of a split
    int lo, hi;                    // the K2 range the launch's stages are sized for
};

constexpr int GP_STEPS = 4;        // 32-k steps a stage
constexpr int GP_WAVES = 4;
constexpr int GP_AROW = GP_STEPS * 32;                // halves of a member row's slice
__host__ __device__ constexpr int gp_buf_bytes(int k2, int tr) { return GP_STEPS * 2 * 32 * k2 * 4 + tr * GP_AROW * 2; }

// The K loop of one program. A stage is 4 steps of the block's trellis tiles and of the member rows, double-buffered in
// shared memory by DMA. A row's slice is 16 units of 16 bytes, stored with unit s at place s ^ (row & 15): a wave's copy
// is four whole rows (contiguous in shared memory, as the DMA needs), and the 16 rows that an MFMA operand reads lie in
// different banks. Rows past nrows are copies of row 0, whose sums are not stored.
template <int CB, int K2, int MG, int TR>
__device__ __forceinline__ void grouped_prompt_body(const GroupedPromptArgs& a, const uint32_t* __restrict__ T,
                                                    const uint16_t* __restrict__ X, const int* rows_sh, int nrows,
                                                    int mat, float scale, unsigned char* smem, int yb) {
    constexpr int TW = 4 * K2;
    constexpr int ROW_WORDS = StagePlan<K2>::ROW_WORDS;
    constexpr int B_WORDS = GP_STEPS * 2 * ROW_WORDS, BUF_BYTES = gp_buf_bytes(K2, TR);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5, c = lane & 15, G = lane >> 4;
    const int NTILES = a.N >> 4, nt0 = yb * 8, steps = a.K >> 5, nst = steps / GP_STEPS;      // K % 128 == 0
    // the copies' offsets, worked out once: a stage moves every trellis unit by whole k-tile rows and every member row
    // by 128 halves
    constexpr int UPR = 2 * TW, TU = 2 * GP_STEPS * UPR, TU_IT = (TU + 255) / 256;
    int t_off[TU_IT];
#pragma unroll
    for (int i = 0; i < TU_IT; ++i) {
        const int u = (wave + i * GP_WAVES) * 64 + lane, r = u / UPR;
        t_off[i] = (r * NTILES + nt0) * TW + (u - r * UPR) * 4;
    }
    constexpr int RQ = MG * 16 / 4;                          // copies of four rows
    int a_off[(RQ + GP_WAVES - 1) / GP_WAVES];
#pragma unroll
    for (int j = 0; j < (RQ + GP_WAVES - 1) / GP_WAVES; ++j) {
        const int m = 4 * (wave + j * GP_WAVES) + (lane >> 4);
        a_off[j] = rows_sh[m < nrows ? m : 0] * a.K + ((c ^ (m & 15)) * 8);
    }
    auto issue = [&](int st) __attribute__((always_inline)) {
        unsigned char* buf = smem + (st & 1) * BUF_BYTES;
        uint32_t* tb = reinterpret_cast<uint32_t*>(buf);
        const uint32_t* Ts = T + (size_t)(2 * GP_STEPS * st) * NTILES * TW;
#pragma unroll
        for (int i = 0; i < TU_IT; ++i) {
            const int u0 = (wave + i * GP_WAVES) * 64;
            if (TU % 256 == 0 || u0 < TU)                    // TU is a multiple of 64
                __builtin_amdgcn_global_load_lds((global_void_ptr)(Ts + t_off[i]), (lds_void_ptr)(tb + u0 * 4), 16, 0,
                                                 CPOL_NT);
        }
        uint16_t* ab = reinterpret_cast<uint16_t*>(buf + B_WORDS * 4);
        const uint16_t* Xs = X + st * GP_AROW;
#pragma unroll
        for (int j = 0; j < (RQ + GP_WAVES - 1) / GP_WAVES; ++j) {
            const int q = wave + j * GP_WAVES;
            if (q < RQ && 4 * q < nrows)
                __builtin_amdgcn_global_load_lds((global_void_ptr)(Xs + a_off[j]),
                                                 (lds_void_ptr)(ab + q * 4 * GP_AROW), 16, 0, 0);
        }
    };
    f32x4 acc[2][MG], tot[2][MG];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int g = 0; g < MG; ++g) {
            acc[j][g] = f32x4{0.f, 0.f, 0.f, 0.f};
            tot[j][g] = f32x4{-0.f, -0.f, -0.f, -0.f};       // -0 + v = v: the first split's sums as they are
        }
    const LanePlan<K2> lp(lane);
    const LdsWords<K2> lw(lp);
    const int lane_base = ((G >> 1) * 8 + 2 * wave) * TW;
    // this lane's A slots of a step: halves 4 (G & 1) .. + 3 of the slice's units u and u + 1, u = 4 * step + 2 (G >> 1)
    const int u0 = (((2 * (G >> 1)) ^ c) * 8) + 4 * (G & 1) + c * GP_AROW;
    const int u1 = (((2 * (G >> 1) + 1) ^ c) * 8) + 4 * (G & 1) + c * GP_AROW;
    int left = a.split_steps;
    issue(0);
    for (int st = 0; st < nst; ++st) {
        wait_stage();
        if (st + 1 < nst) issue(st + 1);
        const unsigned char* buf = smem + (st & 1) * BUF_BYTES;
        const uint32_t* bb = reinterpret_cast<const uint32_t*>(buf) + lane_base;
        const uint16_t* ab = reinterpret_cast<const uint16_t*>(buf + B_WORDS * 4);
#pragma unroll 1
        for (int ls = 0; ls < GP_STEPS; ++ls) {
            const uint32_t* tl = bb + ls * 2 * ROW_WORDS;
            uint32_t w[2][6];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 6; ++i) w[j][i] = tl[j * TW + lw.off[i]];
            typedef __attribute__((address_space(3))) const uint64_t* u64_t;
            const uint16_t* p0 = ab + (u0 ^ (ls * 32));       // unit u ^ c moves with the step's two bits
            const uint16_t* p1 = ab + (u1 ^ (ls * 32));
            f16x8 av[MG];
#pragma unroll
            for (int g = 0; g < MG; ++g) {
                const uint64_t x0 = *(u64_t)(p0 + g * 16 * GP_AROW), x1 = *(u64_t)(p1 + g * 16 * GP_AROW);
                const u32x4 t = {(uint32_t)x0, (uint32_t)(x0 >> 32), (uint32_t)x1, (uint32_t)(x1 >> 32)};
                av[g] = __builtin_bit_cast(f16x8, t);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f16x8 b = decode_b<CB, K2>(w[j], lp);
#pragma unroll
                for (int g = 0; g < MG; ++g)
                    acc[j][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[g], b, acc[j][g], 0, 0, 0);
            }
            if (--left == 0) {                                // the split's last step
                left = a.split_steps;
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int g = 0; g < MG; ++g)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            tot[j][g][i] += acc[j][g][i] * scale;
                            acc[j][g][i] = 0.f;
                        }
            }
        }
    }
    // the program's sums through shared memory, then one member row a 32-lane half
    __syncthreads();
    float* red = reinterpret_cast<float*>(smem);
    store_partials<MG>(red, nrows, tot);
    __syncthreads();
    float* Zm = a.Z + (size_t)mat * a.P * a.N + nt0 * 16 + 4 * l32;
    for (int m = wave * 2 + half; m < nrows; m += 2 * GP_WAVES)
        *reinterpret_cast<float4*>(Zm + (size_t)rows_sh[m] * a.N) = *reinterpret_cast<const float4*>(red + m * 128 + 4 * l32);
}

template <int TR>
__global__ __launch_bounds__(GP_WAVES * 64) __attribute__((amdgpu_waves_per_eu(TR == 64 ? 3 : 4))) void
grouped_prompt_kernel(GroupedPromptArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int rows_sh[TR];
    __shared__ int nrows_sh;
    // a grid smaller than the list (a caller that sized the launch for fewer picks or members than the list was given)
    // would leave listed tiles' partials stale: say so in the status word
    const int bx = blockIdx.x, by = blockIdx.y, mat = blockIdx.z;
    if (bx == 0 && threadIdx.x == 0 && a.tiles[0] > (int)gridDim.x)
        __hip_atomic_fetch_or(&g_moe_prompt_status, ESP_STATUS_TILE_LIST, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (bx >= a.tiles[0]) return;                            // workgroup-uniform
    const int ent = a.tiles[1 + bx], u = ent >> 16, mtile = ent & 0xFFFF;
    const int cnt = a.ucount[0], e = a.uids[u];
    if (threadIdx.x < 64) {
        const int m = threadIdx.x, mm = mtile * TR + m;
        const int code = m < TR && mm < a.maxm ? a.members[(size_t)u * a.maxm + mm] : -1;
        const int rp = code >= 0 ? (code >> 5) * a.slots + (code & 31) : -1;
        if (m < TR) rows_sh[m] = rp;
        const uint64_t valid = __ballot(rp >= 0);            // members come first, -1 padded
        if (m == 0) nrows_sh = __builtin_popcountll(valid);
    }
    if (u >= cnt) return;                                    // workgroup-uniform
    const uint32_t* T = reinterpret_cast<const uint32_t*>(mat ? a.TP[1][e] : a.TP[0][e]);
    const uint16_t* X = mat ? a.X[1] : a.X[0];
    const int k2 = mat ? a.B[1][e] : a.B[0][e], cb = mat ? a.C[1][e] : a.C[0][e];
    __syncthreads();
    const int nrows = __builtin_amdgcn_readfirstlane(nrows_sh);
    if (nrows == 0) return;
    // as esp_grouped: no copy for an expert with no kernel or outside the stages' range; its sums become NaN
    if (!supported(cb, k2) || k2 < a.lo || k2 > a.hi) {
        if (threadIdx.x == 0)
            __hip_atomic_fetch_or(&g_moe_prompt_status, supported(cb, k2) ? ESP_STATUS_WIDTH_RANGE : ESP_STATUS_NO_KERNEL,
                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int l32 = threadIdx.x & 31, hw = threadIdx.x >> 5;
        const float qn = __builtin_nanf("");
        for (int m = hw; m < nrows; m += 2 * GP_WAVES)
            *reinterpret_cast<float4*>(a.Z + ((size_t)mat * a.P + rows_sh[m]) * a.N + by * 128 + 4 * l32) =
                make_float4(qn, qn, qn, qn);
        return;
    }
    switch (cb * 32 + k2) {
#define ESP_GP_CASE(CB_, K2_)                                                                                  \
    case CB_ * 32 + K2_:                                                                                       \
        if (nrows <= 16)                                                                                       \
            grouped_prompt_body<gemm_cb(CB_), K2_, 1, TR>(a, T, X, rows_sh, nrows, mat, gemm_scale(CB_), smem, by);    \
        else if (TR == 32 || nrows <= 32)                                                                      \
            grouped_prompt_body<gemm_cb(CB_), K2_, 2, TR>(a, T, X, rows_sh, nrows, mat, gemm_scale(CB_), smem, by);    \
        else                                                                                                   \
            grouped_prompt_body<gemm_cb(CB_), K2_, TR / 16, TR>(a, T, X, rows_sh, nrows, mat, gemm_scale(CB_), smem,   \
                                                                by);                                           \
        break;
        ESP_CASES(ESP_GP_CASE)
#undef ESP_GP_CASE
        default:
            break;
    }
}

template <int TR>
static int launch_grouped_prompt(const GroupedPromptArgs& a, dim3 grid, int hi, hipStream_t st) {
    const size_t stage = 2 * (size_t)gp_buf_bytes(hi, TR), red = (size_t)TR * 128 * 4, smem = stage > red ? stage : red;
    if (smem > 64 * 1024 && hipFuncSetAttribute((const void*)grouped_prompt_kernel<TR>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess)
        return esp_host::fail(ESP_ERR_HIP, "grouped_prompt: cannot raise the shared memory limit to %zu bytes", smem);
    grouped_prompt_kernel<TR><<<grid, GP_WAVES * 64, smem, st>>>(a);
    return esp_host::launch_check("grouped_prompt");
}

}  // namespace esp

using namespace esp;

namespace esp_host {
// the prompt expert launches' device status word into *out (ORed), cleared if asked (esp_status)
int moe_prompt_status(int clear, hipStream_t st, int* out) {
    int v = 0;
    if (hipMemcpyFromSymbolAsync(&v, HIP_SYMBOL(g_moe_prompt_status), sizeof(int), 0, hipMemcpyDeviceToHost, st) !=
            hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return fail(ESP_ERR_HIP, "status: cannot read the prompt expert launches' status word");
    *out |= v;
    if (clear && v) {
        const int zero = 0;
        if (hipMemcpyToSymbolAsync(HIP_SYMBOL(g_moe_prompt_status), &zero, sizeof(int), 0, hipMemcpyHostToDevice, st) !=
                hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            return fail(ESP_ERR_HIP, "status: cannot clear the prompt expert launches' status word");
    }
    return ESP_OK;
}
}  // namespace esp_host

extern "C" int esp_grouped_prompt(const void* X0, const void* X1, const int64_t* TP0, const int64_t* TP1,
                                  const int32_t* B0, const int32_t* B1, const int32_t* C0, const int32_t* C1,
                                  const int32_t* uids, int64_t nexp_max, const int32_t* ucount, const int32_t* members,
                                  int64_t maxm, const int32_t* tiles, int64_t tile_rows, float* Z, int64_t z_numel,
                                  int64_t mats, int64_t K, int64_t N, int64_t P, int64_t SK, int64_t slots, int64_t lo,
                                  int64_t hi, void* stream) {
    ESP_REQUIRE(X0 && X1 && TP0 && TP1 && B0 && B1 && C0 && C1 && uids && ucount && members && tiles && Z,
                "grouped_prompt: null pointer");
    ESP_REQUIRE(mats == 1 || mats == 2, "mats must be 1 or 2");
    ESP_REQUIRE(SK >= 1 && K > 0 && N > 0 && K % 128 == 0 && K % (32 * SK) == 0 && N % 128 == 0,
                "grouped_prompt: K and N multiples of 128, K in SK equal splits of whole 32-k steps");
    ESP_REQUIRE(P >= 1 && z_numel >= mats * P * N, "Z too small");
    ESP_REQUIRE(P * K < (int64_t(1) << 31), "grouped_prompt: P * K below 2^31");
    ESP_REQUIRE(maxm >= 1 && maxm <= 65536, "members a row of the table: 1 to 65536");
    ESP_REQUIRE(slots >= 1 && slots <= 32, "at most 32 slots a row");
    ESP_REQUIRE(lo >= 2 && hi <= 16 && lo <= hi, "K2 range must lie in [2, 16]");
    ESP_REQUIRE(tile_rows == 32 || tile_rows == 64, "grouped_prompt: tiles of 32 or 64 members");
    ESP_REQUIRE(nexp_max < 65536 && mats * N / 128 <= 65535, "grouped_prompt: at most 65535 expert slots");
    ESP_REQUIRE((((uintptr_t)X0 | (uintptr_t)X1 | (uintptr_t)Z) & 15) == 0,
                "grouped_prompt: X0 / X1 and Z must be 16-byte aligned");
    if (nexp_max <= 0) return esp_host::ok();
    GroupedPromptArgs a{{static_cast<const uint16_t*>(X0), static_cast<const uint16_t*>(X1)},
                        {TP0, TP1},
                        {B0, B1},
                        {C0, C1},
                        uids,
                        ucount,
                        members,
                        tiles,
                        Z,
                        (int)K,
                        (int)N,
                        (int)P,
                        (int)maxm,
                        (int)slots,
                        (int)(K / 32 / SK),
                        (int)lo,
                        (int)hi};
    const int64_t mt = (maxm + tile_rows - 1) / tile_rows, bound = (P + tile_rows - 1) / tile_rows + nexp_max;
    const int64_t cap = nexp_max * mt < bound ? nexp_max * mt : bound;
    const dim3 grid((unsigned)cap, (unsigned)(N / 128), (unsigned)mats);
    hipStream_t st = (hipStream_t)stream;
    return tile_rows == 64 ? launch_grouped_prompt<64>(a, grid, (int)hi, st)
                           : launch_grouped_prompt<32>(a, grid, (int)hi, st);
}
