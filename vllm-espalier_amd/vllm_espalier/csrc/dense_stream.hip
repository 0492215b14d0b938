// esp_dense_stream: a wide dense layer (an LM head) over a few rows, its column blocks cut into equal shares for
// workgroups that fill the device once, with the bits of esp_dense at one K split and 8 waves.
//
// As one workgroup a column block, 1187 blocks on 512 resident workgroups are 2.3 rounds, each with a start of its own
// (arguments, the rows' rotation, the first copies' latency). Here a workgroup rotates the rows once and walks its share of
// the (block, stage) sequence with the copies running ahead across blocks. A share may begin and end inside a block: a
// workgroup first runs the block that it begins at its share's end and hands its accumulators on (exact fp32, so the next
// workgroup's MFMAs continue the chain of sums where it broke off), then its whole blocks, and last the block that its
// predecessor began, whose accumulators are there by then.
//
// No result depends on that order in time. A workgroup whose predecessor's sums stay away past a.wait (its XCD held by
// another stream, a time slice of another process) gives up on them and runs the block from its first stage: the same sums
// in the same order, at most a block's work again. The buffer is all-ones again when the launch ends, whichever of the two
// comes last. Wave w of both holds the same KiB of the sums, with a flag word of its own:
//   the predecessor   stores its KiB, waits until the stores are done, then reads the flag; if the flag is taken (0) it
//                     puts the all-ones back over the KiB and the flag;
//   the successor     takes the flag, waits until that store is done, then looks once more: bytes that are there by now it
//                     puts back to all-ones; if all of them are there, the flag too.
// Bytes that the successor does not see are stored after the flag was taken, so the predecessor sees the flag taken. Bytes
// that it sees may be put back twice.
#include "dense.hpp"

namespace esp {

struct StreamArgs {
    const uint32_t* T;
    const uint16_t* suh;
    const uint16_t* svh;
    float scale;
    const void* x;
    int x_dtype, x_stride;
    void* y;
    int y_dtype, y_stride;                // y at the matrix's first column
    float* part;                          // [workgroups][2][M][128], then a line of flags a workgroup: all-ones between launches
    int64_t wait;                         // clock ticks (10 ns) before a workgroup gives up on its predecessor's sums
    int M, K, NB, xs_stride;
    const uint16_t* nh;                   // the rows are RMSNorm(nh + nd1 + nd2) * nw, as esp_dense_rmsnorm's
    const uint16_t* nd1;
    const uint16_t* nd2;
    const uint16_t* nw;
    uint16_t* nh_out;
    float neps;
};

constexpr int DS_WAVES = 8, DS_KW = 2;    // waves (4 column pairs x 2 k slots)
constexpr int DS_STEPS = 8;               // 32-k steps a stage
constexpr int DS_MAX_ROWS = 6;
__host__ __device__ constexpr int ds_stage_bytes(int k2) { return DS_STEPS * 2 * 32 * k2 * 4; }

// The (block, stage of it) pairs of a workgroup's share in the order it runs them; phase 0: the block it begins last, 1: its
// whole blocks, 2: the block that its predecessor began
struct StreamSeq {
    int b, t, left, phase;
    int b0, nB, bC, tC, nC, SS;
    __device__ __forceinline__ StreamSeq(unsigned g0, unsigned g1, int ss) : SS(ss) {
        const int first = (int)(g0 / (unsigned)ss), last = (int)(g1 / (unsigned)ss), rest = (int)g0 - first * ss;
        b0 = rest ? first + 1 : first;
        nB = (last - b0) * ss;
        bC = first;
        tC = rest;
        nC = rest ? ss - rest : 0;
        b = last;
        t = 0;
        left = (int)g1 - last * ss;
        phase = 0;
        settle();
    }
    __device__ __forceinline__ void settle() {                 // past empty phases
        if (left == 0 && phase == 0) {
            phase = 1;
            b = b0;
            t = 0;
            left = nB;
        }
        if (left == 0 && phase == 1) {
            phase = 2;
            b = bC;
            t = tC;
            left = nC;
        }
    }
    __device__ __forceinline__ void next() {
        ++t;
        if (--left == 0) {
            settle();
        } else if (t == SS) {
            t = 0;
            ++b;
        }
    }
};

// Bound by issue (6.5 lane operations a weight; 2048 -> 151936 at 6 bits, one row: 75.3 us as a workgroup a block, 65.5 here,
// of which reading a step's words ahead is 5; three stages in shared memory instead of two: 71.3 against 69.6 before that).
template <int CB, int K2>
__global__ __launch_bounds__(DS_WAVES * 64, 4) void dense_stream_kernel(StreamArgs a) {
    constexpr int TW = 4 * K2, ROW_WORDS = 8 * TW, UPR = 2 * TW, UNITS = 2 * DS_STEPS * UPR;
    constexpr int UPT = (UNITS + DS_WAVES * 64 - 1) / (DS_WAVES * 64), STAGE_WORDS = ds_stage_bytes(K2) / 4;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float npart[DS_WAVES], ninv[2];
    __shared__ int late;                                       // the predecessor's sums stay away
    uint32_t* const stage = reinterpret_cast<uint32_t*>(smem);
    uint16_t* const xs = reinterpret_cast<uint16_t*>(smem + 2 * ds_stage_bytes(K2));
    float* const red = reinterpret_cast<float*>(smem + 2 * ds_stage_bytes(K2) + (size_t)a.M * a.xs_stride * 2);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l32 = lane & 31, half = lane >> 5, c = lane & 15, G = lane >> 4, pair = wave & 3, kw = wave >> 2;
    const int M = a.M, SS = a.K / (32 * DS_STEPS), NTILES = a.NB * 8, wg = (int)blockIdx.x;
    const unsigned NS = (unsigned)(a.NB * SS);                    // at most 2^18 stages (K * N <= 2^33), 2^12 workgroups
    const unsigned g0 = NS * (unsigned)wg / gridDim.x, g1 = NS * (unsigned)(wg + 1) / gridDim.x;
    int t_off[UPT];
#pragma unroll
    for (int i = 0; i < UPT; ++i) {
        const int u = (wave + i * DS_WAVES) * 64 + lane, r = u / UPR;
        t_off[i] = r * NTILES * TW + (u - r * UPR) * 4;
    }
    if (threadIdx.x == 0) late = 0;
    StreamSeq ahead(g0, g1, SS), cur = ahead;
    auto issue = [&](int buf) __attribute__((always_inline)) {
        const uint32_t* src = a.T + ((size_t)ahead.t * 2 * DS_STEPS * NTILES + (size_t)ahead.b * 8) * TW;
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int u0 = (wave + i * DS_WAVES) * 64;
            if (UNITS % (DS_WAVES * 64) == 0 || u0 < UNITS)             // UNITS is a multiple of 64
                __builtin_amdgcn_global_load_lds((global_void_ptr)(src + t_off[i]),
                                                 (lds_void_ptr)(stage + buf * STAGE_WORDS + u0 * 4), 16, 0, CPOL_NT);
        }
        ahead.next();
    };
    int n = (int)(g1 - g0);
    issue(0);
    // the rows, rotated, in shared memory (dense_program's arithmetic)
    const int chunks = a.K >> 7;
    if (a.nh != nullptr) {
        const bool bf = a.x_dtype == BF16;
        uint4 zq[NORM_CHUNKS];
        norm_rows_inv(a.nh, a.nd1, a.nd2, a.x_stride, M, a.K, a.neps, bf, npart, ninv, zq, xs, a.xs_stride, 0, a.K);
        if (wg == 0) norm_rows_store(zq, M, a.K, a.x_stride, a.nh_out);
        for (int idx = wave * 2 + half; idx < M * chunks; idx += 2 * DS_WAVES) {
            const int r = idx / chunks, kb = (idx - r * chunks) * 128 + 4 * l32;
            uint16_t* xp = xs + (size_t)r * a.xs_stride + kb;
            const RotIn in = norm_rot_in(*reinterpret_cast<const uint2*>(xp), *reinterpret_cast<const uint2*>(a.nw + kb),
                                         *reinterpret_cast<const uint2*>(a.suh + kb), ninv[r], bf);
            *reinterpret_cast<uint2*>(xp) = rot128_apply(in, a.x_dtype, l32);
        }
    } else {
        for (int idx = wave * 2 + half; idx < M * chunks; idx += 2 * DS_WAVES) {
            const int r = idx / chunks, kb = (idx - r * chunks) * 128;
            *reinterpret_cast<uint2*>(xs + (size_t)r * a.xs_stride + kb + 4 * l32) =
                rot128(a.x, a.x_dtype, (size_t)r * a.x_stride + kb, a.suh + kb, l32);
        }
    }
    RowsA<1, true> al;
    al.set(0, xs + (size_t)(c < M ? c : 0) * a.xs_stride + 16 * (G >> 1) + 4 * (G & 1));     // a row past M reads row 0
    al.kbase = 0;

    const LanePlan<K2> lp(lane);
    const LdsWords<K2> lw(lp);
    const int lane_base = ((G >> 1) * 8 + 2 * pair) * TW;
    f32x4 acc[2][1] = {{f32x4{0.f, 0.f, 0.f, 0.f}}, {f32x4{0.f, 0.f, 0.f, 0.f}}};
    // every wave's sums of rows < M to red [k slot][M][128], visible to the workgroup
    auto to_red = [&]() __attribute__((always_inline)) {
        store_partials<1>(red, M, acc);
        lds_barrier();
        acc[0][0] = acc[1][0] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    const DevBuf pb(a.part);
    const int piece = 2 * M * 128, mine = (int)threadIdx.x * 4;           // a KiB each of waves 0 .. M - 1
    const bool carries = wave < M;
    constexpr uint32_t empty = 0xFFFFFFFFu;
    const float4 ones = make_float4(__uint_as_float(empty), __uint_as_float(empty), __uint_as_float(empty),
                                    __uint_as_float(empty));
    auto landed = [&](const float4& u) __attribute__((always_inline)) {
        return __float_as_uint(u.x) != empty && __float_as_uint(u.y) != empty && __float_as_uint(u.z) != empty &&
               __float_as_uint(u.w) != empty;
    };
    auto flag = [&](int w) __attribute__((always_inline)) {               // this wave's of workgroup w
        return reinterpret_cast<int*>(a.part + (size_t)gridDim.x * piece) + (size_t)w * CNT_STRIDE + wave;
    };
    bool begun = false, handed = false;                       // the predecessor's sums are taken over; the own ones stored
    int told = (int)empty;                                    // and the flag read then
    for (int q = 0; q < n; ++q) {
        wait_stage();                                         // the stage landed; every wave is done with the other buffer
        if (q + 1 < n) issue((q + 1) & 1);
        if (handed) {                                         // the stores are done (wait_stage)
            handed = false;
            told = load_dev(flag(wg));
        }
        if (cur.phase == 2 && !begun) {
            begun = true;
            float* p = a.part + (size_t)(wg - 1) * piece + mine;
            bool here = true;
            if (carries) {
                float4 u = pb.load4(p);
                const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
                here = a.wait >= 0 && landed(u);
                while (!here && (int64_t)(__builtin_amdgcn_s_memrealtime() - t0) < a.wait) {
                    __builtin_amdgcn_s_sleep(1);
                    u = pb.load4(p);
                    here = landed(u);
                }
                if (here) {
                    *reinterpret_cast<float4*>(red + mine) = u;
                    pb.store4(p, ones);
                } else {
                    late = 1;
                }
            }
            lds_barrier();
            if (__builtin_amdgcn_readfirstlane(late)) {
                if (carries && lane == 0) store_dev(flag(wg - 1), 0);
                wait_stage();                                 // the flag is taken, and the copies in flight landed
                if (!here && landed(pb.load4(p))) {
                    pb.store4(p, ones);
                    here = true;
                }
                const bool all = __ballot(!here) == 0;
                if (carries && all && lane == 0) store_dev(flag(wg - 1), (int)empty);
                // the block from its first stage; the stages in shared memory are brought again after the ones before them
                cur.t = 0;
                cur.left += cur.tC;
                n += cur.tC;
                ahead = cur;
                issue(q & 1);
                wait_stage();
                if (q + 1 < n) issue((q + 1) & 1);
            } else {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (4 * G + r < M) acc[j][0][r] = red[((size_t)kw * M + 4 * G + r) * 128 + 32 * pair + 16 * j + c];
            }
        }
        const uint32_t* bb = stage + (q & 1) * STAGE_WORDS + lane_base;
        // a step's words and rows are read while the step before is decoded
        uint32_t w[2][2][6];
        f16x8 av[2];
        auto read = [&](int i) __attribute__((always_inline)) {
            const uint32_t* tl = bb + (2 * i + kw) * 2 * ROW_WORDS;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int u = 0; u < 6; ++u) w[i & 1][j][u] = tl[j * TW + lw.off[u]];
            al(0, 32 * (cur.t * DS_STEPS + 2 * i + kw), av[i & 1]);
        };
        read(0);
#pragma unroll
        for (int i = 0; i < DS_STEPS / DS_KW; ++i) {
            if (i + 1 < DS_STEPS / DS_KW) read(i + 1);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[i & 1], decode_b<CB, K2>(w[i & 1][j], lp),
                                                                   acc[j][0], 0, 0, 0);
        }
        if (cur.phase == 0) {
            if (cur.left == 1) {                              // the share's last stage of the block: hand the sums on
                to_red();
                handed = carries;
                if (carries)
                    pb.store4(a.part + (size_t)wg * piece + mine, *reinterpret_cast<const float4*>(red + mine));
            }
        } else if (cur.t == SS - 1) {                         // the block's sums are whole: slot 0's plus slot 1's
            to_red();
            const int r = wave * 2 + half;
            if (r < M) {
                const int col = cur.b * 128 + 4 * l32;
                float4 s = *reinterpret_cast<const float4*>(red + (size_t)r * 128 + 4 * l32);
                const float4 u = *reinterpret_cast<const float4*>(red + ((size_t)M + r) * 128 + 4 * l32);
                s.x += u.x; s.y += u.y; s.z += u.z; s.w += u.w;
                float v[4] = {s.x, s.y, s.z, s.w};
                finish(v, l32, *reinterpret_cast<const uint2*>(a.svh + col), a.scale);
                store4(a.y, a.y_dtype, (size_t)r * a.y_stride + col, v);
            }
        }
        cur.next();
    }
    // a share is at least a block, so a stage followed the one that handed the sums on: the flag was read
    if (told != (int)empty) {
        pb.store4(a.part + (size_t)wg * piece + mine, ones);
        if (lane == 0) store_dev(flag(wg), (int)empty);
    }
}

}  // namespace esp

using namespace esp;

extern "C" int esp_dense_stream(const void* x, int x_dtype, int64_t x_stride, int64_t M, int64_t K, const void* trellis,
                                const void* suh, const void* svh, int64_t N, void* y, int y_dtype, int64_t y_stride,
                                const void* d1, const void* d2, const void* norm_w, double eps, void* h_out, float* part,
                                int64_t part_numel, int64_t wait_us, int64_t k2, int64_t cb, void* stream) {
    ESP_REQUIRE(x && trellis && suh && svh && y && part, "dense_stream: null pointer");
    ESP_REQUIRE(M >= 1 && M <= DS_MAX_ROWS, "dense_stream: 1 to 6 rows");
    ESP_REQUIRE(K > 0 && K % (32 * DS_STEPS) == 0 && K <= 65536 && N > 0 && N % 128 == 0 && N < (int64_t(1) << 24) &&
                    K * N <= (int64_t(1) << 33),
                "dense_stream: K a multiple of 256, N of 128");
    ESP_REQUIRE(x_dtype >= 0 && x_dtype <= 2 && y_dtype >= 0 && y_dtype <= 2, "dense_stream: x / y dtype");
    ESP_REQUIRE(x_stride >= K && y_stride >= N && esp_host::strides_fit(M, x_stride, y_stride),
                "dense_stream: x / y row stride");
    ESP_REQUIRE(((uintptr_t)x % (x_dtype == ESP_F32 ? 16 : 8)) == 0 && x_stride % 4 == 0 &&
                    ((uintptr_t)y % (y_dtype == ESP_F32 ? 16 : 8)) == 0 && y_stride % 4 == 0,
                "dense_stream: x / y 8-byte aligned (16 for fp32) with row strides a multiple of 4 elements");
    ESP_REQUIRE((((uintptr_t)trellis | (uintptr_t)part) & 15) == 0 && (((uintptr_t)suh | (uintptr_t)svh) & 7) == 0,
                "dense_stream: trellis and part 16-byte aligned, suh / svh 8-byte aligned");
    if (!supported((int)cb, (int)k2))
        return esp_host::fail(ESP_ERR_UNSUPPORTED, "unsupported codebook/width: cb=%lld k2=%lld", (long long)cb,
                              (long long)k2);
    if (norm_w) {
        ESP_REQUIRE(h_out && x_dtype != ESP_F32 && M <= 2, "dense_stream: a norm takes bf16 or fp16 rows, at most 2");
        ESP_REQUIRE(K <= NORM_MAX_D && x_stride % 8 == 0 &&
                        ((uintptr_t)x | (uintptr_t)d1 | (uintptr_t)d2 | (uintptr_t)norm_w | (uintptr_t)h_out) % 16 == 0,
                    "dense_stream: norm rows of at most 8192, 16-byte aligned");
    }
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return esp_host::fail(ESP_ERR_HIP, "dense_stream: cannot read the device's compute units");
    StreamArgs a{};
    a.T = static_cast<const uint32_t*>(trellis);
    a.suh = static_cast<const uint16_t*>(suh);
    a.svh = static_cast<const uint16_t*>(svh);
    a.scale = gemm_scale((int)cb);
    a.x = x;
    a.x_dtype = x_dtype;
    a.x_stride = (int)x_stride;
    a.y = y;
    a.y_dtype = y_dtype;
    a.y_stride = (int)y_stride;
    a.part = part;
    a.wait = wait_us < 0 ? -1 : wait_us < 1000000 ? wait_us * 100 : 100000000;       // s_memrealtime counts at 100 MHz
    a.M = (int)M;
    a.K = (int)K;
    a.NB = (int)(N / 128);
    a.xs_stride = (int)K + 8;                                  // pad rows across the LDS banks
    if (norm_w) {
        a.nh = static_cast<const uint16_t*>(x);
        a.nd1 = static_cast<const uint16_t*>(d1);
        a.nd2 = static_cast<const uint16_t*>(d2);
        a.nw = static_cast<const uint16_t*>(norm_w);
        a.nh_out = static_cast<uint16_t*>(h_out);
        a.neps = (float)eps;
    }
    const size_t smem = 2 * (size_t)ds_stage_bytes((int)k2) + (size_t)M * a.xs_stride * 2 + 2 * (size_t)M * 512;
    ESP_REQUIRE(smem <= 160 * 1024 - 1024, "dense_stream: shared memory exceeds 160 KiB");
    // every share at least a block, so a block spans two workgroups at most
    const int per_cu = smem <= 80 * 1024 - 512 ? 2 : 1;
    const int wgs = per_cu * cus < a.NB ? per_cu * cus : a.NB;
    ESP_REQUIRE(wgs < 4096, "dense_stream: at most 4095 workgroups");
    ESP_REQUIRE(part_numel >= (int64_t)wgs * (2 * M * 128 + CNT_STRIDE),
                "dense_stream: part needs 256 floats a row and 32 more for each workgroup (two a compute unit, at most one "
                "a 128-column block)");
    hipStream_t st = (hipStream_t)stream;
    switch (cb * 32 + k2) {
#define ESP_STREAM_CASE(CB_, K2_)                                                                                       \
    case CB_ * 32 + K2_: {                                                                                              \
        auto kern = dense_stream_kernel<gemm_cb(CB_), K2_>;                                                             \
        if (smem > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,      \
                                                    (int)smem) != hipSuccess)                                           \
            return esp_host::fail(ESP_ERR_HIP, "dense_stream: cannot raise the shared memory limit to %zu bytes", smem); \
        kern<<<(unsigned)wgs, DS_WAVES * 64, smem, st>>>(a);                                                            \
        break;                                                                                                          \
    }
        ESP_CASES(ESP_STREAM_CASE)
#undef ESP_STREAM_CASE
    }
    return esp_host::launch_check("dense_stream");
}
