// esp_dense_prompt: a dense layer over a prompt on gfx950 with every weight decoded once, whatever the number of rows,
// and the bits of a launch that splits K: esp_dense (k slots = W / 4) or esp_dense_tile (two k slots).
//
// Two launches. (1) prompt_prep_kernel rotates every row once a matrix (xh, esp_dense_tile's A-fragment order) and
// decodes every weight to fp16 in MFMA B-fragment order: wf[128-column block][32-k step][8 n tiles][64 lanes][8 halves].
// (2) prompt_gemm_kernel is an fp16 GEMM on those fragments: no decode, no shuffles, every LDS read a conflict-free
// 16 bytes a lane.
//
// The sums keep the order of the launch they stand for: of a K split's steps, slot j takes steps j, j + KW, ... in
// order; the slots are added in order, then the splits in order (z and tot below). All of it stays in registers, where
// the split launches exchange fp32 partials between workgroups; a row's bits are the same either way, for any T and any
// place in the prompt. The preparation stores the steps in that order (StepOrder), so the GEMM walks them in a line and
// only counts down to each slot's end.
#include <type_traits>

#include "tile.hpp"

namespace esp {

// The order of the steps: K / 32 = SQ * SK + SR steps, split s takes the next SQ + (s < SR) (at least KW of them), and
// inside a split slot after slot takes its steps, every KW-th one (KW = 1 << kw_log)
struct StepOrder {
    int SQ, SR, kw_log;
    uint32_t by_long, by_short;              // 2^32 / (SQ + 1) and / SQ, rounded up: exact quotients of steps by mulhi
    __device__ __forceinline__ int slot_steps(int ns, int slot) const { return (ns - slot + (1 << kw_log) - 1) >> kw_log; }
    // the place of step st in the order
    __device__ __forceinline__ int place(int st) const {
        const int longer = SR * (SQ + 1);                       // the steps of the splits that take one more
        const int ns = st < longer ? SQ + 1 : SQ;
        const int s0 = st < longer ? (int)((uint64_t)st * by_long >> 32) * ns
                                   : SQ == 1 ? st
                                   : longer + (int)((uint64_t)(st - longer) * by_short >> 32) * ns;
        const int in = st - s0, slot = in & ((1 << kw_log) - 1);
        int before = 0;
        for (int j = 0; j < slot; ++j) before += slot_steps(ns, j);
        return s0 + before + (in >> kw_log);
    }
};

// ---- preparation: rotated rows and decoded weights
// Rotated rows: 8 lanes take one (matrix, row, 128-chunk of K) of unit = ((matrix * RG + row group) * K / 128 + chunk) *
// 16 + row of the group (rows past T are zero): a lane's 16 elements are one k-tile's, which two lanes of the chunk's
// step (l8 / 2) hold in halves, 16 bytes each. place(step) is the step's block among the (matrix, row group)'s in xh.
template <typename PLACE>
__device__ __forceinline__ void tile_rot_unit(unsigned unit, const void* __restrict__ x, int x_dtype, int x_stride, int T,
                                              int K, bool wide, const uint16_t* suh0, const uint16_t* suh1,
                                              const uint16_t* suh2, const uint16_t* suh3, uint16_t* __restrict__ xh,
                                              int RG, const PLACE& place) {
    const int lane = threadIdx.x & 63, l8 = lane & 7, nb = K >> 7;
    const int rr = (int)(unit & 15), ch = (int)((unit >> 4) % nb);
    const int rg = (int)((unit >> 4) / nb % RG), s = (int)((unit >> 4) / nb / RG), r = rg * 16 + rr;
    const uint16_t* suh = s == 0 ? suh0 : s == 1 ? suh1 : s == 2 ? suh2 : suh3;
    uint32_t w[8];
    // every lane of the 8 takes the same branch
    if (r < T) {
        rot128_16<16>(x, x_dtype, (size_t)r * x_stride + ch * 128, suh + ch * 128, wide, lane, w);
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = 0u;
    }
    uint16_t* dst = xh + (((size_t)s * RG + rg) * (K >> 5) + place(ch * 4 + (l8 >> 1))) * TILE_FRAG;
    const int G = 2 * (l8 & 1);                      // the fragment lanes rr + 16 G (k 0-3, 8-11) and G + 1 (4-7, 12-15)
    *reinterpret_cast<uint4*>(dst + (rr + 16 * G) * 8) = make_uint4(w[0], w[1], w[4], w[5]);
    *reinterpret_cast<uint4*>(dst + (rr + 16 * (G + 1)) * 8) = make_uint4(w[2], w[3], w[6], w[7]);
}

constexpr int ROT_UNITS = 32;                        // units a workgroup of 256

// whether rot128_16 may read x and the signs 16 bytes at a time
inline bool rot_wide(const void* x, int64_t x_stride, const uint16_t* const* suh, int n) {
    bool wide = (uintptr_t)x % 16 == 0 && x_stride % 8 == 0;
    for (int i = 0; i < n; ++i) wide = wide && (uintptr_t)suh[i] % 16 == 0;
    return wide;
}

struct PrepArgs {
    StepOrder order;
    const uint32_t* T[MAX_SHARDS];
    const uint16_t* suh[MAX_SHARDS];
    int nb0[MAX_SHARDS], nb[MAX_SHARDS];     // first 128-column block in the launch, blocks
    int n;
    const void* x;
    int x_dtype, x_stride;
    int rows, K, RG, NBT;
    uint16_t* xh;
    uint16_t* wf;
    bool wide;                                // rot128_16's
    unsigned rot_units, rot_wgs;              // rows to rotate, and the workgroups that do; the others decode
};

constexpr int PREP_WAVES = 4;                 // waves of a decoding workgroup, a 32-k step each

// A decoding wave takes one (column block, step): its 16 trellis tiles come to shared memory in whole KiBs, then each
// lane decodes its B operand of the 8 n tiles and stores it as 16 bytes, a wave a KiB.
template <int CB, int K2>
__global__ __launch_bounds__(256) void prompt_prep_kernel(PrepArgs a) {
    __shared__ __align__(16) uint32_t smem[K2 * PREP_WAVES * 64];
    if (blockIdx.x < a.rot_wgs) {
        const unsigned unit = blockIdx.x * ROT_UNITS + (threadIdx.x >> 3);
        if (unit < a.rot_units)
            tile_rot_unit(unit, a.x, a.x_dtype, a.x_stride, a.rows, a.K, a.wide, a.suh[0], a.suh[1], a.suh[2], a.suh[3],
                          a.xh, a.RG, [&](int st) { return a.order.place(st); });
        return;
    }
    constexpr int TW = 4 * K2, ROW = 8 * TW;             // words of a tile, of a k tile of the block
    const int steps = a.K >> 5, groups = steps / PREP_WAVES;                  // K % 128 == 0
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, G = lane >> 4;
    const int unit = (int)(blockIdx.x - a.rot_wgs), nbg = unit / groups, step = (unit - nbg * groups) * PREP_WAVES + wave;
    const uint32_t* T = a.T[0];
    int nb0 = a.nb0[0], nb = a.nb[0];
#pragma unroll
    for (int i = 1; i < MAX_SHARDS; ++i)
        if (i < a.n && nbg >= a.nb0[i]) {
            T = a.T[i];
            nb0 = a.nb0[i];
            nb = a.nb[i];
        }
    const uint32_t* src = T + ((size_t)(2 * step) * (nb * 8) + (nbg - nb0) * 8) * TW;
    uint32_t* words = smem + wave * 2 * ROW;
    constexpr int UNITS = 2 * ROW / 4;                    // 16-byte units of the step
#pragma unroll
    for (int u0 = 0; u0 < UNITS; u0 += 64) {
        const int u = u0 + lane;
        if (UNITS % 64 == 0 || u < UNITS) {
            const int r = u / (ROW / 4), w = (u - r * (ROW / 4)) * 4;
            __builtin_amdgcn_global_load_lds((global_void_ptr)(src + (size_t)r * (nb * 8) * TW + w),
                                             (lds_void_ptr)(words + u0 * 4), 16, 0, CPOL_NT);
        }
    }
    const LanePlan<K2> lp(lane);
    const LdsWords<K2> off(lp);
    uint4* dst = reinterpret_cast<uint4*>(a.wf + ((size_t)nbg * steps + a.order.place(step)) * 8 * TILE_FRAG) + lane;
    wait_stage();
    const uint32_t* tl = words + (G >> 1) * ROW;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        uint32_t w[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) w[i] = tl[t * TW + off.off[i]];
        const u32x4 v = decode_words<CB, K2>(w, lp);
        dst[t * 64] = make_uint4(v.x, v.y, v.z, v.w);
    }
}

// ---- the GEMM
struct PromptArgs {
    const uint16_t* svh[MAX_SHARDS];
    int nb0[MAX_SHARDS], col0[MAX_SHARDS];
    int n;
    float scale;                 // factor of the decoded form's sums (gemm_scale)
    const uint16_t* xh;          // [n][RG][K / 32][64][8]
    const uint16_t* wf;          // [NBT][K / 32][8][64][8]
    void* y;
    int y_dtype, y_stride;
    int T, K, SK, NBT, RG, tiles_m, chunk;
    StepOrder order;
};

constexpr int PG_WAVES = 4;
constexpr int PG_RG = 4;                      // row groups of 16 a workgroup, all of them each wave's
constexpr int PG_NR = 2;                      // n tiles a wave
constexpr int PG_ROWS = PG_RG * 16;
constexpr int PG_UNITS = PG_RG + 8;           // KiB fragments a step: the tile's A blocks and the block's B tiles
constexpr int PG_LPW = PG_UNITS / PG_WAVES;   // a wave's copies of them
constexpr int PG_DEPTH = 4;                   // steps in shared memory
constexpr int PG_BUF = PG_UNITS * TILE_FRAG;  // halves a step
constexpr int PG_SMEM = PG_DEPTH * PG_BUF * 2;
static_assert(PG_UNITS % PG_WAVES == 0, "every wave issues the same copies");
static_assert(PG_SMEM >= PG_ROWS * RED_STRIDE * 4, "the tile's sums fit");

// s_waitcnt with at most VM vector loads and no shared-memory access outstanding
template <int VM>
__device__ __forceinline__ void wait_vm_lgkm0() {
    static_assert(VM < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
}

// A workgroup is 4 waves on a tile of 64 rows and one 128-column block, a wave 32 of the columns. A step's fragments are
// brought to shared memory by global_load_lds, PG_DEPTH steps deep; a wave waits by count for its own copies of the next
// step, then one barrier makes every wave's copies visible and frees the buffer whose fragments the waves hold in
// registers, and the next step's fragments are read while this one multiplies. Every wave issues the same number of
// copies a step (row groups past the prompt and steps past the last are clamped, read and not used), so the counts hold.
//
// SPS > 0: every split is 4 slots of SPS steps (the plans of narrow layers), a loop iteration whose slots the compiler
// knows; 0: any order, counted down at run time, at the price of 20 spilled registers, which come back at each split's end:
// the wait for them there also drains the copies in flight.
//
// Bound by the shared memory: 12 KiB written and 24 KiB read a step are ~290 clocks of its bandwidth against 128 of MFMA, so
// at most 44 % of the matrix peak, of which 30 % are reached at 2048 rows of 2048 -> 5120 (58 us); the reads' latency is
// hidden by three workgroups a CU where the grid holds them. A 128-row tile halves the B reads a row, but its three sets of
// sums (slot, split, total: 192 registers) leave two waves a SIMD: 2048 x 2048 -> 5120, 94 us against 58.
template <int SPS>
__global__ __launch_bounds__(PG_WAVES * 64, 3) void prompt_gemm_kernel(PromptArgs a) {
    __shared__ __align__(16) uint16_t smem[PG_DEPTH * PG_BUF];
    // workgroups go round the XCDs: each takes a run of `chunk` tiles, ordered in groups of 8 column blocks, so an XCD's
    // tiles share rows and columns in its L2
    const int id = (int)(blockIdx.x & 7) * a.chunk + (int)(blockIdx.x >> 3);
    if (id >= a.tiles_m * a.NBT) return;
    const int per = a.tiles_m * 8, grp = id / per, gw = a.NBT - grp * 8 < 8 ? a.NBT - grp * 8 : 8;
    const int in = id - grp * per, mt = in / gw, nbg = grp * 8 + in % gw;

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int c = lane & 15, G = lane >> 4;
    int si = 0;
    const uint16_t* svh = a.svh[0];
    int nb0 = a.nb0[0], col0 = a.col0[0];
#pragma unroll
    for (int i = 1; i < MAX_SHARDS; ++i)
        if (i < a.n && nbg >= a.nb0[i]) {
            si = i;
            svh = a.svh[i];
            nb0 = a.nb0[i];
            col0 = a.col0[i];
        }
    const int ksteps = a.K >> 5, rg0 = mt * PG_RG;
    // this wave's copies of a step: units wave * PG_LPW ..., B tiles first
    const uint16_t* base[PG_LPW];
    int stride[PG_LPW];
#pragma unroll
    for (int i = 0; i < PG_LPW; ++i) {
        const int u = wave * PG_LPW + i;
        if (u < 8) {
            base[i] = a.wf + ((size_t)nbg * ksteps * 8 + u) * TILE_FRAG;
            stride[i] = 8 * TILE_FRAG;
        } else {
            const int rg = rg0 + u - 8 < a.RG ? rg0 + u - 8 : a.RG - 1;
            base[i] = a.xh + ((size_t)si * a.RG + rg) * ksteps * TILE_FRAG;
            stride[i] = TILE_FRAG;
        }
    }
    int issued = 0;                                // steps issued (clamped to the last)
    auto issue = [&](int buf) __attribute__((always_inline)) {       // the next step into buffer buf
#pragma unroll
        for (int i = 0; i < PG_LPW; ++i)
            __builtin_amdgcn_global_load_lds((global_void_ptr)(base[i] + lane * 8),
                                             (lds_void_ptr)(smem + buf * PG_BUF + (wave * PG_LPW + i) * TILE_FRAG), 16, 0, 0);
        if (++issued < ksteps)
#pragma unroll
            for (int i = 0; i < PG_LPW; ++i) base[i] += stride[i];
    };
    struct Frags {
        f16x8 b[PG_NR], a[PG_RG];
    };
    auto read = [&](int buf, Frags& f) __attribute__((always_inline)) {
        const uint16_t* p = smem + buf * PG_BUF + lane * 8;
#pragma unroll
        for (int j = 0; j < PG_NR; ++j) f.b[j] = *(lds_f16x8_ptr)(p + (wave * PG_NR + j) * TILE_FRAG);
#pragma unroll
        for (int g = 0; g < PG_RG; ++g) f.a[g] = *(lds_f16x8_ptr)(p + (8 + g) * TILE_FRAG);
    };
    auto landed = [&](auto vm) __attribute__((always_inline)) {
        wait_vm_lgkm0<decltype(vm)::value>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Sums that start at -0 take their first term's bits (-0 + v = v for every v, +0 and -0 included), so no sum's first
    // term is a case of its own
    typedef f32x4 Sums[PG_NR][PG_RG];
    Sums acc, z, tot;
    auto fill = [&](Sums& d, float v) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PG_NR; ++j)
#pragma unroll
            for (int g = 0; g < PG_RG; ++g) d[j][g] = f32x4{v, v, v, v};
    };
    auto add = [&](Sums& d, const Sums& v) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PG_NR; ++j)
#pragma unroll
            for (int g = 0; g < PG_RG; ++g) d[j][g] += v[j][g];
    };
    Frags f[2];
    auto mul = [&](Sums& d, const Frags& q, auto first) __attribute__((always_inline)) {     // d = A B, or d + A B
#pragma unroll
        for (int j = 0; j < PG_NR; ++j)
#pragma unroll
            for (int g = 0; g < PG_RG; ++g)
                d[j][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    q.a[g], q.b[j], decltype(first)::value ? f32x4{0.f, 0.f, 0.f, 0.f} : d[j][g], 0, 0, 0);
    };
    // step u's fragments are in f[u & 1] (read by every wave, its buffer free): wait for the next step's, read them, and
    // refill the buffer
    auto next = [&](int u) __attribute__((always_inline)) {
        landed(std::integral_constant<int, (PG_DEPTH - 2) * PG_LPW>{});
        read((u + 1) % PG_DEPTH, f[(u + 1) & 1]);
        issue(u % PG_DEPTH);
    };
#pragma unroll
    for (int i = 0; i < PG_DEPTH; ++i) issue(i);
    landed(std::integral_constant<int, (PG_DEPTH - 1) * PG_LPW>{});
    read(0, f[0]);
    fill(tot, -0.f);
    if constexpr (SPS > 0) {
        // splits of 4 slots of SPS steps each: a split an iteration, its slots known to the compiler
        for (int s = 0; s < a.SK; ++s) {
#pragma unroll
            for (int u = 0; u < 4 * SPS; ++u) {
                next(u);
                Sums& d = u < SPS ? z : acc;
                if (u % SPS == 0)
                    mul(d, f[u & 1], std::true_type{});
                else
                    mul(d, f[u & 1], std::false_type{});
                if (u >= SPS && u % SPS == SPS - 1) add(z, acc);
            }
            add(tot, z);
        }
    } else {
        fill(acc, 0.f);
        fill(z, -0.f);
        int slot = 0, split = 0, ns = a.order.SQ + (a.order.SR > 0), left = a.order.slot_steps(ns, 0);
        for (int i = 0; i < ksteps; i += 4) {          // K % 128 == 0
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                next(u);
                mul(acc, f[u & 1], std::false_type{});
                if (--left == 0) {                                    // the slot's last step
                    add(z, acc);
                    fill(acc, 0.f);
                    if (++slot == 1 << a.order.kw_log) {              // and the split's
                        add(tot, z);
                        fill(z, -0.f);
                        slot = 0;
                        ++split;
                        ns = a.order.SQ + (split < a.order.SR);
                    }
                    left = a.order.slot_steps(ns, slot);
                }
            }
        }
    }

    // the tile's sums through shared memory: 8 lanes a row, 16 columns a lane, for the output transform
    const int cb_local = nbg - nb0, l8 = lane & 7;
    const uint2* sp = reinterpret_cast<const uint2*>(svh + cb_local * 128 + 16 * l8);          // 8-byte aligned
    const uint2 s0 = sp[0], s1 = sp[1], s2 = sp[2], s3 = sp[3];
    const uint32_t sw[8] = {s0.x, s0.y, s1.x, s1.y, s2.x, s2.y, s3.x, s3.y};
    float* red = reinterpret_cast<float*>(smem);
    const int ycol = col0 + cb_local * 128 + 16 * l8;
    wait_vm_lgkm0<0>();                                                // every copy landed, every fragment read
    __syncthreads();
#pragma unroll
    for (int g = 0; g < PG_RG; ++g)
#pragma unroll
        for (int j = 0; j < PG_NR; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                red[(g * 16 + 4 * G + i) * RED_STRIDE + (wave * PG_NR + j) * 16 + c] = tot[j][g][i];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PG_ROWS / 32; ++q) {
        const int r = q * 32 + wave * 8 + (lane >> 3);
        float v[16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 t = *reinterpret_cast<const float4*>(red + r * RED_STRIDE + 16 * l8 + 4 * i);
            v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
        }
        fwht128_16<16>(v, lane);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            v[i] *= a.scale;
            v[i] *= HAD_SCALE * h2f((uint16_t)(sw[i >> 1] >> (16 * (i & 1))));
        }
        if (mt * PG_ROWS + r < a.T) {
            const size_t yi = (size_t)(mt * PG_ROWS + r) * a.y_stride + ycol;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float w[4] = {v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
                store4(a.y, a.y_dtype, yi + 4 * i, w);
            }
        }
    }
}

}  // namespace esp

using namespace esp;

extern "C" int esp_dense_prompt(const void* x, int x_dtype, int64_t x_stride, int64_t T, int64_t K, int64_t n_shards,
                                const void* const* trellis, const void* const* suh, const void* const* svh,
                                const int64_t* n_cols, const int64_t* col0, void* y, int y_dtype, int64_t y_stride,
                                int64_t y_cols, void* xh, int64_t xh_numel, void* wf, int64_t wf_numel, int64_t k2,
                                int64_t cb, int64_t SK, int64_t KW, void* stream) {
    ESP_REQUIRE(x && y && xh && wf && trellis && suh && svh && n_cols && col0, "dense_prompt: null pointer");
    ESP_REQUIRE(n_shards >= 1 && n_shards <= MAX_SHARDS, "dense_prompt: 1 to 4 matrices a launch");
    ESP_REQUIRE(T >= 1 && T < (int64_t(1) << 30), "dense_prompt: at least one row");
    ESP_REQUIRE(K > 0 && K % 128 == 0 && SK >= 1 && (KW == 1 || KW == 2 || KW == 4) && SK * KW <= K / 32,
                "dense_prompt: K must be a multiple of 128, with a 32-k step for each of SK * KW slots (KW 1, 2 or 4)");
    ESP_REQUIRE(x_dtype >= 0 && x_dtype <= 2 && y_dtype >= 0 && y_dtype <= 2, "dense_prompt: x / y dtype");
    ESP_REQUIRE(x_stride >= K && y_stride >= y_cols && esp_host::strides_fit(T, x_stride, y_stride),
                "dense_prompt: x / y row stride");
    ESP_REQUIRE(((uintptr_t)x % (x_dtype == ESP_F32 ? 16 : 8)) == 0 && x_stride % 4 == 0 &&
                    ((uintptr_t)y % (y_dtype == ESP_F32 ? 16 : 8)) == 0 && y_stride % 4 == 0 &&
                    ((uintptr_t)xh & 15) == 0 && ((uintptr_t)wf & 15) == 0,
                "dense_prompt: x / y 8-byte aligned (16 for fp32) with row strides a multiple of 4 elements, xh and wf "
                "16-byte aligned");
    if (!supported((int)cb, (int)k2))
        return esp_host::fail(ESP_ERR_UNSUPPORTED, "unsupported codebook/width: cb=%lld k2=%lld", (long long)cb,
                              (long long)k2);
    PrepArgs p{};
    PromptArgs a{};
    int nbt = 0;
    for (int s = 0; s < n_shards; ++s) {
        const int64_t N = n_cols[s];
        ESP_REQUIRE(N > 0 && N % 128 == 0, "dense_prompt: matrix shape");
        ESP_REQUIRE(col0[s] >= 0 && col0[s] + N <= y_cols, "dense_prompt: matrix columns past y");
        ESP_REQUIRE(trellis[s] && suh[s] && svh[s], "dense_prompt: null matrix pointer");
        ESP_REQUIRE(((uintptr_t)trellis[s] & 15) == 0 && ((uintptr_t)suh[s] & 7) == 0 && ((uintptr_t)svh[s] & 7) == 0 &&
                        col0[s] % 4 == 0,
                    "dense_prompt: trellis 16-byte aligned, suh / svh 8-byte aligned, col0 a multiple of 4");
        p.T[s] = static_cast<const uint32_t*>(trellis[s]);
        p.suh[s] = static_cast<const uint16_t*>(suh[s]);
        a.svh[s] = static_cast<const uint16_t*>(svh[s]);
        p.nb0[s] = a.nb0[s] = nbt;
        p.nb[s] = (int)(N / 128);
        a.col0[s] = (int)col0[s];
        nbt += (int)(N / 128);
    }
    const int64_t RG = (T + 15) / 16;
    ESP_REQUIRE(xh_numel >= n_shards * RG * 16 * K, "dense_prompt: xh needs n_shards * ceil(T / 16) * 16 * K halves");
    ESP_REQUIRE(wf_numel >= (int64_t)nbt * 128 * K, "dense_prompt: wf needs K * N halves");
    const int64_t rot_units = n_shards * RG * (K / 128) * 16, rot_wgs = (rot_units + ROT_UNITS - 1) / ROT_UNITS, dec_units = (int64_t)nbt * (K / 32) / PREP_WAVES;
    ESP_REQUIRE(rot_units + dec_units < (int64_t(1) << 31) && (T + PG_ROWS) / PG_ROWS * nbt < (int64_t(1) << 28),
                "dense_prompt: too many rows for one launch");
    p.n = a.n = (int)n_shards;
    p.x = x;
    p.x_dtype = x_dtype;
    p.x_stride = (int)x_stride;
    p.rows = a.T = (int)T;
    p.K = a.K = (int)K;
    p.RG = a.RG = (int)RG;
    p.NBT = a.NBT = nbt;
    p.xh = static_cast<uint16_t*>(xh);
    p.wf = static_cast<uint16_t*>(wf);
    p.rot_units = (unsigned)rot_units;
    p.rot_wgs = (unsigned)rot_wgs;
    p.wide = rot_wide(x, x_stride, p.suh, (int)n_shards);
    a.scale = gemm_scale((int)cb);
    a.xh = static_cast<const uint16_t*>(xh);
    a.wf = static_cast<const uint16_t*>(wf);
    a.y = y;
    a.y_dtype = y_dtype;
    a.y_stride = (int)y_stride;
    a.SK = (int)SK;
    const int SQ = (int)((K / 32) / SK);
    a.order = p.order =
        StepOrder{SQ, (int)((K / 32) % SK), KW == 4 ? 2 : (int)KW - 1, (uint32_t)(((uint64_t(1) << 32) + SQ) / (SQ + 1)),
                  SQ == 1 ? 0u : (uint32_t)(((uint64_t(1) << 32) + SQ - 1) / SQ)};
    hipStream_t st = (hipStream_t)stream;
    switch (cb * 32 + k2) {
#define ESP_PREP_CASE(CB_, K2_)                                                                              \
    case CB_ * 32 + K2_:                                                                                     \
        prompt_prep_kernel<gemm_cb(CB_), K2_><<<(unsigned)(rot_wgs + dec_units), 256, 0, st>>>(p);           \
        break;
        ESP_CASES(ESP_PREP_CASE)
#undef ESP_PREP_CASE
    }
    const int rc = esp_host::launch_check("dense_prompt preparation");
    if (rc) return rc;
    a.tiles_m = (int)((T + PG_ROWS - 1) / PG_ROWS);
    a.chunk = (a.tiles_m * nbt + 7) / 8;
    const unsigned grid = (unsigned)a.chunk * 8;
    if (KW == 4 && K / 32 == SK * 4)
        prompt_gemm_kernel<1><<<grid, PG_WAVES * 64, 0, st>>>(a);
    else if (KW == 4 && K / 32 == SK * 8)
        prompt_gemm_kernel<2><<<grid, PG_WAVES * 64, 0, st>>>(a);
    else
        prompt_gemm_kernel<0><<<grid, PG_WAVES * 64, 0, st>>>(a);
    return esp_host::launch_check("dense_prompt");
}
