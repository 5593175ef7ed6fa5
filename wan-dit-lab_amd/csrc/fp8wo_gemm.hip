// FP8 weight-only linear on gfx950: y = x W^T (W = w_fp8 * w_scale) + bias, x and y bf16. The weight stays in e4m3
// in memory (one byte per value, per output row or per tensor scale); activations keep their bf16 precision. No
// counterpart in the reference, whose FP8 linears quantize the activation too (quantization/fp8.py:1-6, 44-67): the
// mixed-precision mode of the benchmark plan (attention projections FP8 weight-only, FFN W4A4).
//
// Products. Every e4m3 value is exact in bf16 (3 mantissa bits, exponents inside bf16's range), so the weight codes
// are widened to bf16 in registers (v_cvt_scalef32_pk_bf16_fp8, two codes per instruction) and C^T = W X^T runs on
// v_mfma_f32_32x32x16_bf16: each product of a bf16 and an e4m3 value is exact in fp32 (8 + 4 significant bits), sums
// accumulate in fp32, and the per-row scale multiplies the sum once in the epilogue (scale * sum, then + bias, then
// bf16).
//
// Tiles. 256 features x 128 tokens by 8 waves of 64 x 64 (one workgroup per CU, a 4-stage ring of 128 KB), or for the
// smaller products 128 x 128 by 4 waves of 32 features x 128 tokens (two workgroups per CU, 3 stages of 24 KB each;
// every weight row of the tile is then widened by one wave only); a lane owns one token and 16 features per 32 x 32
// subtile. K advances 64 per stage through the LDS ring, fed by direct global->LDS loads (16 bytes per lane, waited for
// with an explicit vmcnt):
//   W stage: [features][64 B] of e4m3, each row's four 16-byte quarters XOR-swizzled by (row / 4) % 4;
//   X stage: [128 tokens][128 B] of bf16, each row's eight 16-byte chunks XOR-swizzled by (row / 2) % 8,
// which spreads the 8- and 16-byte fragment reads of 16 consecutive rows over the banks. Fragments are double-buffered in
// registers across steps and stages. Rows of X past M are loaded from row M - 1 (never written back).
//
// What bounds it: no single unit. The matrix cores are busy for half of the time at 2640 x 9216 x 3072 (they alone would
// take 70 us); a third of the wave cycles wait at the ring's barrier and loads, a third for their turn to issue, LDS waits
// are 1 % (bank conflicts one cycle per active one). A timing copy without the loads takes 115 us, so the operands' way
// into LDS is the largest part that can be named. Measured (graph replays, both sides in turn on one box): 2640 tokens QKV
// 177 -> 141 us (1.06 PFLOP/s; 8192^3 in bf16 through the library GEMM 1.25), o 61.2 -> 48.5; 1392 tokens QKV 104 -> 85, o
// 47.7 -> 37.7; 464 tokens QKV 48.4 -> 37.6, o 35.1 -> 27.0 us. The steps, as each was made: fragments
// double-buffered and the one-instruction widening -8 % at 1392 tokens; the 256 x 128 tiles -12 % at 2640; rows staged to
// whole segments on the way out and the swizzle by row / 2 the rest.
#include "wdl_common.h"

#include <type_traits>

namespace {

using namespace wdl;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int BM = 128, KS = 64;  // tokens of a tile, K of a stage
constexpr int EPI_BF16 = 0, EPI_RESIDUAL = 2;

struct Args {
    const uint16_t* x;
    int64_t ldx;
    const uint8_t* w;
    const float* ws;      // [N] (rows) or [1]
    int64_t ws_step;      // 1 (rows) or 0 (tensor)
    const uint16_t* bias; // [N] or null
    uint16_t* out;
    int64_t ldo;
    const float* gate;    // [N] (gated residual)
    int64_t M, N, K, ntm;
};

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return uint32_t(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}

// 64 lanes x 16 bytes from a wave-uniform base plus a 32-bit per-lane offset to LDS [m0, m0 + 1024)
__device__ __forceinline__ void dma16s(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "{m0}"(lds) : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// eight e4m3 codes (little-endian in two dwords) -> eight bf16 (exact)
__device__ __forceinline__ bf16x8 widen(uint2 c) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    auto two = [](uint32_t w, auto high) {
        return __builtin_bit_cast(uint32_t, bf16x2(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, decltype(high)::value)));
    };
    constexpr std::false_type lo{};
    constexpr std::true_type hi{};
    return __builtin_bit_cast(bf16x8, make_uint4(two(c.x, lo), two(c.x, hi), two(c.y, lo), two(c.y, hi)));
}

// BN features x 128 tokens by NW waves of 32 TN features x 32 TJ tokens, a ring of ST stages
template <int BN, int TN, int TJ, int ST, int EPI>
__global__ __launch_bounds__(BN / (32 * TN) * (4 / TJ) * 64) void fp8wo_gemm_kernel(Args a) {
    constexpr int NWN = BN / (32 * TN), NW = NWN * (4 / TJ);      // waves along the features, all
    constexpr int WST = BN * KS, XST = BM * KS * 2;               // bytes of a W (e4m3) / X (bf16) stage
    constexpr int WL = WST / (NW * 1024), XL = XST / (NW * 1024); // 16-byte loads per lane and stage
    static_assert(WL * NW * 1024 == WST && XL * NW * 1024 == XST, "stages split evenly over the waves");
    constexpr int F = 32 * TN, SROW = F + 4;                      // staged output row (4 values of padding)
    static_assert(NW * 32 * TJ * SROW * 2 <= ST * (WST + XST), "the outputs' staging fits the ring");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[ST * (WST + XST)];

    const int t = threadIdx.x, lane = t % 64, half = lane / 32, tok = lane % 32;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int wn = wave % NWN, wm = wave / NWN;  // the wave's features 32 TN wn .., tokens 32 TJ wm ..
    // Workgroups go round-robin over the 8 XCDs; each XCD takes a contiguous range of the tiles, which run GM token tiles
    // deep over the features: the 32 tiles an XCD's CUs run at a time are about 4 weight slabs by 8 token tiles, 12 operand
    // blocks a stage to fetch into its L2 (slab after slab over all of 2640 tokens it was 23).
    const int64_t total = gridDim.x, pid = blockIdx.x, xcd = pid % 8;
    const int64_t tile = xcd * (total / 8) + min(xcd, total % 8) + pid / 8;
    constexpr int64_t GM = 8;
    const int64_t ntn = a.N / BN, band = tile / (GM * ntn), in = tile % (GM * ntn), gm = min(GM, a.ntm - band * GM);
    const int64_t n0 = in / gm * BN, m0 = (band * GM + in % gm) * BM;
    auto sW = [&](int slot) { return smem + slot * (WST + XST); };
    auto sX = [&](int slot) { return smem + slot * (WST + XST) + WST; };

    // this lane's load offsets: W chunk id = 64 (NW i + wave) + lane: row id / 4, stored quarter id % 4 holds the row's
    // quarter (id % 4) ^ ((row / 4) % 4); X chunk id likewise: row id / 8, stored chunk id % 8 holds chunk
    // (id % 8) ^ ((row / 2) % 8)
    uint32_t woff[WL], xoff[XL];
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int id = 64 * (NW * i + wave) + lane, row = id / 4, q = (id % 4) ^ ((row / 4) % 4);
        woff[i] = uint32_t(row * a.K + 16 * q);
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int id = 64 * (NW * i + wave) + lane, row = id / 8, c = (id % 8) ^ (row / 2 % 8);
        const int64_t m = m0 + row < a.M ? m0 + row : a.M - 1;
        xoff[i] = uint32_t(m * a.ldx * 2 + 16 * c);
    }
    const uint8_t* wtile = a.w + n0 * a.K;
    const int G = int(a.K / KS);
    auto issue = [&](int slot, int g) {
        const int gg = g < G ? g : G - 1;  // past the end: the last stage again (a slot no wave reads any more)
        const uint8_t* wb = wtile + int64_t(gg) * KS;
        const uint8_t* xb = reinterpret_cast<const uint8_t*>(a.x) + int64_t(gg) * KS * 2;
#pragma unroll
        for (int i = 0; i < WL; ++i) dma16s(wb, woff[i], lds_addr(sW(slot) + 1024 * (NW * i + wave)));
#pragma unroll
        for (int i = 0; i < XL; ++i) dma16s(xb, xoff[i], lds_addr(sX(slot) + 1024 * (NW * i + wave)));
    };

    f32x16 acc[TN][TJ];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x16{};

    // fragments of one 16-deep step (quarter s of the rows, k = 16 s + 8 half .. + 7) of the lane's W rows F wn + 32 i +
    // tok and X rows 32 TJ wm + 32 j + tok: two register sets, the next step's reads issued before the current step's
    // MFMAs, also across stages
    const int wsw = ((tok / 4) % 4), xsw = tok / 2 % 8;  // (multiples of 32 leave both unchanged)
    uint2 wf[2][TN];
    bf16x8 bf[2][TJ];
    auto read = [&](int set, int slot, int s) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
            wf[set][i] = *reinterpret_cast<const uint2*>(sW(slot) + (F * wn + 32 * i + tok) * 64 + 16 * (s ^ wsw) + 8 * half);
#pragma unroll
        for (int j = 0; j < TJ; ++j)
            bf[set][j] = *reinterpret_cast<const bf16x8*>(sX(slot) + (32 * TJ * wm + 32 * j + tok) * 128 +
                                                          16 * ((2 * s + half) ^ xsw));
    };
#pragma unroll
    for (int k = 0; k < ST - 1; ++k) issue(k, k);
    wait_vmcnt<(ST - 2) * (WL + XL)>();
    __syncthreads();
    read(0, 0, 0);
    int slot = 0, free = ST - 1;
    for (int g = 0; g < G; ++g) {
        // stage g + 1 has landed for every wave; stage g - 1 is read (its last fragments were in registers a step ago)
        const int next = slot + 1 == ST ? 0 : slot + 1;
        wait_vmcnt<(ST - 3) * (WL + XL)>();
        __syncthreads();
        issue(free, g + ST - 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s < 3) read((s + 1) % 2, slot, s + 1);
            else read(0, next, 0);
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const bf16x8 af = widen(wf[s % 2][i]);
#pragma unroll
                for (int j = 0; j < TJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf[s % 2][j], acc[i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        free = slot;
        slot = next;
    }
    wait_vmcnt<0>();  // the clamped tail loads land before the ring is reused
    __syncthreads();

    // epilogue: element e of subtile (i, j) is feature n0 + F wn + 32 i + 8 (e / 4) + 4 half + e % 4 of token m0 + 32 TJ wm
    // + 32 j + tok. The bf16 results go through the wave's own part of the ring and leave token-major, F / 4 lanes on a
    // token's features in 8-byte pieces (from the MFMA layout a store touches 32 rows).
    uint16_t* const stg = reinterpret_cast<uint16_t*>(smem) + wave * (32 * TJ * SROW);
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int f = 32 * i + 8 * q + 4 * half;
            const int64_t n = n0 + F * wn + f;
            float sc[4], bi[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc[e] = a.ws[(n + e) * a.ws_step];
                bi[e] = a.bias ? bf16_to_f32(a.bias[n + e]) : -0.0f;  // -0: an exact identity of the sum
            }
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                uint16_t r[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) r[e] = f32_to_bf16(acc[i][j][4 * q + e] * sc[e] + bi[e]);
                *reinterpret_cast<uint2*>(stg + (32 * j + tok) * SROW + f) =
                    make_uint2(r[0] | (uint32_t(r[1]) << 16), r[2] | (uint32_t(r[3]) << 16));
            }
        }
    asm volatile("" ::: "memory");  // the writes stay ahead of the reads (one wave: LDS keeps its order)
    constexpr int TPS = 64 / (F / 4);  // tokens per store
    const int f = 4 * (lane % (F / 4));
    const int64_t n = n0 + F * wn + f;
    float gate[4];
    if (EPI == EPI_RESIDUAL)
#pragma unroll
        for (int e = 0; e < 4; ++e) gate[e] = a.gate[n + e];
#pragma unroll
    for (int k = 0; k < 32 * TJ / TPS; ++k) {
        const int tk = k * TPS + lane / (F / 4);
        const int64_t m = m0 + 32 * TJ * wm + tk;
        uint2 w = *reinterpret_cast<const uint2*>(stg + tk * SROW + f);
        if (m >= a.M) continue;
        uint2* const out = reinterpret_cast<uint2*>(a.out + m * a.ldo + n);
        if (EPI == EPI_RESIDUAL) {
            const uint2 old = *out;
            const uint32_t yw[2] = {w.x, w.y}, ow[2] = {old.x, old.y};
            uint32_t rw[2];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const float y0 = bf16_to_f32(uint16_t(yw[d])), y1 = bf16_to_f32(uint16_t(yw[d] >> 16));
                const float o0 = bf16_to_f32(uint16_t(ow[d])), o1 = bf16_to_f32(uint16_t(ow[d] >> 16));
                rw[d] = f32_to_bf16(o0 + y0 * gate[2 * d]) | (uint32_t(f32_to_bf16(o1 + y1 * gate[2 * d + 1])) << 16);
            }
            w = make_uint2(rw[0], rw[1]);
        }
        *out = w;
    }
}

// 256 x 128 tiles (8 waves, one workgroup per CU) move two thirds of the operand bytes of 128 x 128 tiles per product and
// bind less on the L2's delivery: taken where N allows and they occupy at least half of the CUs (measured at the line,
// 132 tiles: o at 1392 tokens 40.7 -> 39.4 us, 144 tiles: QKV at 464 tokens 41.0 -> 38.0 us); fewer leave CUs idle that
// the small tiles use.
template <int EPI>
int launch(const Args& a, hipStream_t stream) {
    const int64_t cus = cu_count(), wide = a.N % 256 == 0 ? a.ntm * (a.N / 256) : 0;
    if (cus > 0 && 2 * wide >= cus) {
        fp8wo_gemm_kernel<256, 2, 2, 4, EPI><<<unsigned(wide), 512, 0, stream>>>(a);
    } else {
        fp8wo_gemm_kernel<128, 1, 4, 3, EPI><<<unsigned(a.ntm * (a.N / 128)), 256, 0, stream>>>(a);
    }
    return check_launch("fp8wo_gemm");
}

}  // namespace

extern "C" int wdl_fp8wo_gemm(const void* x, int64_t ldx, const void* w, const float* w_scale, int scale_rows,
                              const void* bias, int64_t M, int64_t N, int64_t K, void* out, int64_t ldo,
                              int epilogue, const float* gate, hipStream_t stream) {
    if (M < 0 || N <= 0 || K <= 0 || N % 128 || K % KS || ldx < K || ldo < N || ldx % 8 || ldo % 4)
        return fail(WDL_EINVAL, "fp8wo_gemm: bad shape M=%lld N=%lld K=%lld ldx=%lld ldo=%lld", (long long)M,
                    (long long)N, (long long)K, (long long)ldx, (long long)ldo);
    if (!x || !w || !w_scale || !out || (epilogue == EPI_RESIDUAL && !gate))
        return fail(WDL_EINVAL, "fp8wo_gemm: null pointer");
    if (epilogue != EPI_BF16 && epilogue != EPI_RESIDUAL)
        return fail(WDL_EINVAL, "fp8wo_gemm: epilogue must be 0 (bf16) or 2 (gated residual)");
    if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) % 16 ||
        reinterpret_cast<uintptr_t>(out) % 8 || reinterpret_cast<uintptr_t>(bias) % 2)
        return fail(WDL_EINVAL, "fp8wo_gemm: x, w 16-byte aligned, out 8-byte, bias 2-byte");
    if (int64_t(128) * K >= (int64_t(1) << 31) || M * ldx * 2 >= (int64_t(1) << 32))
        return fail(WDL_EINVAL, "fp8wo_gemm: operands beyond 32-bit load offsets");
    if (M == 0) return WDL_OK;
    const Args a{static_cast<const uint16_t*>(x), ldx, static_cast<const uint8_t*>(w), w_scale, scale_rows ? 1 : 0,
                 static_cast<const uint16_t*>(bias), static_cast<uint16_t*>(out), ldo, gate, M, N, K, (M + BM - 1) / BM};
    return epilogue == EPI_RESIDUAL ? launch<EPI_RESIDUAL>(a, stream) : launch<EPI_BF16>(a, stream);
}
