// gemv_mfma.hip -- small-batch IQ4_XS x Q8_1 multiply (2 <= M <= GM_MAX_COLS
// columns) on the gfx950 int8 matrix cores.
//
// Semantics: those of the GEMV / GEMM (real_stock_dp4a_comparator.hip:
// 68-166, 374-443): per 32-weight sub-block the exact int32 dot sumi of the
// IQ4_XS codes with the Q8_1 codes, scaled by fp16(d_w)*(ls-32) and the
// column's fp16 d.
//
// Why a second GEMV.  The dot4 GEMV spends VALU work per weight byte and per
// column, so from 4 columns on it is VALU-bound.  Here one
// v_mfma_i32_32x32x32_i8 takes 32 weight rows x 32 k of one sub-block against
// 32 columns (the A operand is the activations, one token per MFMA row;
// rows past M hold any token and only produce C rows that are never stored),
// so the VALU cost is the decode of the codes into the B operand, the same for
// any M, and per output a subtract, a scale product and a fused add.
//
// Mapping.  A workgroup owns up to 32 weight rows (one MFMA block) of one
// matrix and all columns (8 G of them), and splits K over its waves: wave w takes the
// super-blocks kb = w, w + waves, ... (at any moment the waves stream adjacent
// super-blocks of the same rows), with no barrier before the final sum.  The
// partial sums are added in a fixed order and the split follows the
// matrix's own shape (gm_split), so a row's bits depend neither on the rows
// per workgroup nor on what shares the launch.
//   * Loads are coalesced (each of the 4 weight loads of a block covers the qs
//     of 8 whole rows, the activation loads a token's 256 codes per 8 lanes)
//     and staged in LDS rows of the wave's own, from which the MFMA operands
//     are read.  Staging frees the load registers, so the next block's loads
//     are issued before the current block is computed, without a second set
//     (112 VGPRs at G = 2; the two-set form this replaces measured 20.7 us
//     against 18.6 us on 17408 -> 5120 at M = 8).
//   * The MFMA sums over k, so any order of k that A and B share gives the same
//     int32: lane l (half h = l >> 5) supplies weight row l & 31 with both
//     nibbles of qs bytes 8h .. 8h+7 of the sub-block (weights 8h .. 8h+7 and
//     16+8h .. 16+8h+7), and the A lanes the activation codes of the same 16
//     weights, which the staging puts side by side (one 16-byte read).
//   * The C element e of lane l is token 8*(e>>2) + 4h + (e&3) of its row; past
//     32 columns a second MFMA takes the same B operand, so the decode is not
//     repeated.
//   * The int32 sum comes back as a float without a convert (which issues at
//     half the rate of an add): the accumulator starts at the bits of
//     1/(2 pi) = 0x3E22F983, an inline constant in the middle of the binade
//     [1/8, 1/4), so that sumi (|sumi| < 2^20) counts units of 2^-26 there and
//     one exact subtraction leaves sumi * 2^-26; the weight scale carries 2^26.
#include "iq4xs_device.h"
#include "iq4xs_internal.h"

namespace iq4xs {

constexpr int GM_LDS_MAX = 160 * 1024;

// Activations are staged a whole super-block at a time up to 16 tokens, above
// in halves of 4 sub-blocks: less LDS and fewer registers in flight, hence
// more waves per CU.
constexpr int gm_halves(int G) { return G <= 2 ? 1 : 2; }
// LDS row of one token's staged codes, padded (conflict-free 16-byte reads)
constexpr int gm_arow(int G) { return QK_K / gm_halves(G) + 16; }
constexpr int GM_WROW = 136;  // LDS row of one weight row's 128 qs bytes, padded (conflict-free 8-byte reads)
// per-wave staging bytes: weight rows, token rows, then the super-block's
// column scales [8 sub-blocks][8G tokens]; the final sum reuses them
constexpr int gm_wave_lds(int G) { return 32 * GM_WROW + G * (8 * gm_arow(G) + 8 * 8 * 4); }

constexpr int GM_ZERO_BITS = 0x3E22F983;  // the accumulator's zero (1/(2 pi) as a float)

// Waves per SIMD that the registers are held to (96 to 128 VGPRs up to G = 4,
// 161 and 168 at 5 and 6, 226 and 246 at 7 and 8);
// `more`: the debug export, or two sums per wave (116 VGPRs; two workgroups
// of 8 waves a CU either way).
constexpr int gm_waves_per_simd(int G, bool more) { return G == 1 ? (more ? 4 : 5) : (G == 2 ? 4 : (more || G > 6 ? 2 : G <= 4 ? 4 : 3)); }

// The matrices of one launch (same K and activations): workgroups
// [tile_end[i-1], tile_end[i]) run matrix i.  Entries past the group's count
// repeat its last matrix with tile_end = the grid size, so no workgroup
// selects them.
struct GmGroup {
    const uint8_t* W[GEMV_GROUP_MAX];
    float* Y[GEMV_GROUP_MAX];
    int64_t ldy_m[GEMV_GROUP_MAX];
    int N[GEMV_GROUP_MAX];
    int tile_end[GEMV_GROUP_MAX];
};

// kTwo: two partial sums per wave (GmSplit)
template <int G, bool kDebug, bool kTwo>
__global__ __launch_bounds__(64 * gm_max_waves(G)) __attribute__((amdgpu_waves_per_eu(gm_waves_per_simd(G, kDebug || kTwo))))
void gemv_mfma_kernel(const GmGroup grp, const int8_t* __restrict__ aqs, const uint32_t* __restrict__ ads, int K,
                      int M, int rows, int64_t ldy_n, int32_t* __restrict__ dbg) {
    // sub-blocks unrolled together: above 16 tokens one at a time, since the
    // registers of more reads in flight would cost waves (M = 32, gate + up: 2
    // together 56.6 us, 1 at a time 50.6)
    constexpr int UNR = kDebug || G >= 3 ? 1 : 8;
    constexpr int HALVES = gm_halves(G), SUB = 8 / HALVES, AROW = gm_arow(G);
    extern __shared__ __attribute__((aligned(16))) uint8_t gm_lds[];
    // this workgroup's matrix: scalar selects on the by-value descriptor (a
    // dynamic index into it would go through scratch)
    const uint8_t* __restrict__ W = grp.W[0];
    float* __restrict__ Y = grp.Y[0];
    int64_t ldy_m = grp.ldy_m[0];
    int N = grp.N[0], tile0 = 0;
#pragma unroll
    for (int i = 1; i < GEMV_GROUP_MAX; ++i) {
        if ((int)blockIdx.x >= grp.tile_end[i - 1]) {
            W = grp.W[i];
            Y = grp.Y[i];
            ldy_m = grp.ldy_m[i];
            N = grp.N[i];
            tile0 = grp.tile_end[i - 1];
        }
    }
    const int bpr = K / QK_K, nb = K / QK8_1;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)blockDim.x >> 6;
    uint8_t* sw = gm_lds + wave * gm_wave_lds(G);                   // [32][136] qs of a block's rows
    uint8_t* sact = sw + 32 * GM_WROW;                              // [8G][AROW] activations
    float* sdx = reinterpret_cast<float*>(sact + 8 * G * AROW);  // [8][8G] column scales (0 past M)
    const int r0 = ((int)blockIdx.x - tile0) * rows;
    const int nrow = min(rows, N - r0);  // this workgroup's rows (1 .. 32)
    // Global loads are 32-bit lane offsets from workgroup-uniform bases.  MFMA
    // rows past nrow are clamped to its last row (a repeat of bytes already
    // loaded, so no extra HBM traffic): computed, never stored.
    const uint32_t row_bytes = (uint32_t)bpr * BLOCK_BYTES;
    const uint8_t* wbase = W + (size_t)r0 * row_bytes;

    // an offset kept scalar: the loads then take a scalar base and a 32-bit
    // lane offset, instead of a 64-bit address per lane and load
    auto uniform = [](int off) {
        asm volatile("" : "+s"(off));
        return (uint32_t)off;
    };
    v2u wh;        // d, scales_h, scales_l of row col
    v4i wq[4];     // qs chunk lane % 8 of rows lane/8 + 8i
    // sub-block lane % 8 of token 8g + lane/8, or of a half the 16 codes lane % 8 of it
    v4i xa[G][2 / HALVES];
    uint32_t xd[G];
    auto load_w = [&](int kb) {
        const uint8_t* wk = wbase + uniform(kb * BLOCK_BYTES);
        wh = *reinterpret_cast<const v2u*>(wk + (uint32_t)min(col, nrow - 1) * row_bytes);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            wq[i] = *reinterpret_cast<const v4i_a8*>(
                wk + ((uint32_t)min(8 * i + (lane >> 3), nrow - 1) * row_bytes + 8 + 16 * (lane & 7)));
    };
    auto load_x = [&](int kb, int half) {
        const int8_t* ak = aqs + uniform(kb * QK_K + half * 128);
        const uint32_t* dk = ads + uniform(kb * 8);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t t = (uint32_t)min(8 * g + (lane >> 3), M - 1);
            const uint32_t off = t * (uint32_t)K + (32 / HALVES) * (lane & 7);
#pragma unroll
            for (int i = 0; i < 2 / HALVES; ++i) xa[g][i] = *reinterpret_cast<const v4i*>(ak + off + 16 * i);
            if (half == 0) xd[g] = dk[t * (uint32_t)nb + (lane & 7)];
        }
    };
    // LDS operations of one wave complete in order: the reads below by other
    // lanes of the wave see these writes, and the previous block's reads were
    // issued before them
    uint8_t* xwrite = sact + (lane >> 3) * AROW + (HALVES == 1 ? 32 * (lane & 7) : 32 * ((lane & 7) >> 1) + 8 * (lane & 1));
    const uint8_t* xread = sact + min(col, 8 * G - 1) * AROW + 16 * h;
    uint8_t* wwrite = sw + (lane >> 3) * GM_WROW + 16 * (lane & 7);
    const uint8_t* wread = sw + col * GM_WROW + 8 * h;
    auto stage_x = [&](int half) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            // a sub-block's elements in the order 0-7, 16-23, 8-15, 24-31: the A operand of each lane half
            uint8_t* x = xwrite + 8 * g * AROW;
            if constexpr (HALVES == 1) {
                *reinterpret_cast<v4i*>(x) = v4i{xa[g][0].x, xa[g][0].y, xa[g][1].x, xa[g][1].y};
                *reinterpret_cast<v4i*>(x + 16) = v4i{xa[g][0].z, xa[g][0].w, xa[g][1].z, xa[g][1].w};
            } else {
                *reinterpret_cast<v2u*>(x) = v2u{(uint32_t)xa[g][0].x, (uint32_t)xa[g][0].y};
                *reinterpret_cast<v2u*>(x + 16) = v2u{(uint32_t)xa[g][0].z, (uint32_t)xa[g][0].w};
            }
            const int t = 8 * g + (lane >> 3);
            if (half == 0) sdx[(lane & 7) * 8 * G + t] = t < M ? half_bits_to_float(xd[g] & 0xFFFFu) : 0.0f;
        }
    };
    auto stage_w = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<v2u*>(wwrite + 8 * i * GM_WROW) = v2u{(uint32_t)wq[i].x, (uint32_t)wq[i].y};
            *reinterpret_cast<v2u*>(wwrite + 8 * i * GM_WROW + 8) = v2u{(uint32_t)wq[i].z, (uint32_t)wq[i].w};
        }
    };

    float acc[4 * G];
#pragma unroll
    for (int e = 0; e < 4 * G; ++e) acc[e] = 0.0f;
    auto compute = [&](const v2u hd, int kb, int half) {
        const float dw = half_bits_to_float(hd.x & 0xFFFFu) * 67108864.0f;  // 2^26
#pragma unroll UNR
        for (int i = 0; i < SUB; ++i) {
            const int s = SUB * half + i;
            uint32_t lo0, hi0, lo1, hi1;
            const v2u q = *reinterpret_cast<const v2u*>(wread + 16 * s);
            decode_codes_x(q.x, lo0, hi0);
            decode_codes_x(q.y, lo1, hi1);
            const v4i bw = v4i{(int)lo0, (int)lo1, (int)hi0, (int)hi1};
            v16i z;
#pragma unroll
            for (int e = 0; e < 16; ++e) z[e] = GM_ZERO_BITS;
            const int ls = subblock_ls(hd.x, hd.y, s) - 32;
            const float sa = dw * (float)ls;
            // 32 tokens (4 groups of 8) per MFMA
#pragma unroll
            for (int b = 0; b < (G + 3) / 4; ++b) {
                const uint8_t* xr = b == 0 ? xread : sact + min(32 * b + col, 8 * G - 1) * AROW + 16 * h;
                const v4i ax = *reinterpret_cast<const v4i*>(xr + 32 * i);
                const v16i c = __builtin_amdgcn_mfma_i32_32x32x32_i8(ax, bw, z, 0, 0, 0);
#pragma unroll
                for (int g = 4 * b; g < (4 * b + 4 < G ? 4 * b + 4 : G); ++g) {
                    const v4f bx = *reinterpret_cast<const v4f*>(sdx + s * 8 * G + 8 * g + 4 * h);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int e = 4 * g + j, ce = (int)c[e - 16 * b];
                        const float f = __builtin_bit_cast(float, ce) - __builtin_bit_cast(float, GM_ZERO_BITS);
                        acc[e] = __builtin_fmaf(f, sa * bx[j], acc[e]);
                        if (kDebug) {
                            const int t = 8 * g + 4 * h + j;
                            if (t < M && col < nrow)
                                dbg[((size_t)t * N + r0 + col) * nb + kb * 8 + s] = (ce - GM_ZERO_BITS) * ls;
                        }
                    }
                }
            }
        }
    };
    // with two sums the super-blocks go to acc and alt in turn
    float alt[kTwo ? 4 * G : 1] = {};
    // every load is unconditional (past this wave's last super-block it repeats that one)
    if (wave < bpr) {
        load_x(wave, 0);
        load_w(wave);
        for (int kb = wave; kb < bpr; kb += waves) {
            if constexpr (kTwo) {
#pragma unroll
                for (int e = 0; e < 4 * G; ++e) {
                    const float other = alt[e];
                    alt[e] = acc[e];
                    acc[e] = other;
                }
            }
            const int kn = kb + waves < bpr ? kb + waves : kb;
            const v2u hd = wh;
            stage_x(0);
            load_x(HALVES == 1 ? kn : kb, HALVES - 1);
            stage_w();
            load_w(kn);
            compute(hd, kb, 0);
            if constexpr (HALVES == 2) {
                stage_x(1);
                load_x(kn, 0);
                compute(hd, kb, 1);
            }
        }
    }
    // the partial sums, added in wave order (with two per wave the even ones
    // first), those of twelve waves in two chains of every other one
    __syncthreads();  // the staging is free
    float* red = reinterpret_cast<float*>(gm_lds);  // [waves, or 2 waves][4G][64]
    constexpr int PER = 4 * G * 64;
    static_assert((kTwo ? 2 : 1) * PER * 4 <= gm_wave_lds(G), "the final sum fits the staging");
    if constexpr (kTwo) {
        const bool odd = ((bpr - wave + waves - 1) / waves & 1) == 0;  // the last super-block was an odd one
#pragma unroll
        for (int e = 0; e < 4 * G; ++e) {
            red[wave * PER + e * 64 + lane] = odd ? alt[e] : acc[e];
            red[(waves + wave) * PER + e * 64 + lane] = odd ? acc[e] : alt[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4 * G; ++e) red[wave * PER + e * 64 + lane] = acc[e];
    }
    __syncthreads();
    for (int e = wave; e < 4 * G; e += waves) {  // uniform per wave
        float v = red[e * 64 + lane];
        if (G == 1 && !kTwo && waves == 12) {
            float u = red[PER + e * 64 + lane];
#pragma unroll
            for (int w = 2; w < 12; w += 2) {
                v += red[w * PER + e * 64 + lane];
                u += red[(w + 1) * PER + e * 64 + lane];
            }
            v += u;
        } else if constexpr (kTwo) {  // 8 waves
#pragma unroll
            for (int w = 1; w < 16; ++w) v += red[w * PER + e * 64 + lane];
        } else {
            for (int w = 1; w < waves; ++w) v += red[w * PER + e * 64 + lane];
        }
        const int t = 8 * (e >> 2) + 4 * h + (e & 3);
        if (t < M && col < nrow) Y[(int64_t)t * ldy_m + (int64_t)(r0 + col) * ldy_n] = v;
    }
}

template <int G>
static hipError_t launch_gm(const GmGroup& grp, dim3 grid, GmSplit split, const int8_t* aqs, const uint32_t* ads,
                            int64_t K, int64_t M, int64_t rows, int64_t ldy_n, int32_t* dbg,
                            hipStream_t stream) {
    const int waves = split.waves;
    const size_t lds = (size_t)waves * gm_wave_lds(G);
    static_assert(gm_max_waves(G) * gm_wave_lds(G) <= GM_LDS_MAX, "the staging fits a CU");
    auto launch = [&](auto kernel) -> hipError_t {
        if (lds > 64 * 1024) {  // beyond the default dynamic-LDS limit of a launch
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, GM_LDS_MAX);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), lds, stream, grp, aqs, ads, (int)K, (int)M, (int)rows,
                           ldy_n, dbg);
        return hipGetLastError();
    };
    if constexpr (G == 1)
        if (split.two) return dbg ? launch(&gemv_mfma_kernel<G, true, true>) : launch(&gemv_mfma_kernel<G, false, true>);
    return dbg ? launch(&gemv_mfma_kernel<G, true, false>) : launch(&gemv_mfma_kernel<G, false, false>);
}

// The matrices of one split in one launch.
static hipError_t launch_gm_split(int count, const uint8_t* const* W, float* const* Y, const int64_t* N,
                                  const int64_t* ldy_m, const int8_t* aqs, const uint32_t* ads, int64_t K, int64_t M,
                                  int64_t ldy_n, int32_t* dbg, GmSplit split, hipStream_t stream) {
    const int64_t cus = device_cu_count();
    const int64_t rows = gm_rows(count, N, cus);
    GmGroup grp{};
    int64_t wgs = 0;
    for (int i = 0; i < GEMV_GROUP_MAX; ++i) {
        const int j = i < count ? i : count - 1;
        if (i < count) wgs += (N[j] + rows - 1) / rows;
        if (wgs > 0x7FFFFFFF) return hipErrorInvalidConfiguration;
        grp.W[i] = W[j];
        grp.Y[i] = Y[j];
        grp.ldy_m[i] = ldy_m[j];
        grp.N[i] = (int)N[j];
        grp.tile_end[i] = (int)wgs;
    }
    const dim3 grid((unsigned)wgs);
#define IQ4XS_GM(G) \
    case G: return launch_gm<G>(grp, grid, split, aqs, ads, K, M, rows, ldy_n, dbg, stream)
    switch ((M + 7) / 8) {
        IQ4XS_GM(1);
        IQ4XS_GM(2);
        IQ4XS_GM(3);
        IQ4XS_GM(4);
        IQ4XS_GM(5);
        IQ4XS_GM(6);
        IQ4XS_GM(7);
        IQ4XS_GM(8);
        default: return hipErrorNotSupported;
    }
#undef IQ4XS_GM
}

hipError_t launch_gemv_mfma_group(int count, const uint8_t* const* W, float* const* Y, const int64_t* N,
                                  const int64_t* ldy_m, const int8_t* aqs, const uint32_t* ads, int64_t K,
                                  int64_t M, int64_t ldy_n, int32_t* dbg, hipStream_t stream) {
    clear_launch_error();
    if (count < 1 || count > GEMV_GROUP_MAX || (dbg && count != 1)) return hipErrorInvalidValue;
    if (M < 1 || M > GM_MAX_COLS || K % QK_K || K >= (1 << 24)) return hipErrorNotSupported;
    // the kernel's 32-bit load offsets span 32 rows and GM_MAX_COLS tokens
    if ((int64_t)32 * (K / QK_K) * BLOCK_BYTES >= ((int64_t)1 << 31) || GM_MAX_COLS * K >= ((int64_t)1 << 31))
        return hipErrorNotSupported;
    for (int i = 0; i < count; ++i)
        if (N[i] < 1 || N[i] >= (1 << 30)) return hipErrorNotSupported;
    // one launch per split
    const int G = (int)((M + 7) / 8);
    bool done[GEMV_GROUP_MAX] = {};
    for (int i = 0; i < count; ++i) {
        if (done[i]) continue;
        const GmSplit split = gm_split(N[i], K, G);
        const uint8_t* gW[GEMV_GROUP_MAX];
        float* gY[GEMV_GROUP_MAX];
        int64_t gN[GEMV_GROUP_MAX], gL[GEMV_GROUP_MAX];
        int n = 0;
        for (int j = i; j < count; ++j) {
            if (done[j] || !(gm_split(N[j], K, G) == split)) continue;
            gW[n] = W[j];
            gY[n] = Y[j];
            gN[n] = N[j];
            gL[n] = ldy_m[j];
            ++n;
            done[j] = true;
        }
        const hipError_t e = launch_gm_split(n, gW, gY, gN, gL, aqs, ads, K, M, ldy_n, dbg, split, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_gemv_mfma(const uint8_t* W, const int8_t* aqs, const uint32_t* ads, float* Y, int64_t K,
                            int64_t N, int64_t M, int64_t ldy_m, int64_t ldy_n, int32_t* dbg, hipStream_t stream) {
    return launch_gemv_mfma_group(1, &W, &Y, &N, &ldy_m, aqs, ads, K, M, ldy_n, dbg, stream);
}

}  // namespace iq4xs
