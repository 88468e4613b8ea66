// Quantized GEMM for batched prompt prefill: Y[m][n] = sum_k X[m][k] * W[n][k]
// (+ R[m][n]) for M prompt rows at once against a GGUF Q4_0 / Q8_0 weight
// matrix W [N][K] -- the projections of te_qwen_prefill_prompt_batch
// (reference c/src/qwen.c:630-905), whose per-row meaning is te_model_matvec_f32
// (ops.c:177-269) applied to every row.
//
// Products (gemm_bf16_kernel): one 32-value block of a row against one GGUF
// block of a weight row is two K = 16 steps of v_mfma_f32_32x32x16_bf16 for
// each of two operand parts.  An activation x enters as hi + lo bf16 (hi =
// RNE(x), lo = RNE(x - hi), 8 significant bits each: |x - hi - lo| <= 2^-17
// |x|, with the exponent range of fp32), a weight code (Q4_0's n - 8, Q8_0's
// byte) as one bf16, exactly.  The block's fp32 sum is scaled by the weight
// block's scale d and accumulated in fp32, one FMA per product of the block.
//
// Why two bf16 parts and not integer digits: a block-scaled integer digit
// form (two int8 MFMAs at twice the rate) needs a shift, a conversion and the
// product of two block scales for every sum, four VALU instructions per
// output and block against 64 cycles of MFMA; a bf16 pair carries its own
// exponent, so one FMA is left against 128 cycles of MFMA.
//
// Range: activations are stored times 2^-13 (kActScale) and the weight scales
// times 2^13, so that a block's sum (32 products with codes up to 128) of
// values near FLT_MAX stays finite, as the row's true sum does.  At the other
// end lo is a subnormal bf16 for |x| < 2^-104: an absolute error of 2^-121 there.
//
// Layout of the activation operand (act_off): units of one 32-row tile and one
// 32-value block, [M/32][K/32], 4 KiB each: [hi, lo][K step 0, 1][K half
// 0, 1][32 rows][8 values] bf16 -- the order the MFMA operand is held in, so a
// wave loads one operand as 1 KiB contiguous.
#include "te_hip_common.h"

#include <math.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "te_act_split.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr uint32_t kQ4_0 = 2, kQ8_0 = 8;
constexpr int kActThreads = 256;

__device__ __forceinline__ float half_bits(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

enum ActPre { kActPlain = 0, kActRmsNorm = 1, kActSwiGLU = 2 };

// Eight consecutive floats: two 16-byte loads where `vec`.
__device__ __forceinline__ void load8(const float *p, bool vec, float (&v)[8]) {
    if (vec) {
        const float4 a = *reinterpret_cast<const float4 *>(p);
        const float4 c = *reinterpret_cast<const float4 *>(p + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = c.x, v[5] = c.y, v[6] = c.z, v[7] = c.w;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v[j] = p[j];
        }
    }
}

__device__ __forceinline__ void store8(float *p, bool vec, const float (&v)[8]) {
    if (vec) {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = v[j];
        }
    }
}

// The fp64 sum of squares of a row whose thread t holds columns
// 8t + 2048i .. +7 (i = 0, 1, ...): each thread adds its values in column
// order, the wave's lanes are added by an xor butterfly and the workgroup's
// four waves in wave order.  split_act_kernel<kActRmsNorm> and
// gemm_reduce_rms_kernel both sum this way, so their RMSNorm factors agree
// bit for bit.  (te_rmsnorm_f32, ops.c:272-293, sums in fp64 in index order.)
__device__ __forceinline__ double row_sum_squares(double ss) {
    __shared__ double part[kActThreads / 64];
    for (int off = 32; off > 0; off >>= 1) {
        ss += __shfl_xor(ss, off);
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6] = ss;
    }
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kActThreads / 64; ++w) {
        t += part[w];
    }
    return t;
}

// Row of workgroup id: workgroups go to the XCDs round-robin, and eight
// consecutive rows share each 128-byte line of the operand, so an XCD takes
// consecutive rows (7B layer of 512 rows 654 -> 648 us, 3B Q4_0 prompt of 512
// 9.09 -> 9.06 ms, against row = id).
__host__ __device__ inline size_t xcd_rows(size_t rows) { return (rows + 63) / 64 * 8; }  // per XCD
__device__ __forceinline__ size_t xcd_row(unsigned id, int rows) {
    return (id & 7) * xcd_rows((size_t)rows) + (id >> 3);
}

// x' = pre(x) as the GEMM's hi / lo operand.  Thread t of a workgroup holds
// eight consecutive values of block t / 4 of a pass of 64 blocks; without a
// row-wide norm the gridDim.y workgroups of a row take every gridDim.y-th
// pass, else one workgroup takes the row (the norm's sum first, then the
// operand from a second read of the row).  `vec`: the inputs are 16-byte
// aligned.
constexpr int kActPass = kActThreads * 8;
template <int PRE>
__global__ __launch_bounds__(kActThreads) void split_act_kernel(const float *__restrict__ x,
                                                                const float *__restrict__ x2,
                                                                const float *__restrict__ norm_w, float eps,
                                                                int M, int K, unsigned char *__restrict__ act, bool vec) {
    const size_t row = xcd_row(blockIdx.x, M);
    if (row >= (size_t)M) {
        return;
    }
    const float *xr = x + row * (size_t)K;
    const int c0 = 8 * (int)threadIdx.x;
    float rms = 1.0f;
    if (PRE == kActRmsNorm) {
        double ss = 0.0;
        for (int c = c0; c < K; c += kActPass) {
            float v[8];
            load8(xr + c, vec, v);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const double d = (double)v[j];
                ss += d * d;
            }
        }
        rms = 1.0f / sqrtf((float)(row_sum_squares(ss) / (double)K) + eps);
    }
    for (int c = c0 + blockIdx.y * kActPass; c < K; c += kActPass * gridDim.y) {
        float v[8], w2[8];
        load8(xr + c, vec, v);
        if (PRE == kActRmsNorm) {
            load8(norm_w + c, vec, w2);
        } else if (PRE == kActSwiGLU) {
            load8(x2 + row * (size_t)K + c, vec, w2);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (PRE == kActRmsNorm) {
                v[j] = v[j] * rms * w2[j];
            } else if (PRE == kActSwiGLU) {
                v[j] = v[j] / (1.0f + expf(-v[j])) * w2[j];  // te_swiglu_f32 (ops.c:397-405)
            }
        }
        split_store8(v, row, K >> 5, c, act);
    }
}

// Weight matrices of one launch (same K and type), whose column tiles are
// numbered one after another: segment i holds tiles tile_end[i-1] ..
// tile_end[i]-1.  Split-K partial sums are laid out [split][segment][M][n]
// (n_off: columns before segment i).
constexpr int kMaxGemmSegs = 3;
struct GemmSegsArg {
    const unsigned char *w[kMaxGemmSegs];
    float *out[kMaxGemmSegs];
    const float *resid[kMaxGemmSegs];
    int n[kMaxGemmSegs];
    int tile_end[kMaxGemmSegs];
    int n_off[kMaxGemmSegs + 1];
    int nseg;
};

// Eight weight codes (int8 in two dwords) as bf16, exactly: int8 -> fp32, whose
// upper half is the bf16.
__device__ __forceinline__ uint4 codes_bf16(uint32_t c0, uint32_t c1) {
    uint32_t f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int8_t q = (int8_t)((j < 4 ? c0 : c1) >> (8 * (j & 3)));
        f[j] = __float_as_uint((float)(int)q);
    }
    uint4 r;
    r.x = __builtin_amdgcn_perm(f[1], f[0], 0x07060302u);
    r.y = __builtin_amdgcn_perm(f[3], f[2], 0x07060302u);
    r.z = __builtin_amdgcn_perm(f[5], f[4], 0x07060302u);
    r.w = __builtin_amdgcn_perm(f[7], f[6], 0x07060302u);
    return r;
}

// Four nibbles (one per byte, 0..15) minus 8 as int8: (n + 0x78) ^ 0x80, no carries.
__device__ __forceinline__ uint32_t nibbles_i8(uint32_t n) { return (n + 0x78787878u) ^ 0x80808080u; }

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// grid.x: (weight tile, split, row tile) units, see the index map below; 256 G
// threads = G groups of 4 waves over BM = 32 * WM rows x 128 weight rows; a
// wave's tile is 32 rows x (32 * WM) columns (WM = 4: a group's waves are
// stacked over the rows and share the weight tile; WM = 2: two by two).  Two
// groups take alternate chunks of K and add their sums through LDS at the end:
// two waves per SIMD from one workgroup per CU, with half the split-K partial
// sums of two one-group workgroups (the choice: gemm_plan).
//
// K runs in steps of G chunks of kCh blocks, one chunk per group.  Thread (n, p)
// of the workgroup holds blocks 2p and 2p + 1 of weight row n of the next step
// (36 / 68 bytes) in registers and converts them, a piece per step of the
// second half, into the LDS buffer the group of p / 2 reads next
// (double-buffered, one barrier per step).  LDS holds the converted operand in
// MFMA order, [block][K step][32-row tile][K half][row] in 16-byte pieces (a
// wave reads 1 KiB contiguous; the row's slot is xor 2p, so the 2 G
// threads of a row store to different banks), and the scales d.  The activation
// operand goes from global memory to registers, kCh - 1 blocks ahead.
//
// What bounds it: MFMA, VALU and the board's power together.  A loop of these
// MFMAs alone on random operands runs at 1.75 PFLOP/s (the clock falls to 1.8
// GHz); with the FMAs and LDS reads of a step 1.45, with the conversion 1.3.
// Gate and up of 512 rows at 3B (2 x 11008 x 2048 Q4_0, 92 GFLOP of MFMA) take
// 98-104 us, Q8_0 108-117 us, against 146 and 171 us with the block-scaled int8 digits
// this replaced; converting the weights costs 15 us of it, their loads 5.
//
// GLU: sg.w[0] / sg.w[1] are the gate / up matrices (n rows each); the tile's
// 128 weight rows are 32 gate, 32 up, 32 gate, 32 up, so a lane holds both
// products of an output; the epilogue writes silu(gate) * up (te_swiglu_f32's
// operations) as the next GEMM's operand.  One K split.
//
// W4: rows are 4-byte aligned and hold an even number of blocks; else the
// blocks are read as 16-bit words.
constexpr int kCh = 4;
constexpr int kBN = 128;
template <uint32_t TYPE, int WM, int G, bool GLU, bool W4>
__global__ __launch_bounds__(256 * G, G == 1 ? 2 : 1) void gemm_bf16_kernel(GemmSegsArg sg, size_t row_bytes,
                                                           const unsigned char *__restrict__ act, int M, int K, int per,
                                                           int m_tiles, int units, int n_tiles, float *part,
                                                           unsigned char *glu_out) {
    constexpr int BB = TYPE == kQ4_0 ? 18 : 34;  // bytes per GGUF block
    constexpr int DW = 2 * BB / 4;               // dwords of a pair of blocks
    constexpr int NT = WM;                       // 32-column tiles per wave
    __shared__ __align__(16) uint4 wb_lds[G][2][kCh][2][2 * kBN];
    __shared__ float sd_lds[G][2][kCh][kBN];
    // Workgroups go to the XCDs round-robin; the row tiles of one (weight
    // tile, split) unit stay on one XCD, whose L2 then reads its weights once.
    const int xcd = (int)blockIdx.x & 7, slot_id = (int)blockIdx.x >> 3;
    const int unit = slot_id / m_tiles * 8 + xcd;
    const int m_t = slot_id % m_tiles;
    if (unit >= units) {
        return;
    }
    const int z = unit / n_tiles, tile = unit % n_tiles;
    int seg = 0;
#pragma unroll
    for (int i = 1; i < kMaxGemmSegs; ++i) {
        seg += (i < sg.nseg && tile >= sg.tile_end[i - 1]) ? 1 : 0;
    }
    const int N = sg.n[seg];
    const int n_wg = (tile - (seg > 0 ? sg.tile_end[seg - 1] : 0)) * (GLU ? kBN / 2 : kBN);
    const int tid = threadIdx.x & 255, wave = tid >> 6, lane = tid & 63;
    const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int lr = lane & 31, kh = lane >> 5;
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = (m_t * WM + wm) * 32;
    const bool active = m0 < M;
    const int nb = K / 32;
    const int kb0 = z * per, kb1 = min(nb, kb0 + per);
    // chunks of each group: chunk c is blocks kb0 + (G c + group) kCh ..
    const int n_chunks = (kb1 - kb0 + G * kCh - 1) / (G * kCh);
    auto &wb = wb_lds[group];
    auto &sd = sd_lds[group];

    // ---- weights: global -> registers -> converted in LDS
    // (the 2 G threads of a row read consecutive blocks, the groups' next
    // chunks; sp: the pair of blocks, of group sp / 2)
    const int sn = (int)threadIdx.x / (2 * G), sp = (int)threadIdx.x % (2 * G);
    auto &wb_st = wb_lds[sp >> 1];
    auto &sd_st = sd_lds[sp >> 1];
    const unsigned char *wrow;
    {
        const int i = sn >> 5;
        const int row = min(GLU ? n_wg + (i >> 1) * 32 + (sn & 31) : n_wg + sn, N - 1);
        wrow = (GLU ? sg.w[i & 1] : sg.w[seg]) + (size_t)row * row_bytes;
    }
    uint32_t wreg[DW];
    // load i of chunk c's pair (kLoads in all): 16 bytes, the last one dword.
    // Blocks past the split's end are read from its last ones (no branch
    // around the loads) and not used.
    constexpr int kLoads = (DW + 3) / 4;
    auto load_w = [&](int c, int i) {
        const int b = kb0 + G * c * kCh + 2 * sp;
        if (W4) {
            const unsigned char *p = wrow + (size_t)min(b, kb1 - 2) * BB;
            if (4 * i + 4 <= DW) {
                const u32x4_a4 v = *reinterpret_cast<const u32x4_a4 *>(p + 16 * i);
                wreg[4 * i] = v[0], wreg[4 * i + 1] = v[1], wreg[4 * i + 2] = v[2], wreg[4 * i + 3] = v[3];
            } else {
                wreg[DW - 1] = *reinterpret_cast<const uint32_t *>(p + 4 * (DW - 1));
            }
        } else {
            const uint16_t *h0 = reinterpret_cast<const uint16_t *>(wrow + (size_t)min(b, kb1 - 1) * BB);
            const uint16_t *h1 = reinterpret_cast<const uint16_t *>(wrow + (size_t)min(b + 1, kb1 - 1) * BB);
            uint32_t half[8] = {};
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = 8 * i + k;  // 16-bit word of the pair
                if (e < BB) {
                    half[k] = e < BB / 2 ? h0[e] : h1[e - BB / 2];
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (4 * i + k < DW) {
                    wreg[4 * i + k] = half[2 * k] | half[2 * k + 1] << 16;
                }
            }
        }
    };
    // piece q of the thread's pair of blocks: its block q / 4, K step (q / 2) % 2,
    // K half q % 2; piece 0 of a block also stores its scale
    constexpr int kPieces = 8;
    auto store_w = [&](int buf, int q) {
        const int i = q >> 2, s = (q >> 1) & 1, h = q & 1;
        const int blk = 2 * (sp & 1) + i;
        if ((q & 3) == 0) {
            sd_st[buf][blk][sn] = half_bits(i == 0 ? wreg[0] & 0xffffu : wreg[BB / 4] >> 16) * kActUnscale;
        }
        auto code = [&](int k) {  // dword k of the block's codes
            return i == 0 ? __builtin_amdgcn_alignbyte(wreg[k + 1], wreg[k], 2) : wreg[BB / 4 + 1 + k];
        };
        uint4 v;
        if (TYPE == kQ4_0) {
            v = codes_bf16(nibbles_i8((code(2 * h) >> (4 * s)) & 0x0f0f0f0fu),
                           nibbles_i8((code(2 * h + 1) >> (4 * s)) & 0x0f0f0f0fu));
        } else {
            v = codes_bf16(code(4 * s + 2 * h), code(4 * s + 2 * h + 1));
        }
        wb_st[buf][blk][s][64 * (sn >> 5) + 32 * h + ((sn & 31) ^ (2 * sp))] = v;
    };

    // ---- activations: global -> registers, kCh - 1 blocks ahead
    const unsigned char *a_base = act + (((size_t)(min(m0, (M - 1) & ~31) >> 5) * nb) << 12) + lane * 16;
    uint4 areg[kCh][4];
    auto load_a = [&](int b, int slot, int i) {
        areg[slot][i] = *reinterpret_cast<const uint4 *>(a_base + ((size_t)min(b, kb1 - 1) << 12) + 1024 * i);
    };

    // A step is one 32 x 32 tile of one block: four MFMAs, under which the
    // previous step's sums are scaled and added, the next step's weights are
    // read from LDS and (second half of a chunk) a piece of the next chunk is
    // converted.
    constexpr int kSteps = kCh * NT;
    v16f acc[NT], prev = {};
    float prev_d = 0.0f;
    bf16x8 bw[2][2];
    float bd[2];
    auto load_b = [&](int buf, int step) {
        const int bb = step / NT, tile = wn * NT + step % NT, slot = 64 * tile + (lane ^ (4 * group + 2 * (bb >> 1)));
        bw[step & 1][0] = __builtin_bit_cast(bf16x8, wb[buf][bb][0][slot]);
        bw[step & 1][1] = __builtin_bit_cast(bf16x8, wb[buf][bb][1][slot]);
        bd[step & 1] = sd[buf][bb][32 * tile + lr];
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] = v16f{};
    }
    if (n_chunks > 0) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            load_w(0, i);
        }
#pragma unroll
        for (int i = 0; i < 4 * (kCh - 1); ++i) {
            load_a(kb0 + group * kCh + i / 4, i / 4, i % 4);
        }
#pragma unroll
        for (int q = 0; q < kPieces; ++q) {
            store_w(0, q);
        }
    }
    __syncthreads();
    // One chunk.  LAST: nothing follows, so nothing is loaded or converted for a
    // next one, and blocks past the split's end are skipped.  (The last chunk in
    // the common form loaded and converted itself again, and padded its blocks:
    // much of a short K range.  1 x 64 x 64 8.1 -> 6.5 us, 200 x 2048 x 512 Q4_0
    // 14.0 -> 13.0; 3B Q8_0 layer of 64 rows 102.0 -> 98.6, 7B Q8_0 layer of 512 647
    // -> 631, 3B Q4_0 prompt of 512 8645 -> 8379.)
    auto chunk = [&](const int c, auto last) {
        constexpr bool LAST = decltype(last)::value;
        const int buf = c & 1;
        const int live = LAST ? kb1 - (kb0 + (G * c + group) * kCh) : kCh;
        load_b(buf, 0);
#pragma unroll
        for (int step = 0; step < kSteps; ++step) {
            const int bb = step / NT, t = step % NT;
            if (LAST && bb >= live) {
                continue;
            }
            // One step's share of the global loads: a burst of them would hold
            // the wave (and, in step with it, the others) at their issue.
            // Activations are kCh - 1 blocks ahead: loads return in order, so
            // waiting for activations issued after the weights (from HBM) waits
            // for the weights too.
            if (!LAST || bb == 0) {
#pragma unroll
                for (int i = 0; i < 4 / NT; ++i) {
                    load_a(kb0 + (G * c + group) * kCh + (bb == 0 ? kCh - 1 : G * kCh + bb - 1),
                           (bb + kCh - 1) % kCh, t * (4 / NT) + i);
                }
            }
            if (!LAST) {
#pragma unroll
                for (int i = 0; i < kLoads; ++i) {
                    if (step == i * (kSteps / 2) / kLoads) {
                        load_w(c + 1, i);
                    }
                }
            }
            if (step + 1 < kSteps) {
                load_b(buf, step + 1);
            }
            // the loads are issued here, not sunk towards their use
            __builtin_amdgcn_sched_barrier(0);
            const bf16x8 b0 = bw[step & 1][0], b1 = bw[step & 1][1];
            v16f s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, areg[bb][0]), b0, v16f{},
                                                             0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, areg[bb][1]), b1, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, areg[bb][2]), b0, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, areg[bb][3]), b1, s, 0, 0, 0);
            const int tp = (t + NT - 1) % NT;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[tp][r] = fmaf(prev[r], prev_d, acc[tp][r]);
            }
            // pieces over the second half of the chunk's steps
            constexpr int kPer = kPieces / (kSteps / 2);
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                if (!LAST && step >= kSteps / 2) {
                    store_w(buf ^ 1, (step - kSteps / 2) * kPer + i);
                }
            }
            prev = s;
            prev_d = bd[step & 1];
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    };
    for (int c = 0; c + 1 < n_chunks; ++c) {
        chunk(c, std::false_type{});
    }
    chunk(n_chunks - 1, std::true_type{});
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc[NT - 1][r] = fmaf(prev[r], prev_d, acc[NT - 1][r]);
    }
    // Each group finishes the tiles it owns: the other's sums of them come
    // through LDS (group 0's first, then group 1's)
    auto owns = [&](int g, int t) { return G == 1 || (NT == 4 ? t / 2 == g : GLU ? g == 0 : t == g); };
    if constexpr (G == 2) {
        float4 *xs = reinterpret_cast<float4 *>(&wb_lds[0][0][0][0][0]);
        static_assert(sizeof(wb_lds) >= NT * 4 * 16 * 64 * sizeof(float), "the exchange fits the weight stages");
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (!owns(group, t)) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    xs[((t * 4 + wave) * 4 + q) * 64 + lane] =
                        make_float4(acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (owns(group, t)) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = xs[((t * 4 + wave) * 4 + q) * 64 + lane];
                    acc[t][4 * q] += v.x, acc[t][4 * q + 1] += v.y, acc[t][4 * q + 2] += v.z, acc[t][4 * q + 3] += v.w;
                }
            }
        }
    }
    // lane holds column lr of rows 8 * (r / 4) + 4 * kh + r % 4 of each 32 x 32 tile
    if constexpr (GLU) {
        // silu(gate) * up, split and turned through LDS into the operand's
        // order (rows of 32 + 1 dwords: hi | lo << 16)
        uint32_t *xch = reinterpret_cast<uint32_t *>(&wb_lds[G - 1][0][0][0][0]) + (group * 4 + wave) * (32 * 33);
        static_assert(sizeof(wb_lds[0]) >= NT * 4 * 16 * 64 * sizeof(float) && sizeof(wb_lds[0]) >= G * 4 * 32 * 33 * 4,
                      "the exchange and the turned tiles each fit one group's weight stages");
        const int nb_out = N / 32;
#pragma unroll
        for (int p = 0; p < NT / 2; ++p) {
            const int b = n_wg / 32 + wn * (NT / 2) + p;
            if (!owns(group, 2 * p) || !active || b >= nb_out) {
                continue;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float g = acc[2 * p][r], u = acc[2 * p + 1][r];
                const float v = g / (1.0f + expf(-g)) * u;  // te_swiglu_f32 (ops.c:397-405)
                xch[(8 * (r >> 2) + 4 * kh + (r & 3)) * 33 + lr] = split_pack(v);
            }
            // only this wave's own slice: its writes before its reads
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            unsigned char *dst = glu_out + (((size_t)(m0 >> 5) * nb_out + b) << 12) + lane * 16;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t e[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    e[j] = xch[lr * 33 + 16 * s + 8 * kh + j];
                }
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    hi[j] = __builtin_amdgcn_perm(e[2 * j + 1], e[2 * j], 0x05040100u);
                    lo[j] = __builtin_amdgcn_perm(e[2 * j + 1], e[2 * j], 0x07060302u);
                }
                *reinterpret_cast<uint4 *>(dst + 1024 * s) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                *reinterpret_cast<uint4 *>(dst + 2048 + 1024 * s) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            }
        }
        return;
    }
    if (!active) {
        return;
    }
    const bool one = units == n_tiles;  // one split
    float *dst = one ? sg.out[seg] : part + ((size_t)z * sg.n_off[sg.nseg] + sg.n_off[seg]) * M;
    const float *resid = one ? sg.resid[seg] : nullptr;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int col = n_wg + 32 * (wn * NT + t) + lr;
        if (owns(group, t) && col < N) {
            // Every residual before the first store: out may be resid, so a load
            // after a store would wait for it, 16 * NT round trips one by one
            // (an element is one lane's alone; rows past M load row M - 1).  512 x
            // 18944 x 64 with a residual 53.8 -> 24.3 us, two 0.5B layers of 512 rows
            // 215.4 -> 207.4.
            float rv[16] = {};
            if (resid != nullptr) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = min(m0 + 8 * (r >> 2) + 4 * kh + (r & 3), M - 1);
                    rv[r] = resid[(size_t)row * N + col];
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + 8 * (r >> 2) + 4 * kh + (r & 3);
                if (row < M) {
                    dst[(size_t)row * N + col] = resid != nullptr ? rv[r] + acc[t][r] : acc[t][r];
                }
            }
        }
    }
}

// part[0][i] + part[1][i] + ... + part[splits-1][i], added in split order,
// for W consecutive elements at i (W = 4: 16-byte loads); the splits' loads
// are issued eight at a time.
template <int W>
struct Vals {
    float v[W];
};
template <int W>
__device__ __forceinline__ Vals<W> load_vals(const float *p) {
    Vals<W> r;
    if constexpr (W == 4) {
        const float4 a = *reinterpret_cast<const float4 *>(p);
        r.v[0] = a.x, r.v[1] = a.y, r.v[2] = a.z, r.v[3] = a.w;
    } else {
        r.v[0] = *p;
    }
    return r;
}
template <int W>
__device__ __forceinline__ void store_vals(float *p, const Vals<W> &r) {
    if constexpr (W == 4) {
        *reinterpret_cast<float4 *>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
    } else {
        *p = r.v[0];
    }
}
template <int W>
__device__ __forceinline__ Vals<W> sum_splits(const float *__restrict__ part, int splits, size_t count, size_t i) {
    Vals<W> a = load_vals<W>(part + i);
    for (int z0 = 1; z0 < splits; z0 += 8) {
        Vals<W> b[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (z0 + u < splits) {
                b[u] = load_vals<W>(part + (size_t)(z0 + u) * count + i);
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (z0 + u < splits) {
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    a.v[j] += b[u].v[j];
                }
            }
        }
    }
    return a;
}

// out = (resid +) the splits' partial sums, added in split order, for every
// segment of a segmented launch (element i of the [segment][M][n] order),
// W elements per thread (W = 4: every pointer 16-byte aligned and every
// segment boundary M * n_off a multiple of 4, so four elements never straddle
// one).
template <int W>
__global__ __launch_bounds__(256) void gemm_reduce_segs_kernel(const float *__restrict__ part, int splits, int M,
                                                               GemmSegsArg sg) {
    const size_t count = (size_t)M * sg.n_off[sg.nseg];
    for (size_t i = (blockIdx.x * (size_t)256 + threadIdx.x) * W; i < count; i += (size_t)gridDim.x * 256 * W) {
        int seg = 0;
#pragma unroll
        for (int t = 1; t < kMaxGemmSegs; ++t) {
            seg += (t < sg.nseg && i >= (size_t)M * sg.n_off[t]) ? 1 : 0;
        }
        Vals<W> a = sum_splits<W>(part, splits, count, i);
        const size_t j = i - (size_t)M * sg.n_off[seg];
        if (sg.resid[seg] != nullptr) {
            const Vals<W> r = load_vals<W>(sg.resid[seg] + j);
#pragma unroll
            for (int k = 0; k < W; ++k) {
                a.v[k] = r.v[k] + a.v[k];
            }
        }
        store_vals<W>(sg.out[seg] + j, a);
    }
}

// gemm_reduce_kernel's sums for one row (resid + the splits' partial sums in
// split order -> out), then that row's RMSNorm operand into act, exactly as
// split_act_kernel<kActRmsNorm> computes it from out: thread t holds columns
// 8t .. 8t + 7 of each of P passes of kActPass, summed into the fp64 sum of
// squares in row_sum_squares's order, and splits them as split_act_kernel's
// thread t does.  One workgroup per row, N <= P * kActPass, N % 32 == 0,
// splits <= rms_splits(P) (what the registers hold).  Every load, the norm weights' included, is issued before the
// first store (out may be resid), so all of a thread's loads are in flight
// together.  Bound by its two rounds of latency (loads, the row's sum) and the
// launch; two passes of 256 threads rather than 512 threads keep
// split_act_kernel's sum order.  P = 2 against the separate sums and operand
// launches, 7B, two layers (three such places): Q4_0 181 rows 613.9 -> 610.3
// us, 12 rows 321.5 -> 319.4, Q8_0 21 rows 395.2 -> 392.4.
constexpr int kRmsSplits = 16;  // also the most splits of a launch
// (P = 2: 228 VGPRs, two waves per SIMD; a 7B down takes up to 9 splits)
constexpr int rms_splits(int passes) { return passes == 1 ? kRmsSplits : 12; }
template <int P>
__global__ __launch_bounds__(kActThreads) void gemm_reduce_rms_kernel(const float *__restrict__ part, int splits,
                                                                      size_t count, const float *resid, float *out,
                                                                      int M, int N, const float *__restrict__ norm_w,
                                                                      float eps, unsigned char *__restrict__ act,
                                                                      bool vec) {
    constexpr int S = rms_splits(P);
    const size_t row = xcd_row(blockIdx.x, M);
    if (row >= (size_t)M) {
        return;
    }
    const int c0 = 8 * (int)threadIdx.x;
    const size_t o0 = row * (size_t)N;
    float pv[P][S][8], rv[P][8] = {}, wv[P][8];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = c0 + i * kActPass;
        const int cl = c < N ? c : 0;  // threads past the row load column 0 and store nothing
#pragma unroll
        for (int z = 0; z < S; ++z) {
            if (z < splits) {
                load8(part + (size_t)z * count + o0 + cl, vec, pv[i][z]);
            }
        }
        if (resid != nullptr) {
            load8(resid + o0 + cl, vec, rv[i]);
        }
        load8(norm_w + cl, vec, wv[i]);
    }
    float xv[P][8];
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const bool mine = c0 + i * kActPass < N;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float a = pv[i][0][j];
#pragma unroll
            for (int z = 1; z < S; ++z) {
                if (z < splits) {
                    a += pv[i][z][j];
                }
            }
            xv[i][j] = resid != nullptr ? rv[i][j] + a : a;
            const double d = (double)xv[i][j];
            ss += mine ? d * d : 0.0;
        }
    }
#pragma unroll
    for (int i = 0; i < P; ++i) {
        if (c0 + i * kActPass < N) {
            store8(out + o0 + c0 + i * kActPass, vec, xv[i]);
        }
    }
    const float rms = 1.0f / sqrtf((float)(row_sum_squares(ss) / (double)N) + eps);
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int c = c0 + i * kActPass;
        if (c < N) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                xv[i][j] = xv[i][j] * rms * wv[i][j];
            }
            split_store8(xv[i], row, N >> 5, c, act);
        }
    }
}

// out = (resid +) the splits' partial sums, added in split order, W
// elements per thread (W = 4: count % 4 == 0 and every pointer 16-byte
// aligned).
template <int W>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float *__restrict__ part, int splits, size_t count,
                                                          const float *resid, float *out) {
    for (size_t i = (blockIdx.x * (size_t)256 + threadIdx.x) * W; i < count; i += (size_t)gridDim.x * 256 * W) {
        Vals<W> a = sum_splits<W>(part, splits, count, i);
        if (resid != nullptr) {
            const Vals<W> r = load_vals<W>(resid + i);
#pragma unroll
            for (int k = 0; k < W; ++k) {
                a.v[k] = r.v[k] + a.v[k];
            }
        }
        store_vals<W>(out + i, a);
    }
}

}  // namespace

namespace te_hip {

static bool aligned16(const void *p) {
    return ((uintptr_t)p & 15u) == 0;
}

// 32-row tiles, hi and lo; 16 bytes so that any pointer has an aligned base
size_t act_buffer_bytes(size_t rows, size_t cols) { return (rows + 31) / 32 * 32 * cols * 4 + 16; }

te_status launch_split_act(int pre, const float *x, const float *x2, const float *norm_w, float eps, size_t rows,
                           size_t cols, void *act, hipStream_t stream) {
    if (rows == 0 || cols == 0 || cols % 32 != 0 || rows > 0x7fffffffu || cols > (1u << 24)) {
        return TE_STATUS_UNSUPPORTED;
    }
    unsigned char *a = act_base(act);
    const bool vec = aligned16(x) && (pre != kActSwiGLU || aligned16(x2)) && (pre != kActRmsNorm || aligned16(norm_w));
    // without a row-wide norm, the row's passes of kActPass values are spread over workgroups
    const dim3 grid((unsigned)(8 * xcd_rows(rows)), pre == kActRmsNorm ? 1u : (unsigned)std::max<size_t>(1, cols / kActPass));
    if (pre == kActRmsNorm) {
        split_act_kernel<kActRmsNorm><<<grid, kActThreads, 0, stream>>>(x, x2, norm_w, eps, (int)rows, (int)cols, a, vec);
    } else if (pre == kActSwiGLU) {
        split_act_kernel<kActSwiGLU><<<grid, kActThreads, 0, stream>>>(x, x2, norm_w, eps, (int)rows, (int)cols, a, vec);
    } else {
        split_act_kernel<kActPlain><<<grid, kActThreads, 0, stream>>>(x, x2, norm_w, eps, (int)rows, (int)cols, a, vec);
    }
    return launch_status();
}

// Rows per workgroup (32 * wm), groups per workgroup, K splits and their
// length, from the estimated time of a launch.  A (weight tile, split) unit and
// its row tiles stay on one XCD, so the rounds of one workgroup per CU are
// counted per XCD (28 weight tiles x 3 splits x 3 row tiles: 252 workgroups,
// but 33 on some XCDs, measured 145 us against 111 with 2 splits).
//   One round: two groups per workgroup.  A pair of chunks takes 3.4 us at 128
//   rows on 64 CUs and 4.9 on all 256 (the clock falls), 2.5 and 3.0 at 64.
//   More: two one-group workgroups per CU, which fill each other's waits (512
//   x 22016 x 2048 Q4_0 107-111 us against 110 in two-group workgroups, Q8_0
//   111-113 against 116; 512 x 37888 x 3584 274-276 against 276-277, 296-299
//   against 302-304); a round's pair takes 4.2 and 2.8 us.
// The partial sums are written and read back at 2.7 TB/s.
struct GemmPlan {
    int wm, groups;
    size_t per, splits;  // blocks of K per split, a multiple of two chunks
};
static GemmPlan gemm_plan(size_t rows, size_t n, size_t n_tiles, size_t nb, size_t splits_max) {
    const size_t pairs = (nb + 2 * kCh - 1) / (2 * kCh);
    const double cus = (double)device_compute_units();
    GemmPlan best = {};
    double best_us = 0.0;
    for (int wm = 2; wm <= 4; wm += 2) {
        const size_t m_tiles = (rows + 32 * wm - 1) / (32 * wm);
        for (size_t want = 1; want <= std::min<size_t>(splits_max, kRmsSplits); ++want) {
            const size_t per = (pairs + want - 1) / want;
            const size_t splits = (pairs + per - 1) / per;
            const double per_xcd = (double)((n_tiles * splits + 7) / 8 * m_tiles);
            const double rounds = ceil(per_xcd * 8.0 / cus);
            const double busy = std::min(1.0, per_xcd * 8.0 / cus);
            const double pair_us = rounds > 1.0 ? (wm == 4 ? 4.2 : 2.8) : wm == 4 ? 3.0 + 1.9 * busy : 2.1 + 0.9 * busy;
            const double us = rounds * (pair_us * (double)per + 3.5) +
                              (splits > 1 ? 2.0 + (double)(splits * rows * n) * 8.0 / 2.7e6 : 0.0);
            if (best.wm == 0 || us < best_us) {
                best_us = us;
                best = {wm, rounds > 1.0 ? 1 : 2, per * 2 * kCh, splits};
            }
        }
    }
    return best;
}

// One gemm_bf16_kernel launch.
static te_status launch_tiles(uint32_t ggml_type, bool glu, bool w4, const GemmSegsArg &sg, size_t row_bytes,
                              const void *act, size_t rows, size_t k, const GemmPlan &plan, size_t n_tiles,
                              float *part, void *glu_out, hipStream_t stream) {
    const size_t wm = (size_t)plan.wm;
    const size_t m_tiles = (rows + 32 * wm - 1) / (32 * wm);
    const size_t units = n_tiles * plan.splits;
    const size_t blocks = (units + 7) / 8 * 8 * m_tiles;
    if (blocks > 0x7fffffffu) {
        return TE_STATUS_UNSUPPORTED;
    }
    auto go = [&](auto type, auto wmc, auto g, auto gluc, auto w4c) {
        gemm_bf16_kernel<decltype(type)::value, decltype(wmc)::value, decltype(g)::value, decltype(gluc)::value,
                         decltype(w4c)::value>
            <<<(unsigned)blocks, 256 * decltype(g)::value, 0, stream>>>(
                sg, row_bytes, act_base(const_cast<void *>(act)), (int)rows, (int)k, (int)plan.per, (int)m_tiles,
                (int)units, (int)n_tiles, part, glu_out == nullptr ? nullptr : act_base(glu_out));
    };
    auto with_w4 = [&](auto type, auto wmc, auto g, auto gluc) {
        if (w4) {
            go(type, wmc, g, gluc, std::true_type{});
        } else {
            go(type, wmc, g, gluc, std::false_type{});
        }
    };
    auto with_glu = [&](auto type, auto wmc, auto g) {
        if (glu) {
            with_w4(type, wmc, g, std::true_type{});
        } else {
            with_w4(type, wmc, g, std::false_type{});
        }
    };
    auto with_g = [&](auto type, auto wmc) {
        if (plan.groups == 2) {
            with_glu(type, wmc, std::integral_constant<int, 2>{});
        } else {
            with_glu(type, wmc, std::integral_constant<int, 1>{});
        }
    };
    auto with_wm = [&](auto type) {
        if (wm == 2) {
            with_g(type, std::integral_constant<int, 2>{});
        } else {
            with_g(type, std::integral_constant<int, 4>{});
        }
    };
    if (ggml_type == kQ4_0) {
        with_wm(std::integral_constant<uint32_t, kQ4_0>{});
    } else {
        with_wm(std::integral_constant<uint32_t, kQ8_0>{});
    }
    return launch_status();
}

// Whether a tensor's rows can be read as dwords holding whole pairs of blocks.
static bool rows_w4(const void *w, size_t row_bytes) { return ((uintptr_t)w & 3u) == 0 && row_bytes % 4 == 0; }

te_status launch_gemm_q_segs(uint32_t ggml_type, const GemmSeg *segs, int nseg, const void *act, size_t rows,
                             size_t k, float *partials, size_t partial_bytes, hipStream_t stream,
                             const GemmRmsDigits *post) {
    if ((ggml_type != kQ4_0 && ggml_type != kQ8_0) || k % 32 != 0 || rows == 0 || rows > 0x7fffffffu ||
        k > (1u << 24) || nseg < 1 || nseg > kMaxGemmSegs) {
        return TE_STATUS_UNSUPPORTED;
    }
    if (post != nullptr && nseg != 1) {
        return TE_STATUS_INVALID_ARGUMENT;  // the operand is of one output
    }
    const size_t row_bytes = k / 32 * (ggml_type == kQ4_0 ? 18 : 34);
    bool w4 = true;
    size_t n_total = 0, tiles_n = 0;
    for (int i = 0; i < nseg; ++i) {
        if (segs[i].n == 0 || segs[i].n > 0x7fffffffu || ((size_t)segs[i].w & 1u) != 0 ||
            (segs[i].resid != nullptr) != (segs[0].resid != nullptr)) {
            return TE_STATUS_UNSUPPORTED;
        }
        w4 = w4 && rows_w4(segs[i].w, row_bytes);
        n_total += segs[i].n;
        tiles_n += (segs[i].n + kBN - 1) / kBN;
    }
    if (n_total > 0x7fffffffu) {
        return TE_STATUS_UNSUPPORTED;
    }
    const size_t splits_max =
        partials == nullptr ? 1 : std::max<size_t>(1, partial_bytes / (rows * n_total * sizeof(float)));
    const GemmPlan plan = gemm_plan(rows, n_total, tiles_n, k / 32, splits_max);
    const size_t splits = plan.splits;
    GemmSegsArg sg = {};
    sg.nseg = nseg;
    int tile_end = 0;
    for (int i = 0; i < nseg; ++i) {
        sg.w[i] = static_cast<const unsigned char *>(segs[i].w);
        sg.out[i] = segs[i].out;
        sg.resid[i] = segs[i].resid;
        sg.n[i] = (int)segs[i].n;
        tile_end += (int)((segs[i].n + kBN - 1) / kBN);
        sg.tile_end[i] = tile_end;
        sg.n_off[i + 1] = sg.n_off[i] + (int)segs[i].n;
    }
    const size_t n = segs[0].n;
    float *out = segs[0].out;
    const float *res = segs[0].resid;
    te_status st = launch_tiles(ggml_type, false, w4, sg, row_bytes, act, rows, k, plan, tiles_n, partials,
                                nullptr, stream);
    if (st != TE_STATUS_OK) {
        return st;
    }
    // the RMSNorm operand of a single output: fused into the split-K sums
    // where the row fits the fused kernel, else from out afterwards
    const bool rms = post != nullptr && nseg == 1 && n % 32 == 0;
    bool rms_done = false;
    if (splits > 1) {
        const size_t count = rows * n_total;
        bool vec = aligned16(partials) && count % 4 == 0;
        for (int i = 0; i < nseg; ++i) {
            vec = vec && aligned16(sg.out[i]) && aligned16(sg.resid[i]) && (rows * (size_t)sg.n_off[i + 1]) % 4 == 0;
        }
        const int width = vec ? 4 : 1;
        const unsigned blocks = (unsigned)std::min<size_t>((count / width + 255) / 256, 4096);
        const char *env = getenv("TE_HIP_GEMM_REDUCE_RMS");
        // one pass of a row up to 2048 wide, two up to 4096 (the 7B width); wider
        // rows take two launches, as the registers hold no third pass
        const size_t passes = (n + kActPass - 1) / kActPass;
        if (rms && passes <= 2 && splits <= (size_t)rms_splits((int)passes) && !(env != nullptr && env[0] == '0')) {
            auto *kernel = passes == 1 ? gemm_reduce_rms_kernel<1> : gemm_reduce_rms_kernel<2>;
            kernel<<<(unsigned)(8 * xcd_rows(rows)), kActThreads, 0, stream>>>(
                partials, (int)splits, count, res, out, (int)rows, (int)n, post->norm_w, post->eps, act_base(post->act_out),
                vec && aligned16(post->norm_w));
            rms_done = true;
        } else if (nseg == 1) {
            if (vec) {
                gemm_reduce_kernel<4><<<blocks, 256, 0, stream>>>(partials, (int)splits, count, res, out);
            } else {
                gemm_reduce_kernel<1><<<blocks, 256, 0, stream>>>(partials, (int)splits, count, res, out);
            }
        } else if (vec) {
            gemm_reduce_segs_kernel<4><<<blocks, 256, 0, stream>>>(partials, (int)splits, (int)rows, sg);
        } else {
            gemm_reduce_segs_kernel<1><<<blocks, 256, 0, stream>>>(partials, (int)splits, (int)rows, sg);
        }
        st = launch_status();
    }
    if (st == TE_STATUS_OK && post != nullptr && !rms_done) {
        st = launch_split_act(kActRmsNorm, out, nullptr, post->norm_w, post->eps, rows, n, post->act_out, stream);
    }
    return st;
}

te_status launch_gemm_q(const void *weights, uint32_t ggml_type, const void *act, size_t rows, size_t n, size_t k,
                        float *out, const float *resid, float *partials, size_t partial_bytes, hipStream_t stream) {
    const GemmSeg seg = {weights, out, resid, n};
    return launch_gemm_q_segs(ggml_type, &seg, 1, act, rows, k, partials, partial_bytes, stream, nullptr);
}

te_status launch_gemm_q_rms(const void *weights, uint32_t ggml_type, const void *act, size_t rows, size_t n,
                            size_t k, float *out, const float *resid, float *partials, size_t partial_bytes,
                            const float *norm_w, float eps, void *act_out, hipStream_t stream) {
    const GemmSeg seg = {weights, out, resid, n};
    const GemmRmsDigits post = {norm_w, eps, act_out};
    return launch_gemm_q_segs(ggml_type, &seg, 1, act, rows, k, partials, partial_bytes, stream, &post);
}

te_status launch_gemm_glu_q(uint32_t ggml_type, const void *gate_w, const void *up_w, const void *act, size_t rows,
                            size_t n, size_t k, void *act_out, hipStream_t stream, bool *launched) {
    *launched = false;
    const size_t row_bytes = k / 32 * (ggml_type == kQ4_0 ? 18 : 34);
    const size_t n_tiles = (n + kBN / 2 - 1) / (kBN / 2);
    const size_t tiles = n_tiles * ((rows + 127) / 128);
    const char *env = getenv("TE_HIP_GEMM_GLU");
    if ((ggml_type != kQ4_0 && ggml_type != kQ8_0) || k % 32 != 0 || n % 32 != 0 || rows == 0 ||
        rows > 0x7fffffffu || n > 0x7fffffffu || k > (1u << 24) || ((size_t)gate_w & 1u) != 0 ||
        ((size_t)up_w & 1u) != 0 || (env != nullptr && env[0] == '0') ||
        (tiles < (size_t)device_compute_units() / 2 && !(env != nullptr && env[0] == '1'))) {
        return TE_STATUS_OK;  // not launched: the caller runs the two GEMMs and the SwiGLU operand
    }
    GemmSegsArg sg = {};
    sg.nseg = 1;
    sg.w[0] = static_cast<const unsigned char *>(gate_w);
    sg.w[1] = static_cast<const unsigned char *>(up_w);
    sg.n[0] = (int)n;
    sg.tile_end[0] = (int)n_tiles;
    sg.n_off[1] = (int)n;
    const bool w4 = rows_w4(gate_w, row_bytes) && rows_w4(up_w, row_bytes);
    GemmPlan plan = gemm_plan(rows, n, n_tiles, k / 32, 1);
    // The groups that one projection's tiles take in one K split: where the two
    // GEMMs run unsplit too, the sums are theirs bit for bit (the layer flow's
    // partials let them split K at few rows, 3B and 1.5B at 8-64: not there).
    // Where the pair's own tiles exceed the CUs and one projection's do not, its
    // own plan would take one-group workgroups, two per CU; the override against
    // that, two layers, us: 7B 8 / 64 / 128 rows Q4_0 284 : 290, 325 : 333, 448 :
    // 442, Q8_0 374 : 405, 405 : 438, 519 : 543; 3B Q4_0 129 / 256 rows 270 : 263,
    // 311 : 301; 1.5B 129 / 256 192 : 187, 250 : 235; 0.5B 512 rows 207 : 196.
    plan.groups = gemm_plan(rows, n, (n + kBN - 1) / kBN, k / 32, 1).groups;
    *launched = true;
    return launch_tiles(ggml_type, true, w4, sg, row_bytes, act, rows, k, plan, n_tiles, nullptr, act_out, stream);
}

}  // namespace te_hip

// Test entry point: Y = pre(X) * W^T (+ R) through the two launches above, on
// device pointers; `act` is scratch of te_hip_gemm_act_bytes(rows, k) bytes.
extern "C" size_t te_hip_gemm_act_bytes(size_t rows, size_t k) {
    return te_hip::act_buffer_bytes(rows, k);
}

extern "C" te_status te_hip_gemm_q_f32(const void *weights, uint32_t ggml_type, const float *x, const float *x2,
                                       const float *norm_w, float epsilon, int pre, size_t rows, size_t n, size_t k,
                                       float *out, const float *resid, void *act, float *partials,
                                       size_t partial_bytes, void *stream) {
    if (weights == nullptr || x == nullptr || out == nullptr || act == nullptr || pre < 0 || pre > 2 ||
        (pre == kActRmsNorm && (norm_w == nullptr || !(epsilon > 0.0f))) || (pre == kActSwiGLU && x2 == nullptr)) {
        return TE_STATUS_INVALID_ARGUMENT;
    }
    hipStream_t s = te_hip::as_stream(stream);
    te_status st = te_hip::launch_split_act(pre, x, x2, norm_w, epsilon, rows, k, act, s);
    if (st != TE_STATUS_OK) {
        return st;
    }
    return te_hip::launch_gemm_q(weights, ggml_type, act, rows, n, k, out, resid, partials, partial_bytes, s);
}
