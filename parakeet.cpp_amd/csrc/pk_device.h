// pk_device.h -- device code of the MI355X transducer greedy decode.
//
// Included once, by pk_decode.hip.  See that file for the host side and the
// overall structure; this file holds the data layout, the building blocks
// (MFMA tiles over q8_0 / f16 weights, argmax keys, domain barrier, coherent
// loads and stores) and the kernels.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "exchange_word.h"
#include "parakeet_hip.h"

namespace pkdev {

constexpr int kWave = 64;
constexpr int kBlock = 512;                 // 8 waves per workgroup, one workgroup per CU
constexpr int kWaves = kBlock / kWave;
constexpr int kTile = 16;                   // MFMA tile edge (rows = outputs, columns = utterances)
constexpr int kMaxNT = 2;                   // utterance tiles per domain
constexpr int kDomCap = kTile * kMaxNT;     // utterances per domain
constexpr int kColCap = kDomCap;            // joint columns per domain and iteration (argmax key slots)
constexpr int kSmallB = 4;                  // LSTM batch at or below which layer 0 runs redundantly
constexpr int kIdxBits = 14;                // argmax key: index field
constexpr int kStampShift = 46;             // argmax key: 14 index + 32 value bits below the stamp
constexpr unsigned kMaxStamp = (1u << 18) - 1;
constexpr int kFlagStride = 32;             // words between barrier flags (128 B, one L2 line)
// error word of a launch whose ordinary dispatch was not co-resident (never returned to a caller:
// the host relaunches the call cooperatively)
constexpr int kStatusNotResident = 0x7001;
constexpr int kKPad = 8;                    // halves of padding per staged row (bank spread)

// Flags in the per-utterance control word.
constexpr int kFlagZeroHC = 1;              // LSTM input state is zero (init / EOU reset)
constexpr int kFlagTokOverflow = 2;
constexpr int kFlagSegOverflow = 4;
constexpr int kFlagTraceOverflow = 8;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A weight matrix [rows][K] laid out as MFMA fragments: for row tile t and
// K block kb (32 columns), lane l holds the 8 consecutive weights of row
// 16t + l%16 starting at column 32kb + 8(l/16).  f16: 8 halves per lane,
// [t][kb][lane]; f32: two f16 planes holding hi = f16(w), lo = f16(w - hi).
// q8_0: 8 bytes q ^ 0x80 per lane and block (the int8 values offset by 128, so
// the conversion needs no xor), stored per unit of kQ8Unit = 5 blocks as one
// kQ8UnitBytes record [t][unit]: lane l's 16 bytes of blocks 0-1 (1 KB for the
// 64 lanes), of blocks 2-3 (1 KB), its 8 bytes of block 4 (512 B), then the
// block scales (the stored f16 bits), 16 bytes per row r = d[16t + r] of
// blocks 0-4 and three zeros.  A unit is then 4 wave loads (16 + 16 + 8 bytes
// of quants, 16 bytes of scales per lane) instead of 10: the products are paced
// by the number of vector memory instructions per CU, not by bytes.
//
// Products are computed transposed: the staged activations are the MFMA A
// operand (rows = utterances) and the weight fragment the B operand (columns =
// weight rows), so a D fragment lane holds ONE weight row (l%16) for four
// utterances (4(l/16) .. +3) and a q8_0 block needs one scale per lane.
struct TMat {
    const void *a;                 // fragment plane (f32 weights: the hi plane, then the lo plane)
    const void *a_lo;              // f32 weights: the lo plane (a + one plane)
    const unsigned short *scale;   // q8_0 block scales, f16 bits
    int type;                      // PK_TYPE_Q8_0, PK_TYPE_F16, PK_TYPE_F32
    int rows, tiles, KB;           // KB: stored K blocks of 32 per tile row (q8_0: padded to whole units)
    int KBa;                       // K blocks that hold weights (K / 32); blocks KBa .. KB-1 are zero
    int lds_off;                   // byte offset of this workgroup's tiles in its LDS weight cache, -1: not cached
};

constexpr int kQ8Unit = 5, kQ8UnitBytes = 2 * 1024 + 512 + 16 * 16;   // q8_0 unit record (see TMat)
constexpr int kQ8Scales = 2560;                                        // offset of its scales

// Bytes of one tile row of a matrix (KB stored blocks), as stored and as cached
// in LDS: q8_0 unit records; f16 fragments; f32 hi then lo fragments.
__host__ __device__ constexpr int tile_bytes(int type, int KB) {
    return type == PK_TYPE_Q8_0 ? KB / kQ8Unit * kQ8UnitBytes : type == PK_TYPE_F16 ? KB * 1024 : KB * 2048;
}

struct KParams {
    int kind, H, L, J, V1, Dn, Vo, blank, eou, eob, max_sym, n_dur;
    int durations[PK_MAX_DURATIONS];
    const float *eproj;                      // [V1][4H] W_ih0 . embed[v] + b_ih0 + b_hh0, unit-major
    TMat w_ih[PK_MAX_LAYERS], w_hh[PK_MAX_LAYERS];   // unit-major gate rows (w_ih[0] unused)
    const float *b_lstm[PK_MAX_LAYERS];      // b_ih + b_hh (unit-major), layers >= 1
    TMat w_pred, w_out;
    const float *b_pred, *b_out;
    const unsigned char *special;
    int n_special;
    // slot state (persistent between calls)
    float *slot_h;       // [slots][L][H]
    float *slot_c;       // [slots][L][H]
    float *slot_pp;      // [slots][J]  b_p + W_p . h[L-1]
    float *slot_r;       // [slots][L][4H]  W_hh . h (no bias), unit-major rows
    int *slot_ctrl;      // [slots][PK_CTRL_N]
    // batch
    int n_utts;
    const float *encp;           // [rows][J] b_e + W_e . enc
    long long encp_rows;
    const long long *encp_row;   // [n_utts]
    const int *T;
    const int *slot;
    const float *blank_bias;     // nullable
    const int *tokens_base;      // nullable
    int *tokens; int token_cap;
    int *n_tokens; int *steps;
    int *segs; int seg_cap; int *n_segs;
    int *trace; int trace_cap;
    float *logits; int logit_steps;   // nullable debug tap [n_utts][logit_steps][Vo]
    float *lcol;                 // tap staging [n_dom][kColCap][Vo]: each joint column's logits of one
                                 // iteration, copied to the row of the step that takes the column
    const int *reset;            // nullable [n_utts]: 1 = fresh state whatever the slot holds
    int *ctrl_out;               // nullable [n_utts][PK_CTRL_N]: control words after the call
    // exchange buffers of one launch (one allocation from hs, xchg_bytes long; coherent accesses).
    // State by batch index, read and written by the workgroup that owns the units except where
    // layer 0 runs redundantly:
    float *hs;           // [L][n][H]      h of every layer (for the slots at the end)
    float *cx;           // [2][n][H]      c of layer 0, ping-pong by utterance parity
    float *rx;           // [2][n][4H]     W_hh0 . h0 (no bias), unit-major rows, ping-pong like cx
    // Data every workgroup of a domain waits for, word by word (kEmpty until written):
    float *hx;           // [L - hl0][2][n_dom][H/4][rows][4]  h of one LSTM step by list position; the
                         // 4 units x rows of a tile are one producer's whole lines
    float *ppx;          // [2][n_dom][J/16][prows][16]  b_p + W_p . h by domain utterance and parity
    int rows, prows;     // row capacities (powers of two >= utterances per domain; rows >= 8)
    int hl0;             // first layer of hx: 1 where layer 0 always runs redundantly
    unsigned xchg_bytes;
    // domains: independent utterance groups, each on dom_size workgroups
    int n_dom, dom_size, nt;
    const int *dom_n;            // [n_dom] utterances per domain
    const int *dom_list;         // [n_dom][kDomCap] batch indices
    const int *wg_dom;           // [nwg] domain of a workgroup
    const int *wg_rank;          // [nwg] rank inside its domain
    const int *dom_wg;           // [n_dom][dom_size] workgroup of each rank
    // sync
    unsigned *flags;             // [nwg * kFlagStride]
    // argmax keys by iteration parity, stamped with the iteration: each workgroup's best token key
    // per joint column, and the duration keys of the one or two ranks that own duration rows
    unsigned long long *keys;    // [2][n_dom][P][cols] then [2][n_dom][2][cols]
    int cols;                    // column capacity: 16 or 32
    int dur_rank[2], n_durk;     // ranks that own duration rows (n_durk of them)
    int *status;                 // [0] error code, [1] iterations, [2] overflow, [3] trace overflow,
                                 // [9] co-residency decision (cleared per launch)
    unsigned arrive_ticks;       // ordinary dispatch: limit of the arrival wait (100 MHz ticks); 0: none
    int spec;                    // blank-run columns: spare joint columns evaluate later frames
    int max_iter;
    int red_slots;               // LDS partial slots: a phase runs in passes of red_slots / (units per item) items
    int st_n, st_k;              // LDS state of layers >= 1: utterance and owned-tile capacity
    int bias_floats;             // LDS bias table size (floats)
    int wcache_bytes;            // LDS weight cache per workgroup (0: weights are read from L2)
    unsigned long long *prof;    // nullable: per-phase wall-clock totals of workgroup 0 (100 MHz ticks)
};

// Phase timers (workgroup 0 only, when p.prof is set): totals kept in LDS,
// written to p.prof when the loop ends.
enum { kPrL0 = 0, kPrStage0, kPrL1, kPrStage1, kPrPred, kPrJStage, kPrJCompute, kPrKeys, kPrDecide, kPrN };

// ---------------------------------------------------------------- memory helpers

// Buffer resource over [base, base + bytes): out-of-range lanes read 0 and
// drop stores, so a bad index cannot fault.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

// Agent-coherent (SC1) loads / stores: used for every buffer written by one
// workgroup and read by another inside a launch.  Plain loads elsewhere keep
// weights cached in L2 (nothing in the loop invalidates the L2).
constexpr int kSC1 = 16;
__device__ __forceinline__ float4 ld4_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, kSC1));
}
__device__ __forceinline__ void st4_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off, float4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), r,
                                           byte_off, 0, kSC1);
}
// Offset past every buffer range: loads return 0 and stores are dropped.
constexpr unsigned kBad = 0x80000000u;
__device__ __forceinline__ float4 ld4(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0));
}
__device__ __forceinline__ float ld1_coh(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, kSC1));
}
__device__ __forceinline__ float ld_coh(const float *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coh(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup barrier for LDS traffic only: each wave waits for its own LDS
// operations (lgkmcnt 0) but not for its global loads and stores, which stay
// in flight across it (s_barrier carries no implicit wait on gfx950); data of
// other workgroups is waited for word by word.  The signal fences keep the
// compiler from moving memory accesses across it.
__device__ __forceinline__ void lds_sync() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);   // gfx9 encoding: lgkmcnt(0), vmcnt and expcnt unconstrained
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// ---------------------------------------------------------------- MFMA tiles

// 8 int8 stored as q ^ 0x80 = q + 128 (two dwords) -> 8 exact f16: the byte
// becomes the low mantissa byte of 1024.0 (0x64xx), then 1152 is subtracted.
__device__ __forceinline__ half8 q8_to_half8(uint2 q) {
    const unsigned x0 = q.x, x1 = q.y;
    const half2v off = {(_Float16)1152.0f, (_Float16)1152.0f};
    half2v p0 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, x0, 0x04010400u)) - off;
    half2v p1 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, x0, 0x04030402u)) - off;
    half2v p2 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, x1, 0x04010400u)) - off;
    half2v p3 = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, x1, 0x04030402u)) - off;
    return half8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

__device__ __forceinline__ void split_f16(float x, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);
}

// DPP quad permutation of a float: lane i of each quad reads quad lane perm_i.
template <int CTRL>
__device__ __forceinline__ float quad_perm(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// 4x4 transpose inside each quad of lanes: afterwards element j of quad lane p
// is what element p of quad lane j was.  Two butterfly stages (partner p^1,
// then p^2), each exchanging the two elements whose index bit differs from p's.
__device__ __forceinline__ f32x4 quad_transpose(f32x4 a) {
    const int p = threadIdx.x & 3;
    {
        const bool odd = p & 1;
        const float r0 = quad_perm<0xB1>(odd ? a[0] : a[1]);   // quad_perm [1,0,3,2]
        const float r1 = quad_perm<0xB1>(odd ? a[2] : a[3]);
        if (odd) { a[0] = r0; a[2] = r1; } else { a[1] = r0; a[3] = r1; }
    }
    {
        const bool hi = p & 2;
        const float r0 = quad_perm<0x4E>(hi ? a[0] : a[2]);    // quad_perm [2,3,0,1]
        const float r1 = quad_perm<0x4E>(hi ? a[1] : a[3]);
        if (hi) { a[0] = r0; a[1] = r1; } else { a[2] = r0; a[3] = r1; }
    }
    return a;
}

// Maximum of a 64-bit value over the lanes that agree modulo `step` (a power of two up to 16),
// in every lane.  Below 16 by rotations inside a DPP row of 16 lanes, then by the row and half
// swaps: no LDS round trip (a shuffle is one, about 0.05 us, and an argmax takes up to six).
typedef unsigned long long u64;
template <int CTRL>
__device__ __forceinline__ u64 row_ror_max(u64 v) {
    const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)v, CTRL, 0xF, 0xF, false);
    const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(v >> 32), CTRL, 0xF, 0xF, false);
    const u64 o = ((u64)hi << 32) | lo;
    return o > v ? o : v;
}
__device__ __forceinline__ u64 lanes_max(u64 v, int step) {
    if (step <= 8) v = row_ror_max<0x128>(v);   // row_ror:8
    if (step <= 4) v = row_ror_max<0x124>(v);
    if (step <= 2) v = row_ror_max<0x122>(v);
    if (step <= 1) v = row_ror_max<0x121>(v);
    if (step <= 16) {   // rows 0, 1 and rows 2, 3
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
        const u64 a = ((u64)hi[0] << 32) | lo[0], b = ((u64)hi[1] << 32) | lo[1];
        v = a > b ? a : b;
    }
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
    const u64 a = ((u64)hi[0] << 32) | lo[0], b = ((u64)hi[1] << 32) | lo[1];
    return a > b ? a : b;
}

// Inclusive prefix sum over the wave: shifts inside a DPP row, then the rows' last lanes passed on.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int v) {
    return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ int wave_scan(int v) {
    v = dpp_add<0x111, 0xF>(v);   // row_shr:1
    v = dpp_add<0x112, 0xF>(v);
    v = dpp_add<0x114, 0xF>(v);
    v = dpp_add<0x118, 0xF>(v);
    v = dpp_add<0x142, 0xA>(v);   // row_bcast:15 into rows 1 and 3
    return dpp_add<0x143, 0xC>(v);   // row_bcast:31 into rows 2 and 3
}

// Staged activation block: 16 utterance rows of K values as f16 (hi, lo).
// Only rows 0 .. n-1 are staged; product columns n .. 15 are not used.
struct Act {
    _Float16 *hi, *lo;
    int kp;     // row stride in halves (K + kKPad)
    int n;      // live rows
};

// Four values split as in split_f16 (packed conversions).
__device__ __forceinline__ void put4(const Act &x, int row, int k, float4 v) {
    const f32x4 f = {v.x, v.y, v.z, v.w};
    const half4 h = __builtin_convertvector(f, half4);
    const half4 l = __builtin_convertvector(f - __builtin_convertvector(h, f32x4), half4);
    *reinterpret_cast<half4 *>(x.hi + row * x.kp + k) = h;
    *reinterpret_cast<half4 *>(x.lo + row * x.kp + k) = l;
}

// ---------------------------------------------------------------- argmax keys

// Order-preserving map of an f32 onto u32 (-0 folded onto +0).
__device__ __forceinline__ unsigned ordered_bits(float v) {
    if (v == 0.0f) v = 0.0f;
    const unsigned b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// Larger key = larger value, then smaller index: the reference's first-index rule.
__device__ __forceinline__ unsigned long long make_key(unsigned ordered, int idx) {
    return ((unsigned long long)ordered << kIdxBits) | (unsigned long long)((1 << kIdxBits) - 1 - idx);
}
__device__ __forceinline__ int key_index(unsigned long long key) {
    return (1 << kIdxBits) - 1 - (int)(key & ((1u << kIdxBits) - 1));
}
__device__ __forceinline__ unsigned key_stamp(unsigned long long key) { return (unsigned)(key >> kStampShift); }

// Gate nonlinearities from the hardware base-2 exponential (v_exp_f32) and
// reciprocal (v_rcp_f32), each within about 1 ulp: sigmoid(x) = 1 / (1 + e^-x),
// tanh(x) = 2 sigmoid(2x) - 1.  Absolute error stays below ~1e-7, far inside
// the state tolerance, and saturates correctly for large |x| (e^-x -> inf / 0).
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
__device__ __forceinline__ float sigmoidf_(float x) { return __builtin_amdgcn_rcpf(1.0f + exp_fast(-x)); }
__device__ __forceinline__ float tanh_fast(float x) { return 2.0f * sigmoidf_(2.0f * x) - 1.0f; }

__device__ __forceinline__ void cell(float gi, float gf, float gg, float go, float c_prev, float &c_new, float &h_new) {
    c_new = sigmoidf_(gf) * c_prev + sigmoidf_(gi) * tanh_fast(gg);
    h_new = sigmoidf_(go) * tanh_fast(c_new);
}

// ---------------------------------------------------------------- prepare-time kernels

// out[v][r] = bias0[r] + bias1[r] + W[r, :] . E[v, :] in f32: the layer-0
// input projection of every vocabulary row (W_ih0 . embed[v] + b_ih0 + b_hh0).
// Operands are dense f32 here (dequantised on the host from the stored bytes).
__global__ void __launch_bounds__(256) embed_proj_kernel(const float *__restrict w, const float *__restrict e,
                                                         int rows, int V, int K, const float *__restrict b0,
                                                         const float *__restrict b1, float *__restrict out) {
    const int v0 = blockIdx.x * 16, r0 = blockIdx.y * 64;
    __shared__ float es[16][65];
    __shared__ float ws[64][65];
    const int tid = threadIdx.x;
    const int tv = tid / 16, tr = tid % 16;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 64) {
        for (int i = tid; i < 16 * 64; i += 256) {
            const int vv = i / 64, k = i % 64;
            es[vv][k] = (v0 + vv < V && k0 + k < K) ? e[(size_t)(v0 + vv) * K + k0 + k] : 0.0f;
        }
        for (int i = tid; i < 64 * 64; i += 256) {
            const int rr = i / 64, k = i % 64;
            ws[rr][k] = (r0 + rr < rows && k0 + k < K) ? w[(size_t)(r0 + rr) * K + k0 + k] : 0.0f;
        }
        __syncthreads();
        for (int k = 0; k < 64; ++k) {
            const float x = es[tv][k];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = fmaf(ws[tr * 4 + j][k], x, acc[j]);
        }
        __syncthreads();
    }
    const int v = v0 + tv;
    if (v >= V) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = r0 + tr * 4 + j;
        if (r < rows) out[(size_t)v * rows + r] = acc[j] + (b0[r] + b1[r]);
    }
}

// Zero n 32-bit words (clears the flags, keys and status words of a call).
__global__ void __launch_bounds__(256) fill_zero_kernel(unsigned *__restrict p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0u;
}

// ---------------------------------------------------------------- enc_proj

// encp[rows of utterance u] = b_e + W_e . enc[row] for every frame: an MFMA
// GEMM with f32 accuracy.  Frames (f32) are split into f16 hi + lo.  How W_e
// arrives, by its storage (kEp*):
//   quantised  the block integers as exact f16 [J][D] and the block scales as
//              f32 [D/32][J]: per K block p = q.lo(q.hi), acc += scale * p;
//   f16        as stored [J][D]: acc += w.hi, then w.lo;
//   f32        hi and lo planes [J][D]: acc += hi.hi, hi.lo (frames' lo), lo.hi
//              (the lo.lo term is below f32 rounding).
// K blocks of 32 in order, one accumulator per output: the three kernels below
// run the same instructions per output, so their rows are equal bit for bit and
// the host chooses between them by row count alone.
// Against hi and lo planes of the dequantised weights for every storage type, a K
// block takes 2 MFMAs instead of 3 and its error against 64 bits falls (joint
// logits of TDT-0.6b q8_0: 3.0e-7 against 4.1e-7 relative): the integers are exact,
// while the lo plane of a small weight is a subnormal f16.
// d_enc % 32 == 0.  Output rows are the frames of all utterances packed in order
// (utterance u owns rows dst_row[u] .. dst_row[u] + T[u]), so short windows of
// many utterances share tiles; a row's utterance is the last u with
// dst_row[u] <= row.  Threads of the whole grid also zero `clear_words` 32-bit
// words at `clear` (the decode loop's status, barrier flags and argmax keys),
// which saves the loop a separate fill.
enum { kEpQuant = 0, kEpHalf = 1, kEpFull = 2 };
struct EncProj {
    const _Float16 *w, *w_lo;       // see above (w_lo: f32 only)
    const float *w_scale;           // quantised only
    const float *bias, *enc;
    int J, d_enc, n_utts;
    const long long *src_row, *dst_row;
    long long rows;
    float *out;
    unsigned *clear;
    size_t clear_words;
};
constexpr int kEpK = 32, kEpStride = kEpK + 8;   // K step; LDS row stride in halves

__device__ __forceinline__ void ep_clear(const EncProj &e, size_t thread, size_t threads) {
    for (size_t i = thread; i < e.clear_words; i += threads) e.clear[i] = 0u;
}
// First value of output row r's frame (rows past the last: the last row, never stored).
__device__ __forceinline__ const float *ep_src(const EncProj &e, long long r) {
    r = r < e.rows ? r : e.rows - 1;
    int lo = 0, hi = e.n_utts - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (e.dst_row[mid] <= r) lo = mid;
        else hi = mid - 1;
    }
    return e.enc + (size_t)(e.src_row[lo] + (r - e.dst_row[lo])) * e.d_enc;
}
__device__ __forceinline__ void ep_split(const float4 &a, const float4 &b, half8 &h, half8 &l) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        h[i] = (_Float16)v[i];
        l[i] = (_Float16)(v[i] - (float)h[i]);
    }
}
// One K block of a 16x16 output tile (scale: kEpQuant, the lane's column).
template <int W>
__device__ __forceinline__ f32x4 ep_mma(half8 a_h, half8 a_l, half8 b, half8 b_lo, float scale, f32x4 acc) {
    if constexpr (W == kEpQuant) {
        f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_h, b, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_l, b, p, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = fmaf(scale, p[i], acc[i]);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_h, b, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_l, b, acc, 0, 0, 0);
        if constexpr (W == kEpFull) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_h, b_lo, acc, 0, 0, 0);
    }
    return acc;
}
// Bias of output column col (past the last: the last one's, never stored).  Loaded before the
// products: behind the epilogue's stores, which may alias it, each load waits by itself (20 in a
// wave of the wide kernel: 10,240 rows of TDT-0.6b q8_0 55 us instead of 47; 64 x 64 tiles, 4 in a
// wave: 4,096 rows 36 instead of 34).
__device__ __forceinline__ float ep_bias(const EncProj &e, int col) { return e.bias[min(col, e.J - 1)]; }
// D fragment of a tile: a lane holds output column `col` of rows row .. row + 3.
__device__ __forceinline__ void ep_store(const EncProj &e, long long row, int col, f32x4 acc, float bc) {
    if (col >= e.J) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (row + i < e.rows) e.out[(size_t)(row + i) * e.J + col] = acc[i] + bc;
}

// Middle row counts: workgroup of 64 output rows x 64 outputs, 4 waves of 16
// rows, K steps of 32 through LDS.  The global loads of K step k+1 are issued
// before the products of step k (one register set ahead), so each step waits
// for LDS and the matrix cores rather than for memory.
constexpr int kEpTile = 64;
template <int W>
__global__ void __launch_bounds__(256) enc_proj_kernel(EncProj e) {
    __shared__ __attribute__((aligned(16))) _Float16 ah[kEpTile * kEpStride], al[kEpTile * kEpStride];
    __shared__ __attribute__((aligned(16))) _Float16 bh[kEpTile * kEpStride],
        bl[W == kEpFull ? kEpTile * kEpStride : 8];
    __shared__ float bs[W == kEpQuant ? kEpTile : 1];
    ep_clear(e, ((size_t)blockIdx.z * gridDim.x + blockIdx.x) * 256 + threadIdx.x, (size_t)gridDim.x * gridDim.z * 256);
    const long long m0 = (long long)blockIdx.x * kEpTile;
    const int n0 = blockIdx.z * kEpTile;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int sr = tid / 4, sc = (tid % 4) * 8;   // staging: row / column of this thread's 8 values
    const float *src = ep_src(e, m0 + sr) + sc;
    const size_t wrow = (size_t)min(n0 + sr, e.J - 1) * e.d_enc + sc;
    const int scol = min(n0 + tid, e.J - 1);
    // one K step's global operands of this thread
    float4 v0, v1;
    half8 wh, wl;
    float ws = 0.f;
    auto fetch = [&](int k0) {
        v0 = *reinterpret_cast<const float4 *>(src + k0);
        v1 = *reinterpret_cast<const float4 *>(src + k0 + 4);
        wh = *reinterpret_cast<const half8 *>(e.w + wrow + k0);
        if constexpr (W == kEpFull) wl = *reinterpret_cast<const half8 *>(e.w_lo + wrow + k0);
        if constexpr (W == kEpQuant)
            if (tid < kEpTile) ws = e.w_scale[(size_t)(k0 / kEpK) * e.J + scol];
    };
    f32x4 acc[4];
    float bias[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        bias[t] = ep_bias(e, n0 + t * 16 + (lane & 15));
    }
    fetch(0);
    for (int k0 = 0; k0 < e.d_enc; k0 += kEpK) {
        {
            half8 h, l;
            ep_split(v0, v1, h, l);
            *reinterpret_cast<half8 *>(ah + sr * kEpStride + sc) = h;
            *reinterpret_cast<half8 *>(al + sr * kEpStride + sc) = l;
            *reinterpret_cast<half8 *>(bh + sr * kEpStride + sc) = wh;
            if constexpr (W == kEpFull) *reinterpret_cast<half8 *>(bl + sr * kEpStride + sc) = wl;
            if constexpr (W == kEpQuant)
                if (tid < kEpTile) bs[tid] = ws;
        }
        __syncthreads();
        if (k0 + kEpK < e.d_enc) fetch(k0 + kEpK);   // in flight during this step's products
        const int ao = (wave * 16 + (lane & 15)) * kEpStride + (lane >> 4) * 8;
        const half8 a_h = *reinterpret_cast<const half8 *>(ah + ao);
        const half8 a_l = *reinterpret_cast<const half8 *>(al + ao);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int bo = (t * 16 + (lane & 15)) * kEpStride + (lane >> 4) * 8;
            const half8 b = *reinterpret_cast<const half8 *>(bh + bo);
            half8 b_lo = half8{};
            if constexpr (W == kEpFull) b_lo = *reinterpret_cast<const half8 *>(bl + bo);
            acc[t] = ep_mma<W>(a_h, a_l, b, b_lo, W == kEpQuant ? bs[t * 16 + (lane & 15)] : 0.f, acc[t]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
        ep_store(e, m0 + wave * 16 + (lane >> 4) * 4, n0 + t * 16 + (lane & 15), acc[t], bias[t]);
}

// Large row counts (batched offline decoding): workgroup of 128 output rows x
// 320 outputs, 8 waves of 64 x 80 (4 x 5 tiles).  A frame is split and staged
// J / 320 times instead of J / 64 times and read from LDS by 4 waves instead of
// one per 4 tiles; per K step a wave reads 13 KB of fragments from LDS for 40
// MFMAs (f32: 18 KB for 60), with 64 x 64 tiles 6 KB for 8 (f32: 10 KB for 12).  Two LDS buffers, one barrier per K step:
// step k+1 is written from registers and step k+2's loads are issued before the
// products of step k (loads one more step ahead measured the same).  Workgroups
// that share rows sit on one XCD (ids 8 apart), one after the other, so the second
// reads the frames from its L2.
// 131,072 rows, D = 1024, J = 640: q8_0 433 us, f16 384 us, f32 535 us (0.79, 0.89,
// 0.96 PFLOP/s of MFMA; a large library product reaches 1.21 on the same card), 1245,
// 1234 and 1375 us with enc_proj_kernel.  It is bound by the workgroup's serial K
// steps, about 1.3 us each, so a launch takes 43 us however few its rows are: up to
// 8,192 rows the 64 x 64 tiles are as fast or faster (47 us either way; 5,120 rows: 40
// against 46; 16,384: 89 against 51), and a launch of few columns leaves most of its
// waves empty, hence the host's rule between the two (enc_proj_rule.h).
constexpr int kEwRows = 128, kEwCols = 320, kEwThreads = 512;
template <int W>
__global__ void __launch_bounds__(kEwThreads) enc_proj_wide_kernel(EncProj e) {
    __shared__ __attribute__((aligned(16))) _Float16 ah[2][kEwRows * kEpStride], al[2][kEwRows * kEpStride];
    __shared__ __attribute__((aligned(16))) _Float16 bh[2][kEwCols * kEpStride],
        bl[2][W == kEpFull ? kEwCols * kEpStride : 8];
    __shared__ float bs[2][W == kEpQuant ? kEwCols : 1];
    ep_clear(e, (size_t)blockIdx.x * kEwThreads + threadIdx.x, (size_t)gridDim.x * kEwThreads);
    const int n_col = (e.J + kEwCols - 1) / kEwCols, group = blockIdx.x / (8 * n_col), in = blockIdx.x % (8 * n_col);
    const long long m0 = (long long)(group * 8 + (in & 7)) * kEwRows;
    const int n0 = (in >> 3) * kEwCols;
    if (m0 >= e.rows) return;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wr = (wave >> 2) * 64, wn = (wave & 3) * 80;   // this wave's rows and columns of the tile
    const int sr = tid / 4, sc = (tid % 4) * 8;              // staging: one row's 8 values, 3 columns' 8 values
    const float *src = ep_src(e, m0 + sr) + sc;
    constexpr int kChunks = kEwCols * 4, kPer = (kChunks + kEwThreads - 1) / kEwThreads;
    size_t wrow[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) wrow[i] = (size_t)min(n0 + (tid + i * kEwThreads) / 4, e.J - 1) * e.d_enc + sc;
    const int scol = min(n0 + tid, e.J - 1);
    float4 v0, v1;
    half8 wh[kPer], wl[kPer];
    float ws = 0.f;
    auto fetch = [&](int k0) {
        v0 = *reinterpret_cast<const float4 *>(src + k0);
        v1 = *reinterpret_cast<const float4 *>(src + k0 + 4);
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            wh[i] = *reinterpret_cast<const half8 *>(e.w + wrow[i] + k0);
            if constexpr (W == kEpFull) wl[i] = *reinterpret_cast<const half8 *>(e.w_lo + wrow[i] + k0);
        }
        if constexpr (W == kEpQuant) ws = e.w_scale[(size_t)(k0 / kEpK) * e.J + scol];
    };
    auto stage = [&](int b) {
        half8 h, l;
        ep_split(v0, v1, h, l);
        *reinterpret_cast<half8 *>(ah[b] + sr * kEpStride + sc) = h;
        *reinterpret_cast<half8 *>(al[b] + sr * kEpStride + sc) = l;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int col = (tid + i * kEwThreads) / 4;
            if ((i + 1) * kEwThreads > kChunks && col >= kEwCols) break;
            *reinterpret_cast<half8 *>(bh[b] + col * kEpStride + sc) = wh[i];
            if constexpr (W == kEpFull) *reinterpret_cast<half8 *>(bl[b] + col * kEpStride + sc) = wl[i];
        }
        if constexpr (W == kEpQuant)
            if (tid < kEwCols) bs[b][tid] = ws;
    };
    f32x4 acc[4][5];
    float bias[5];
#pragma unroll
    for (int n = 0; n < 5; ++n) {
        bias[n] = ep_bias(e, n0 + wn + n * 16 + (lane & 15));
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int steps = e.d_enc / kEpK, last = e.d_enc - kEpK;
    fetch(0);
    stage(0);
    fetch(min(kEpK, last));   // (steps past the last reload it)
    lds_sync();
    const int fo = (lane & 15) * kEpStride + (lane >> 4) * 8;
    for (int s = 0; s < steps; ++s) {
        const int b = s & 1;
        // the other buffer's readers, step s-1, are behind the last barrier
        if (s + 1 < steps) stage(b ^ 1);
        fetch(min((s + 2) * kEpK, last));
        half8 a_h[4], a_l[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            a_h[t] = *reinterpret_cast<const half8 *>(ah[b] + (wr + t * 16) * kEpStride + fo);
            a_l[t] = *reinterpret_cast<const half8 *>(al[b] + (wr + t * 16) * kEpStride + fo);
        }
#pragma unroll
        for (int n = 0; n < 5; ++n) {
            const int bo = (wn + n * 16) * kEpStride + fo;
            const half8 w = *reinterpret_cast<const half8 *>(bh[b] + bo);
            half8 w_lo = half8{};
            if constexpr (W == kEpFull) w_lo = *reinterpret_cast<const half8 *>(bl[b] + bo);
            const float scale = W == kEpQuant ? bs[b][wn + n * 16 + (lane & 15)] : 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t][n] = ep_mma<W>(a_h[t], a_l[t], w, w_lo, scale, acc[t][n]);
        }
        lds_sync();
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int n = 0; n < 5; ++n)
            ep_store(e, m0 + wr + t * 16 + (lane >> 4) * 4, n0 + wn + n * 16 + (lane & 15), acc[t][n], bias[n]);
}

// Few rows (streaming chunks, short windows).  There the tiled kernels above run
// on a few dozen workgroups, each paying workgroup barriers and an LDS round trip
// per K step.  Here each wave owns one 16x16 output block and loads its operands
// straight into MFMA fragment registers, kEnSteps K steps per batch, the next
// batch in flight while the current one is multiplied: no LDS and no barrier.
// Workgroup: 4 waves, 16 rows x 64 outputs.
constexpr int kEnSteps = 4;   // K steps per batch of the narrow kernel
template <int W>
__global__ void __launch_bounds__(256) enc_proj_narrow_kernel(EncProj e) {
    ep_clear(e, ((size_t)blockIdx.z * gridDim.x + blockIdx.x) * 256 + threadIdx.x, (size_t)gridDim.x * gridDim.z * 256);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const long long m0 = (long long)blockIdx.x * 16;
    const int n0 = (blockIdx.z * 4 + wave) * 16;
    if (n0 >= e.J) return;
    const int col = n0 + (lane & 15), cc = min(col, e.J - 1);
    const int ks = (lane >> 4) * 8;
    const int nsteps = e.d_enc / kEpK, nb = (nsteps + kEnSteps - 1) / kEnSteps;
    // Every lane loads: a row past the last reads the last frame row and a column past J
    // reads W_e row J - 1.  Row i of an MFMA product depends only on row i of A, and column j
    // only on column j of B, so those lanes' values reach only outputs never stored.
    const float *src = ep_src(e, m0 + (lane & 15)) + ks;
    const _Float16 *bhp = e.w + (size_t)cc * e.d_enc + ks;
    const _Float16 *blp = W == kEpFull ? e.w_lo + (size_t)cc * e.d_enc + ks : nullptr;
    struct Batch {
        float4 a0[kEnSteps], a1[kEnSteps];
        half8 bh[kEnSteps], bl[kEnSteps];
        float s[kEnSteps];
    };
    // batch b's operands (a batch past the last reloads the last one, so no load sits
    // behind a branch and the compiler's wait counts stay exact)
    auto load = [&](int b, Batch &x) {
        b = b < nb ? b : nb - 1;
#pragma unroll
        for (int s = 0; s < kEnSteps; ++s) {
            int st = b * kEnSteps + s;
            st = st < nsteps ? st : nsteps - 1;
            const int k = st * kEpK;
            x.a0[s] = *reinterpret_cast<const float4 *>(src + k);
            x.a1[s] = *reinterpret_cast<const float4 *>(src + k + 4);
            x.bh[s] = *reinterpret_cast<const half8 *>(bhp + k);
            x.bl[s] = half8{};
            if constexpr (W == kEpFull) x.bl[s] = *reinterpret_cast<const half8 *>(blp + k);
            x.s[s] = W == kEpQuant ? e.w_scale[(size_t)st * e.J + cc] : 0.f;
        }
    };
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    const float bias = ep_bias(e, col);
    auto mul = [&](int b, const Batch &x) {
#pragma unroll
        for (int s = 0; s < kEnSteps; ++s) {
            if (b * kEnSteps + s >= nsteps) break;
            half8 h, l;
            ep_split(x.a0[s], x.a1[s], h, l);
            acc = ep_mma<W>(h, l, x.bh[s], x.bl[s], x.s[s], acc);
        }
    };
    Batch X, Y;
    load(0, X);
    for (int b = 0; b < nb; b += 2) {
        load(b + 1, Y);
        mul(b, X);
        load(b + 2, X);
        if (b + 1 < nb) mul(b + 1, Y);
    }
    ep_store(e, m0 + (lane >> 4) * 4, col, acc, bias);
}

// ---------------------------------------------------------------- decode loop

// Control state of an utterance of the domain: lane ul of wave 0 holds utterance ul's for
// the whole launch, in registers (the other waves' copies are not used).  The decisions
// are a serial chain in which every workgroup waits; with this state in LDS every field
// was a dependent round trip of 0.05 us.  The lists go out as the byte offsets their
// readers need (Ctl::lrow, crow), one LDS read instead of list entry, fields and products.
// Measured with the joint's epilogue on ordered bits (joint_phase), us per iteration before
// and after: B=1 13.61 -> 12.57, B=24 (TDT-1.1b f16) 18.29 -> 17.11, EOU-120m B=16 13.06 ->
// 11.93, B=64 19.83 -> 19.39, B=256 32.12 -> 31.22, B=512 41.69 -> 39.57.
struct Utt {
    int t, T, sym, pend, flags, ntok, steps;
    int cur;                      // parity of the utterance's state once its pending token (if any) is taken
    int keep;                     // 1: the last decision kept the prediction output
    int stp;                      // 1: the utterance took an LSTM step in this launch
    // joint columns: column col is the utterance at its frame t; columns sbase .. sbase + sn - 1
    // are the same utterance at frames t + 1 .. t + sn
    int col, sbase, sn;
};

struct Ctl {                      // per-workgroup state of its domain
    // the lists of an iteration, as the byte offsets their readers need
    int4 cnt;                     // LSTM list length (-1: the launch ends, see ok), joint list length, joint
                                  // columns, log2 of the first, rounded up
    // LSTM list row: E' row of the pending token; c_0 row of the old state (-1: zero state) and of the
    // new one; h row | parity << 6 | zero state << 5 | domain utterance
    int4 lrow[kDomCap];
    int4 crow[kColCap];           // joint column: encp row, ppx row, blank offset (f32 bits), -
    // per domain utterance, for the whole launch
    int b[kDomCap];               // batch index
    unsigned erow[kDomCap];       // first encp row (byte offset)
    float bbias[kDomCap];         // blank logit offset
    int tbase[kDomCap];           // tokens before this call (EOU segment indices)
    int nseg[kDomCap], segst[kDomCap], last[kDomCap];   // EOU (lane ul of wave 0)
    int cur[kDomCap];             // parity of the state at the start and at the end
    int mark[kDomCap];            // start: 1 = zero state; end: 1 = took an LSTM step
    int dur[PK_MAX_DURATIONS];    // duration values (the decision step reads them from LDS)
    int n;
    int dom, rank, P;
    int ok;                       // 0: a wait ended without its data (error or time-out)
    // this workgroup's tiles of an LSTM matrix, of W_p and of W_o (fixed for the
    // launch; computed once, since each is an integer division)
    int own_lstm, own_pred, own_out;
    int pass[PK_MAX_LAYERS + 1];  // items per pass of the phase consuming layer l's output (l < L), of W_o (L)
    unsigned mag_p;               // udiv multiplier for P
    unsigned wmask;               // bit ul: this workgroup writes utterance ul's outputs (ul % P == rank)
    int tq_n, tq_col[kColCap], tq_b[kColCap], tq_step[kColCap];   // logit tap: (column, utterance, step)
                                                                  // of this iteration's decisions
    unsigned long long wgkey[kColCap][2];   // this workgroup's best key per joint column and head
    unsigned long long prof[kPrN];
};
// Row word of the LSTM list (rows of h are multiples of 128 bytes).
constexpr int kRowUl = 31, kRowZero = 32, kRowCur = 64, kRowMask = ~127;

__device__ __forceinline__ void pmark(const KParams &p, Ctl &s, unsigned long long &last, int k) {
    if (!p.prof) return;
    lds_sync();
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const unsigned long long now = __builtin_amdgcn_s_memrealtime();
        s.prof[k] += now - last;
        last = now;
    }
}

// Checkpoint timeline (built with -DPK_TIMELINE, read with PK_PROFILE_PHASES=1):
// workgroup 0 sums, per wave and checkpoint, the time since the start of the
// iteration over iterations 40 .. 295; the host prints the per-wave means.
// TL(k) is relative to the phase base set by TLBASE, TLA(k) absolute.  The
// checkpoints add LDS traffic and waits of their own, so their times are
// upper bounds.
constexpr int kTl = 32;
#ifdef PK_TIMELINE
__device__ __forceinline__ unsigned long long *tl_sum() { __shared__ unsigned long long b[kWaves * kTl]; return b; }
__device__ __forceinline__ int *tl_ctl() { __shared__ int c[2 + kTl]; return c; }
__device__ __forceinline__ unsigned long long *tl_t0() { __shared__ unsigned long long t; return &t; }
#define TLX(k, rel) do { int *c_ = tl_ctl(); if (c_[0]) { const int w_ = threadIdx.x >> 6; \
    if ((threadIdx.x & 63) == 0) { const int kk_ = ((rel) ? c_[1] : 0) + (k); \
    tl_sum()[w_ * kTl + kk_] += __builtin_amdgcn_s_memrealtime() - *tl_t0(); if (w_ == 0) c_[2 + kk_]++; } } } while (0)
#define TLBASE(b) do { if (threadIdx.x == 0) tl_ctl()[1] = (b); } while (0)
#else
#define TLX(k, rel) do { } while (0)
#define TLBASE(b) do { } while (0)
#endif
#define TL(k) TLX(k, 1)
#define TLA(k) TLX(k, 0)

// State offsets (floats): c_0 / h_0 of parity buf, W_hh0 . h_0.
__device__ __forceinline__ size_t cx_off(const KParams &p, int buf, int b) { return ((size_t)buf * p.n_utts + b) * p.H; }
__device__ __forceinline__ size_t rx_off(const KParams &p, int buf, int b) {
    return ((size_t)buf * p.n_utts + b) * 4 * p.H;
}
__device__ __forceinline__ size_t hs_off(const KParams &p, int layer, int b) {
    return ((size_t)layer * p.n_utts + b) * p.H;
}
// Exchange offsets (floats): the 4 units of tile t for list row u; the 16 rows
// of pred tile t for domain utterance ul.
__device__ __forceinline__ unsigned hx_at(const KParams &p, int dom, int layer, int half, int t, int u) {
    return ((((unsigned)((layer - p.hl0) * 2 + half) * p.n_dom + dom) * (p.H / 4) + t) * p.rows + u) * 4u;
}
__device__ __forceinline__ unsigned ppx_at(const KParams &p, int dom, int half, int t, int ul) {
    return ((((unsigned)half * p.n_dom + dom) * (p.J / kTile) + t) * p.prows + ul) * (unsigned)kTile;
}
// Compact the LSTM list (pending token) and the joint list (frames left).
// Then the joint columns: one per joint-list utterance at its frame t, and
// (spec) the column tiles' spare columns dealt out evenly as frames t + 1,
// t + 2, ... to the utterances in a run of blanks (last decision kept the
// prediction output), up to their last frame.  A blank decision keeps the
// prediction output, so the logits of the next frame are already in a spare
// column: the decision step walks a run of blanks in one iteration instead of
// one iteration per blank.
__device__ __forceinline__ void build_lists(const KParams &p, Ctl &s, Utt &u) {
    if (threadIdx.x < kWave) {
        const int lane = threadIdx.x, ul = min(lane, kDomCap - 1);
        const bool fl = lane < s.n && u.pend >= 0;
        const bool fj = lane < s.n && u.t < u.T;
        const unsigned long long bl = __ballot(fl), bj = __ballot(fj);
        const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
        const int il = __popcll(bl & below), ij = __popcll(bj & below);
        const int b = s.b[ul];
        if (fl) {
            const bool zero = u.flags & kFlagZeroHC;
            const int row = p.H * 4;   // bytes of a c_0 row
            s.lrow[il] = make_int4(u.pend * 4 * row, zero ? -1 : ((u.cur ^ 1) * p.n_utts + b) * row,
                                   (u.cur * p.n_utts + b) * row,
                                   b * row | (u.cur ? kRowCur : 0) | (zero ? kRowZero : 0) | lane);
        }
        const int nj = __popcll(bj);
        // an utterance in a blank run takes q spare columns: an even share of the
        // spare columns of the tiles, capped at the frames it has left
        const int spare = p.spec != 0 && nj > 0 ? ((nj + kTile - 1) / kTile) * kTile - nj : 0;
        const bool fe = fj && spare > 0 && u.keep != 0;
        const unsigned long long be = __ballot(fe);
        int total = 0;
        int4 c = make_int4((int)(s.erow[ul] + (unsigned)u.t * (unsigned)(p.J * 4)),
                           (int)(ppx_at(p, s.dom, u.cur, 0, ul) * 4u), __float_as_int(s.bbias[ul]), 0);
        if (fj) s.crow[ij] = c;
        u.col = ij;
        u.sbase = u.sn = 0;
        if (be != 0ull) {   // some utterance is in a run of blanks (wave-uniform)
            const int ne = __popcll(be), ie = __popcll(be & below);
            int q = 0;
            if (fe) {
                // spare / ne (both at most 32: the half keeps the product off the integers)
                const int each = (int)(((float)spare + 0.5f) * __builtin_amdgcn_rcpf((float)ne));
                q = each + (ie < spare - each * ne ? 1 : 0);
                q = min(q, u.T - u.t - 1);
            }
            // prefix sum of q over the joint list (lanes in list order)
            const int incl = wave_scan(q);
            if (fj) {
                u.sbase = nj + incl - q;
                u.sn = q;
                for (int o = 1; o <= q; ++o) {
                    c.x += p.J * 4;
                    s.crow[u.sbase + o - 1] = c;
                }
            }
            total = __builtin_amdgcn_readlane(incl, kWave - 1);
        }
        if (lane == 0) {
            const int nl = __popcll(bl);
            s.cnt = make_int4(s.ok ? nl : -1, nj, nj + total, nl <= 1 ? 0 : 32 - __builtin_clz((unsigned)(nl - 1)));
        }
    }
    lds_sync();
}

// A wait that does not end by itself: every 64 polls the error word and the
// clock are read, and after ~2 s the launch ends with PK_ERR_TIMEOUT (s.ok is
// checked once per iteration; waits that follow end at their 64th poll).
__device__ __forceinline__ bool wait_over(const KParams &p, Ctl &s, unsigned &n, unsigned long long &t0) {
    if ((++n & 63u) != 0u) return false;
    const unsigned long long now = __builtin_amdgcn_s_memrealtime();   // 100 MHz
    if (t0 == 0ull) t0 = now;
    if (__hip_atomic_load(p.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
        s.ok = 0;
        return true;
    }
    if (now - t0 > 200000000ull) {
        __hip_atomic_store(p.status, PK_ERR_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s.ok = 0;
        return true;
    }
    return false;
}

// Domain barrier before the first iteration: every member publishes its epoch
// in its own flag word and every member polls all members' flags (thread t
// polls rank t).  No cache-wide fences: cross-workgroup data is stored and
// loaded coherently (SC1), and each thread waits for its own stores
// (s_waitcnt 0) before arriving.  Returns false if the error word is set or the
// wait exceeds ~2 s.
__device__ __forceinline__ bool dom_sync(const KParams &p, Ctl &s, unsigned &epoch) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    ++epoch;
    if (threadIdx.x == 0)
        __hip_atomic_store(p.flags + (size_t)blockIdx.x * kFlagStride, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x < s.P) {
        unsigned *f = p.flags + (size_t)p.dom_wg[s.dom * s.P + threadIdx.x] * kFlagStride;
        unsigned n = 0;
        unsigned long long t0 = 0ull;
        while (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < epoch)
            if (wait_over(p, s, n, t0)) break;
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    return s.ok != 0;
}

// Exchange between the workgroups of a domain inside an iteration.
//
// Every value that other workgroups need (h of each layer, the prediction
// output, the argmax keys) is waited for word by word: a consumer loads the
// words it stages until none of them is empty.  One device-coherent store and
// the load that sees it replace the store, its acknowledgement, a barrier (flag
// store, polls of every member's flag) and the staging load behind it.  Layouts
// give each producer whole lines of 128 bytes: a tile's rows are stored by one
// wave, so no line is invalidated under its readers by another workgroup's store.
// (The prediction output of a domain of one utterance is the exception: a tile is
// then 64 bytes, and two neighbouring ranks share a line.)
// Measured per exchange with nothing else in flight (store, wait, staged rows):
// 16 rows over 64 workgroups 1.84 us against 2.71 us with a barrier, over 16
// workgroups 2.07 against 2.57, one row over 256 workgroups 1.75 against 2.15.
//
// Words become empty again in time: h of an LSTM step sits in one of two halves
// (hx), and its producer empties the half of the previous step when the next one
// begins; the prediction output of an utterance sits in the half of its parity
// (ppx), and its producer empties the old half when it writes the new one.  By
// then every reader is done: the argmax keys are exchanged at the end of each
// iteration, and a workgroup stores its keys after its last staging.  It also
// waits for all of its own stores before that, so a workgroup that has seen
// every key sees every word emptied or written in the iteration.

// (exchange_word.h: kEmpty, filled_word, any_empty)
__device__ __forceinline__ float filled(float v) { return __uint_as_float(filled_word(__float_as_uint(v))); }
__device__ __forceinline__ bool has_empty(float4 v) {
    return any_empty(__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w));
}
__device__ __forceinline__ float4 empty4() {
    const float e = __uint_as_float(kEmpty);
    return make_float4(e, e, e, e);
}

constexpr int kCopyB = 4;   // float4 per thread in flight when copying state

struct Bufs {
    __amdgpu_buffer_rsrc_t hx, cx, ppx, rx, ep, encp, keys;
};

// Staging: loads of kStageMax float4 per thread in flight; a thread converts
// and drops each as it arrives and loads the rest again.
constexpr int kStageMax = 5;

// h of layer lc for list rows c0 .. c0+nc-1 (nc <= 16) into an activation block.
// A wave covers 4 tiles x 16 rows (16 tiles x 4 rows for short lists): 1 KB in a
// row of the exchange buffer.
__device__ __forceinline__ void stage_h(const KParams &p, Ctl &s, const Bufs &B, const Act &x, int lc, int half,
                                        int c0, int nc) {
    const int lg = nc <= 4 ? 2 : 4;
    const int u = threadIdx.x & ((1 << lg) - 1), t0 = threadIdx.x >> lg, step = kBlock >> lg, ntile = p.H / 4;
    const unsigned base = hx_at(p, s.dom, lc, half, 0, c0 + u) * 4u, stride = (unsigned)p.rows * 16u;
    for (int b0 = 0; b0 < ntile; b0 += step * kStageMax) {
        unsigned pend = 0u, n = 0u;
        unsigned long long since = 0ull;
#pragma unroll
        for (int j = 0; j < kStageMax; ++j)
            if (u < nc && b0 + t0 + step * j < ntile) pend |= 1u << j;
        while (pend != 0u) {
            float4 v[kStageMax];
#pragma unroll
            for (int j = 0; j < kStageMax; ++j)
                v[j] = ld4_coh(B.hx, (pend >> j) & 1u ? base + (unsigned)(b0 + t0 + step * j) * stride : kBad);
#pragma unroll
            for (int j = 0; j < kStageMax; ++j)
                if (((pend >> j) & 1u) && !has_empty(v[j])) {
                    put4(x, u, (b0 + t0 + step * j) * 4, v[j]);
                    pend &= ~(1u << j);
                }
            if (pend != 0u && wait_over(p, s, n, since)) break;
        }
    }
}

// ---------------------------------------------------------------- MFMA phase engine
//
// A phase multiplies weight row tiles ("items") by one staged 16-utterance
// activation block.  Items 0 .. n_a-1 are tiles rank, rank+P, ... of matrix A,
// items n_a .. n_items-1 the same of matrix B (same storage type and K).  Each
// item's K blocks are cut into S units of kUnitOf blocks (f32 weights count
// every K block twice, once per f16 plane).  Items are taken in passes of as
// many items as the LDS partial slots hold.  Within a pass the units are
// numbered K-major -- unit u = chunk * nj + item -- and every wave takes a
// contiguous range of them, so a wave reads one chunk's activation fragments
// from LDS once and reuses them from registers for every item of its range.
// Each unit leaves one 16x16 partial in LDS slot (item - j0) * S + chunk; the
// pass's reduce sums an item's partials in chunk order (a fixed order, so
// results do not depend on timing) and runs the epilogue.  The weight
// fragments of a wave's next unit are loaded before its current unit is
// multiplied, so one unit's L2 latency hides behind the previous unit's
// products.

// K blocks per unit, by weight storage.  Measured: q8_0 5 (beats 4, 8 and 10 at B=1/64/256);
// f16 and f32 4 (TDT-1.1b f16 at B=256: 49.9 vs 60.5 ms per launch with 5).
template <bool Q8> constexpr int kUnitOf = Q8 ? 5 : 4;
__host__ __device__ constexpr int unit_blocks(int type) { return type == PK_TYPE_Q8_0 ? 5 : 4; }

// One matrix's fragment sources for a phase: buffer descriptors (q8_0: the
// quants and the block scales; f16: the plane twice; f32: the hi and lo
// planes) and the base of this workgroup's LDS-cached tiles, set up once.
struct MatSrc {
    __amdgpu_buffer_rsrc_t r0, r1;
    const unsigned char *lds;
    int KB;
    unsigned plane;   // f32: bytes of the hi plane (the lo plane's offset)
};
template <bool Q8, bool CACHED>
__device__ __forceinline__ MatSrc mat_src(const TMat &m, bool two, const unsigned char *wc) {
    MatSrc s;
    if (Q8) {
        s.r0 = rsrc(m.a, (unsigned)m.tiles * (unsigned)tile_bytes(PK_TYPE_Q8_0, m.KB));
        s.r1 = s.r0;
    } else {   // f32: both planes under one descriptor (the lo plane follows the hi plane)
        const unsigned bytes = (unsigned)m.tiles * m.KB * kWave * 16u;
        s.r0 = rsrc(m.a, two ? 2 * bytes : bytes);
        s.r1 = s.r0;
    }
    s.lds = CACHED ? wc + m.lds_off : nullptr;
    s.KB = m.KB;
    s.plane = (unsigned)m.tiles * m.KB * kWave * 16u;
    return s;
}

// Fragments of one unit, blocks sb0 .. sb0+kUnitOf-1 of tile `tile` (local index
// li in the LDS cache).  q8_0: the unit's record, four loads.  f16 / f32: FULL,
// all kUnitOf blocks exist (K is a whole number of units), so every offset is a
// lane constant plus a wave-uniform base plus an immediate; otherwise blocks
// past nb read as zero (buffer loads past the range return 0; cached blocks are
// zeroed).  Matrices are stored in whole units, so only FULL is instantiated.
template <bool Q8, bool CACHED, bool FULL>
__device__ __forceinline__ void unit_load_src(const MatSrc &m, bool two, int tile, int li, int sb0, int nb, int lane,
                                              uint4 (&f)[kUnitOf<Q8>]) {
    if constexpr (Q8) {   // one unit record (matrices are stored in whole units: every block exists)
        static_assert(kUnitOf<Q8> == kQ8Unit, "q8_0 units are the stored records");
        const int uc = sb0 / kQ8Unit;
        uint4 qa, qb, sc;
        uint2 qc;
        if (CACHED) {
            const unsigned char *rec = m.lds + ((size_t)li * (m.KB / kQ8Unit) + uc) * kQ8UnitBytes;
            qa = *reinterpret_cast<const uint4 *>(rec + lane * 16);
            qb = *reinterpret_cast<const uint4 *>(rec + 1024 + lane * 16);
            qc = *reinterpret_cast<const uint2 *>(rec + 2048 + lane * 8);
            sc = *reinterpret_cast<const uint4 *>(rec + kQ8Scales + (lane & 15) * 16);
        } else {
            const int rec = (tile * (m.KB / kQ8Unit) + uc) * kQ8UnitBytes;   // wave-uniform
            qa = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(m.r0, lane * 16, rec, 0));
            qb = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(m.r0, lane * 16 + 1024, rec, 0));
            qc = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(m.r0, lane * 8 + 2048, rec, 0));
            sc = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(m.r0, (lane & 15) * 16 + kQ8Scales,
                                                                                 rec, 0));
        }
        f[0] = make_uint4(qa.x, qa.y, sc.x & 0xffffu, 0u);
        f[1] = make_uint4(qa.z, qa.w, sc.x >> 16, 0u);
        f[2] = make_uint4(qb.x, qb.y, sc.y & 0xffffu, 0u);
        f[3] = make_uint4(qb.z, qb.w, sc.y >> 16, 0u);
        f[4] = make_uint4(qc.x, qc.y, sc.z & 0xffffu, 0u);
        return;
    }
    if (CACHED) {
#pragma unroll
        for (int j = 0; j < kUnitOf<Q8>; ++j) {
            const bool ok = FULL || j < nb;
            const int sb = ok ? sb0 + j : sb0;
            uint4 v;
            {
                const int kb = two ? sb >> 1 : sb;
                const int plane = two ? (sb & 1) : 0;
                v = *reinterpret_cast<const uint4 *>(m.lds + (((size_t)li * m.KB + kb) * (two ? 2 : 1) + plane) * 1024 +
                                                     lane * 16);
            }
            f[j] = ok ? v : make_uint4(0u, 0u, 0u, 0u);
        }
        return;
    }
    {
#pragma unroll
        for (int j = 0; j < kUnitOf<Q8>; ++j) {
            const int sb = sb0 + j;
            const int kb = two ? sb >> 1 : sb;
            const bool ok = FULL || j < nb;
            // f32: odd sub-blocks read the lo plane, m.plane bytes past the hi plane
            const unsigned o = ok ? (unsigned)(((tile * m.KB + kb) * kWave + lane) * 16) +
                                        ((two && (sb & 1)) ? m.plane : 0u)
                                  : kBad;
            f[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(m.r0, o, 0, 0));
        }
    }
}

// The activation fragments of a unit's K blocks (all reads issued at once).
template <int U>
__device__ __forceinline__ void unit_act(const Act &x, int xo, bool two, int sb0, int nb, half8 (&ah)[U],
                                         half8 (&al)[U]) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int sb = min(sb0 + j, sb0 + nb - 1);
        const int kb = two ? sb >> 1 : sb;
        ah[j] = *reinterpret_cast<const half8 *>(x.hi + xo + kb * 32);
        al[j] = *reinterpret_cast<const half8 *>(x.lo + xo + kb * 32);
    }
}

// acc += (unit's weight blocks) . (activation blocks), transposed (lane: one
// weight row, four utterances).  Zero blocks past nb add nothing.  q8_0: the
// products of all blocks are issued first (independent MFMA pairs), then each
// is scaled by its block's d; f16/f32: two independent accumulation chains (hi
// and lo activations) added at the end.
template <bool Q8>
__device__ __forceinline__ f32x4 unit_mma(const uint4 (&f)[kUnitOf<Q8>], const half8 (&ah)[kUnitOf<Q8>],
                                          const half8 (&al)[kUnitOf<Q8>],
                                          bool two, int sb0, f32x4 acc) {
    if (Q8) {
        f32x4 p[kUnitOf<Q8>];
#pragma unroll
        for (int j = 0; j < kUnitOf<Q8>; ++j) {
            const half8 w = q8_to_half8(make_uint2(f[j].x, f[j].y));
            p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j], w, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            p[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[j], w, p[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < kUnitOf<Q8>; ++j) {
            const float d = (float)__builtin_bit_cast(_Float16, (unsigned short)f[j].z);
            acc += d * p[j];
        }
        return acc;
    }
    // f16 weights: hi and lo activations; f32 weights: the lo plane (odd
    // sub-blocks) skips the lo activations (lo x lo is below f32 rounding)
    f32x4 lo = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kUnitOf<Q8>; ++j) {
        const half8 w = __builtin_bit_cast(half8, f[j]);
        const half8 b2 = (two && ((sb0 + j) & 1)) ? half8{} : al[j];
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[j], w, acc, 0, 0, 0);
        lo = __builtin_amdgcn_mfma_f32_16x16x32_f16(b2, w, lo, 0, 0, 0);
    }
    return acc + lo;
}

// Wavefront-reduction GEMV form of unit_mma for column tiles with at most
// kGemvCols live utterances (q8_0 weights): VALU dot products instead of a
// 16-column MFMA tile of which at most kGemvCols columns are live.  Lane l
// takes weight row l % 16 and the K slice 8 (l / 16) .. +7 of every block (the
// fragment it loaded), multiplies it with each live utterance's activations
// (hi + lo, exact in f32) in f32, scales by the block's d, and the four lanes
// of a row sum their slices with two shuffles.  The partial lands in the
// layout unit_mma produces (lane l < 16: row l, utterances 0 .. 3), so the
// reduce and the epilogues are the same; columns 4 .. 15 read as zero.
constexpr int kGemvCols = 4;
template <int U>
__device__ __forceinline__ f32x4 unit_gemv(const uint4 (&f)[U], const Act &x, int sb0, int nb, int lane) {
    const int g = lane >> 4;
    float acc[kGemvCols] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const unsigned q0 = f[j].x, q1 = f[j].y;
        // the stored bytes are q + 128: exact small integers in f32
        const float w[8] = {(float)(q0 & 0xffu) - 128.f, (float)((q0 >> 8) & 0xffu) - 128.f,
                            (float)((q0 >> 16) & 0xffu) - 128.f, (float)(q0 >> 24) - 128.f,
                            (float)(q1 & 0xffu) - 128.f, (float)((q1 >> 8) & 0xffu) - 128.f,
                            (float)((q1 >> 16) & 0xffu) - 128.f, (float)(q1 >> 24) - 128.f};
        const float d = (float)__builtin_bit_cast(_Float16, (unsigned short)f[j].z);
        // blocks past the weights' K (zero scales, matrices padded to whole units) read the last
        // real block's activations, which are finite
        const int ko = (sb0 + min(j, nb - 1)) * 32 + g * 8;
#pragma unroll
        for (int u = 0; u < kGemvCols; ++u) {
            if (u >= x.n) break;   // wave-uniform
            const half8 h = *reinterpret_cast<const half8 *>(x.hi + u * x.kp + ko);
            const half8 l = *reinterpret_cast<const half8 *>(x.lo + u * x.kp + ko);
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) sum = fmaf(w[i], (float)h[i] + (float)l[i], sum);
            acc[u] = fmaf(d, sum, acc[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < kGemvCols; ++u) {
        acc[u] += __shfl_xor(acc[u], 16, kWave);
        acc[u] += __shfl_xor(acc[u], 32, kWave);
    }
    return lane < kTile ? f32x4{acc[0], acc[1], acc[2], acc[3]} : f32x4{0.f, 0.f, 0.f, 0.f};
}

// Wave w's unit range [c0, c1) of N units.  Waves w and w + 4 share SIMD w & 3,
// and the older one (w < 4) wins the issue arbitration: for equal ranges the
// younger one finishes 15-30 % later, and the reduce waits for it.  So each SIMD
// gets an even quarter of the units, and its older wave takes the odd unit and,
// with at least 12 units per SIMD, 19 % more than half (76 / 128).  Partials are
// reduced in chunk order, so the split does not change results.  Measured
// against an even split over the 8 waves (two A/Bs chained): B=256, ragged
// B=512 and TDT-1.1b f16 about -3 %, B=64 -0.5 %, B=1 +1.5 %; a 28 % skew
// gained no more.
static_assert(kWaves == 8, "wave_range pairs waves w and w + 4 on SIMD w & 3");
__device__ __forceinline__ void wave_range(int N, int w, int &c0, int &c1) {
    const int j = w & 3, a = (N * j) >> 2, b = (N * (j + 1)) >> 2, len = b - a;
    const int d = N >= 48 ? 12 : 0;
    const int o = (len * (64 + d) + 64) >> 7;   // the older wave's share of its SIMD's range
    c0 = w < 4 ? a : a + o;
    c1 = w < 4 ? a + o : b;
}

// Partials of items j0 .. j1-1 (one pass), K-major, next unit's weights prefetched.
template <bool Q8, bool CACHED, bool FULL, bool GV = false>
__device__ __forceinline__ void phase_partials(const TMat &A, int n_a, const TMat &Bm, int j0, int j1, int rank, int P,
                                               const Act &x, f32x4 *red, const unsigned char *wc) {
    // wave-uniform unit bookkeeping: the weight buffer descriptors stay in SGPRs
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool two = !Q8 && A.type == PK_TYPE_F32;
    const int KBe = two ? 2 * A.KB : A.KB;
    const int KBa = two ? 2 * A.KBa : A.KBa;          // blocks with weights (activations past them are never read)
    constexpr int U = kUnitOf<Q8>;
    const int S = (KBe + U - 1) / U;                  // units per item
    const int nj = j1 - j0, N = nj * S;
    int c0, c1;
    wave_range(N, wave, c0, c1);
    if (c0 >= c1) return;
    // Column c of the product depends only on row c of the activations; rows
    // past x.n are not staged (they hold older values) and the columns they
    // feed are never read.
    const int xo = (lane & 15) * x.kp + (lane >> 4) * 8;
    const MatSrc sA = mat_src<Q8, CACHED>(A, two, wc), sB = mat_src<Q8, CACHED>(Bm, two, wc);
    auto load = [&](int item, int c, uint4 (&f)[U]) {
        const bool in_a = item < n_a;
        const int li = in_a ? item : item - n_a;
        const int sb0 = c * U;
        unit_load_src<Q8, CACHED, FULL>(in_a ? sA : sB, two, rank + li * P, li, sb0, min(U, KBe - sb0), lane, f);
    };
    half8 ah[U], al[U];
    uint4 fa[U], fb[U];
    // u = c * nj + i: c < S, so short wave-uniform loops instead of divisions
    int u = c0, c = 0, i = c0, cur = -1;
    while (i >= nj) {
        i -= nj;
        ++c;
    }
    // f16 / f32 from L2: the prefetch past the range reloads the wave's last unit,
    // an address the compiler cannot equate with the set in flight (reloading the
    // current unit, it copies that set instead, waiting for its loads)
    int cl = 0, il = c1 - 1;
    while (il >= nj) {
        il -= nj;
        ++cl;
    }
    load(j0 + i, c, fa);
    // one unit: issue the next unit's loads into fn, then multiply fc
    auto step = [&](uint4 (&fc)[U], uint4 (&fn)[U]) {
        int nc = c, ni = i + 1;
        if (ni == nj) {
            ni = 0;
            ++nc;
        }
        // q8_0 from L2: issued on every step (the last one reloads the current
        // unit).  With a conditional prefetch the compiler's wait counts after
        // the join assume no prefetch, so each unit's products would also wait
        // for the next unit's first loads.  (Measured: B=256 q8_0 -6 %; the f16
        // and LDS-cached paths are faster with the conditional form.)
        if (u + 1 < c1) load(j0 + ni, nc, fn);
        else if (Q8 && !CACHED) load(j0 + i, c, fn);
        else if (!CACHED) load(j0 + il, cl, fn);   // f16 / f32: the wave's last unit (see below)
        const int sb0 = c * U;
        if constexpr (GV) {
            red[(i * S + c) * kWave + lane] = unit_gemv<U>(fc, x, sb0, min(U, KBa - sb0), lane);
        } else {
            if (c != cur) {
                unit_act(x, xo, two, sb0, min(U, KBa - sb0), ah, al);
                cur = c;
            }
            red[(i * S + c) * kWave + lane] = unit_mma<Q8>(fc, ah, al, two, sb0, f32x4{0.f, 0.f, 0.f, 0.f});
        }
        ++u;
        c = nc;
        i = ni;
    };
    while (true) {
        step(fa, fb);
        if (u >= c1) break;
        step(fb, fa);
        if (u >= c1) break;
    }
    TL(2);
}

// Sum each item's partials of one pass in chunk order and run epi(item, acc);
// items are dealt round robin over the waves.  Opens with a barrier (all
// partials written); the caller's next barrier (before any new partials or
// staging) closes it.
template <class EpiFn>
__device__ __forceinline__ void phase_reduce(int j0, int j1, int S, const f32x4 *red, EpiFn epi) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    lds_sync();
    TL(3);
    for (int it = j0 + wave; it < j1; it += kWaves) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int c = 0; c < S; ++c) acc += red[((it - j0) * S + c) * kWave + lane];
        epi(it, acc);
    }
    TL(4);
}

// Weight classes the decode loop is compiled for: each instantiation carries
// only the phase engines its matrices need (a smaller kernel with its own
// register allocation).  kWcAny serves models whose phases mix storage types.
// kWcQ8Gemv: all-q8_0 decoders with the wavefront-reduction GEMV form for column
// tiles of at most kGemvCols live utterances (its own instantiation, so the
// default kernels keep their registers; selected by PK_GEMV=1 for comparisons:
// the MFMA form measured faster at every batch size).
enum { kWcQ8 = 0, kWcHalf = 1, kWcAny = 2, kWcQ8Gemv = 3 };

// Products of one phase for this workgroup, then the epilogue per item, in
// passes of at most `batch` items (red_slots / S, computed once per launch).
template <int WC, class EpiFn>
__device__ __forceinline__ void run_phase(const TMat &A, int n_a, const TMat &Bm, int n_items, int rank, int P,
                                          const Act &x, f32x4 *red, const unsigned char *wc, int batch, EpiFn epi) {
    if (n_items <= 0) return;
    // both matrices of a phase are in the LDS weight cache or neither
    const bool cached = wc != nullptr && A.lds_off >= 0;
    const int KBe = A.type == PK_TYPE_F32 ? 2 * A.KB : A.KB;
    const int U = (WC == kWcQ8 || WC == kWcQ8Gemv) ? kUnitOf<true> : WC == kWcHalf ? kUnitOf<false> : unit_blocks(A.type);
    const int S = (KBe + U - 1) / U;
    for (int j0 = 0; j0 < n_items; j0 += batch) {
        const int j1 = min(n_items, j0 + batch);
        if (j0 > 0) lds_sync();   // the previous pass's reduce has read its slots
        // matrices are stored with whole units of K blocks (zero blocks past
        // K / 32), so unit loads are never masked
        auto q8 = [&]() {
            if (WC == kWcQ8Gemv && x.n <= kGemvCols) {
                if (cached) phase_partials<true, true, true, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
                else phase_partials<true, false, true, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
            } else if (cached) {
                phase_partials<true, true, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
            } else {
                phase_partials<true, false, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
            }
        };
        auto half = [&]() {
            if (cached) phase_partials<false, true, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
            else phase_partials<false, false, true>(A, n_a, Bm, j0, j1, rank, P, x, red, wc);
        };
        if constexpr (WC == kWcQ8 || WC == kWcQ8Gemv) q8();
        else if constexpr (WC == kWcHalf) half();
        else if (A.type == PK_TYPE_Q8_0) q8();
        else half();
        phase_reduce(j0, j1, S, red, epi);
    }
}

// Tiles of a matrix with `tiles` row tiles owned by rank r of P: t = r, r+P, ...
__device__ __forceinline__ int owned(int tiles, int r, int P) { return tiles > r ? (tiles - r + P - 1) / P : 0; }

// n / d without a division, for n * d < 2^32: with m = floor(2^32 / d) + 1,
// floor(n * m / 2^32) = floor(n / d + n * e / 2^32) (0 < e <= 1), and the added
// term stays below 1 / d, the distance from n / d up to the next integer.
__host__ __device__ inline unsigned udiv_magic(unsigned d) { return d <= 1 ? 0u : (unsigned)(0x100000000ull / d + 1); }
__device__ __forceinline__ int udiv(int n, unsigned m, int d) { return d <= 1 ? n : (int)__umulhi((unsigned)n, m); }

// Units (kUnitOf K blocks) per tile row of a matrix.
__device__ __forceinline__ int units_per_item(const TMat &m) {
    const int KBe = m.type == PK_TYPE_F32 ? 2 * m.KB : m.KB, U = unit_blocks(m.type);
    return (KBe + U - 1) / U;
}

// LSTM state of layers >= 1 kept in LDS by the workgroup that owns the units:
// for layer l, utterance ul (domain index) and owned tile k (tile rank + kP,
// units 4t .. 4t+3): R_l rows 16t .. 16t+15 (W_hh_l . h_l, unit-major), then
// c_l of the 4 units.  Those units' gates are produced (the recurrent product
// of the phase that consumes h_l) and consumed (the cell update) by the same
// workgroup, so they never travel through memory inside a launch.
constexpr int kStFloats = kTile + 4;

struct Lds {
    Act act[1 + PK_MAX_LAYERS];   // staged activation blocks
    float *st;                    // [L-1][st_n][st_k][kStFloats] LDS state of layers >= 1
    float *bias;                  // epilogue bias rows of this workgroup's tiles (see bias_table)
    f32x4 *red;                   // [red_slots][kWave] per-(item, chunk) partials of one pass
    const unsigned char *wcache;  // weight cache (nullptr when the tiles do not fit)
};

// Epilogue bias rows of this workgroup's tiles, in LDS for the whole launch:
// the 16 rows of each owned tile of W_ih_l (b_ih_l + b_hh_l, l = 1 .. L-1;
// 4H/16 tiles each), then of W_p (b_p; J/16 tiles), then of W_o (b_o).
// The rows of matrix m start at float kTile * m * own_lstm (m = 0 .. L-2 the
// LSTM layers 1 .. L-1, m = L-1 W_p) and W_o's at kTile * ((L-1) * own_lstm +
// own_pred): H and J are multiples of 32, so own_lstm and own_pred count the
// 4H/16 and J/16 tiles used here.
__device__ __forceinline__ void bias_table(const KParams &p, int rank, int P, float *tab) {
    const int n_lstm = owned(p.H / 4, rank, P), n_pred = owned(p.J / kTile, rank, P);
    const int n_out = owned(p.w_out.tiles, rank, P);
    const int nl = (p.L - 1) * n_lstm * kTile, np = n_pred * kTile, no = n_out * kTile;
    for (int i = threadIdx.x; i < nl + np + no; i += kBlock) {
        float v;
        if (i < nl) {
            const int l = 1 + i / (n_lstm * kTile), r = i % (n_lstm * kTile);
            v = p.b_lstm[l][(rank + (r / kTile) * P) * kTile + r % kTile];
        } else if (i < nl + np) {
            const int r = i - nl;
            v = p.b_pred[(rank + (r / kTile) * P) * kTile + r % kTile];
        } else {
            const int r = i - nl - np;
            const int row = (rank + (r / kTile) * P) * kTile + r % kTile;
            v = row < p.Vo ? p.b_out[row] : 0.0f;
        }
        tab[i] = v;
    }
}

// Copy this workgroup's tiles of m (rank, rank+P, ...) into its LDS cache:
// per K block the fragment, then (q8_0) the 16 block scales.  kCacheB 16-byte
// chunks per thread are loaded before any is stored.
constexpr int kCacheB = 8;
// 16-byte chunk c of this workgroup's cached image of m: its tiles in order,
// each as stored (q8_0 unit records, f16 fragments; f32: per K block the hi
// then the lo fragment).
__device__ __forceinline__ const unsigned char *cache_src(const TMat &m, int rank, int P, int chunks, int c) {
    const int ch = c % chunks, li = c / chunks;   // chunks: of one tile
    const size_t t = (size_t)(rank + li * P);      // global tile
    if (m.type != PK_TYPE_F32) return static_cast<const unsigned char *>(m.a) + t * (size_t)chunks * 16 + ch * 16;
    const int kb = ch / 128, part = ch % 128;      // f32: 128 chunks per block (64 hi, 64 lo)
    return static_cast<const unsigned char *>(part < 64 ? m.a : m.a_lo) + (t * m.KB + kb) * 1024 + (part % 64) * 16;
}
__device__ __forceinline__ void cache_matrix(const TMat &m, int rank, int P, unsigned char *wc) {
    if (m.lds_off < 0) return;
    const int n = owned(m.tiles, rank, P);
    const int chunks = tile_bytes(m.type, m.KB) / 16;
    const int nchunk = n * chunks;
    if (nchunk == 0) return;
    for (int base = 0; base < nchunk; base += kCacheB * kBlock) {
        uint4 v[kCacheB];
#pragma unroll
        for (int j = 0; j < kCacheB; ++j)   // clamped: chunks past the end reload the last one
            v[j] = *reinterpret_cast<const uint4 *>(cache_src(m, rank, P, chunks, min(base + (int)threadIdx.x + j * kBlock, nchunk - 1)));
#pragma unroll
        for (int j = 0; j < kCacheB; ++j) {
            const int c = base + threadIdx.x + j * kBlock;
            if (c < nchunk) *reinterpret_cast<uint4 *>(wc + m.lds_off + (size_t)c * 16) = v[j];
        }
    }
}

// Row mapping of the joint's staging: a wave covers one pred tile (16 values)
// of 16 columns, 1 KB in a row of ppx; thread t takes column (t / 4) % 16,
// values 4 (t % 4) .. +3 of pred tiles t / 64, t / 64 + 8, ...
// The encp rows of the first round (column tile 0) are loaded at the start of
// the iteration: the list rebuild has fixed every column's frame, and the loads
// complete during layer 0, whose own loads take as long, instead of at the
// joint's staging.
__device__ __forceinline__ void encp_prefetch(const KParams &p, const Ctl &s, const Bufs &B, int ncol, float4 (&e)[kStageMax]) {
    const int J = p.J, ntile = J / kTile, g = threadIdx.x & 3, u = (threadIdx.x >> 2) & 15, t0 = threadIdx.x >> 6;
    const bool live = u < min(kTile, ncol);
    const unsigned erow = (unsigned)s.crow[live ? u : 0].x;
#pragma unroll
    for (int j = 0; j < kStageMax; ++j) {
        const int t = t0 + kWaves * j;
        e[j] = ld4(B.encp, live && t < ntile ? erow + (unsigned)(t * kTile + g * 4) * 4 : kBad);
    }
}

// Joint + argmax for this workgroup's output tiles.  Utterances are processed
// 16 at a time (one MFMA column tile).
template <int WC>
__device__ __forceinline__ void joint_phase(const KParams &p, Ctl &s, const Bufs &B, const Lds &S, unsigned stamp, int ncol,
                            const float4 (&epre)[kStageMax], unsigned long long &tlast) {
    const int J = p.J, lane = threadIdx.x & (kWave - 1);
    if (threadIdx.x < 2 * kColCap) s.wgkey[threadIdx.x / 2][threadIdx.x % 2] = 0ull;
    const int n_out = s.own_out;
    for (int c0 = 0; c0 < ncol; c0 += kTile) {
        const int nc = min(kTile, ncol - c0);
        Act x = S.act[0];
        x.n = nc;
        // stage hidden = relu(encp[t] + pp) for this column tile
        {
            const int ntile = J / kTile, g = threadIdx.x & 3, u = (threadIdx.x >> 2) & 15, t0 = threadIdx.x >> 6;
            const bool live = u < nc;
            const int2 row = *reinterpret_cast<const int2 *>(&s.crow[c0 + (live ? u : 0)]);
            const unsigned erow = (unsigned)row.x, prow = (unsigned)row.y + g * 16u;
            const unsigned stride = (unsigned)p.prows * kTile * 4u;
            for (int b0 = 0; b0 < ntile; b0 += kWaves * kStageMax) {
                float4 e[kStageMax];
                unsigned pend = 0u, n = 0u;
                unsigned long long since = 0ull;
#pragma unroll
                for (int j = 0; j < kStageMax; ++j) {
                    const int t = b0 + t0 + kWaves * j;
                    const bool ok = live && t < ntile;
                    e[j] = (c0 == 0 && b0 == 0) ? epre[j]
                                                : ld4(B.encp, ok ? erow + (unsigned)(t * kTile + g * 4) * 4 : kBad);
                    if (ok) pend |= 1u << j;
                }
                while (pend != 0u) {
                    float4 q[kStageMax];
#pragma unroll
                    for (int j = 0; j < kStageMax; ++j)
                        q[j] = ld4_coh(B.ppx, (pend >> j) & 1u ? prow + (unsigned)(b0 + t0 + kWaves * j) * stride : kBad);
#pragma unroll
                    for (int j = 0; j < kStageMax; ++j)
                        if (((pend >> j) & 1u) && !has_empty(q[j])) {
                            float4 v = make_float4(e[j].x + q[j].x, e[j].y + q[j].y, e[j].z + q[j].z, e[j].w + q[j].w);
                            v.x = (0.0f < v.x) ? v.x : 0.0f;
                            v.y = (0.0f < v.y) ? v.y : 0.0f;
                            v.z = (0.0f < v.z) ? v.z : 0.0f;
                            v.w = (0.0f < v.w) ? v.w : 0.0f;
                            put4(x, u, (b0 + t0 + kWaves * j) * kTile + g * 4, v);
                            pend &= ~(1u << j);
                        }
                    if (pend != 0u && wait_over(p, s, n, since)) break;
                }
            }
        }
        TLBASE(21);
        lds_sync();
        TL(0);
        pmark(p, s, tlast, kPrJStage);
        // after the epilogue's quad transpose (see quad_transpose) a lane holds
        // rows 4g .. 4g+3 of a tile for utterance u of the column tile; its blank
        // offset is loaded before the products
        const int u = 4 * (lane >> 4) + (lane & 3), g = (lane >> 2) & 3;
        const float bb = u < nc ? __int_as_float(s.crow[c0 + u].z) : 0.0f;
        // (b_out is zero-padded to whole tiles)
        const float *btab = S.bias + kTile * ((p.L - 1) * s.own_lstm + s.own_pred);
        TL(1);
        // debug logit tap: this lane's column (spare columns included) into the staging rows;
        // the decision step copies a column to the row of the step that takes it
        float *ltap = nullptr;
        if (p.logits && u < nc) ltap = p.lcol + ((size_t)s.dom * kColCap + c0 + u) * p.Vo;
        // each lane keeps the best value (as ordered bits, never 0) and row of each head:
        // its rows come in ascending order, so "greater" keeps the first index; the four
        // lanes of one utterance then combine, and one LDS atomic per utterance and
        // head follows.  (64-bit keys per row, with the head, the range and the blank
        // tested row by row, made the reduce of a 24-tile pass 2.4 us; with one test per
        // tile and 32-bit compares the joint's products and reduce fall from 11.0 to
        // 10.2 us at B = 256 and from 17.1 to 15.9 at B = 512.)
        unsigned top0 = 0u, top1 = 0u;
        int row0 = 0, row1 = 0;
        run_phase<WC>(p.w_out, n_out, p.w_out, n_out, s.rank, s.P, x, S.red, S.wcache, s.pass[p.L],
                  [&](int k, f32x4 acc) {
                      acc = quad_transpose(acc);   // every lane of the wave takes part
                      const int tile = s.rank + k * s.P, first = tile * kTile;   // wave-uniform
                      const float4 bias4 = *reinterpret_cast<const float4 *>(btab + k * kTile + g * 4);
                      float v[4] = {acc[0] + bias4.x, acc[1] + bias4.y, acc[2] + bias4.z, acc[3] + bias4.w};
                      if ((unsigned)(p.blank - first) < (unsigned)kTile) {
#pragma unroll
                          for (int i = 0; i < 4; ++i)
                              if (first + g * 4 + i == p.blank) v[i] += bb;
                      }
                      if (ltap) {
#pragma unroll
                          for (int i = 0; i < 4; ++i)
                              if (first + g * 4 + i < p.Vo) st_coh(ltap + first + g * 4 + i, v[i]);
                      }
                      if (first + kTile <= p.V1) {   // token rows only
#pragma unroll
                          for (int i = 0; i < 4; ++i) {
                              const unsigned o = max(ordered_bits(v[i]), 1u);
                              const bool better = o > top0;
                              top0 = better ? o : top0;
                              row0 = better ? first + g * 4 + i : row0;
                          }
                      } else {
#pragma unroll
                          for (int i = 0; i < 4; ++i) {
                              const int row = first + g * 4 + i;
                              const unsigned o = max(ordered_bits(v[i]), 1u);
                              const bool b0 = row < p.V1 && o > top0, b1 = row >= p.V1 && row < p.Vo && o > top1;
                              top0 = b0 ? o : top0;
                              row0 = b0 ? row : row0;
                              top1 = b1 ? o : top1;
                              row1 = b1 ? row - p.V1 : row1;
                          }
                      }
                  });
        // the lanes of utterance u differ in bits 2 and 3
        u64 best0 = top0 != 0u ? make_key(top0, row0) : 0ull, best1 = top1 != 0u ? make_key(top1, row1) : 0ull;
        best0 = row_ror_max<0x124>(row_ror_max<0x128>(best0));
        best1 = row_ror_max<0x124>(row_ror_max<0x128>(best1));
        if (g == 0 && u < nc) {
            if (best0) atomicMax(&s.wgkey[c0 + u][0], best0);
            if (best1) atomicMax(&s.wgkey[c0 + u][1], best1);
        }
        // the keys stored next say that this workgroup's other stores of the iteration have landed
        if (c0 + kTile >= ncol) __builtin_amdgcn_s_waitcnt(0);
        lds_sync();
        TLA(27);
        pmark(p, s, tlast, kPrJCompute);
    }
    // this workgroup's stamped best token key of every joint column, one line per
    // workgroup; the duration keys from the ranks that own duration rows
    if (threadIdx.x < 2 * ncol) {
        const int u = threadIdx.x >> 1, head = threadIdx.x & 1;
        const unsigned long long k = ((unsigned long long)stamp << kStampShift) | s.wgkey[u][head];
        const size_t par = stamp & 1;
        if (head == 0) {
            __hip_atomic_store(p.keys + ((par * p.n_dom + s.dom) * s.P + s.rank) * p.cols + u, k, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        } else {
            for (int d = 0; d < p.n_durk; ++d)
                if (p.dur_rank[d] == s.rank)
                    __hip_atomic_store(p.keys + (size_t)2 * p.n_dom * s.P * p.cols +
                                           ((par * p.n_dom + s.dom) * 2 + d) * p.cols + u,
                                       k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    TLA(28);
}

// Layer 0 from the precomputed input projection: gates = E'[token] + R0,
// elementwise per unit.  redundant: every unit for every listed utterance,
// h' also written into the layer-1 activation block; otherwise only this
// workgroup's unit tiles.  Work item: unit g of list row u of a tile, so a wave
// stores whole tiles of the exchange buffer.
// Owners store h', c' coherently.
// Each thread issues the loads of up to kL0 units before computing any.
constexpr int kL0 = 3;
__device__ __forceinline__ void lstm_layer0(const KParams &p, Ctl &s, const Lds &S, const Bufs &B, bool redundant,
                                            int half, int nl, int lgn) {
    const int H = p.H;
    const int n_work = (redundant ? H / 4 : s.own_lstm) << (lgn + 2);
    for (int base = 0; base < n_work; base += kL0 * kBlock) {
        float4 e[kL0], r[kL0];
        float c_prev[kL0];
#pragma unroll
        for (int q = 0; q < kL0; ++q) {   // no branches: unused loads take kBad and return 0
            const int i = base + threadIdx.x + q * kBlock;
            const int k = i >> (lgn + 2), u = (i >> 2) & ((1 << lgn) - 1);
            const int j = 4 * (redundant ? k : s.rank + k * s.P) + (i & 3);
            const bool ok = i < n_work && u < nl;
            const int2 row = *reinterpret_cast<const int2 *>(&s.lrow[u < nl ? u : 0]);
            const bool st = ok && row.y >= 0;
            e[q] = ld4(B.ep, ok ? (unsigned)(row.x + 16 * j) : kBad);
            r[q] = ld4_coh(B.rx, st ? (unsigned)(4 * row.y + 16 * j) : kBad);
            c_prev[q] = ld1_coh(B.cx, st ? (unsigned)(row.y + 4 * j) : kBad);
        }
#pragma unroll
        for (int q = 0; q < kL0; ++q) {
            const int i = base + threadIdx.x + q * kBlock;
            const int k = i >> (lgn + 2), u = (i >> 2) & ((1 << lgn) - 1), g = i & 3;
            if (i >= n_work || u >= nl) continue;
            const int tile = redundant ? k : s.rank + k * s.P, j = 4 * tile + g;
            const int2 row = *(reinterpret_cast<const int2 *>(&s.lrow[u]) + 1);
            float c_new, h_new;
            cell(e[q].x + r[q].x, e[q].y + r[q].y, e[q].z + r[q].z, e[q].w + r[q].w, c_prev[q], c_new, h_new);
            if (redundant) {   // straight into the layer-1 activation block
                const Act &x = S.act[1];
                split_f16(h_new, x.hi[u * x.kp + j], x.lo[u * x.kp + j]);
            } else {
                st_coh(p.hx + hx_at(p, s.dom, 0, half, tile, u) + g, filled(h_new));
            }
            // owner of the tile (always, when only this workgroup's units are listed)
            if (!redundant || tile - udiv(tile, s.mag_p, s.P) * s.P == s.rank) {
                st_coh(p.cx + (row.x >> 2) + j, c_new);
                st_coh(p.hs + ((row.y & kRowMask) >> 2) + j, h_new);
            }
        }
    }
}

// Items of the phase that consumes layer lc's new output h_lc' (staged in x):
//   consumer tiles   W_ih_{lc+1} (LSTM layer lc+1, cell update in the epilogue:
//                    the four rows a lane holds are the four gates of one unit)
//                    or W_p (pred projection) when lc is the last layer;
//   recurrent tiles  W_hh_lc . h_lc' -> R_lc for the utterance's next step
//                    (R_0 in the half of rx of the new parity).
// Column tile: utterances lst[c0 .. c0+nc).
// Both matrices have K = H and the same storage type.
// LDS state of layer l (>= 1), utterance ul, owned tile k.
__device__ __forceinline__ float *st_at(const KParams &p, const Lds &S, int l, int ul, int k) {
    return S.st + ((size_t)((l - 1) * p.st_n + ul) * p.st_k + k) * kStFloats;
}

template <int WC>
__device__ __forceinline__ void consume_layer(const KParams &p, Ctl &s, const Lds &S, const Bufs &B, const Act &x,
                                              int lc, int half, int c0, int nc) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool last = lc == p.L - 1;
    const TMat &wc = last ? p.w_pred : p.w_ih[lc + 1];
    const TMat &wr = p.w_hh[lc];
    const int n_c = last ? s.own_pred : s.own_lstm, n_r = s.own_lstm;
    // the epilogue quad-transposes the (transposed) D fragment, after which a
    // lane holds rows 4g .. 4g+3 of a tile (the four gates of one unit, or four
    // pred rows) for one utterance u of the column tile
    const int layer = lc + 1, u = 4 * (lane >> 4) + (lane & 3), g = (lane >> 2) & 3;
    // this lane's utterance (a valid index for every lane; lanes u >= nc store nothing)
    const int2 row = *(reinterpret_cast<const int2 *>(&s.lrow[c0 + min(u, nc - 1)]) + 1);
    const int ul = row.y & kRowUl, cur = (row.y & kRowCur) ? 1 : 0;
    const bool zero = row.y & kRowZero;
    // bias rows of the consumer tiles (LDS table): lane rows row0 .. row0+3 are
    // the pred rows, or the four gates of unit j = row0 / 4
    const float *btab = S.bias + kTile * lc * s.own_lstm;
    TL(1);
    run_phase<WC>(wc, n_c, wr, n_c + n_r, s.rank, s.P, x, S.red, S.wcache, s.pass[lc],
              [&](int it, f32x4 acc) {
                  acc = quad_transpose(acc);   // every lane of the wave takes part
                  if (u >= nc) return;
                  if (it >= n_c) {          // recurrent product for the next step
                      const int k = it - n_c;
                      if (lc == 0) {        // R_0: read by the layer-0 update of every workgroup (global)
                          const int row0 = (s.rank + k * s.P) * kTile + g * 4;
                          st4_coh(B.rx, (unsigned)(4 * row.x + 4 * row0),
                                  make_float4(acc[0], acc[1], acc[2], acc[3]));
                      } else {              // R_lc: LDS state of this workgroup
                          *reinterpret_cast<float4 *>(st_at(p, S, lc, ul, k) + g * 4) =
                              make_float4(acc[0], acc[1], acc[2], acc[3]);
                      }
                      return;
                  }
                  const int row0 = (s.rank + it * s.P) * kTile + g * 4;
                  const float4 bias = *reinterpret_cast<const float4 *>(btab + it * kTile + g * 4);
                  if (last) {               // pred projection: rows row0 .. row0+3 of pp; the old ones emptied
                      const int t = s.rank + it * s.P;
                      st4_coh(B.ppx, (ppx_at(p, s.dom, cur, t, ul) + g * 4) * 4u,
                              make_float4(filled(acc[0] + bias.x), filled(acc[1] + bias.y), filled(acc[2] + bias.z),
                                          filled(acc[3] + bias.w)));
                      st4_coh(B.ppx, (ppx_at(p, s.dom, cur ^ 1, t, ul) + g * 4) * 4u, empty4());
                      return;
                  }
                  // cell update of unit j = row0 / 4 of layer `layer`: R and c_prev from the LDS state
                  float *st = st_at(p, S, layer, ul, it);
                  float4 r = *reinterpret_cast<const float4 *>(st + g * 4);
                  float c_prev = st[kTile + g];
                  if (zero) {
                      r = make_float4(0.f, 0.f, 0.f, 0.f);
                      c_prev = 0.0f;
                  }
                  float c_new, h_new;
                  cell((acc[0] + r.x) + bias.x, (acc[1] + r.y) + bias.y, (acc[2] + r.z) + bias.z,
                       (acc[3] + r.w) + bias.w, c_prev, c_new, h_new);
                  st[kTile + g] = c_new;
                  st_coh(p.hx + hx_at(p, s.dom, layer, half, s.rank + it * s.P, c0 + u) + g, filled(h_new));
                  st_coh(p.hs + (size_t)layer * p.n_utts * p.H + ((row.y & kRowMask) >> 2) + row0 / 4, h_new);
              });
}

// Empty this workgroup's tiles of h (every layer) in one half of hx, rows below n.
__device__ __forceinline__ void empty_h(const KParams &p, const Ctl &s, const Bufs &B, int half, int n) {
    const int lr = __builtin_ctz((unsigned)p.rows), per = s.own_lstm << lr;
    for (int l = p.hl0; l < p.L; ++l)
        for (int i = threadIdx.x; i < per; i += kBlock) {
            const int u = i & (p.rows - 1), t = s.rank + (i >> lr) * s.P;
            if (u < n) st4_coh(B.hx, hx_at(p, s.dom, l, half, t, u) * 4u, empty4());
        }
}

// One LSTM step (all layers), the pred projection and the recurrent products
// for every utterance of the LSTM list.  A small list in a whole-device
// domain runs layer 0 redundantly in every workgroup (no exchange between
// layers 0 and 1); otherwise layer 0 is split by unit tiles.  Each later phase
// stages one layer's full new output as it arrives and runs the tiles that
// consume it.  half: the half of hx this step uses; n_prev: list length of the
// previous step, whose half is emptied here.
template <int WC>
__device__ __forceinline__ void lstm_and_pred(const KParams &p, Ctl &s, const Bufs &B, const Lds &S, int half,
                                              int n_prev, int nl, int lgn, unsigned long long &tlast) {
    const int L = p.L;
    const bool redundant = nl <= kSmallB && p.n_dom == 1;
    lstm_layer0(p, s, S, B, redundant, half, nl, lgn);
    empty_h(p, s, B, half ^ 1, n_prev);
    TLA(1);
    pmark(p, s, tlast, kPrL0);
    for (int lc = 0; lc < L; ++lc) {
        const bool local = lc == 0 && redundant;     // h_0' is in LDS already
        for (int c0 = 0; c0 < nl; c0 += kTile) {
            const int nc = min(kTile, nl - c0);
            Act x = S.act[1];
            x.n = nc;
            // (redundant layer 0 wrote h_0' into the block itself.)  The block's last readers, the
            // previous products, are behind the barrier that opens their reduce.
            if (!local) stage_h(p, s, B, x, lc, half, c0, nc);
            TLBASE(2 + 8 * lc);
            lds_sync();
            TL(0);
            pmark(p, s, tlast, lc == 0 ? kPrStage0 : kPrStage1);
            consume_layer<WC>(p, s, S, B, x, lc, half, c0, nc);
            TL(6);
        }
        pmark(p, s, tlast, lc == L - 1 ? kPrPred : kPrL1);
    }
}

// The domain's best key per joint column and head.  Token keys: lane groups of
// `pairs` threads load two columns of one rank each (16 bytes) until both carry
// this iteration's stamp, every rank of the domain; then the wave's maximum per
// column and one LDS atomic max per wave.  Duration keys come from the ranks that
// own duration rows.  The stamp is the arrival signal: a workgroup that has seen
// every rank's keys knows that all of them are done with the iteration's staged
// data.  A rank cannot overwrite a key before every workgroup has read it: it
// stores the same half again two iterations on, after the keys of the next.
// Where one wave's loads cover every rank (domains of few workgroups, few columns) wave 0, which
// decides, gathers alone: no combining through LDS and no barrier before the decisions (with the
// prefix sum of the spare columns by DPP: B=1 -2 % of a call, B=256 and B=512 -2 %).
constexpr int kKeyRounds = 4;
__device__ __forceinline__ void gather_keys(const KParams &p, Ctl &s, const Bufs &B, unsigned stamp, int ncol) {
    lds_sync();   // this workgroup's key stores have read s.wgkey
    const int P = s.P, nc = ncol, lane = threadIdx.x & (kWave - 1);
    const int lgp = nc <= 2 ? 0 : 31 - __builtin_clz((unsigned)(nc - 1));   // log2 of the column pairs, rounded up
    const int pairs = 1 << lgp, cp = threadIdx.x & (pairs - 1), r0 = threadIdx.x >> lgp;
    const bool alone = P << lgp <= kWave * kKeyRounds;
    if (alone && threadIdx.x >= kWave) return;
    const int step = (alone ? kWave : kBlock) >> lgp;
    const unsigned dom = (stamp & 1) * p.n_dom + s.dom;
    const unsigned base = (dom * P * p.cols + 2 * cp) * 8u, stride = (unsigned)p.cols * 8u;
    const bool two = 2 * cp + 1 < nc, one = 2 * cp < nc;
    // the duration word of this thread, polled with its first round
    const int lc = __builtin_ctz((unsigned)p.cols), dc = threadIdx.x & (p.cols - 1), dd = threadIdx.x >> lc;
    bool want_d = dd < p.n_durk && dc < nc;
    const unsigned doff = (2u * p.n_dom * P * p.cols + (dom * 2 + dd) * p.cols + dc) * 8u;
    unsigned long long best0 = 0ull, best1 = 0ull, kd = 0ull;
    for (int rb = 0; rb < P; rb += step * kKeyRounds) {
        unsigned pend = 0u, n = 0u;
        unsigned long long since = 0ull;
#pragma unroll
        for (int q = 0; q < kKeyRounds; ++q)
            if (one && rb + r0 + step * q < P) pend |= 1u << q;
        while (pend != 0u || want_d) {
            typedef unsigned long long u64x2 __attribute__((ext_vector_type(2)));
            u64x2 v[kKeyRounds];
#pragma unroll
            for (int q = 0; q < kKeyRounds; ++q)
                v[q] = __builtin_bit_cast(u64x2, ld4_coh(B.keys, (pend >> q) & 1u
                                                                     ? base + (unsigned)(rb + r0 + step * q) * stride
                                                                     : kBad));
            const unsigned long long d = __builtin_bit_cast(
                unsigned long long, __builtin_amdgcn_raw_buffer_load_b64(B.keys, want_d ? doff : kBad, 0, kSC1));
#pragma unroll
            for (int q = 0; q < kKeyRounds; ++q)
                if (((pend >> q) & 1u) && key_stamp(v[q][0]) == stamp && (!two || key_stamp(v[q][1]) == stamp)) {
                    best0 = v[q][0] > best0 ? v[q][0] : best0;
                    best1 = two && v[q][1] > best1 ? v[q][1] : best1;
                    pend &= ~(1u << q);
                }
            if (want_d && key_stamp(d) == stamp) {
                kd = d;
                want_d = false;
            }
            if ((pend != 0u || want_d) && wait_over(p, s, n, since)) break;
        }
    }
    if (kd != 0ull) atomicMax(&s.wgkey[dc][1], kd);
    best0 = lanes_max(best0, pairs);
    best1 = lanes_max(best1, pairs);
    if (lane < pairs) {
        if (best0 != 0ull) atomicMax(&s.wgkey[2 * cp][0], best0);
        if (best1 != 0ull) atomicMax(&s.wgkey[2 * cp + 1][0], best1);
    }
    if (!alone) lds_sync();
    else __atomic_signal_fence(__ATOMIC_SEQ_CST);   // (a wave's LDS operations complete in order)
}

// Apply the argmax results of iteration `stamp` to every utterance of the joint
// list: src/parakeet_tdt.cpp:936-967 (TDT) and src/parakeet_eou.cpp:275-332 (EOU).
// One utterance per lane of wave 0.  Its first decision is column u.col (frame t);
// while the decision keeps the prediction output (a TDT blank; an EOU blank, <EOB>
// or special piece) and the next frame's column was evaluated, the walk goes
// on with that column, one step per column, exactly as later iterations would.
__device__ __forceinline__ void decide_steps(const KParams &p, Ctl &s, Utt &u, unsigned stamp) {
    const int ul = threadIdx.x;
    if (ul >= s.n || u.t >= u.T) return;
    const int b = s.b[ul];
    const bool writer = ((s.wmask >> ul) & 1u) != 0u;
    const int t0 = u.t;
    int col = u.col;
    while (true) {
        const unsigned long long kt = s.wgkey[col][0], kd = s.wgkey[col][1];
        if (key_stamp(kt) != stamp || (p.Dn > 0 && key_stamp(kd) != stamp)) {
            __hip_atomic_store(p.status, PK_ERR_DEVICE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            u.t = u.T;
            break;
        }
        const int tok = key_index(kt);
        const int di = p.Dn > 0 ? key_index(kd) : -1;
        const int step = u.steps++;
        if (p.logits && step < p.logit_steps) {
            const int q = atomicAdd(&s.tq_n, 1);
            s.tq_col[q] = col;
            s.tq_b[q] = b;
            s.tq_step[q] = step;
        }
        if (writer && p.trace) {
            if (step < p.trace_cap) {
                p.trace[((size_t)b * p.trace_cap + step) * 2] = tok;
                p.trace[((size_t)b * p.trace_cap + step) * 2 + 1] = di;
            } else {
                u.flags |= kFlagTraceOverflow;
            }
        }
        bool keep = false;   // the prediction output stays: the next frame may follow at once
        if (p.kind == PK_KIND_TDT) {
            const int dur = p.n_dur > 0 ? s.dur[di] : di;
            const int adv = dur > 1 ? dur : 1;
            if (tok == p.blank) {
                u.t += adv;
                u.sym = 0;
                keep = true;
            } else {
                const int n = u.ntok++;
                if (writer) {
                    if (n < p.token_cap) p.tokens[(size_t)b * p.token_cap + n] = tok;
                    else u.flags |= kFlagTokOverflow;
                }
                u.pend = tok;
                u.cur ^= 1;
                u.sym += 1;
                if (dur > 0 || u.sym >= p.max_sym) {
                    u.t += adv;
                    u.sym = 0;
                }
            }
        } else {
            const int max_syms = p.max_sym > 1 ? p.max_sym : 1;
            bool frame_done = false;
            if (tok == p.blank || tok == p.eob) {
                frame_done = true;
                keep = true;
            } else if (tok == p.eou) {
                const int total = s.tbase[ul] + u.ntok;
                if (total > s.segst[ul]) {
                    const int ns = s.nseg[ul]++;
                    if (writer) {
                        if (p.segs && ns < p.seg_cap) p.segs[(size_t)b * p.seg_cap + ns] = total;
                        else u.flags |= kFlagSegOverflow;
                    }
                    s.segst[ul] = total;
                }
                u.flags |= kFlagZeroHC;
                u.pend = p.blank;
                u.cur ^= 1;
                s.last[ul] = p.blank;
                frame_done = true;
            } else if (tok >= 0 && tok < p.n_special && p.special[tok]) {
                frame_done = true;
                keep = true;
            } else {
                const int n = u.ntok++;
                if (writer) {
                    if (n < p.token_cap) p.tokens[(size_t)b * p.token_cap + n] = tok;
                    else u.flags |= kFlagTokOverflow;
                }
                u.pend = tok;
                u.cur ^= 1;
                s.last[ul] = tok;
                u.sym += 1;
                if (u.sym >= max_syms) frame_done = true;
            }
            if (frame_done) {          // the next frame starts with sym = 0 (src/parakeet_eou.cpp:269)
                u.t += 1;
                if (u.t < u.T) u.sym = 0;
            }
        }
        // the next decision's frame offset from t0, if its column was evaluated
        u.keep = keep ? 1 : 0;
        if (!keep || u.t >= u.T) break;
        const int o = u.t - t0;
        if (o > u.sn) break;
        col = u.sbase + o - 1;
    }
}

// Logit tap: the staged logits of each column a decision took go to the row of
// that decision's step.  Every workgroup copies the rows of its own W_o tiles,
// the ones it staged (so no other workgroup's stores are read).
__device__ __forceinline__ void tap_copy(const KParams &p, Ctl &s) {
    __builtin_amdgcn_s_waitcnt(0);   // this workgroup's staging stores are complete
    lds_sync();
    const int rows = s.own_out * kTile;
    for (int e = threadIdx.x; e < s.tq_n * rows; e += kBlock) {
        const int q = e / rows, r = e - q * rows;
        const int row = (s.rank + (r / kTile) * s.P) * kTile + r % kTile;
        if (row >= p.Vo) continue;
        const float v = ld_coh(p.lcol + ((size_t)s.dom * kColCap + s.tq_col[q]) * p.Vo + row);
        p.logits[((size_t)s.tq_b[q] * p.logit_steps + s.tq_step[q]) * p.Vo + row] = v;
    }
    lds_sync();
    if (threadIdx.x == 0) s.tq_n = 0;
}

__device__ __forceinline__ void decide(const KParams &p, Ctl &s, Utt &u, unsigned stamp) {
    if (threadIdx.x < kWave && s.ok) decide_steps(p, s, u, stamp);
    if (p.logits) {
        lds_sync();
        tap_copy(p, s);
    }
}

// Co-residency of an ordinary dispatch.  The loop's barriers need every
// workgroup of the grid resident at once, which a cooperative launch
// guarantees and an ordinary dispatch does not (a long kernel on another
// stream may hold CUs).  Each workgroup stores an arrival flag (word 1 of its
// barrier flag slot).  Workgroup 0 watches every flag, one thread per
// workgroup, for up to p.arrive_ticks, and proposes "go" if all arrived,
// "abort" if not; any other workgroup that has waited twice that long for a
// decision proposes "abort" (workgroup 0 itself may be the one not resident).
// One compare-and-swap on the decision word settles it, and every workgroup
// follows it.  On "abort" no workgroup has written anything but these words;
// the winner of the abort sets the error word to kStatusNotResident, and the
// host relaunches the call cooperatively.  A workgroup that starts after the
// decision reads it and leaves.  Every wait is bounded by the tick limit.
constexpr unsigned kArriveGo = 1u, kArriveAbort = 2u;
__device__ __forceinline__ void propose(const KParams &p, unsigned *dec, unsigned want) {
    unsigned z = 0u;
    if (__hip_atomic_compare_exchange_strong(dec, &z, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) &&
        want == kArriveAbort)
        __hip_atomic_store(p.status, kStatusNotResident, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool coresident(const KParams &p) {
    __shared__ unsigned s_dec;
    __shared__ int s_all;
    unsigned *dec = reinterpret_cast<unsigned *>(p.status + 9);
    if (threadIdx.x == 0) {
        s_all = 1;
        __hip_atomic_store(p.flags + (size_t)blockIdx.x * kFlagStride + 1, 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    if (blockIdx.x == 0) {   // the decider (gridDim.x <= the block size)
        __syncthreads();
        if (threadIdx.x < gridDim.x) {
            const unsigned *f = p.flags + (size_t)threadIdx.x * kFlagStride + 1;
            const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
            while (__hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
                if (__builtin_amdgcn_s_memrealtime() - t0 > p.arrive_ticks) {
                    s_all = 0;
                    break;
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) propose(p, dec, s_all ? kArriveGo : kArriveAbort);
    }
    if (threadIdx.x == 0) {
        const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
        unsigned d;
        while ((d = __hip_atomic_load(dec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0u)
            if (__builtin_amdgcn_s_memrealtime() - t0 > 2ull * p.arrive_ticks) propose(p, dec, kArriveAbort);
        s_dec = d;
    }
    __syncthreads();
    return s_dec == kArriveGo;
}

template <int WC>
__global__ void __launch_bounds__(kBlock) decode_loop_kernel(KParams p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    __shared__ Ctl s;
    if (p.arrive_ticks != 0u && !coresident(p)) return;
    const int wg = blockIdx.x;
    const int H = p.H, L = p.L, J = p.J, n_all = p.n_utts;
    unsigned epoch = 0;
    Bufs B;
    B.hx = rsrc(p.hx, (unsigned)((size_t)2 * (L - p.hl0) * p.n_dom * H * p.rows * 4));
    B.cx = rsrc(p.cx, (unsigned)((size_t)2 * n_all * H * 4));
    B.ppx = rsrc(p.ppx, (unsigned)((size_t)2 * p.n_dom * J * p.prows * 4));
    B.rx = rsrc(p.rx, (unsigned)((size_t)2 * n_all * 4 * H * 4));
    B.keys = rsrc(p.keys, (unsigned)((size_t)2 * p.n_dom * (p.dom_size + 2) * p.cols * 8));
    B.ep = rsrc(p.eproj, (unsigned)((size_t)p.V1 * 4 * H * 4));
    B.encp = rsrc(p.encp, (unsigned)(p.encp_rows * J * 4));

    // LDS: one activation block (the joint's hidden block and the LSTM phases'
    // block are never live together), per-(item, wave) partials, then the
    // weight cache
    Lds S;
    unsigned char *wcache = nullptr;
    {
        unsigned char *q = lds_raw;
        for (int a = 0; a <= 1; ++a) {
            const int K = a == 0 ? J : H;
            const int kp = K + kKPad;
            S.act[a].hi = reinterpret_cast<_Float16 *>(q);
            S.act[a].lo = S.act[a].hi + kTile * kp;
            S.act[a].kp = kp;
            S.act[a].n = kTile;
        }
        q += (size_t)kTile * ((J > H ? J : H) + kKPad) * 2 * 2;
        S.st = reinterpret_cast<float *>(q);
        q += (size_t)(L - 1) * p.st_n * p.st_k * kStFloats * 4;
        S.bias = reinterpret_cast<float *>(q);
        q += (size_t)p.bias_floats * 4;
        S.red = reinterpret_cast<f32x4 *>(q);
        q += (size_t)p.red_slots * kWave * sizeof(f32x4);
        if (p.wcache_bytes > 0) wcache = q;
        S.wcache = wcache;
    }

    if (threadIdx.x < kPrN) s.prof[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) s.tq_n = 0;
#ifdef PK_TIMELINE
    if (threadIdx.x < kWaves * kTl) tl_sum()[threadIdx.x] = 0ull;
    if (threadIdx.x < 2 + kTl) tl_ctl()[threadIdx.x] = 0;
#endif
    if (threadIdx.x == 0) {
        s.dom = p.wg_dom[wg];
        s.rank = p.wg_rank[wg];
        s.P = p.dom_size;
        s.n = p.dom_n[s.dom];
        s.own_lstm = owned(p.w_hh[0].tiles, s.rank, s.P);
        s.own_pred = owned(p.w_pred.tiles, s.rank, s.P);
        s.own_out = owned(p.w_out.tiles, s.rank, s.P);
        for (int lc = 0; lc < p.L; ++lc)
            s.pass[lc] = p.red_slots / units_per_item(lc == p.L - 1 ? p.w_pred : p.w_ih[lc + 1]);
        s.pass[p.L] = p.red_slots / units_per_item(p.w_out);
        s.mag_p = udiv_magic(s.P);
        s.ok = 1;
        unsigned wm = 0;
        for (int ul = 0; ul < kDomCap; ++ul) wm |= (ul % s.P == s.rank ? 1u : 0u) << ul;
        s.wmask = wm;
    }
    if (threadIdx.x < PK_MAX_DURATIONS) s.dur[threadIdx.x] = threadIdx.x < p.n_dur ? p.durations[threadIdx.x] : 0;
    __syncthreads();
    Utt u{};
    u.pend = -1;
    if (threadIdx.x < s.n) {
        const int ul = threadIdx.x, b = p.dom_list[s.dom * kDomCap + ul];
        const int slot = p.slot[b];
        const int *ctrl = p.slot_ctrl + (size_t)slot * PK_CTRL_N;
        const bool init = ctrl[PK_CTRL_INIT] != 0 && !(p.reset && p.reset[b]);
        u.T = p.T[b];
        u.cur = init ? 0 : 1;   // (a fresh utterance's first step is pending)
        u.sym = init ? ctrl[PK_CTRL_SYM] : 0;
        if (p.kind == PK_KIND_EOU && u.T > 0) u.sym = 0;   // reset per frame (src/parakeet_eou.cpp:269)
        const int carry = init ? ctrl[PK_CTRL_CARRY] : 0;
        u.pend = init ? -1 : p.blank;
        u.flags = init ? 0 : kFlagZeroHC;
        if (p.kind == PK_KIND_TDT) u.t = carry > 0 ? min(carry, u.T) : 0;
        s.b[ul] = b;
        s.erow[ul] = (unsigned)((size_t)p.encp_row[b] * J * 4);
        s.bbias[ul] = p.blank_bias ? p.blank_bias[b] : 0.0f;
        s.tbase[ul] = p.tokens_base ? p.tokens_base[b] : 0;
        s.nseg[ul] = 0;
        s.last[ul] = init ? ctrl[PK_CTRL_LAST] : -1;
        s.segst[ul] = init ? ctrl[PK_CTRL_SEGSTART] : 0;
        s.mark[ul] = init ? 0 : 1;
    }
    __syncthreads();
    // copy c_0, R_0 and pp of this workgroup's utterances from their slots into the
    // exchange buffers (kCopyB loads in flight per thread, then the stores), and empty
    // the words the loop waits for: the other half of pp, this workgroup's tiles of h
    for (int ul = s.rank; ul < s.n; ul += s.P) {
        const int b = s.b[ul], slot = p.slot[b];
        const bool fresh = s.mark[ul] != 0;
        const float *src_c = p.slot_c + (size_t)slot * L * H, *src_r = p.slot_r + (size_t)slot * L * 4 * H,
                    *src_p = p.slot_pp + (size_t)slot * J;
        const int nq = fresh ? 0 : (H + 4 * H + J) / 4;
        for (int q0 = 0; q0 < nq; q0 += kCopyB * kBlock) {
            float4 v[kCopyB];
#pragma unroll
            for (int j = 0; j < kCopyB; ++j) {
                const int i = 4 * min(q0 + (int)threadIdx.x + j * kBlock, nq - 1);
                v[j] = *reinterpret_cast<const float4 *>(i < H ? src_c + i : i < 5 * H ? src_r + (i - H) : src_p + (i - 5 * H));
            }
#pragma unroll
            for (int j = 0; j < kCopyB; ++j) {
                const int q = q0 + threadIdx.x + j * kBlock, i = 4 * q;
                if (q >= nq) continue;
                if (i < H) st4_coh(B.cx, (unsigned)((cx_off(p, 0, b) + i) * 4), v[j]);
                else if (i < 5 * H) st4_coh(B.rx, (unsigned)((rx_off(p, 0, b) + (i - H)) * 4), v[j]);
                else st4_coh(B.ppx, (ppx_at(p, s.dom, 0, (i - 5 * H) / kTile, ul) + (i - 5 * H) % kTile) * 4u,
                             make_float4(filled(v[j].x), filled(v[j].y), filled(v[j].z), filled(v[j].w)));
            }
        }
        for (int i = 4 * threadIdx.x; i < J; i += 4 * kBlock)
            st4_coh(B.ppx, (ppx_at(p, s.dom, 1, i / kTile, ul) + i % kTile) * 4u, empty4());
    }
    empty_h(p, s, B, 0, s.n);
    empty_h(p, s, B, 1, s.n);
    bias_table(p, s.rank, s.P, S.bias);
    // LDS state of layers >= 1: R and c of this workgroup's unit tiles for every utterance of the domain
    if (L > 1) {
        const int n_own = owned(p.w_hh[1].tiles, s.rank, s.P);
        const int n_st = (L - 1) * s.n * n_own * kStFloats;
        for (int i = threadIdx.x; i < n_st; i += kBlock) {
            const int e = i % kStFloats, k = (i / kStFloats) % n_own, ul = (i / kStFloats / n_own) % s.n;
            const int l = 1 + i / (kStFloats * n_own * s.n);
            const int slot = p.slot[s.b[ul]], t = s.rank + k * s.P;
            st_at(p, S, l, ul, k)[e] = e < kTile ? p.slot_r[((size_t)slot * L + l) * 4 * H + t * kTile + e]
                                                 : p.slot_c[((size_t)slot * L + l) * H + t * 4 + (e - kTile)];
        }
    }
    if (wcache) {      // this workgroup's weight tiles, read from LDS for the whole launch
        for (int l = 1; l < L; ++l) cache_matrix(p.w_ih[l], s.rank, s.P, wcache);
        for (int l = 0; l < L; ++l) cache_matrix(p.w_hh[l], s.rank, s.P, wcache);
        cache_matrix(p.w_pred, s.rank, s.P, wcache);
        cache_matrix(p.w_out, s.rank, s.P, wcache);
    }
    build_lists(p, s, u);
    bool ok = dom_sync(p, s, epoch);

    unsigned iter = 0;
    int half = 0, n_prev = 0;   // half of hx of the next LSTM step; list length of the previous one
    unsigned long long tlast = __builtin_amdgcn_s_memrealtime();
    while (ok) {
        const int nl = __builtin_amdgcn_readfirstlane(s.cnt.x), nj = __builtin_amdgcn_readfirstlane(s.cnt.y),
                  ncol = __builtin_amdgcn_readfirstlane(s.cnt.z), lgn = __builtin_amdgcn_readfirstlane(s.cnt.w);
        if (nl < 0) {
            ok = false;
            break;
        }
        if (nl == 0 && nj == 0) break;
        if ((int)iter >= p.max_iter) {
            if (threadIdx.x == 0)
                __hip_atomic_store(p.status, PK_ERR_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ok = false;
            break;
        }
        ++iter;
#ifdef PK_TIMELINE
        if (p.prof) {
            if (threadIdx.x == 0) {
                tl_ctl()[0] = (blockIdx.x == 0 && iter >= 40 && iter < 40 + 256) ? 1 : 0;
                *tl_t0() = __builtin_amdgcn_s_memrealtime();
            }
            lds_sync();
        }
#endif
        float4 epre[kStageMax];
        if (nj > 0) encp_prefetch(p, s, B, ncol, epre);
        if (nl > 0) {
            lstm_and_pred<WC>(p, s, B, S, half, n_prev, nl, lgn, tlast);
            half ^= 1;
            n_prev = nl;
            if (u.pend >= 0) {   // the step is taken
                u.pend = -1;
                u.flags &= ~kFlagZeroHC;
                u.stp = 1;
            }
        }
        if (nj > 0) {
            joint_phase<WC>(p, s, B, S, iter, ncol, epre, tlast);
            gather_keys(p, s, B, iter, ncol);
            TLA(29);
            pmark(p, s, tlast, kPrKeys);
            decide(p, s, u, iter);
        }
        if (nj == 0) lds_sync();   // (behind the keys' barrier otherwise)
        build_lists(p, s, u);
        TLA(31);
        pmark(p, s, tlast, kPrDecide);
    }
    if (p.prof && wg == 0 && threadIdx.x < kPrN) p.prof[threadIdx.x] = s.prof[threadIdx.x];
#ifdef PK_TIMELINE
    if (p.prof && wg == 0 && threadIdx.x < kWaves * kTl) p.prof[kPrN + threadIdx.x] = tl_sum()[threadIdx.x];
    if (p.prof && wg == 0 && threadIdx.x < kTl) p.prof[kPrN + kWaves * kTl + threadIdx.x] = tl_ctl()[2 + threadIdx.x];
#endif
    if (threadIdx.x < s.n) {
        s.cur[threadIdx.x] = u.cur;
        s.mark[threadIdx.x] = u.stp;
    }
    __builtin_amdgcn_s_waitcnt(0);   // this workgroup's state stores have landed
    __syncthreads();
    if (!ok || !s.ok) return;

    if (L > 1) {       // layers >= 1: R and c of this workgroup's unit tiles, from its LDS state
        const int n_own = owned(p.w_hh[1].tiles, s.rank, s.P);
        const int n_st = (L - 1) * s.n * n_own * kStFloats;
        for (int i = threadIdx.x; i < n_st; i += kBlock) {
            const int e = i % kStFloats, k = (i / kStFloats) % n_own, ul = (i / kStFloats / n_own) % s.n;
            const int l = 1 + i / (kStFloats * n_own * s.n);
            const int slot = p.slot[s.b[ul]], t = s.rank + k * s.P;
            const float v = st_at(p, S, l, ul, k)[e];
            if (e < kTile) p.slot_r[((size_t)slot * L + l) * 4 * H + t * kTile + e] = v;
            else p.slot_c[((size_t)slot * L + l) * H + t * 4 + (e - kTile)] = v;
        }
    }
    // h of every layer, c_0, R_0 and pp of this workgroup's tiles, for the utterances that took a
    // step (the others' slots hold them already)
    {
        const __amdgpu_buffer_rsrc_t bx = rsrc(p.hs, p.xchg_bytes);
        const int per = L + 1 + 4, n1 = s.n * s.own_lstm * per, n2 = s.n * s.own_pred * 4;
        for (int i = threadIdx.x; i < n1 + n2; i += kBlock) {
            float *dst;
            long long x;   // float offset from p.hs
            int ul;
            if (i < n1) {
                const int e = i % per, k = (i / per) % s.own_lstm, j = 4 * (s.rank + k * s.P);
                ul = i / per / s.own_lstm;
                const int b = s.b[ul], slot = p.slot[b], cur = s.cur[ul];
                if (e < L) {
                    dst = p.slot_h + ((size_t)slot * L + e) * H + j;
                    x = (long long)hs_off(p, e, b) + j;
                } else if (e == L) {
                    dst = p.slot_c + (size_t)slot * L * H + j;
                    x = (p.cx - p.hs) + (long long)cx_off(p, cur, b) + j;
                } else {
                    const int row = 4 * j + 4 * (e - L - 1);
                    dst = p.slot_r + (size_t)slot * L * 4 * H + row;
                    x = (p.rx - p.hs) + (long long)rx_off(p, cur, b) + row;
                }
            } else {
                const int q = i - n1, g = q & 3, k = (q >> 2) % s.own_pred, t = s.rank + k * s.P;
                ul = (q >> 2) / s.own_pred;
                dst = p.slot_pp + (size_t)p.slot[s.b[ul]] * J + t * kTile + g * 4;
                x = (p.ppx - p.hs) + (long long)ppx_at(p, s.dom, s.cur[ul], t, ul) + g * 4;
            }
            if (s.mark[ul]) *reinterpret_cast<float4 *>(dst) = ld4_coh(bx, (unsigned)(x * 4));
        }
    }
    if (threadIdx.x < s.n && ((s.wmask >> threadIdx.x) & 1u) != 0u) {   // outputs and control words
        const int ul = threadIdx.x, b = s.b[ul];
        int *ctrl = p.slot_ctrl + (size_t)p.slot[b] * PK_CTRL_N;
#pragma unroll
        for (int k = 0; k < PK_CTRL_N; ++k) {
            const int v = k == PK_CTRL_INIT ? 1
                        : k == PK_CTRL_SYM ? u.sym
                        : k == PK_CTRL_CARRY ? ((p.kind == PK_KIND_TDT) ? max(0, u.t - u.T) : 0)
                        : k == PK_CTRL_LAST ? s.last[ul]
                        : k == PK_CTRL_SEGSTART ? s.segst[ul] : 0;
            ctrl[k] = v;
            if (p.ctrl_out) p.ctrl_out[(size_t)b * PK_CTRL_N + k] = v;
        }
        p.n_tokens[b] = u.ntok;
        p.steps[b] = u.steps;
        if (p.n_segs) p.n_segs[b] = s.nseg[ul];
        if (u.flags & (kFlagTokOverflow | kFlagSegOverflow))
            __hip_atomic_store(p.status + 2, PK_ERR_OVERFLOW, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (u.flags & kFlagTraceOverflow)
            __hip_atomic_store(p.status + 3, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (threadIdx.x == 0) atomicMax(p.status + 1, (int)iter);
}

}  // namespace pkdev
