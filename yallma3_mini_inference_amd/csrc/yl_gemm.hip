// yl_gemm.hip -- quantized matmul over several tokens (prompts, chat turns,
// and yl_matmul with a batch) on int8 MFMA, bit-identical to
// matmul_q8_slices (weight_type.rs:122-226).
//
// The reference sums, for each output (token t, row c), the block terms
//     term_b = ((float)isum_b * w_scale[c][b]) * x_scale[t][b]
// in ascending block order into an f32 accumulator, where isum_b is the
// exact int32 dot of one 32-element block.  v_mfma_i32_32x32x32_i8 and
// v_mfma_i32_16x16x32_i8 have K = 32: one instruction yields exactly the
// tile's block dots of one block, and each lane then folds its 16 (or 4)
// dots into as many f32 accumulators in block order with the reference's
// two roundings.  The f32 work per output and block is the bound, not the
// MFMA: with f16 scales (Q8_0, Q4_0) one fused multiply-add on a biased dot
// (the convert folded away; see `bias` in k_gemm), one product and one sum;
// with f32 scales a convert, two products and one sum.
//
// Tile: a workgroup of GM x GN wavefronts; each wavefront owns one MFMA tile
// of T tokens x T weight rows.  MFMA lane layout (gfx950), g = l / T:
// operand lane l holds row l%T (token for A, weight row for B) and, of the
// block's 32 bytes, 8*g .. +7 (T = 16) or 16*g .. +15 (T = 32); result
// register i of lane l is (token 4*g + i (T = 16) or (i%4) + 8*(i/4) + 4*g
// (T = 32), weight row l%T).  A lane's weight row is fixed, so one converted
// weight scale serves all its outputs of a tile, and the activation scales
// of its tokens come by 16-byte LDS reads.
//
// Stages of KB blocks (activations, weights, both scale vectors) stream into
// LDS by LDS DMA, NST stages deep, so no register holds data in flight.
// Rows are stored as 16-byte units in rotated order (gm_unit): the DMA reads
// a row's KB*32 contiguous bytes with consecutive lanes, and the operand
// reads of 16 rows fall on distinct LDS banks (unrotated, a 1000-token gate
// projection of the 1B shape took 150 us instead of 73).  Loads go through
// buffer descriptors that end with the arrays: the last stage may reach past
// a row (into the next one; unused) or past the matrix (reads as 0).
// Q4_0 weights keep the reference nibble order and are unpacked in registers
// to int8 in k order (values 0..15, no offset).
// Q8 with f32 scales (lm.rs, safetensors): per block (kQ8S), or per group
// of 2 or 4 blocks (kQ8S64, kQ8S128), whose block MFMAs accumulate into one
// int32 tile -- the group's exact dot -- before its one f32 term; the
// activations are quantized in the same groups.
#include <hip/hip_runtime.h>

#include "yl_blocks.h"
#include "yl_device.h"
#include "yl_internal.h"

namespace yl {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// 32-blocks per scale group
template <int WF>
constexpr int gm_bpg() { return WF == kQ8S64 ? 2 : (WF == kQ8S128 ? 4 : 1); }

// One tile configuration: T x T MFMA tiles, one per wavefront, GM x GN
// wavefronts, KB blocks per stage, NST stages, registers for OCC wavefronts
// per SIMD; DEEP: a stage's operands read ahead (see k_gemm).
template <int T_, int GM_, int GN_, int KB_, int NST_, int OCC_, bool DEEP_ = false>
struct GmCfg {
    static constexpr bool DEEP = DEEP_;
    static constexpr int T = T_, GM = GM_, GN = GN_, KB = KB_, NST = NST_, OCC = OCC_;
    static constexpr int NW = GM * GN, TM = T * GM, TN = T * GN;
};

// What one stage holds in LDS, and the DMA instructions that fill it.
template <int WF, class C>
struct GmStage {
    static constexpr int G = gm_bpg<WF>();
    static constexpr bool kF32 = WF == kQ8S || WF == kQ8S64 || WF == kQ8S128;
    static constexpr int UA = 2 * C::KB;                       // 16-byte units per activation row
    static constexpr int UB = WF == kQ4 ? C::KB : 2 * C::KB;   // and per weight row
    static constexpr int A = C::TM * UA * 16, B = C::TN * UB * 16;
    // activation scales [token / 16][group][16] f32
    static constexpr int XW = C::KB / G;
    static constexpr int XS = (C::TM * XW * 4 + 255) / 256 * 256;
    // weight scales: f16 as WW dwords per row from the aligned dword that
    // holds the stage's first scale (one more than the blocks need: an odd
    // nb puts every other row half a dword off), f32 as [group][row]
    static constexpr int WW = kF32 ? C::KB / G : C::KB / 2 + 1;
    static constexpr int WS = (C::TN * WW * 4 + 255) / 256 * 256;
    static constexpr int bytes = A + B + XS + WS;
    // 16-byte-lane DMA instructions (1 KiB each), then 4-byte-lane ones
    // (256 B), dealt to the wavefronts in turn; every wavefront issues the
    // same number (the last ones repeat, with identical bytes)
    static constexpr int nA = A / 1024, nB = B / 1024, nX = XS / 256, nW = WS / 256;
    static constexpr int k16 = (nA + nB + C::NW - 1) / C::NW, k4 = (nX + nW + C::NW - 1) / C::NW;
    static constexpr int dma = k16 + k4;
    static_assert(A % 1024 == 0 && B % 1024 == 0 && C::KB % G == 0 && (C::KB == 2 || C::KB == 4), "stage shapes");
    static_assert((C::NST - 2) * dma < 64, "stage waits count DMA instructions in 6 bits");
};

// Unit p of row `row` in a stage of U units per row: rotated by the row so
// that the same unit of 16 consecutive rows covers all 64 banks once.
template <int U>
__device__ __forceinline__ int gm_unit(int row, int p) { return row * U + (p ^ ((row / (16 / U)) & (U - 1))); }

// this wavefront's DMA of the current stage has landed when at most `later`
// younger stages (D instructions each) are still in flight
template <int D, int NST>
__device__ __forceinline__ void gm_wait(int later) {
    static_assert(NST >= 2 && NST <= 4, "waits below");
    if (later <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (NST == 3 || later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NST >= 4 ? 2 * D : 0) : "memory");
}

// 4 Q4_0 bytes (8 nibbles, byte j = elements 2j | 2j+1 << 4) -> 8 int8 in
// element order
__device__ __forceinline__ uint2 q4_unpack8(uint32_t p) {
    const uint32_t lo = p & 0x0f0f0f0fu, hi = (p >> 4) & 0x0f0f0f0fu;
    // v_perm_b32(hi, lo, sel): byte k of the result = byte sel_k of {hi:lo}
    // (lo = bytes 0..3, hi = bytes 4..7)
    const uint32_t x = __builtin_amdgcn_perm(hi, lo, 0x05010400u);   // lo0 hi0 lo1 hi1
    const uint32_t y = __builtin_amdgcn_perm(hi, lo, 0x07030602u);   // lo2 hi2 lo3 hi3
    return make_uint2(x, y);
}

// A raw buffer descriptor over `bytes` from `base` (uniform values).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gm_rsrc(const void* base, size_t bytes) {
    const uint64_t p = (uint64_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(bytes < 0xffffff00ull ? bytes : 0xffffff00ull));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), (short)0, (int)n, 0x00020000);
}

#if defined(__HIP_DEVICE_COMPILE__)
// One MFMA tile size T (16 or 32): operand and result registers, and the
// token of result register i (of lane group g = lane / T) within the tile.
template <int T>
struct GmMfma;
template <>
struct GmMfma<16> {
    using op = long;    // 8 bytes of the block per lane
    using res = v4i;
    static __device__ __forceinline__ res mul(op a, op b, res c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0); }
};
template <>
struct GmMfma<32> {
    using op = v4i;     // 16 bytes
    using res = v16i;
    static __device__ __forceinline__ res mul(op a, op b, res c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
};
#endif

template <int WF, int EPI, class C>
__global__ __launch_bounds__(64 * C::NW) __attribute__((amdgpu_waves_per_eu(C::OCC, C::OCC))) void k_gemm(GemvArgs a,
                                                                                                     int M) {
    // (device pass only: the host pass has no gfx950 MFMA builtins and
    // needs just the launch stub)
#if defined(__HIP_DEVICE_COMPILE__)
    using S = GmStage<WF, C>;
    constexpr int T = C::T, KB = C::KB, G = S::G, NW = C::NW;
    constexpr int R = T * T / 64;   // result registers per tile
    constexpr bool kDeep = C::DEEP;
    using MF = GmMfma<T>;
    extern __shared__ __align__(16) unsigned char gsm[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rt = lane % T, lg = lane / T;
    const int wm = wave % C::GM, wn = wave / C::GM;
    const int c0 = blockIdx.x * C::TN, t0 = blockIdx.y * C::TM;
    const int tw = t0 + T * wm, cw = c0 + T * wn;   // this wavefront's first token and row
    const int nst = (a.nb + KB - 1) / KB;

    // ---- DMA plan: each instruction's lane offset, once ----
    const int ng = a.nb / G;   // scales per row
    const __amdgpu_buffer_rsrc_t rA = gm_rsrc(a.xq + (size_t)t0 * a.n, (size_t)(M - t0) * a.n);
    const __amdgpu_buffer_rsrc_t rX = gm_rsrc(a.xs + (size_t)t0 * ng, (size_t)(M - t0) * ng * 4);
    const int rowb = WF == kQ4 ? a.n / 2 : a.n;   // weight bytes per row
    const __amdgpu_buffer_rsrc_t rB = gm_rsrc(a.qs + (size_t)c0 * rowb, (size_t)(a.o - c0) * rowb);
    // (the f16 scale array is padded past its last dword)
    const __amdgpu_buffer_rsrc_t rW = S::kF32 ? gm_rsrc(a.sf + (size_t)c0 * ng, (size_t)(a.o - c0) * ng * 4)
                                              : gm_rsrc(a.d + (size_t)c0 * a.nb, ((size_t)(a.o - c0) * a.nb * 2 + 3) & ~(size_t)3);
    // instruction k of this wavefront is number wave + k * NW of its list;
    // its kind is known at compile time except where a round spans both
    auto first_kind = [&](int k, int n0, int n) {   // 1: of the first array, 0: of the second, -1: by wavefront
        return k * NW + NW <= n0 ? 1 : (k * NW >= n0 || n0 == n ? 0 : -1);
    };
    auto offA_of = [&](int j) {
        const int u = 64 * j + lane, row = u / S::UA;
        const int p = gm_unit<S::UA>(row, u % S::UA) - row * S::UA;   // (the rotation is its own inverse)
        return (min(t0 + row, M - 1) - t0) * a.n + 16 * p;
    };
    auto offB_of = [&](int j) {
        const int u = 64 * (j - S::nA) + lane, row = u / S::UB;
        const int p = gm_unit<S::UB>(row, u % S::UB) - row * S::UB;
        return (min(c0 + row, a.o - 1) - c0) * rowb + 16 * p;
    };
    auto offX_of = [&](int j) {
        const int u = min(64 * j + lane, C::TM * S::XW - 1);
        const int tok = u / (T * S::XW) * T + u % T, xi = u / T % S::XW;
        return ((min(t0 + tok, M - 1) - t0) * ng + xi) * 4;
    };
    auto offW_of = [&](int j) {
        const int u = min(64 * (j - S::nX) + lane, C::TN * S::WW - 1);
        if constexpr (S::kF32) return ((min(c0 + u % C::TN, a.o - 1) - c0) * ng + u / C::TN) * 4;
        else return ((((min(c0 + u / S::WW, a.o - 1) - c0) * a.nb) >> 1) + u % S::WW) * 4;
    };
    int v16[S::k16], v4[S::k4];
#pragma unroll
    for (int k = 0; k < S::k16; k++) {
        const int j = min(wave + k * NW, S::nA + S::nB - 1), kind = first_kind(k, S::nA, S::nA + S::nB);
        v16[k] = kind == 1 || (kind < 0 && j < S::nA) ? offA_of(j) : offB_of(j);
    }
#pragma unroll
    for (int k = 0; k < S::k4; k++) {
        const int j = min(wave + k * NW, S::nX + S::nW - 1), kind = first_kind(k, S::nX, S::nX + S::nW);
        v4[k] = kind == 1 || (kind < 0 && j < S::nX) ? offX_of(j) : offW_of(j);
    }
    // DMA of stage s into LDS buffer b
    auto issue = [&](int s, int b) {
        auto* buf = (__attribute__((address_space(3))) unsigned char*)(gsm) + b * S::bytes;
        const int oA = s * (KB * 32), oB = WF == kQ4 ? s * (KB * 16) : s * (KB * 32);
        const int oX = s * (S::XW * 4), oW = S::kF32 ? s * (S::XW * 4) : s * (KB * 2);
#pragma unroll
        for (int k = 0; k < S::k16; k++) {
            const int j = min(wave + k * NW, S::nA + S::nB - 1), kind = first_kind(k, S::nA, S::nA + S::nB);
            if (kind == 1 || (kind < 0 && j < S::nA)) __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, buf + j * 1024, 16, v16[k], oA, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rB, buf + j * 1024, 16, v16[k], oB, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < S::k4; k++) {
            const int j = min(wave + k * NW, S::nX + S::nW - 1), kind = first_kind(k, S::nX, S::nX + S::nW);
            auto* dst = buf + S::A + S::B + j * 256;
            if (kind == 1 || (kind < 0 && j < S::nX)) __builtin_amdgcn_raw_ptr_buffer_load_lds(rX, dst, 4, v4[k], oX, 0, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rW, dst, 4, v4[k], oW, 0, 0);
        }
    };

    // accumulators: acc[i] = (token tw + 4lg + tok_of(i), row cw + rt)
    float acc[R];
    // token offset of register i in a tile, beyond the lane group's 4 * lg
    auto tok_of = [](int i) { return T == 16 ? i : (i & 3) + 8 * (i >> 2); };
    int pos = 0;
    if constexpr (EPI == kEpiQkvRope) pos = a.state->pos;
    // QKV rows: the lane's stored column within q or k (RoPE pair order) and
    // its pair index
    [[maybe_unused]] int kcol = 0, qkcol = 0, qpair = 0;
    if constexpr (EPI == kEpiQkvRope) {
        const int c = cw + rt, att = a.att_dim;
        const int scol = c < att ? c : c - att;   // stored row within q or k
        kcol = qk_column(c - att, a.head_size, a.hf_rows);
        qkcol = qk_column(scol, a.head_size, a.hf_rows);
        qpair = (scol % a.head_size) >> 1;
    }
    // (lane coordinates opaque per use: the initial values' and the epilogue's
    // addresses are then computed where they are used, not kept across the K
    // loop)
    auto opaque = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    auto init_acc = [&]() {
        const int tl = opaque(tw + 4 * lg), c = opaque(cw + rt);
#pragma unroll
        for (int i = 0; i < R; i++) {
            float v = 0.0f;
            const int t = tl + tok_of(i);
            if constexpr (EPI == kEpiStore) {
                if (t < M && c < a.o && c < a.accumulate_cols) v = a.out[(size_t)t * a.o + c];
            } else if constexpr (EPI == kEpiQkvRope) {
                // K/V rows accumulate into the cache (forward.rs:166-169);
                // q rows start at 0.  A tile's rows are all q, all k or all
                // v (att_dim and kv_dim are multiples of 32), so the branches
                // are uniform; token t0 stands in for the rows past M in the
                // (then unused) loads.
                const int att = a.att_dim, kv = a.kv_dim;
                if (cw >= att && cw < a.o) {
                    const int tc = t < M ? t : t0;
                    const float u = cw < att + kv ? a.k_cache[(size_t)kcol * a.kv_ld + pos + tc]
                                                  : a.v_cache[(size_t)(pos + tc) * kv + (c - att - kv)];
                    if (t < M) v = u;
                }
            }
            acc[i] = v;
        }
    };

    // f16 block scales (Q8_0, Q4_0): every block dot starts from the int32
    // bits of the float 3*2^22 instead of 0, so the MFMA's result reads as the
    // float f = 3*2^22 + isum, exactly (|isum| <= 32*128*128 < 2^22).  Then
    //     fma(f, ws, -3*2^22*ws) = round(isum * ws),
    // one rounding of the exact product (3*2^22*ws is exact for an f16 ws):
    // the convert drops out of the per-output work (3 VALU operations
    // instead of 4).  The value equals (float)isum * ws, except that an exact
    // cancellation gives +0 where isum = 0 or ws = 0 gives the product's
    // signed zero.  A zero term's sign changes the sum only while the
    // accumulator is -0, and an accumulator that does not start at -0 never
    // becomes -0 (+0 + -0 = +0, and x + -x = +0).  A non-finite scale makes
    // f * ws - 3*2^22*ws a NaN (f > 0), which the accumulator keeps.  So the
    // fused pass is exact unless a -0 initial value or a non-finite scale is
    // present; a lane that sees the former or ends with a NaN flags it, and
    // the workgroup then reloads its initial values (only the epilogue writes
    // them) and runs the reference's form.  The bias tuple is opaque to the
    // compiler, so it stays in registers rather than being rematerialized
    // before each MFMA.
    constexpr bool kBias = WF == kQ8 || WF == kQ4;
    constexpr float kBiasF = 12582912.0f;   // 3 * 2^22, bits 0x4B400000
    __shared__ int redo;
    typename MF::res bias = {};
    if constexpr (kBias) {
#pragma unroll
        for (int i = 0; i < R; i++) bias[i] = 0x4B400000;
        asm volatile("" : "+v"(bias));
        if (threadIdx.x == 0) redo = 0;   // ordered before any flag by the first stage's barrier
    }

    int neg_zero = 0;   // this lane saw a -0 initial value

    // lane offsets of the operand reads within a stage
    const int offA = T * wm * S::UA * 16, offB = S::A + T * wn * S::UB * 16;
    const int wsh = (((int)rt & a.nb & 1)) << 4;   // an odd nb: odd rows' scales start in the high half

    // the K loop: FUSED.value selects the biased form above
    auto run = [&](auto FUSED) {
    constexpr bool kFused = decltype(FUSED)::value;
    typename MF::res gd;   // group dot (or the block's, G = 1)

    // one block's operands: both int8 rows, the activation scales of the
    // lane's tokens (with a group's last block) and the raw weight scale
    struct Ops {
        typename MF::op av, bv;
        vf4 xv[R / 4];
        uint32_t ws;
    };
    // byte offset of this lane's share of block blk in row rt of a tile
    auto lane_off = [&](int blk) {
        return T == 16 ? gm_unit<S::UA>(rt, 2 * blk + (lg >> 1)) * 16 + 8 * (lg & 1) : gm_unit<S::UA>(rt, 2 * blk + lg) * 16;
    };
    auto load_ops = [&](const unsigned char* buf, int blk, uint32_t w, Ops& o) {
        o.av = *reinterpret_cast<const typename MF::op*>(buf + offA + lane_off(blk));
        const unsigned char* bt = buf + offB;
        if constexpr (WF != kQ4) {
            o.bv = *reinterpret_cast<const typename MF::op*>(bt + lane_off(blk));
        } else if constexpr (T == 16) {   // (the nibbles; unpacked by block())
            o.bv = *reinterpret_cast<const uint32_t*>(bt + gm_unit<S::UB>(rt, blk) * 16 + 4 * lg);
        } else {
            const uint2 u = *reinterpret_cast<const uint2*>(bt + gm_unit<S::UB>(rt, blk) * 16 + 8 * lg);
            o.bv = v4i{(int)u.x, (int)u.y, 0, 0};
        }
        if (G == 1 || blk % G == G - 1) {
            const float* xl = reinterpret_cast<const float*>(buf + S::A + S::B) + 4 * lg;
#pragma unroll
            for (int i = 0; i < R / 4; i++)
                o.xv[i] = *reinterpret_cast<const vf4*>(xl + (wm * S::XW + blk / G) * T + 8 * i);
            if constexpr (S::kF32)
                o.ws = reinterpret_cast<const uint32_t*>(buf + S::A + S::B + S::XS)[blk / G * C::TN + T * wn + rt];
            else o.ws = w;
        }
    };
    // Q4_0: the nibbles read, to int8
    auto unpack = [&](Ops& o) {
        if constexpr (WF == kQ4) {
            if constexpr (T == 16) {
                o.bv = __builtin_bit_cast(long, q4_unpack8((uint32_t)o.bv));
            } else {
                const uint2 x = q4_unpack8((uint32_t)o.bv.x), y = q4_unpack8((uint32_t)o.bv.y);
                o.bv = v4i{(int)x.x, (int)x.y, (int)y.x, (int)y.y};
            }
        }
    };
    // block blk's weight scale from its raw word, and the fused form's constant
    auto scale = [&](uint32_t raw, int blk, float& ws, float& cb) {
        if constexpr (S::kF32) ws = __uint_as_float(raw);
        else ws = f16_to_f32((uint16_t)(raw >> (16 * (blk & 1))));
        if constexpr (kFused) {
            // opaque: otherwise the compiler folds the f16 convert into each
            // FMA (v_fma_mix_f32)
            asm volatile("" : "+v"(ws));
            cb = fmul(-kBiasF, ws);
        }
    };
    // the tile's terms onto its sums.  The three (four) steps run over the
    // outputs one step at a time, so that no instruction waits on the one
    // before it.
    auto fold = [&](const typename MF::res& d, float ws, float cb, const vf4 (&xv)[R / 4]) {
        float term[R];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < R; i++) {
            if constexpr (kFused) term[i] = __builtin_fmaf(__int_as_float(d[i]), ws, cb);
            else term[i] = fmul((float)d[i], ws);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < R; i++) term[i] = fmul(term[i], xv[i / 4][i % 4]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < R; i++) acc[i] = fadd(acc[i], term[i]);
        __builtin_amdgcn_sched_barrier(0);
    };
    // the block's product and terms; `next` (the next block's reads) is
    // issued while the MFMA runs
    auto block = [&](int blk, Ops& o, auto next) {
        float wsc, cb;
        unpack(o);
        scale(o.ws, blk, wsc, cb);
        const typename MF::res zero = {};
        // (the first block of a group starts from zero, the others' dots join
        // it; the term follows the group's last)
        gd = MF::mul(o.av, o.bv, G > 1 && blk % G ? gd : (kFused ? bias : zero));
        __builtin_amdgcn_sched_barrier(0);
        next();
        if (G == 1 || blk % G == G - 1) fold(gd, wsc, cb, o.xv);
    };

#pragma unroll
    for (int s = 0; s < C::NST - 1; s++)
        if (s < nst) issue(s, s);
    if constexpr (kFused) {
        // (the initial values are older loads than the stages')
        int flag = 0;
#pragma unroll
        for (int i = 0; i < R; i++) flag |= __float_as_uint(acc[i]) == 0x80000000u;
        neg_zero = flag;
        asm volatile("" : "+v"(neg_zero));   // decided here: the initial values do not outlive the loop
    }
    int cur = 0;   // LDS buffer of stage s
    // stage s is in LDS, and the stage NST - 1 later on its way
    auto arrive = [&](int s) -> const unsigned char* {
        gm_wait<S::dma, C::NST>(min(C::NST - 2, nst - 1 - s));
        lds_barrier();   // every wavefront's DMA of stage s landed; stage s-1's buffer is free
        const int nxt = cur == 0 ? C::NST - 1 : cur - 1;   // (s + NST - 1) % NST
        if (s + C::NST - 1 < nst) issue(s + C::NST - 1, nxt);
        const unsigned char* buf = gsm + cur * S::bytes;
        cur = cur == C::NST - 1 ? 0 : cur + 1;
        return buf;
    };
    // the stage's f16 weight scales of this lane's row, two to a word
    uint32_t wraw[KB / 2];
    auto load_scales = [&](const unsigned char* buf) {
        if constexpr (!S::kF32) {
            const uint32_t* p = reinterpret_cast<const uint32_t*>(buf + S::A + S::B + S::XS) + (T * wn + rt) * S::WW;
            uint32_t w[S::WW];
#pragma unroll
            for (int i = 0; i < S::WW; i++) w[i] = p[i];
#pragma unroll
            for (int i = 0; i < KB / 2; i++) wraw[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], wsh);
        }
    };
    const int full = a.nb / KB;
    if constexpr (kDeep) {
        // a 16 x 16 tile's block (12 VALU instructions) is shorter than the
        // latencies around it, so a whole stage's operands are read while the
        // previous stage is folded, and its MFMAs issued back to back ahead
        // of its folds
        Ops q[2][KB];
        auto load_stage = [&](int s, Ops (&o)[KB]) {
            const unsigned char* buf = arrive(s);
            load_scales(buf);
#pragma unroll
            for (int blk = 0; blk < KB; blk++) load_ops(buf, blk, wraw[blk / 2], o[blk]);
        };
        auto step = [&](int s, Ops (&o)[KB], Ops (&nx)[KB]) {
            typename MF::res d[KB / G];
#pragma unroll
            for (int blk = 0; blk < KB; blk++) {
                unpack(o[blk]);
                const typename MF::res zero = {};
                d[blk / G] = MF::mul(o[blk].av, o[blk].bv, blk % G ? d[blk / G] : kFused ? bias : zero);
            }
            if (s + 1 < full) load_stage(s + 1, nx);
#pragma unroll
            for (int blk = G - 1; blk < KB; blk += G) {
                float wsc, cb;
                scale(o[blk].ws, blk, wsc, cb);
                fold(d[blk / G], wsc, cb, o[blk].xv);
            }
        };
        if (full > 0) load_stage(0, q[0]);
        int s = 0;
        for (; s + 1 < full; s += 2) {
            step(s, q[0], q[1]);
            step(s + 1, q[1], q[0]);
        }
        if (s < full) step(s, q[0], q[1]);
    } else
    for (int s = 0; s < full; s++) {
        const unsigned char* buf = arrive(s);
        load_scales(buf);
        // the next block's operands are read while this one is folded
        Ops o[2];
        load_ops(buf, 0, wraw[0], o[0]);
#pragma unroll
        for (int blk = 0; blk < KB; blk++) {
            block(blk, o[blk & 1], [&] {
                if (blk + 1 < KB) load_ops(buf, blk + 1, wraw[(blk + 1) / 2], o[(blk + 1) & 1]);
            });
        }
    }
    // the blocks of a last, partial stage
    if (full < nst) {
        const unsigned char* buf = arrive(full);
        load_scales(buf);
#pragma unroll 1
        for (int blk = 0; blk < a.nb - full * KB; blk++) {
            uint32_t w = wraw[0];
            if constexpr (KB > 2) w = blk >= 2 ? wraw[1] : w;
            Ops o;
            load_ops(buf, blk, w, o);
            block(blk, o, [] {});
        }
    }
    };

    // (16 x 16 tiles read the residual ahead of the K loop, off the tail; the
    // 16 registers of a 32 x 32 tile's spilled there, 5 to 12 of them)
    constexpr bool kResidEarly = EPI == kEpiResid && R == 4;
    [[maybe_unused]] float resid[R];
    if constexpr (kResidEarly) {
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int t = min(tw + 4 * lg + tok_of(i), M - 1), c = min(cw + rt, a.o - 1);
            resid[i] = a.x[(size_t)t * a.o + c];
        }
    }
    init_acc();
    if constexpr (kBias) {
        run(std::true_type{});
        bool flag = neg_zero != 0;
#pragma unroll
        for (int i = 0; i < R; i++) flag = flag || acc[i] != acc[i];
        if (flag) redo = 1;
        __syncthreads();   // every flag is in; every wavefront is done with the LDS stages
        if (redo) {
            init_acc();
            wait_vm_all();   // (stage waits count DMA instructions only)
            run(std::false_type{});
        }
    } else {
        run(std::false_type{});
    }

    const int tl = opaque(tw + 4 * lg), c = opaque(cw + rt);
    if constexpr (EPI == kEpiSwiglu) {
        // SwiGLU (forward.rs:220-237) of the 64-row groups [32 gate | 32 up],
        // with expf's constants in registers.  A group's rows are spread over
        // wavefronts: exchange the sums through LDS (the stages are done),
        // then one 32-lane half per (token, group)
        const ExpfK ek = expf_k_regs();
        static_assert(C::TN % 64 == 0, "whole 64-row groups per workgroup");
        constexpr int LD = C::TN + 4;
        float* ex = reinterpret_cast<float*>(gsm);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < R; i++) ex[(tl - t0 + tok_of(i)) * LD + c - c0] = acc[i];
        __syncthreads();
        constexpr int NG = C::TN / 64;
        const int l32 = threadIdx.x & 31;
        for (int it = threadIdx.x >> 5; it < C::TM * NG; it += 2 * NW) {
            const int t = t0 + it / NG, q = it % NG, grp = c0 / 64 + q;
            const bool ok = t < M && c0 + 64 * q < a.o;
            const float g = ex[(it / NG) * LD + 64 * q + l32], u = ex[(it / NG) * LD + 64 * q + 32 + l32];
            const float den = fadd(1.0f, expf_rn(-g, ek));
            const float h = fmul(g / den, u);
            const size_t base = (size_t)t * a.hidden + (size_t)grp * kGroup;
            if (a.h_f32 && ok) a.h_f32[base + l32] = h;
            if (!a.hq) continue;   // f32 h only (quantized afterwards in the model's groups)
            const float am = fmaxf(group_max(fabsf(h), 32), 0.0f);
            const float sc = a.h_fmt == kQ4 ? group_scale<kQ4>(am) : group_scale<kQ8>(am);
            const int8_t qv = (int8_t)(a.h_fmt == kQ4 ? quant_one<kQ4>(h, sc) : quant_one<kQ8>(h, sc));
            if (ok) {
                a.hq[base + l32] = qv;
                if (l32 == 0) a.hs[(size_t)t * (a.hidden / kGroup) + grp] = sc;
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int t = tl + tok_of(i);
            const bool tok_ok = t < M;
            const float v = acc[i];
            if constexpr (EPI == kEpiQkvRope) {
                // rope_gguf (util.rs:653-718) on q and k pairs (2j, 2j+1):
                // the pair partner is the neighbouring lane
                const float other = dpp_mov<0xB1>(v);
                // (uniform branches on the tile, as in the initial values)
                const int att = a.att_dim, kv = a.kv_dim, hd = a.head_size;
                if (cw >= att + kv) {
                    if (tok_ok && cw < a.o) a.v_cache[(size_t)(pos + t) * kv + (c - att - kv)] = v;
                } else {
                    const int tc = tok_ok ? t : t0;
                    const float cs = a.rope_cos[(size_t)(pos + tc) * (hd >> 1) + qpair];
                    const float sn = a.rope_sin[(size_t)(pos + tc) * (hd >> 1) + qpair];
                    const float v0 = (rt & 1) ? other : v, v1 = (rt & 1) ? v : other;
                    const float r = (rt & 1) ? fadd(fmul(v0, sn), fmul(v1, cs)) : fmul(v0, cs) - fmul(v1, sn);
                    if (tok_ok) {
                        if (cw < att) a.q_out[(size_t)t * att + qkcol] = r;
                        else a.k_cache[(size_t)qkcol * a.kv_ld + pos + t] = r;
                    }
                }
            } else if (tok_ok && c < a.o) {
                if constexpr (EPI == kEpiStore) a.out[(size_t)t * a.o + c] = v;
                if constexpr (EPI == kEpiResid) {
                    // residual add (forward.rs:196-204 / 245-253)
                    float* xp = a.x + (size_t)t * a.o + c;
                    *xp = fadd(kResidEarly ? resid[i] : *xp, v);
                }
            }
        }
    }

#endif
}

// ------------------------------------------------------------ dispatch ----

template <int WF, int EPI, class C>
static hipError_t launch_gemm_cfg(const GemvArgs& a, int M, hipStream_t st) {
    // the stages, or the sums SwiGLU exchanges
    constexpr int stages = C::NST * GmStage<WF, C>::bytes, ex = EPI == kEpiSwiglu ? C::TM * (C::TN + 4) * 4 : 0;
    constexpr int smem = stages > ex ? stages : ex;
    static_assert(smem <= 64 * 1024 - 64, "dynamic LDS of a launch without the attribute");
    const dim3 grid((a.o + C::TN - 1) / C::TN, (M + C::TM - 1) / C::TM);
    hipLaunchKernelGGL((k_gemm<WF, EPI, C>), grid, dim3(64 * C::NW), smem, st, a, M);
    return hipGetLastError();
}

// Tile configurations, by the number of 16 x 16 output tiles (what one
// wavefront can own at least): the K loop is one serial chain per output, so
// a short batch is bound by the chain's latency and by how many CUs stream
// weights, and wants one tile per workgroup; more tiles than wavefront slots
// want larger ones, which read each weight and activation byte fewer times.
// Measured (Q8_0, us, rotating weight copies; o x n, M tokens; "before" is
// 64- or 128-token x 128-row tiles of 32 x 32 x 32 MFMAs):
//                         One    Pair   Quad   Wide  Wide2  before
//   2048 x 8192, M 41     24.9   30.2   34.2   54.2          115
//   3072 x 2048, M 41      8.9    9.8   10.9   16.7           38
//   16384 x 2048, M 24    14.0   11.9   14.5   17.4
//   2048 x 2048, M 200    12.7   11.1   11.6   17.1
//   2048 x 2048, M 400    23.5   15.8   14.6   17.3
//   2048 x 8192, M 512                  48.9   56.6   72.1   103
//   16384 x 2048, M 64    28.1   17.7   15.2   17.8           37
//   16384 x 2048, M 100   44.6   28.6   26.7   20.6
//   8192 x 8192, M 300                 134.8   92.6  112.5   127
//   3072 x 2048, M 2000                 82.9   53.9   55.0    66.8
//   8192 x 2048, M 1000                110.8   70.0   68.6    71.9
//   16384 x 2048, M 2000               450.9  293.2  286.2   290.1
// Q4_0 and the f32-scaled formats take the same bounds: over 12 shapes of 16 to
// 2000 tokens Q4_0 is nowhere slower than before, nor are whole prompts of 4 to
// 1900 tokens with f32 scales (4 layers of the 1B shape, 100 tokens, group size
// 32 / 64 / 128: 1368 / 1215 / 1245 -> 520 / 495 / 483 us).
// The large grids stay far from the f32 floor (97 us for the last row at 2
// cycles per VALU instruction): with parts of the loop taken out in a timing
// copy (8192 x 8192, M 1000, Wide), the f32 folds alone take 126 us, the
// MFMAs add 29, the operand reads 26, barriers 16 and the LDS DMA 45 (a DMA
// instruction occupies the L1 for 64 lane accesses whatever its width).
using GmOne = GmCfg<16, 1, 1, 4, 3, 2, true>;    // 16 tokens x 16 rows, 1 wavefront
using GmPair = GmCfg<16, 2, 2, 4, 4, 4>;         // 32 x 32, 4 wavefronts
using GmQuad = GmCfg<16, 4, 2, 4, 3, 4>;         // 64 x 32, 8 wavefronts
using GmWide = GmCfg<32, 2, 2, 4, 2, 4>;         // 64 x 64, 4 wavefronts of one 32 x 32 tile
using GmWide2 = GmCfg<32, 2, 4, 4, 2, 4>;        // 64 x 128, 8 wavefronts: a quarter less traffic per output
// SwiGLU needs whole 64-row groups: as many 16-token rows of wavefronts as
// the batch has
using GmGate1 = GmCfg<16, 1, 4, 4, 4, 2, true>;  // 16 x 64
using GmGate2 = GmCfg<16, 2, 4, 4, 4, 4>;        // 32 x 64
using GmGate4 = GmCfg<16, 4, 4, 4, 3, 4>;        // 64 x 64

template <int WF, int EPI>
static hipError_t launch_gemm_k(const GemvArgs& a, int M, hipStream_t st) {
    const long tiles = (long)((a.o + 15) / 16) * ((M + 15) / 16);
    if constexpr (EPI == kEpiSwiglu) {
        if (M <= 16) return launch_gemm_cfg<WF, EPI, GmGate1>(a, M, st);
        if (M <= 32) return launch_gemm_cfg<WF, EPI, GmGate2>(a, M, st);
        if (M <= 64 || tiles <= 4096) return launch_gemm_cfg<WF, EPI, GmGate4>(a, M, st);
    } else {
        if (tiles <= 1536) return launch_gemm_cfg<WF, EPI, GmOne>(a, M, st);
        if (tiles <= 2048) return launch_gemm_cfg<WF, EPI, GmPair>(a, M, st);
        if (tiles <= 4608) return launch_gemm_cfg<WF, EPI, GmQuad>(a, M, st);
    }
    if (tiles < 28672) return launch_gemm_cfg<WF, EPI, GmWide>(a, M, st);
    return launch_gemm_cfg<WF, EPI, GmWide2>(a, M, st);
}

bool gemm_supported(const GemvArgs& a, int wfmt, int epi, int M) {
    if (M < 1 || a.n % 32 || a.nb != a.n / 32 || a.nb < 1) return false;
    // (odd block counts and short batches: only rows the GEMV takes too)
    if (a.n > 16384 && (a.nb % 2 || M < 16)) return false;
    if (wfmt != kQ8 && wfmt != kQ4 && wfmt != kQ8S && wfmt != kQ8S64 && wfmt != kQ8S128) return false;
    if ((wfmt == kQ8S64 && a.nb % 2) || (wfmt == kQ8S128 && a.nb % 4)) return false;
    if (epi == kEpiSwiglu && !a.hq && !a.h_f32) return false;
    if (epi == kEpiSwiglu && (a.o % 64 || a.hidden * 2 != a.o)) return false;
    if (epi == kEpiQkvRope && (a.head_size % 2 || a.att_dim % 32 || a.kv_dim % 32)) return false;
    return true;
}

// The GEMV's time grows with tokens x rows x blocks (about 4 ps per token and
// row-block in Q8_0, 1.7 ps in Q4_0; less while its rows do not fill the chip,
// up to 64 blocks or 4096 rows, and more with one wavefront per row, up to
// 2048 rows of 128 blocks and more), the GEMM's below a full chip only with
// the chain, about 0.1 us per block.  They meet at the tokens x rows below.
// Measured, us, GEMV / GEMM (rows x columns Q8_0 unless named, tokens):
//   2048 x 2048, 15    7.2 / 8.7      8192 x 2048, 4     12.2 / 10.1
//   4096 x 2048, 8     8.8 / 9.3      6144 x 2048, 5     10.1 / 9.1
//   3072 x 2048, 12    9.0 / 8.8      3072 x 4096, 8     12.0 / 14.3
//   4096 x 4096, 6     16.3 / 14.0    6144 x 4096, 4     14.0 / 14.6
//   2048 x 8192, 8     23.4 / 24.1    2048 x 8192, 12    33.3 / 24.1
//   4096 x 8192, 5     24.2 / 25.0    4096 x 8192, 6     29.8 / 25.0
//   Q4_0 4096 x 4096, 12   13.6 / 15.5   Q4_0 6144 x 4096, 12   20.2 / 16.0
// With a normalization (`norm`: the QKV and gate/up rows of a model) the GEMV
// normalizes in every workgroup and the GEMM behind a kernel of its own.
// Whole prompts, us, GEMV / GEMM: four layers of the 1B shape, QKV at 14
// tokens 455 / 364; six of dim 1024, gate/up at 8 tokens 363 / 328; SmolLM2,
// gate/up at 8 tokens 1202 / 1258.
bool gemm_preferred(int wfmt, int o, int nb, int M, bool norm) {
    if (M >= 16 || M < 4) return M >= 16;
    long bound;
    if (norm) bound = wfmt == kQ4 ? 112000 : 40000;
    else if (wfmt == kQ4) bound = 56000;
    else if (nb <= 64) bound = o <= 4096 ? 33000 : 30000;
    else if (nb >= 128 && o <= 2048) bound = 20000;
    else bound = nb <= 128 ? 25000 : 22000;
    return (long)M * o >= bound;
}

hipError_t launch_gemm(const GemvArgs& a, int wfmt, int epi, int M, hipStream_t st) {
    if (!gemm_supported(a, wfmt, epi, M)) return hipErrorInvalidValue;
#define YL_GEMM_EPI(WF)                                                        \
    switch (epi) {                                                             \
    case kEpiStore: return launch_gemm_k<WF, kEpiStore>(a, M, st);            \
    case kEpiQkvRope: return launch_gemm_k<WF, kEpiQkvRope>(a, M, st);        \
    case kEpiResid: return launch_gemm_k<WF, kEpiResid>(a, M, st);            \
    case kEpiSwiglu: return launch_gemm_k<WF, kEpiSwiglu>(a, M, st);          \
    default: return hipErrorInvalidValue;                                      \
    }
    if (wfmt == kQ8) { YL_GEMM_EPI(kQ8) }
    if (wfmt == kQ8S) { YL_GEMM_EPI(kQ8S) }
    if (wfmt == kQ8S64) { YL_GEMM_EPI(kQ8S64) }
    if (wfmt == kQ8S128) { YL_GEMM_EPI(kQ8S128) }
    YL_GEMM_EPI(kQ4)
#undef YL_GEMM_EPI
}

}  // namespace yl
