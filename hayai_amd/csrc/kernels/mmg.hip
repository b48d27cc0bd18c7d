// Many tokens through one weight matrix on the matrix cores, every GGUF format (gfx950):
//   hh_mmg_amax                 per token its largest magnitude, which its f16 operands' power of
//                               two is made of (h's is collected by gate/up as it stores h)
//   hh_mmg_conv                 tokens [b][n] f32 -> token stages (below)
//   hh_mmg_<fmt>_<mode>         Y[t][r] = W[r] . X[t] (execute_quant_gemv_batched, crates/
//                               hayai-core/src/orchestrator.rs:240-269)
//   hh_mmg_<fmt>_<mode>_gu      h[t][r] = act(W_gate[r] . X[t]) * (W_up[r] . X[t]) (prefill_
//                               batched's gate/up, crates/hayai-core/src/prefill_wave.rs:569-584)
//   hh_mmg_sum, hh_mmg_sum_act  the sums of split columns, in split order
// (Compiled after mm_common.hip: its vector types and hh_split_f16.)
//
// Arithmetic.  Weights enter the f16 matrix cores as the exact integers of their format and
// meet their f32 scale after the products: w = d * code, code = q - 8 (Q4_0), q (Q8_0), sc q
// (Q4_K, <= 945), (2 s + 1) * +-grid (IQ2_XXS <= 1333, IQ3_XXS <= 1922), and for Q6_K sc (q - 32)
// up to 4096 as its f16 rounding plus the remainder (-1, 0 or 1), each exact.  A token's
// elements are scaled by one power of two (its largest magnitude into [512, 1024)) and split
// into two f16, hi + lo, which carry 22 bits; products are summed in f32 by the matrix cores
// over one scale block (32 or 256 columns), then d times that is added to the running sum.
// Measured against 64 bits (2-norm): 6e-8 to 1.7e-7 a product, 1.5e-7 to 4e-7 an FFN; for rows that the
// one-token kernels sum in f32 no more than theirs, by short sums (hh_mmg_fine, and at most 512
// columns to a split).
// The Q4_K minimum is dmin * sum_j m_j X_j with X_j the f32 sum of the token's 32 elements of
// sub-block j, as hi + lo f16: one MFMA per superblock (k slots 0..7 hi, 8..15 lo).
//
// MFMA mapping (v_mfma_f32_32x32x16_f16): A = 32 token rows, B = 32 weight rows, so that lane l
// holds outputs of weight row l % 32 only and d is one register per lane.  Lane l supplies k
// slots 8 (l / 32) .. + 7 of its token / its weight row.  A 32-column group takes two steps;
// half h = l / 32 of a weight row's lanes decodes 16 of the group's 32 columns from bytes that
// are contiguous in the block, and the stage is written in the order that gives:
//   columns 16 h + 8 step + e  (Q8_0, Q4_K, Q6_K, IQ)   or   16 step + 8 h + e  (Q4_0),
//   e natural (Q8_0, IQ) or 0 2 1 3 4 6 5 7 (nibble pairs of a dword).
// Weights go from global memory to registers to the matrix core (Q4_K with one token tile by way
// of LDS, hh_mmg_body); tokens pass through LDS, shared by the workgroup's four waves.  A wave owns
// 64 weight rows (32 of gate and the same 32 of up), so each 1 KB token fragment read from LDS
// feeds two MFMAs.
//
// Modes (chosen by the token count alone, plan_mmg): h<TT>: TT tiles of 32 tokens, hi and lo as
// two MFMAs; s16: 16 tokens, hi in A rows 0..15 and lo in rows 16..31 of one MFMA, added at the end.
//
// What bounds it: at hundreds of tokens the matrix cores, busy for 45 to 49 % of a CU's active cycles
// (Q4_K, Q6_K), with the weight decode beside them at two waves per SIMD.  8B FFN, 512 tokens, 2 x 180
// GFLOP of hi and lo: 0.43 ms IQ2_XXS, 0.60 ms Q6_K, 0.93 ms Q8_0 with its splits, 390 .. 840 TFLOP/s
// (one token at a time these took 12 .. 39 ms).  With few tokens the loads: a lane's row is a line of
// its own in every instruction (Q8_0, 77 tokens: matrix cores 13 % busy, waits 24 %); at 4..16 tokens
// the weight stream's latency (8B Q6_K FFN, 16 tokens: 82 us against 779 us).
//
// MoE (hh_mmg_moe_*): the (token, slot) pairs of an expert in tiles of 16 or 32, one launch over
// every (tile, row group).  128 experts of 2048 x 768, 512 tokens: 1220 -> 225 us a layer.
//
// Token stages: [tile][128-column chunk][group 0..3][step 0..1][hi, lo][lane][8 f16], for Q4_K
// followed after every second chunk by the sums [lane][8 f16] (lane half 0: hi of sub-blocks
// 0..7, half 1: lo).
typedef float hh_f16v __attribute__((ext_vector_type(16)));

enum { HH_MMG_H = 0, HH_MMG_S16 = 1, HH_MMG_F = 2 };
#define HH_MMG_WSLOT 9216u  // a wave's 64 Q4_K rows of one superblock in LDS

struct hh_mmg_args {
    const uint8_t* w0;       // GEMM: W; gate/up: W_gate
    const uint8_t* w1;       // GEMM: W; gate/up: W_up
    const uint8_t* xs;       // token stages
    const float* amax;       // per token: what its scaling was made of
    float* pmax;             // gate/up: [row group][ldt] the group's largest magnitude of each token's h
    float* y;                // kc == 1: Y [b][m] or h [b][m]; else the splits' sums
    uint64_t row_bytes;
    uint64_t tile_bytes;     // stage bytes of one token tile
    uint64_t part_stride;    // kc > 1: floats between two splits' sums
    uint64_t up_stride;      // kc > 1, gate/up: floats from gate's sums to up's
    uint32_t m, n, b;
    uint32_t nch;            // 128-column chunks (the last may be partly past n)
    uint32_t cpk;            // chunks per split (even for formats of 256-column blocks)
    uint32_t kc;             // splits
    uint32_t groups;         // row groups
    uint32_t ttiles;         // token tile groups
    int32_t act;
    uint32_t ldt;
    // MoE: tiles of one expert's pairs (hh_mmg_moe_args); w0 / w1 are expert 0's matrices
    const int4* trec;
    const int32_t* order;
    uint64_t expert_stride;
};

// Bytes at any address (2-byte aligned in GGUF formats): the hardware takes unaligned loads.
HH_DEV uint4 hh_ldu16(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
HH_DEV uint2 hh_ldu8(const uint8_t* p) {
    uint2 v;
    __builtin_memcpy(&v, p, 8);
    return v;
}
HH_DEV uint32_t hh_ldu4(const uint8_t* p) {
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

HH_DEV hh_h2 hh_h2_all(float v) { return hh_h2{(_Float16)v, (_Float16)v}; }
HH_DEV hh_h8 hh_h8_of(hh_h2 a, hh_h2 b, hh_h2 c, hh_h2 d) { return hh_h8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y}; }
// bytes i and j of v as the f16 pair 1024 + byte
template <uint32_t I, uint32_t J>
HH_DEV hh_h2 hh_bytes_h2(uint32_t v) {
    return hh_h2_bits(__builtin_amdgcn_perm(0x64646464u, v, I | (4u << 8) | (J << 16) | (4u << 24)));
}

// Masks and exponent bits of the decodes, held in registers: a gfx9 VOP3 instruction takes no
// literal, so only so is (v & mask) | bits one v_and_or_b32.
struct hh_mmg_k {
    uint32_t lo, hi, magic;  // 0x000F000F, 0x00F000F0 (scalar), 0x64006400 (vector)
    uint32_t b30;            // 0x30303030 (scalar)
    HH_DEV void set() {
        asm volatile("s_mov_b32 %0, 0x000F000F" : "=s"(lo));
        asm volatile("s_mov_b32 %0, 0x00F000F0" : "=s"(hi));
        asm volatile("s_mov_b32 %0, 0x30303030" : "=s"(b30));
        asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    }
};

// ---- weight formats -------------------------------------------------------------------
// Raw: one chunk's bytes of one row as loaded (ready: what is taken from them once); load(p, ch,
// ...) of chunk ch of the row at p (half h); frag(raw, g, s): the B operand of step s of the chunk's group g; scale(raw, g):
// the d of the block that group g closes.  NB: B operands per step.  RUN: groups (32 columns) that
// the matrix cores sum before d.
// The 32-column formats: lane half h loads the two whole blocks 4 ch + 2 h, + 1 (consecutive
// bytes: 3 loads for Q4_0, 5 for Q8_0, where a load of each half block and each d took 8), and
// `ready` exchanges halves with the lane of the same row: then every lane has its half of all four.
// With its 64 lanes in 64 places every load holds the address unit for as long as 64 lines take.
// When it was made, 8B FFN: 512 tokens Q8_0 888 -> 717 us, Q4_0 593 -> 455 us; 16 tokens Q4_0 92 -> 72.
HH_DEV void hh_swap32(uint32_t& a, uint32_t& b) {  // a's upper 32 lanes with b's lower 32
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// Two blocks of QW code dwords each: w[0] low half d of the first, then its codes at half a dword,
// w[QW] high half d of the second, then its codes.  After `ready` w[0 ..] groups 0, 2, w[QW] and dx
// the four d, w[QW + 1 ..] groups 1, 3 (in place, for a copy would stay live beside it: two token
// tiles of Q8_0 are at 256 registers and spill about ten even so).
template <uint32_t QW>
struct hh_mmg_pair {
    static constexpr uint32_t BB = 4 * QW + 2;
    uint32_t w[2 * QW + 1], dx;
    HH_DEV static void put(uint32_t* o, uint4 v) { o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w; }
    HH_DEV void load(const uint8_t* p, uint32_t ch, uint32_t h, uint32_t nblk) {
        const uint32_t k = 4 * ch + 2 * h;
        if (4 * ch + 4 <= nblk) {
            const uint8_t* b = p + k * BB;
#pragma unroll
            for (uint32_t i = 0; i < QW / 2; i++) put(w + 4 * i, hh_ldu16(b + 16 * i));
            w[2 * QW] = hh_ldu4(b + 8 * QW);
        } else {  // the row's end: block by block, d = 0 past it
            uint32_t c[2][QW], d[2];
#pragma unroll
            for (uint32_t i = 0; i < 2; i++) {
                const uint8_t* b = p + min(k + i, nblk - 1) * BB;
                d[i] = k + i < nblk ? hh_ld_u16(b) : 0u;
#pragma unroll
                for (uint32_t j = 0; j < QW; j += 4) put(c[i] + j, hh_ldu16(b + 2 + 4 * j));
            }
            w[0] = d[0] | c[0][0] << 16;
#pragma unroll
            for (uint32_t i = 1; i < QW; i++) w[i] = __builtin_amdgcn_alignbit(c[0][i], c[0][i - 1], 16);
            w[QW] = c[0][QW - 1] >> 16 | d[1] << 16;
#pragma unroll
            for (uint32_t i = 0; i < QW; i++) w[QW + 1 + i] = c[1][i];
        }
    }
    HH_DEV void ready() {
        const uint32_t d = (w[0] & 0xFFFFu) | (w[QW] & 0xFFFF0000u);
#pragma unroll
        for (uint32_t i = 0; i < QW; i++) w[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], 16);
        w[QW] = dx = d;
        hh_swap32(w[QW], dx);
#pragma unroll
        for (uint32_t i = 0; i < QW / 2; i++) {
            hh_swap32(w[i], w[QW / 2 + i]);
            hh_swap32(w[QW + 1 + i], w[QW + 1 + QW / 2 + i]);
        }
    }
    HH_DEV uint32_t code(int g, int i) const { return w[(g & 1 ? QW + 1 : 0) + (g & 2 ? QW / 2 : 0) + i]; }
    HH_DEV float scale(int g) const {
        const uint32_t d = g & 2 ? dx : w[QW];
        return hh_f16(g & 1 ? d >> 16 : d & 0xFFFFu);
    }
};

struct hh_mmg_q4_0 {
    static constexpr bool SUPER = false, MINS = false, TABLES = false, READY = true, ROWS_LDS = false;
    static constexpr int RUN = 1;
    static constexpr int NB = 1;
    typedef hh_mmg_pair<4> Raw;
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t h, uint32_t nblk) {
        r.load(p, ch, h, nblk);
    }
    template <uint32_t HALF>
    HH_DEV static void ready(Raw& r) {
        r.ready();
    }
    HH_DEV static float scale(const Raw& r, int g) { return r.scale(g); }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t, const char*, const hh_mmg_k& k, hh_h8* f) {
        const uint32_t v[4] = {r.code(g, 0), r.code(g, 0) >> 8, r.code(g, 1), r.code(g, 1) >> 8};
        hh_h2 o[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (s == 0)  // 1024 + q, q - 8
                o[i] = hh_h2_bits((v[i] & k.lo) | k.magic) - hh_h2_all(1032.f);
            else  // 1024 + 16 q, q - 8 (exact: the FMA rounds only its result)
                o[i] = __builtin_elementwise_fma(hh_h2_bits((v[i] & k.hi) | k.magic), hh_h2_all(0.0625f),
                                                 hh_h2_all(-72.f));
        }
        f[0] = hh_h8_of(o[0], o[1], o[2], o[3]);
    }
};

struct hh_mmg_q8_0 {
    static constexpr bool SUPER = false, MINS = false, TABLES = false, READY = true, ROWS_LDS = false;
    static constexpr int RUN = 1;
    static constexpr int NB = 1;
    typedef hh_mmg_pair<8> Raw;
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t h, uint32_t nblk) {
        r.load(p, ch, h, nblk);
    }
    template <uint32_t HALF>
    HH_DEV static void ready(Raw& r) {
        r.ready();
    }
    HH_DEV static float scale(const Raw& r, int g) { return r.scale(g); }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t, const char*, const hh_mmg_k& k, hh_h8* f) {
        const uint32_t a = r.code(g, 2 * s) ^ 0x80808080u, b = r.code(g, 2 * s + 1) ^ 0x80808080u;
        const hh_h2 z = hh_h2_all(1152.f);  // 1024 + (q + 128)
        f[0] = hh_h8_of(hh_bytes_h2<0, 1>(a) - z, hh_bytes_h2<2, 3>(a) - z, hh_bytes_h2<0, 1>(b) - z,
                        hh_bytes_h2<2, 3>(b) - z);
    }
};

struct hh_mmg_q4_k {
    static constexpr bool SUPER = true, MINS = true, TABLES = false, READY = true, ROWS_LDS = true;
    static constexpr int RUN = 8;
    static constexpr int NB = 1;
    struct Raw {
        uint4 q[2];
        uint4 hd;
        uint32_t sch;  // the chunk's four sub-block scales
    };
    template <uint32_t HALF>
    HH_DEV static void ready(Raw& r) {
        r.sch = HALF ? (r.hd.w & 0x0F0F0F0Fu) | ((r.hd.y >> 2) & 0x30303030u) : r.hd.y & 0x3F3F3F3Fu;
    }
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t h, uint32_t) {
        const uint8_t* b = p + (ch >> 1) * 144u;
        r.hd = hh_ld16(b);
        r.q[0] = hh_ld16(b + 16 + 64 * HALF + 16 * h);
        r.q[1] = hh_ld16(b + 48 + 64 * HALF + 16 * h);
    }
    // one row's superblock in LDS (both halves' raw)
    HH_DEV static void load_lds(Raw& r0, Raw& r1, const char* b, uint32_t h) {
        const uint4* v = reinterpret_cast<const uint4*>(b);
        r0.hd = r1.hd = v[0];
        r0.q[0] = v[1 + h], r0.q[1] = v[3 + h];
        r1.q[0] = v[5 + h], r1.q[1] = v[7 + h];
    }
    HH_DEV static float scale(const Raw& r, int) { return hh_f16(r.hd.x & 0xFFFFu); }
    HH_DEV static float min_scale(const Raw& r) { return hh_f16(r.hd.x >> 16); }
    // the minima m_0 .. m_7 (get_scale_min_k4, q4k.rs:34-43), the same in both lane halves
    HH_DEV static hh_h8 mins(const Raw& r) {
        const uint32_t lo = r.hd.z & 0x3F3F3F3Fu, hi = ((r.hd.w >> 4) & 0x0F0F0F0Fu) | ((r.hd.z >> 2) & 0x30303030u);
        const hh_h2 z = hh_h2_all(1024.f);
        return hh_h8_of(hh_bytes_h2<0, 1>(lo) - z, hh_bytes_h2<2, 3>(lo) - z, hh_bytes_h2<0, 1>(hi) - z,
                        hh_bytes_h2<2, 3>(hi) - z);
    }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t, const char*, const hh_mmg_k& k, hh_h8* f) {
        // sub-blocks 2p (low nibbles) and 2p + 1 (high) of the 32 qs bytes p
        const uint4 q = r.q[g >> 1];
        const uint32_t a = s ? q.z : q.x, b = s ? q.w : q.y;
        const uint32_t v[4] = {a, a >> 8, b, b >> 8};
        const uint32_t sel = (uint32_t)g | (4u << 8) | ((uint32_t)g << 16) | (4u << 24);
        const hh_h2 sc = hh_h2_bits(__builtin_amdgcn_perm(0x64646464u, r.sch, sel)) - hh_h2_all(1024.f);
        const hh_h2 mul = (g & 1) ? sc * hh_h2_all(0.0625f) : sc;
        const hh_h2 off = mul * hh_h2_all(-1024.f);
        const uint32_t mask = (g & 1) ? k.hi : k.lo;
        hh_h2 o[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
            o[i] = __builtin_elementwise_fma(hh_h2_bits((v[i] & mask) | k.magic), mul, off);
        f[0] = hh_h8_of(o[0], o[1], o[2], o[3]);
    }
};

struct hh_mmg_q6_k {
    static constexpr bool SUPER = true, MINS = false, TABLES = false, READY = false, ROWS_LDS = false;
    static constexpr int RUN = 8;
    static constexpr int NB = 2;
    struct Raw {
        uint4 a, b, qh;
        uint2 sc;
        uint32_t d;
    };
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t h, uint32_t) {
        const uint8_t* b = p + (ch >> 1) * 210u;
        const uint32_t n = HALF;
        r.a = hh_ldu16(b + 64 * n + 16 * h);
        r.b = hh_ldu16(b + 64 * n + 32 + 16 * h);
        r.qh = hh_ldu16(b + 128 + 32 * n + 16 * h);
        r.sc = hh_ldu8(b + 192 + 8 * n);
        r.d = hh_ld_u16(b + 208);
    }
    HH_DEV static float scale(const Raw& r, int) { return hh_f16(r.d); }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t h, const char*, const hh_mmg_k& k, hh_h8* f) {
        const uint4 l = (g & 1) ? r.b : r.a;
        const uint32_t la = s ? l.z : l.x, lb = s ? l.w : l.y, ha = s ? r.qh.z : r.qh.x, hb = s ? r.qh.w : r.qh.y;
        // scale byte 2 g + h of the chunk's eight
        const uint32_t sw = (g & 2) ? r.sc.y : r.sc.x;
        const float scf = (float)(int8_t)(sw >> (16 * (g & 1) + 8 * h));
        const hh_h2 sc = hh_h2_all(scf);
        // bits 2 g, 2 g + 1 of each qh byte to bits 4, 5
        const uint32_t ta = g == 0 ? ha << 4 : g == 1 ? ha << 2 : g == 2 ? ha : ha >> 2;
        const uint32_t tb = g == 0 ? hb << 4 : g == 1 ? hb << 2 : g == 2 ? hb : hb >> 2;
        const uint32_t q[2] = {(ta & k.b30) | (((g & 2) ? la >> 4 : la) & 0x0F0F0F0Fu),
                               (tb & k.b30) | (((g & 2) ? lb >> 4 : lb) & 0x0F0F0F0Fu)};
        hh_h2 hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = q[i >> 1];
            const hh_h2 t = ((i & 1) ? hh_bytes_h2<2, 3>(v) : hh_bytes_h2<0, 1>(v)) - hh_h2_all(1056.f);
            hi[i] = t * sc;                                        // rounded to f16
            lo[i] = __builtin_elementwise_fma(t, sc, -hi[i]);      // the rest, exact
        }
        f[0] = hh_h8_of(hi[0], hi[1], hi[2], hi[3]);
        f[1] = hh_h8_of(lo[0], lo[1], lo[2], lo[3]);
    }
};

// IQ tables as f16: the codebook entries' magnitudes, and per sign index a mask of sign bits.
constexpr uint16_t hh_f16_of_small(uint32_t v) {  // an integer below 2048 as f16 bits
    uint32_t e = 0;
    while ((v >> (e + 1)) != 0) e++;
    return v == 0 ? (uint16_t)0 : (uint16_t)(((e + 15) << 10) | ((v << (10 - e)) & 0x3FFu));
}
struct hh_mmg_iq2_tab {
    uint16_t grid[256 * 8];
    uint16_t sign[128 * 8];
};
struct hh_mmg_iq3_tab {
    uint16_t grid[256 * 4];
    uint16_t sign[128 * 8];
};
constexpr void hh_mmg_signs(uint16_t* s) {
    for (uint32_t i = 0; i < 128; i++) {
        uint32_t par = 0;
        for (uint32_t k = 0; k < 7; k++) par ^= (i >> k) & 1u;
        for (uint32_t k = 0; k < 8; k++) s[8 * i + k] = ((k < 7 ? (i >> k) & 1u : par) != 0) ? 0x8000u : 0u;
    }
}
constexpr hh_mmg_iq2_tab hh_mmg_make_iq2() {
    constexpr uint64_t g[256] = {HH_IQ2XXS_GRID_VALUES};
    hh_mmg_iq2_tab t{};
    for (uint32_t i = 0; i < 256; i++)
        for (uint32_t k = 0; k < 8; k++) t.grid[8 * i + k] = hh_f16_of_small((uint32_t)(g[i] >> (8 * k)) & 0xFFu);
    hh_mmg_signs(t.sign);
    return t;
}
constexpr hh_mmg_iq3_tab hh_mmg_make_iq3() {
    constexpr uint32_t g[256] = {HH_IQ3XXS_GRID_VALUES};
    hh_mmg_iq3_tab t{};
    for (uint32_t i = 0; i < 256; i++)
        for (uint32_t k = 0; k < 4; k++) t.grid[4 * i + k] = hh_f16_of_small((g[i] >> (8 * k)) & 0xFFu);
    hh_mmg_signs(t.sign);
    return t;
}
__device__ const __attribute__((aligned(16))) hh_mmg_iq2_tab hh_mmg_iq2_table = hh_mmg_make_iq2();
__device__ const __attribute__((aligned(16))) hh_mmg_iq3_tab hh_mmg_iq3_table = hh_mmg_make_iq3();

HH_DEV hh_h8 hh_mmg_iq_frag(uint4 grid, uint4 sign, uint32_t aux) {
    const hh_h2 sc = hh_h2_all((float)(2u * (aux >> 28) + 1u));
    return hh_h8_of(hh_h2_bits(grid.x ^ sign.x) * sc, hh_h2_bits(grid.y ^ sign.y) * sc,
                    hh_h2_bits(grid.z ^ sign.z) * sc, hh_h2_bits(grid.w ^ sign.w) * sc);
}

struct hh_mmg_iq2_xxs {
    static constexpr bool SUPER = true, MINS = false, TABLES = true, READY = false, ROWS_LDS = false;
    static constexpr int RUN = 8;
    static constexpr int NB = 1;
    static constexpr uint32_t TAB = sizeof(hh_mmg_iq2_tab);
    HH_DEV static const uint8_t* table() { return (const uint8_t*)&hh_mmg_iq2_table; }
    struct Raw {
        uint2 q[4];
        uint32_t d;
    };
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t, uint32_t) {
        const uint8_t* b = p + (ch >> 1) * 66u;
#pragma unroll
        for (uint32_t g = 0; g < 4; g++) r.q[g] = hh_ldu8(b + 2 + 8 * (4 * HALF + g));
        r.d = hh_ld_u16(b);
    }
    // d * (0.5 + s) * 0.25 = d / 8 * (2 s + 1)
    HH_DEV static float scale(const Raw& r, int) { return hh_f16(r.d) * 0.125f; }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t h, const char* tab, const hh_mmg_k&, hh_h8* f) {
        const uint32_t l = 2 * h + (uint32_t)s, aux = r.q[g].y;
        const uint32_t idx = (r.q[g].x >> (8 * l)) & 0xFFu, sg = (aux >> (7 * l)) & 127u;
        f[0] = hh_mmg_iq_frag(*reinterpret_cast<const uint4*>(tab + idx * 16),
                              *reinterpret_cast<const uint4*>(tab + 4096 + sg * 16), aux);
    }
};

struct hh_mmg_iq3_xxs {
    static constexpr bool SUPER = true, MINS = false, TABLES = true, READY = false, ROWS_LDS = false;
    static constexpr int RUN = 8;
    static constexpr int NB = 1;
    static constexpr uint32_t TAB = sizeof(hh_mmg_iq3_tab);
    HH_DEV static const uint8_t* table() { return (const uint8_t*)&hh_mmg_iq3_table; }
    struct Raw {
        uint32_t q[4];
        uint4 aux;
        uint32_t d;
    };
    template <uint32_t HALF>
    HH_DEV static void load(Raw& r, const uint8_t* p, uint32_t ch, uint32_t h, uint32_t) {
        const uint8_t* b = p + (ch >> 1) * 98u;
        const uint32_t n = HALF;
#pragma unroll
        for (uint32_t g = 0; g < 4; g++) r.q[g] = hh_ldu4(b + 2 + 8 * (4 * n + g) + 4 * h);
        r.aux = hh_ldu16(b + 66 + 16 * n);
        r.d = hh_ld_u16(b);
    }
    // d * (0.5 + s) * 0.5 = d / 4 * (2 s + 1)
    HH_DEV static float scale(const Raw& r, int) { return hh_f16(r.d) * 0.25f; }
    template <uint32_t HALF>
    HH_DEV static void frag(const Raw& r, int g, int s, uint32_t h, const char* tab, const hh_mmg_k&, hh_h8* f) {
        const uint32_t l = 2 * h + (uint32_t)s;
        const uint32_t aux = g == 0 ? r.aux.x : g == 1 ? r.aux.y : g == 2 ? r.aux.z : r.aux.w;
        const uint32_t i0 = (r.q[g] >> (16 * s)) & 0xFFu, i1 = (r.q[g] >> (16 * s + 8)) & 0xFFu;
        const uint2 a = *reinterpret_cast<const uint2*>(tab + i0 * 8), b = *reinterpret_cast<const uint2*>(tab + i1 * 8);
        f[0] = hh_mmg_iq_frag(make_uint4(a.x, a.y, b.x, b.y),
                              *reinterpret_cast<const uint4*>(tab + 2048 + ((aux >> (7 * l)) & 127u) * 16), aux);
    }
};

// For rows that the one-token kernels sum in f32 (MmgForm::Fine): 64 columns (Q6_K, with its
// remainders, 32) to a sum of the matrix cores, whose additions over 256 alone lose more than an
// f32 product does.  2048 x 3840, 24 tokens, against 64 bits: IQ2_XXS 1.74e-7 -> 1.06e-7 (one token
// 1.28e-7), Q6_K 1.82e-7 -> 1.05e-7 (1.13e-7).
template <class F>
struct hh_mmg_fine : F {
    static constexpr int RUN = F::NB > 1 ? 1 : 2;
};
typedef hh_mmg_fine<hh_mmg_q6_k> hh_mmg_q6_k_fine;
typedef hh_mmg_fine<hh_mmg_iq2_xxs> hh_mmg_iq2_xxs_fine;
typedef hh_mmg_fine<hh_mmg_iq3_xxs> hh_mmg_iq3_xxs_fine;

// ---- tokens -> stages -----------------------------------------------------------------

struct hh_mmg_conv_args {
    const float* x;        // [b][n]
    uint8_t* xs;           // stages
    float* amax;           // per token: its largest magnitude
    const float* pmax;     // h: gate/up's [pgroups][ldt] largest magnitudes over its row groups,
                           // from which amax is made (and written) here; null: amax is given
    uint64_t tile_bytes;
    uint32_t b, n, nch;
    uint32_t rows;         // tokens per tile: 32, or 16 (mode s16)
    uint32_t mins;         // write the sub-block sums
    uint32_t half_major;   // column order 16 h + 8 step + e (else 16 step + 8 h + e)
    uint32_t paired;       // e in the order 0 2 1 3 4 6 5 7
    uint32_t pgroups, ldt;
    uint32_t single;       // mode f: hi alone, the sums as two bf16
};

struct hh_mmg_amax_args {
    const float* x;  // [b][n]
    float* amax;     // per token
    uint32_t n, pad;
};

// A token's amax: the largest of its finite magnitudes.  amax in [2^(k-1), 2^k) -> up = 2^(10 - k):
// the largest magnitude into [512, 1024), so that a sum of 32 elements stays below f16's largest
// value; infinities stay what they are under any factor.  A token of zeros keeps the factor 1.
HH_DEV float hh_mmg_mag(float x) { return fabsf(x) < __builtin_inff() ? fabsf(x) : 0.f; }
HH_DEV int hh_mmg_exp(float amax) {
    if (amax == 0.f) return 0;
    int k;
    (void)frexpf(amax, &k);
    return min(max(10 - k, -120), 120);
}
HH_DEV float hh_wave_max(float v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// A workgroup of 256 threads: the amax of x[0, n).
template <class MAG>
HH_DEV float hh_mmg_wave_amax(const float* x, uint32_t n, MAG mag) {
    float v = 0.f;
    if ((((uintptr_t)x | n) & 3u) == 0 && ((uintptr_t)x & 15u) == 0) {
        const float4* x4 = reinterpret_cast<const float4*>(x);
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < n / 4; i += 256) {
            const float4 u = x4[i];
            v = fmaxf(v, fmaxf(fmaxf(mag(u.x), mag(u.y)), fmaxf(mag(u.z), mag(u.w))));
        }
    } else {
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < n; i += 256) v = fmaxf(v, mag(x[i]));
    }
    return hh_wave_max(v);
}
HH_DEV void hh_mmg_token_amax(const float* x, uint32_t n, float* amax) {
    __shared__ float red[4];
    float v = hh_mmg_wave_amax(x, n, [](float e) { return fabsf(e); });  // (fmaxf leaves NaN out)
    if (v == __builtin_inff()) v = hh_mmg_wave_amax(x, n, hh_mmg_mag);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    if (threadIdx.x == 0) *amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
extern "C" __global__ void __launch_bounds__(256) hh_mmg_amax(const hh_mmg_amax_args a) {
    hh_mmg_token_amax(a.x + (size_t)blockIdx.x * a.n, a.n, a.amax + blockIdx.x);
}
HH_DEV float hh_mmg_up(float amax) { return ldexpf(1.f, hh_mmg_exp(amax)); }
HH_DEV float hh_mmg_down(float amax) { return ldexpf(1.f, -hh_mmg_exp(amax)); }

// f32 -> bf16 bits, to nearest even (infinities stay; a NaN keeps a set mantissa bit)
HH_DEV uint32_t hh_bf16(float v) {
    const uint32_t b = __float_as_uint(v);
    if ((b & 0x7FFFFFFFu) >= 0x7F800000u) return (b >> 16) | ((b & 0x7FFFFFu) ? 0x40u : 0u);
    return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}

// v = hi + lo.  An infinity is in lo, with the largest finite hi: hi meets Q6_K's remainders too, most
// of which are 0, and lo only the codes' own products.
HH_DEV void hh_mmg_split(float v, _Float16& hi, _Float16& lo) {
    hi = (_Float16)__builtin_amdgcn_fmed3f(v, -65504.f, 65504.f);
    lo = (_Float16)(v - (float)hi);
}

// One chunk of one tile, by a workgroup of `threads`.  row(tok, &src, &up): the tile's token tok
// as its f32 row and factor, false past the tokens (zeros; columns past n are zeros too).
template <class ROW>
HH_DEV void hh_mmg_conv_chunk(uint8_t* tile, const hh_mmg_conv_args& a, uint32_t ch, bool vec, uint32_t threads,
                              ROW row) {
    const bool s16 = a.rows == 16;
    const uint32_t chunk_bytes = (s16 || a.single ? 8u : 16u) * 1024u;
    uint8_t* st = tile + (a.mins ? (size_t)(ch >> 1) * (2 * chunk_bytes + 1024u) + (ch & 1u) * chunk_bytes
                                 : (size_t)ch * chunk_bytes);
    for (uint32_t p = threadIdx.x; p < (s16 ? 256u : 512u); p += threads) {
        // piece p: group, step, lane half, token
        const uint32_t tok = p % a.rows, h = (p / a.rows) & 1u, step = (p / a.rows >> 1) & 1u, g = p / a.rows >> 2;
        const uint32_t col = 128 * ch + 32 * g + (a.half_major ? 16 * h + 8 * step : 16 * step + 8 * h);
        float v[8];
        const float* src;
        float up;
        if (col < a.n && row(tok, src, up)) {
            src += col;
            if (vec) {
                const float4 u0 = reinterpret_cast<const float4*>(src)[0], u1 = reinterpret_cast<const float4*>(src)[1];
                v[0] = u0.x, v[1] = u0.y, v[2] = u0.z, v[3] = u0.w, v[4] = u1.x, v[5] = u1.y, v[6] = u1.z, v[7] = u1.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = src[e];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] *= up;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = 0.f;
        }
        if (a.paired) {
            float s = v[1];
            v[1] = v[2], v[2] = s;
            s = v[5];
            v[5] = v[6], v[6] = s;
        }
        hh_h8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            _Float16 x0, x1;
            hh_mmg_split(v[e], x0, x1);
            hi[e] = a.single ? (_Float16)v[e] : x0;
            lo[e] = x1;
        }
        const uint32_t gs = g * 2 + step;
        if (s16) {
            *reinterpret_cast<hh_h8*>(st + gs * 1024u + (32 * h + tok) * 16u) = hi;
            *reinterpret_cast<hh_h8*>(st + gs * 1024u + (32 * h + 16 + tok) * 16u) = lo;
        } else if (a.single) {
            *reinterpret_cast<hh_h8*>(st + gs * 1024u + (32 * h + tok) * 16u) = hi;
        } else {
            *reinterpret_cast<hh_h8*>(st + gs * 2048u + (32 * h + tok) * 16u) = hi;
            *reinterpret_cast<hh_h8*>(st + gs * 2048u + 1024u + (32 * h + tok) * 16u) = lo;
        }
    }
    if (!a.mins) return;
    uint8_t* sums = tile + (size_t)(ch >> 1) * (2 * chunk_bytes + 1024u) + 2 * chunk_bytes;
    const uint32_t q = threadIdx.x;  // token row, group
    if (q >= 128) return;
    const uint32_t r = q % 32, g = q / 32, j = 4 * (ch & 1u) + g;
    float s = 0.f;
    const float* src;
    float up;
    if (r < a.rows && row(r, src, up)) {
        src += 128 * ch + 32 * g;
        for (int e = 0; e < 32; e++) s += src[e] * up;
    }
    if (a.single) {
        const uint32_t hi = hh_bf16(s), lo = hh_bf16(s - __uint_as_float(hi << 16));
        *reinterpret_cast<uint16_t*>(sums + r * 16 + j * 2) = (uint16_t)hi;
        *reinterpret_cast<uint16_t*>(sums + 512 + r * 16 + j * 2) = (uint16_t)lo;
        return;
    }
    _Float16 hi, lo;
    hh_mmg_split(s, hi, lo);
    *reinterpret_cast<_Float16*>(sums + r * 16 + j * 2) = hi;  // s16: rows 16..31 are zeros
    *reinterpret_cast<_Float16*>(sums + 512 + r * 16 + j * 2) = lo;
}

// The factors of a tile's rows into LDS; index(row): the row's place in amax / pmax.
template <class IDX>
HH_DEV void hh_mmg_ups(float* ups, const hh_mmg_conv_args& a, uint32_t count, bool store, IDX index) {
    __shared__ float red[8][32];
    const uint32_t row = threadIdx.x % 32, part = threadIdx.x / 32;
    if (a.pmax) {
        float v = 0.f;
        if (row < count) {
            const float* p = a.pmax + index(row);
#pragma unroll 4
            for (uint32_t g = part; g < a.pgroups; g += 8) v = fmaxf(v, p[(size_t)g * a.ldt]);
        }
        red[part][row] = v;
        __syncthreads();
    }
    if (part == 0 && row < count) {
        float v;
        if (a.pmax) {
            v = red[0][row];
#pragma unroll
            for (int k = 1; k < 8; k++) v = fmaxf(v, red[k][row]);
            if (store) a.amax[index(row)] = v;
        } else {
            v = a.amax[index(row)];
        }
        ups[row] = hh_mmg_up(v);
    }
    __syncthreads();
}

// One workgroup per (token tile, chunk).
extern "C" __global__ void __launch_bounds__(256) hh_mmg_conv(const hh_mmg_conv_args a) {
    __shared__ float ups[32];
    const uint32_t tile = blockIdx.x / a.nch, ch = blockIdx.x % a.nch;
    const uint32_t t0 = tile * a.rows, count = t0 < a.b ? min(a.rows, a.b - t0) : 0u;
    hh_mmg_ups(ups, a, count, ch == 0, [&](uint32_t row) { return t0 + row; });
    hh_mmg_conv_chunk(a.xs + tile * a.tile_bytes, a, ch, ((uintptr_t)a.x & 15u) == 0, 256,
                      [&](uint32_t tok, const float*& src, float& up) {
                          if (tok >= count) return false;
                          src = a.x + (size_t)(t0 + tok) * a.n;
                          up = ups[tok];
                          return true;
                      });
}

// MoE: tiles of one expert's (token, slot) pairs.  trec[0].x: how many; trec[1 + tile]: the
// expert, the tile's first position in `order`, its pairs.
struct hh_mmg_moe_args {
    hh_mmg_conv_args c;      // x: tokens [T][n] and their amax; h: tile rows [tile][rows][n] and theirs
    const int4* trec;
    const int32_t* order;
    float* amax_row;         // x: per tile row, its token's amax
    uint32_t k, pad;         // slots per token; 0: h
};
// One workgroup per (tile, chunk).  x: each row is its pair's token; h: the row itself.
extern "C" __global__ void __launch_bounds__(256) hh_mmg_moe_conv(const hh_mmg_moe_args a) {
    __shared__ float ups[32];
    const uint32_t tile = blockIdx.x / a.c.nch, ch = blockIdx.x % a.c.nch;
    if (tile >= (uint32_t)a.trec[0].x) return;
    const int4 rec = a.trec[1 + tile];
    auto token = [&](uint32_t row) {
        return a.k ? (uint32_t)a.order[rec.y + (int)row] / a.k : tile * a.c.rows + row;
    };
    hh_mmg_ups(ups, a.c, (uint32_t)rec.z, ch == 0, token);
    hh_mmg_conv_chunk(a.c.xs + tile * a.c.tile_bytes, a.c, ch, true, 256,
                      [&](uint32_t tok, const float*& src, float& up) {
                          if ((int)tok >= rec.z) return false;
                          src = a.c.x + (size_t)token(tok) * a.c.n;
                          up = ups[tok];
                          return true;
                      });
    if (a.k && ch == 0 && (int)threadIdx.x < rec.z)
        a.amax_row[tile * a.c.rows + threadIdx.x] = a.c.amax[token(threadIdx.x)];
}

template <uint32_t V>
struct hh_uint_c {
    static constexpr uint32_t value = V;
};

// ---- the product ----------------------------------------------------------------------

// Tokens' LDS copies in flight and all LDS reads of this wave done, then the workgroup meets.
HH_DEV void hh_mmg_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// What the outputs of a workgroup's N token rows need, into LDS while the first loads are on
// their way: the factors back, and for MoE's down the pairs.  Read from memory at the end, four
// rows at a time, each read's latency was in the way (MoE above: gate/up 128 -> 112 us, down
// 78 -> 58).
template <uint32_t N>
struct __attribute__((aligned(16))) hh_mmg_tokens {
    float down[N];
    uint32_t pair[N];
    HH_DEV void set(const hh_mmg_args& a, uint32_t tg, int4 rec, bool pairs) {
        const uint32_t t = threadIdx.x;
        if (t >= N) return;
        down[t] = hh_mmg_down(a.amax[tg * N + t]);  // padded to whole tiles
        if (pairs) pair[t] = (uint32_t)a.order[rec.y + min((int)t, rec.z - 1)];
    }
};

// The sums of a wave's 64 weight rows and TT token tiles to memory (gate/up: the activation,
// and the row group's largest |h| of each token).
template <int MODE, int TT, bool GU, bool MOE>
HH_DEV void hh_mmg_store(const hh_mmg_args& a, const hh_f16v (&sum)[2][TT], const uint32_t (&row)[2], int4 rec,
                         uint32_t tg, uint32_t grp, uint32_t kci,
                         const hh_mmg_tokens<TT * (MODE == HH_MMG_S16 ? 16 : 32)>& tok) {
    constexpr uint32_t ROWS = MODE == HH_MMG_S16 ? 16 : 32;  // tokens per tile
    extern __shared__ __attribute__((aligned(16))) char hh_smem[];
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t r = lane & 31u, h = lane >> 5;
    // outputs: lane's weight row, tokens 8 (i / 4) + 4 h + i % 4 of each tile
    float* const out = a.y + (a.kc > 1 ? kci * a.part_stride : 0);
    const bool fuse = GU && (MOE || a.kc == 1);
    float* const wmax = reinterpret_cast<float*>(hh_smem) + wave * 2 * (TT * ROWS);  // gate/up: per token
    if (fuse) hh_mmg_sync();  // the token buffers are read
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
#pragma unroll
        for (int i4 = 0; i4 < (MODE == HH_MMG_S16 ? 2 : 4); i4++) {
            const uint32_t in = 8 * i4 + 4 * h, t0 = (tg * TT + tt) * ROWS + in;
            const float4 d4 = *reinterpret_cast<const float4*>(tok.down + tt * ROWS + in);
            const float dn[4] = {d4.x, d4.y, d4.z, d4.w};
            uint32_t to[4] = {t0, t0 + 1, t0 + 2, t0 + 3};
            if constexpr (MOE && !GU) {  // the pairs
                const uint4 p4 = *reinterpret_cast<const uint4*>(tok.pair + in);
                to[0] = p4.x, to[1] = p4.y, to[2] = p4.z, to[3] = p4.w;
            }
            float v[2][4];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    v[q][k] = sum[q][tt][4 * i4 + k];
                    if constexpr (MODE == HH_MMG_S16) v[q][k] += sum[q][tt][4 * i4 + k + 8];
                    v[q][k] *= dn[k];
                }
            float hv[4];
            if (fuse) {
                // four at a time under one branch: each is a long chain
                if (a.act == HH_ACT_GELU_TANH) {
#pragma unroll
                    for (int k = 0; k < 4; k++) hv[k] = hh_act_mul(v[0][k], v[1][k], HH_ACT_GELU_TANH);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++) hv[k] = hh_act_mul(v[0][k], v[1][k], HH_ACT_SILU);
                }
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool live = MOE ? (int)(in + k) < rec.z : to[k] < a.b;
                const size_t at = (size_t)to[k] * a.m;
                if (fuse) {
                    if (live && row[0] < a.m) out[at + row[0]] = hv[k];
                } else if (live) {
                    if (row[0] < a.m) out[at + row[0]] = v[0][k];
                    if (row[1] < a.m) out[(GU ? a.up_stride : 0) + at + row[1]] = v[1][k];
                }
            }
            if (fuse) {
                // over the wave's 32 rows (a token is the same in a lane half)
                // its two 16-lane rows by DPP: LDS shuffles here cost 10 us of a 150 us launch
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    float x = row[0] < a.m ? hh_mmg_mag(hv[k]) : 0.f;
                    x = fmaxf(x, hh_dpp<0xB1>(x));   // quad_perm [1,0,3,2]
                    x = fmaxf(x, hh_dpp<0x4E>(x));   // quad_perm [2,3,0,1]
                    x = fmaxf(x, hh_dpp<0x124>(x));  // row_ror:4
                    x = fmaxf(x, hh_dpp<0x128>(x));  // row_ror:8
                    if ((r & 15u) == 0) wmax[(r >> 4) * (TT * ROWS) + tt * ROWS + in + k] = x;
                }
            }
        }
    }
    if (fuse) {
        hh_mmg_sync();
        if (tid < TT * ROWS) {
            const float* w = reinterpret_cast<const float*>(hh_smem) + tid;
            float v = w[0];
#pragma unroll
            for (int k = 1; k < 8; k++) v = fmaxf(v, w[k * (TT * ROWS)]);
            a.pmax[(size_t)grp * a.ldt + tg * (TT * ROWS) + tid] = v;
        }
    }
}

// Infinities as the largest finite values.
HH_DEV hh_h8 hh_finite(hh_h8 v) {
    const _Float16 m = (_Float16)65504.f;
    const hh_h8 top = {m, m, m, m, m, m, m, m};
    return __builtin_elementwise_max(__builtin_elementwise_min(v, top), -top);
}

template <class F, int MODE, int TT, bool GU, bool MOE = false>
HH_DEV void hh_mmg_body(const hh_mmg_args& a) {
    constexpr int NA = MODE == HH_MMG_H ? 2 : 1;
    constexpr uint32_t CB = 8u * NA * 1024u;            // stage bytes of a (tile, chunk)
    constexpr uint32_t SUMS = F::MINS ? 1024u : 0u;
    constexpr uint32_t BUF = TT * (CB + SUMS);
    constexpr bool WL = F::ROWS_LDS && TT == 1;
    __shared__ hh_mmg_tokens<TT * (MODE == HH_MMG_S16 ? 16 : 32)> tokens;
    extern __shared__ __attribute__((aligned(16))) char hh_smem[];
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t r = lane & 31u, h = lane >> 5;
    // workgroup -> (row group, split, token tiles): the token tiles of one (row group, split) sit
    // on one XCD one after another, so its weights come from memory once and from L2 after
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    uint32_t tg, grp, kci;
    int4 rec{};
    if constexpr (MOE) {
        // each XCD takes a contiguous share of (tile, row group): the tiles of one expert run
        // close together on one L2
        const uint32_t all = (uint32_t)a.trec[0].x * a.groups, share = (all + 7u) / 8u;
        const uint32_t i = xcd * share + slot;
        if (slot >= share || i >= all) return;
        tg = i / a.groups;
        grp = i % a.groups;
        kci = 0;
        rec = a.trec[1 + tg];
    } else {
        const uint32_t unit = slot / a.ttiles * 8u + xcd;
        tg = slot % a.ttiles;
        if (unit >= a.groups * a.kc) return;
        grp = unit / a.kc;
        kci = unit % a.kc;
    }
    const uint32_t c0 = kci * a.cpk, c1 = min(c0 + a.cpk, a.nch);
    const uint32_t nblk = a.n / 32;

    uint32_t row[2];
    const uint8_t* wp[2];
    row[0] = GU ? grp * 128 + wave * 32 + r : grp * 256 + wave * 64 + r;
    row[1] = GU ? row[0] : row[0] + 32;
    const size_t ex = MOE ? (size_t)rec.x * a.expert_stride : 0;
    wp[0] = a.w0 + ex + (size_t)min(row[0], a.m - 1) * a.row_bytes;
    wp[1] = a.w1 + ex + (size_t)min(row[1], a.m - 1) * a.row_bytes;

    if constexpr (F::TABLES) {
        char* tab = hh_smem + 2 * BUF;
        for (uint32_t i = tid; i < F::TAB / 16; i += 256)
            reinterpret_cast<uint4*>(tab)[i] = reinterpret_cast<const uint4*>(F::table())[i];
    }
    const char* const tab = hh_smem + 2 * BUF;

    auto copy = [&](uint32_t ch, auto buf_c) {
        constexpr uint32_t buf = decltype(buf_c)::value;
        const size_t at = F::MINS ? (size_t)(ch >> 1) * (2 * CB + SUMS) + buf * CB : (size_t)ch * CB;
#pragma unroll
        for (uint32_t i = 0; i < TT * CB / 4096u; i++) {
            const uint32_t u = i * 4 + wave, tt = u / (CB / 1024u), o = u % (CB / 1024u);
            const uint8_t* src = a.xs + (size_t)(tg * TT + tt) * a.tile_bytes + at + o * 1024u + lane * 16u;
            char* dst = hh_smem + buf * BUF + tt * (CB + SUMS) + o * 1024u;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
        }
        if constexpr (F::MINS && buf == 1) {
            if (wave < TT) {
                const uint8_t* src = a.xs + (size_t)(tg * TT + wave) * a.tile_bytes + at + CB + lane * 16u;
                char* dst = hh_smem + buf * BUF + wave * (CB + SUMS) + CB;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                                 (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
            }
        }
    };

    hh_mmg_k kk;
    kk.set();
    hh_f16v sum[2][TT], part[2][TT];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) sum[q][tt][i] = part[q][tt][i] = 0.f;

    // one chunk out of LDS buffer `buf`: for formats of 256-column blocks the first or second
    // half of one (splits start at even chunks)
    auto compute = [&](typename F::Raw* raw, auto buf_c) {
        constexpr uint32_t buf = decltype(buf_c)::value;
        constexpr bool open = buf == 0, close = buf == 1;
        if constexpr (F::READY) {
#pragma unroll
            for (int q = 0; q < 2; q++) F::template ready<buf>(raw[q]);
        }
        const char* st = hh_smem + buf * BUF + lane * 16u;
#pragma unroll
        for (int g = 0; g < 4; g++) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                hh_h8 wf[2][F::NB];
#pragma unroll
                for (int q = 0; q < 2; q++) F::template frag<buf>(raw[q], g, s, h, tab, kk, wf[q]);
                const bool fresh = s == 0 && (F::RUN == 8 ? open && g == 0 : g % F::RUN == 0);
                hh_h8 x[NA][TT];
#pragma unroll
                for (int k = 0; k < NA; k++)
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        x[k][tt] = *reinterpret_cast<const hh_h8*>(st + tt * (CB + SUMS) + (g * 2 + s) * (NA * 1024) +
                                                                   k * 1024);
                // what the weights' remainders meet: hi.  In s16 its tile holds lo too, and they are made
                // finite here (8B Q6_K FFN, 16 tokens 80.7 -> 82.3 us; zeros for lo by way of LDS 87.6)
                hh_h8 xrem[TT];
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
                    xrem[tt] = F::NB > 1 && MODE == HH_MMG_S16 ? hh_finite(x[0][tt]) : x[0][tt];
                // hi of every tile, then lo, then the weights' remainders: no product waits for
                // the one before it
#pragma unroll
                for (int k = 0; k < NA + F::NB - 1; k++)
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
#pragma unroll
                        for (int q = 0; q < 2; q++) {
                            hh_f16v c = part[q][tt];
                            if (fresh && k == 0) {
#pragma unroll
                                for (int i = 0; i < 16; i++) c[i] = 0.f;
                            }
                            part[q][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                                k < NA ? x[k][tt] : xrem[tt], wf[q][k < NA ? 0 : 1], c, 0, 0, 0);
                        }
            }
            if (F::RUN < 8 ? g % F::RUN == F::RUN - 1 : close && g == 3) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const float d = F::scale(raw[q], g);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
#pragma unroll
                        for (int i = 0; i < 16; i++) sum[q][tt][i] = fmaf(d, part[q][tt][i], sum[q][tt][i]);
                }
            }
        }
        if constexpr (F::MINS) {
            if (close) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const hh_h8 mf = F::mins(raw[q]);
                    const float dm = -F::min_scale(raw[q]);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) {
                        const hh_h8 xs = *reinterpret_cast<const hh_h8*>(st + tt * (CB + SUMS) + CB);
                        hh_f16v c;
#pragma unroll
                        for (int i = 0; i < 16; i++) c[i] = 0.f;
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs, mf, c, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 16; i++) sum[q][tt][i] = fmaf(dm, c[i], sum[q][tt][i]);
                    }
                }
            }
        }
    };

    typename F::Raw raw[2][2];  // [buffer][row tile]
    constexpr hh_uint_c<0> B0{};
    constexpr hh_uint_c<1> B1{};
    if constexpr (WL) {
        // A superblock of the wave's 64 rows comes as nine runs of whole pieces, about 14 lines
        // each, where twelve loads of a lane's own row took 64 lines each, and is on its way for
        // two chunks instead of one.  Only where a workgroup has one token tile: two workgroups
        // of a CU fit LDS beside each other so.  512-token MoE layer 258 -> 246 us when it was made.
        char* const slot = hh_smem + 2 * BUF + wave * HH_MMG_WSLOT;
        const uint8_t* src[9];  // piece 64 i + lane of the slot: row / 9, 16 bytes each
#pragma unroll
        for (uint32_t i = 0; i < 9; i++) {
            const uint32_t p = 64 * i + lane, rr = p / 9, q = rr / 32;
            const uint32_t at = GU ? grp * 128 + wave * 32 + rr % 32 : grp * 256 + wave * 64 + rr;
            src[i] = (q ? a.w1 : a.w0) + ex + (size_t)min(at, a.m - 1) * a.row_bytes + (c0 >> 1) * 144u + p % 9 * 16u;
        }
        auto rows = [&]() {
#pragma unroll
            for (uint32_t i = 0; i < 9; i++) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src[i],
                                                 (__attribute__((address_space(3))) void*)(slot + i * 1024u), 16, 0, 0);
                src[i] += 144;
            }
        };
        copy(c0, B0);
        rows();
        tokens.set(a, tg, rec, MOE && !GU);
        for (uint32_t ch = c0; ch < c1; ch += 2) {
            hh_mmg_sync();  // chunk ch's tokens and the superblock's rows have landed, buffer 1 is free
#pragma unroll
            for (int q = 0; q < 2; q++) F::load_lds(raw[0][q], raw[1][q], slot + (q * 32 + r) * 144u, h);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slot is read
            asm volatile("" ::: "memory");
            copy(ch + 1, B1);
            const bool more = ch + 2 < c1;
            if (more) rows();
            compute(raw[0], B0);
            asm volatile("" ::: "memory");
            if (more)
                __builtin_amdgcn_s_waitcnt(0x0079);  // vmcnt(9) lgkmcnt(0): the tokens; the rows stay in flight
            else
                __builtin_amdgcn_s_waitcnt(0x0070);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (more) copy(ch + 2, B0);
            compute(raw[1], B1);
        }
        hh_mmg_store<MODE, TT, GU, MOE>(a, sum, row, rec, tg, grp, kci, tokens);
        return;
    }
    copy(c0, B0);
#pragma unroll
    for (int q = 0; q < 2; q++) F::template load<0>(raw[0][q], wp[q], c0, h, nblk);
    tokens.set(a, tg, rec, MOE && !GU);
    for (uint32_t ch = c0; ch < c1; ch += 2) {
        // chunk ch's tokens have landed for every wave, and buffer 1 is free
        hh_mmg_sync();
        const bool two = F::SUPER || ch + 1 < c1;
        if (two) {
            copy(ch + 1, B1);
#pragma unroll
            for (int q = 0; q < 2; q++) F::template load<1>(raw[1][q], wp[q], ch + 1, h, nblk);
        }
        compute(raw[0], B0);
        if (!two) break;
        hh_mmg_sync();
        if (ch + 2 < c1) {
            copy(ch + 2, B0);
#pragma unroll
            for (int q = 0; q < 2; q++) F::template load<0>(raw[0][q], wp[q], ch + 2, h, nblk);
        }
        compute(raw[1], B1);
    }

    hh_mmg_store<MODE, TT, GU, MOE>(a, sum, row, rec, tg, grp, kci, tokens);
}

// ---- Q4_K, one f16 per token element --------------------------------------------------
// For all-Q4_K batches past 64 tokens, whose activations the 17..64-token kernels hold in 8
// bits: here one f16 (11 bits), so half the matrix-core steps of mode h.  128 tokens per
// workgroup; there is no room for a second accumulator per output at two waves per SIMD, so one
// runs through all superblocks in units of the current superblock's d: at each new superblock it
// is multiplied by d_before / d (f32), and the products stay those of exact integers sc q.  In
// the same units the minimum is -(dmin / d) m_j X_j, whose factors enter the bf16 matrix core as
// two bf16 each (f32's range, 16 bits).  8B FFN, 512 tokens: 558 us as 8 passes of 8-bit tokens,
// 269 us here (669 TFLOP/s, matrix cores 45 % busy); error against 64 bits 1.2e-2 -> 5e-4.  A superblock with d = 0 keeps the unit before it and
// zero scales.
typedef __bf16 hh_b8 __attribute__((ext_vector_type(8)));

template <bool GU>
HH_DEV void hh_mmf_body(const hh_mmg_args& a) {
    typedef hh_mmg_q4_k F;
    constexpr int TT = 4;
    constexpr uint32_t CB = 8192u, SUMS = 1024u, BUF = TT * (CB + SUMS);
    extern __shared__ __attribute__((aligned(16))) char hh_smem[];
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t r = lane & 31u, h = lane >> 5;
    __shared__ hh_mmg_tokens<TT * 32> tokens;
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    const uint32_t unit = slot / a.ttiles * 8u + xcd, tg = slot % a.ttiles;  // as hh_mmg_body
    if (unit >= a.groups * a.kc) return;
    const uint32_t grp = unit / a.kc, kci = unit % a.kc;
    const uint32_t c0 = kci * a.cpk, c1 = min(c0 + a.cpk, a.nch);
    uint32_t row[2];
    const uint8_t* wp[2];
    row[0] = GU ? grp * 128 + wave * 32 + r : grp * 256 + wave * 64 + r;
    row[1] = GU ? row[0] : row[0] + 32;
    wp[0] = a.w0 + (size_t)min(row[0], a.m - 1) * a.row_bytes;
    wp[1] = a.w1 + (size_t)min(row[1], a.m - 1) * a.row_bytes;

    auto copy = [&](uint32_t ch, auto buf_c) {
        constexpr uint32_t buf = decltype(buf_c)::value;
        const size_t at = (size_t)(ch >> 1) * (2 * CB + SUMS) + buf * CB;
        // a wave copies one tile: 8 KB, and in the second half the superblock's sums
        const uint8_t* src = a.xs + (size_t)(tg * TT + wave) * a.tile_bytes + at + lane * 16u;
        char* dst = hh_smem + buf * BUF + wave * (CB + SUMS);
#pragma unroll
        for (uint32_t i = 0; i < (buf ? 9u : 8u); i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + i * 1024u),
                                             (__attribute__((address_space(3))) void*)(dst + i * 1024u), 16, 0, 0);
    };
    hh_mmg_k kk;
    kk.set();
    hh_f16v acc[2][TT];
    float u[2] = {1.f, 1.f};  // the accumulators' unit
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[q][tt][i] = 0.f;

    // a new superblock: its unit, and zero scales where d is zero
    uint32_t zero[2];  // mask of the scales: 0 where d is
    auto open = [&](const typename F::Raw* raw) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const float d = F::scale(raw[q], 0);
            const float n = d != 0.f ? d : u[q];
            zero[q] = d != 0.f ? 0xFFFFFFFFu : 0u;
            const float f = u[q] / n;
            u[q] = n;
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[q][tt][i] *= f;
        }
    };
    auto compute = [&](typename F::Raw* raw, auto buf_c) {
        constexpr uint32_t buf = decltype(buf_c)::value;
        const char* st = hh_smem + buf * BUF + lane * 16u;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            F::ready<buf>(raw[q]);
            raw[q].sch &= zero[q];
        }
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                hh_h8 wf[2], x[TT];
#pragma unroll
                for (int q = 0; q < 2; q++) F::template frag<buf>(raw[q], g, s, h, nullptr, kk, &wf[q]);
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
                    x[tt] = *reinterpret_cast<const hh_h8*>(st + tt * (CB + SUMS) + (g * 2 + s) * 1024);
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
#pragma unroll
                    for (int q = 0; q < 2; q++)
                        acc[q][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[tt], wf[q], acc[q][tt], 0, 0, 0);
            }
        if constexpr (buf == 1) {
            // the minima, in units of u
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const hh_h8 m = F::mins(raw[q]);
                const float rho = -F::min_scale(raw[q]) / u[q];
                union {
                    uint16_t b[8];
                    hh_b8 v;
                } hi, lo;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float f = rho * (float)m[j];
                    const uint32_t t = __float_as_uint(f) >> 16;  // truncated: the rest is exact
                    hi.b[j] = (uint16_t)t;
                    lo.b[j] = (uint16_t)(__float_as_uint(f - __uint_as_float(t << 16)) >> 16);
                }
#pragma unroll
                for (int tt = 0; tt < TT; tt++) {
                    const hh_b8 xs = *reinterpret_cast<const hh_b8*>(st + tt * (CB + SUMS) + CB);
                    acc[q][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, hi.v, acc[q][tt], 0, 0, 0);
                    acc[q][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xs, lo.v, acc[q][tt], 0, 0, 0);
                }
            }
        }
    };
    typename F::Raw raw[2][2];  // [half][row tile]
    constexpr hh_uint_c<0> B0{};
    constexpr hh_uint_c<1> B1{};
    copy(c0, B0);
#pragma unroll
    for (int q = 0; q < 2; q++) F::load<0>(raw[0][q], wp[q], c0, h, 0);
    tokens.set(a, tg, int4{}, false);
    for (uint32_t ch = c0; ch < c1; ch += 2) {
        hh_mmg_sync();
        copy(ch + 1, B1);
#pragma unroll
        for (int q = 0; q < 2; q++) F::load<1>(raw[1][q], wp[q], ch + 1, h, 0);
        open(raw[0]);
        compute(raw[0], B0);
        hh_mmg_sync();
        if (ch + 2 < c1) {
            copy(ch + 2, B0);
#pragma unroll
            for (int q = 0; q < 2; q++) F::load<0>(raw[0][q], wp[q], ch + 2, h, 0);
        }
        compute(raw[1], B1);
    }
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[q][tt][i] *= u[q];
    hh_mmg_store<HH_MMG_F, TT, GU, false>(a, acc, row, int4{}, tg, grp, kci, tokens);
}

struct hh_mmg_sum_args {
    const float* part;     // [kc][b][m] (gate/up: gate's, then up's at up_stride)
    float* y;              // [b][m]
    uint64_t stride;       // floats between two splits
    uint64_t up_stride;
    float* pmax;           // sum_act: [256-row group][ldt] largest magnitudes of each token's h
    uint32_t m;
    uint32_t kc;
    int32_t act;
    uint32_t ldt;
};
// s += v with c, what the additions have lost so far (Kahan): 4096 columns of Q8_0 in up to 32 splits,
// 8 tokens, 1.28e-7 -> 7.8e-8 against 64 bits (one token 1.1e-7), in the same time.
HH_DEV void hh_mmg_add(float& s, float& c, float v) {
    const float y = v + c, t = s + y;
    c = fabsf(t) < __builtin_inff() ? y - (t - s) : 0.f;
    s = t;
}
// grid.y: tokens
extern "C" __global__ void __launch_bounds__(256) hh_mmg_sum(const hh_mmg_sum_args a) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= a.m) return;
    const uint64_t i = (uint64_t)blockIdx.y * a.m + r;
    float s = 0.f, c = 0.f;
#pragma unroll 4
    for (uint32_t k = 0; k < a.kc; k++) hh_mmg_add(s, c, a.part[k * a.stride + i]);
    a.y[i] = s;
}
extern "C" __global__ void __launch_bounds__(256) hh_mmg_sum_act(const hh_mmg_sum_args a) {
    const uint32_t r = blockIdx.x * 256 + threadIdx.x;
    const uint64_t i = (uint64_t)blockIdx.y * a.m + min(r, a.m - 1);
    float g = 0.f, u = 0.f, gc = 0.f, uc = 0.f;
#pragma unroll 4
    for (uint32_t k = 0; k < a.kc; k++) {
        hh_mmg_add(g, gc, a.part[k * a.stride + i]);
        hh_mmg_add(u, uc, a.part[k * a.stride + a.up_stride + i]);
    }
    const float h = hh_act_mul(g, u, a.act);
    if (r < a.m) a.y[i] = h;
    __shared__ float red[4];
    const float v = hh_wave_max(r < a.m ? hh_mmg_mag(h) : 0.f);
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        a.pmax[(size_t)blockIdx.x * a.ldt + blockIdx.y] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

#define HH_MMG_KERNEL(FMT, NAME, MODE, TT, WPE)                                                                  \
    extern "C" __global__ void __launch_bounds__(256, WPE) hh_mmg_##FMT##_##NAME(const hh_mmg_args a) {          \
        hh_mmg_body<hh_mmg_##FMT, MODE, TT, false>(a);                                                          \
    }                                                                                                           \
    extern "C" __global__ void __launch_bounds__(256, WPE) hh_mmg_##FMT##_##NAME##_gu(const hh_mmg_args a) {     \
        hh_mmg_body<hh_mmg_##FMT, MODE, TT, true>(a);                                                           \
    }
#define HH_MMG_ONE_TILE(FMT, WPE)             \
    HH_MMG_KERNEL(FMT, s16, HH_MMG_S16, 1, WPE) \
    HH_MMG_KERNEL(FMT, h1, HH_MMG_H, 1, WPE)
#define HH_MMG_FORMAT(FMT, WPE) \
    HH_MMG_ONE_TILE(FMT, WPE)   \
    HH_MMG_KERNEL(FMT, h2, HH_MMG_H, 2, 2)
HH_MMG_FORMAT(q4_0, 2)
HH_MMG_FORMAT(q8_0, 2)
HH_MMG_FORMAT(q4_k, 2)
HH_MMG_FORMAT(q6_k, 3)
HH_MMG_FORMAT(iq2_xxs, 3)
HH_MMG_FORMAT(iq3_xxs, 3)
HH_MMG_ONE_TILE(q6_k_fine, 2)  // (two tiles spill)
HH_MMG_FORMAT(iq2_xxs_fine, 2)
HH_MMG_FORMAT(iq3_xxs_fine, 2)
#define HH_MMG_MOE(NAME, MODE, WPE)                                                                               \
    extern "C" __global__ void __launch_bounds__(256, WPE) hh_mmg_moe_##NAME(const hh_mmg_args a) {              \
        hh_mmg_body<hh_mmg_q4_k, MODE, 1, false, true>(a);                                                      \
    }                                                                                                           \
    extern "C" __global__ void __launch_bounds__(256, WPE) hh_mmg_moe_##NAME##_gu(const hh_mmg_args a) {         \
        hh_mmg_body<hh_mmg_q4_k, MODE, 1, true, true>(a);                                                       \
    }
HH_MMG_MOE(s16, HH_MMG_S16, 2)
HH_MMG_MOE(h1, HH_MMG_H, 2)
extern "C" __global__ void __launch_bounds__(256, 2) hh_mmg_q4_k_f4(const hh_mmg_args a) { hh_mmf_body<false>(a); }
extern "C" __global__ void __launch_bounds__(256, 2) hh_mmg_q4_k_f4_gu(const hh_mmg_args a) { hh_mmf_body<true>(a); }
