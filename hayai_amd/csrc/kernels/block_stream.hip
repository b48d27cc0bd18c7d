// One token through large Q8_0 / Q4_0 matrices at f32 accuracy (gfx950):
//   hh_bst_<fmt>_<pair|wide>      y = W . x (+ residual)  (ggml_gemv_*, compute.rs:281-461)
//   hh_bst_<fmt>_<pair|wide>_gu   h = act(W_gate . x) * (W_up . x), x optionally RMSNorm'ed first
//                     (stream_infer.rs:3752-3806, hybrid_infer.rs:883-936)
// (Compiled after q4k.hip: hh_dpp.)
//
// What bounds it: the weight stream.  The blocks are 34 and 18 bytes, and a lane that loads its
// own block (gemv.hip) asks for 64 pieces at that stride, misaligned: the address units, not HBM,
// set the pace (8B Q8_0 gate/up 41 us, 3.0 TB/s, here 28 us; down 30 us, 2.1 TB/s, here 16 us; a
// block with RMSNorm and residual 78 -> 45 us, Q4_0 60 -> 39 us).  Here a wave copies a
// whole row slice, 16 bytes per lane and contiguous, into its own LDS ring by global->LDS DMA
// (no registers held, D rows in flight), and each lane then takes its two blocks from LDS: the
// dwords that cover them and one v_alignbit each.  Rows start at any even address: a copy begins
// at the 16 bytes that hold the slice's first byte, and the matrix's last bytes, which whole 16-byte
// pieces would pass, are put in by hand.  Arithmetic as gemv.hip: codes as f32, FMA
// with x held in registers, one scale per block, f32 sums.
//
// Work split: one workgroup per CU, 8 compute waves in teams of W per row, workgroup w taking
// rows w, w + G, ... so that the grid sweeps the matrix.  A lane holds two blocks per item.
// Wide: they are blocks lane and lane + 64 of one row's slice (slices of 65..128 blocks).  Pair:
// the same block of two rows, gate and up of one row or two rows of a GEMV (slices of at most 64
// blocks: with the second block idle instead, a 2048-column row cost a 4096-column one's time).
// Four more waves bring x into LDS (and normalize it) while the first rows are on their way:
// loads that a compute wave issued after its DMA would wait for it, in order.

struct hh_bst_args {
    const uint8_t* w0;    // GEMV: W; gate/up: W_gate (2-byte aligned)
    const uint8_t* w1;    // gate/up: W_up
    const float* x;       // [n]
    const float* norm;    // gate/up: RMSNorm weight or null (16-byte aligned, as x)
    const float* res;     // GEMV: residual to add or null
    float* y;             // [m]
    uint64_t row_bytes;
    uint32_t m, n;
    uint32_t waves;       // W: waves per row (1, 2, 4, 8)
    uint32_t sb;          // blocks per slice (pair: at most 64, wide: 128)
    uint32_t depth;       // D: items in flight per wave (2..4)
    uint32_t pad;
    float eps;
    int32_t act;
};

#define HH_BST_XSTRIDE 36u  // dwords per 32-element block of x in LDS: 16-byte reads without conflicts

typedef _Float16 hh_bst_h2 __attribute__((ext_vector_type(2)));

// A select, and no branch around the product (8B Q4_0 block 79 -> 77 us).
HH_DEV float hh_bst_live(float v, bool live) {
    asm volatile("" : "+v"(v));
    return live ? v : 0.f;
}

struct hh_bst_q8_0_t {
    static constexpr uint32_t BB = 34, DW = 9;
    // block bytes p (dword 0 holds d and codes 0, 1 after the shift): d * sum(q x), or 0 for a lane
    // past the slice (whose x is its last block's, infinite perhaps)
    HH_DEV static float dot(const uint32_t (&v)[DW], const float* xr, bool live) {
        // four chains of 8: with two of 16 a 512-column product was 1.0e-7 from 64 bits, here 0.91e-7
        // (two 8B blocks 2.07e-7, 1.97e-7; the time is the same)
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const uint32_t byte = 2 + i;
            const float q = (float)((int32_t)(v[byte / 4] << (24 - 8 * (byte % 4))) >> 24);
            acc[i / 4 % 4] = fmaf(q, xr[i], acc[i / 4 % 4]);
        }
        return hh_bst_live(hh_f16(v[0] & 0xFFFFu) * ((acc[0] + acc[1]) + (acc[2] + acc[3])), live);
    }
};
struct hh_bst_q4_0_t {
    static constexpr uint32_t BB = 18, DW = 5;
    // q - 8 as exact f16 pairs (1024 + q less 1032; 1024 + 16 q over 16 less 72), which
    // v_fma_mix_f32 takes as they are.  sum(q x) - 8 sum(x) instead is 10 % faster and cancels: 10
    // times the error against 64 bits and more (two 8B blocks 69 us, 3.5e-6; so 78 us, 1e-7).
    HH_DEV static float dot(const uint32_t (&v)[DW], const float* xr, bool live) {
        float al = 0.f, ah = 0.f;
        const hh_bst_h2 z = {(_Float16)1032.f, (_Float16)1032.f};
        const hh_bst_h2 m = {(_Float16)0.0625f, (_Float16)0.0625f}, o = {(_Float16)-72.f, (_Float16)-72.f};
        auto low = [&](uint32_t w) { return __builtin_bit_cast(hh_bst_h2, (w & 0x000F000Fu) | 0x64006400u) - z; };
        auto high = [&](uint32_t w) {
            return __builtin_elementwise_fma(__builtin_bit_cast(hh_bst_h2, (w & 0x00F000F0u) | 0x64006400u), m, o);
        };
#pragma unroll
        for (int j = 0; j < 5; j++) {
            // dword j: codes 4 j - 2 .. 4 j + 1 (dword 0: d below codes 0, 1; dword 4: 14, 15)
            const hh_bst_h2 l = low(v[j]), l8 = low(v[j] >> 8), g = high(v[j]), g8 = high(v[j] >> 8);
            const int c = 4 * j - 2;
            if (j > 0) {
                al = fmaf((float)l[0], xr[c], al), al = fmaf((float)l8[0], xr[c + 1], al);
                ah = fmaf((float)g[0], xr[16 + c], ah), ah = fmaf((float)g8[0], xr[17 + c], ah);
            }
            if (j < 4) {
                al = fmaf((float)l[1], xr[c + 2], al), al = fmaf((float)l8[1], xr[c + 3], al);
                ah = fmaf((float)g[1], xr[18 + c], ah), ah = fmaf((float)g8[1], xr[19 + c], ah);
            }
        }
        return hh_bst_live(hh_f16(v[0] & 0xFFFFu) * (al + ah), live);
    }
};

// At most n vector memory operations of this wave still outstanding.
template <uint32_t N>
HH_DEV void hh_bst_wait() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
    asm volatile("" ::: "memory");
}
HH_DEV void hh_bst_lds_wait() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // LDS only: the DMA stays in flight
    asm volatile("" ::: "memory");
}

template <class F, bool GU, bool PAIR>
HH_DEV void hh_bst_body(const hh_bst_args& a) {
    extern __shared__ __attribute__((aligned(16))) char hh_smem[];
    __shared__ float ssq[4];
    const uint32_t tid = threadIdx.x, lane = tid % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t G = gridDim.x, w = blockIdx.x, W = a.waves;
    const uint32_t nblk = a.n / 32;
    const uint32_t S = (a.sb * F::BB + 45u) & ~15u;  // LDS bytes of a slice: its cover and a read past it
    constexpr uint32_t NR = PAIR ? 2 : 1;           // slices per item
    constexpr uint32_t K = ((PAIR ? 64 : 128) * F::BB + 30u + 1023u) / 1024u;  // DMA operations per slice
    constexpr uint32_t NM = GU ? 2 : 1;             // matrices
    constexpr uint32_t RI = GU || !PAIR ? 1 : 2;    // rows per item
    float* const xs = reinterpret_cast<float*>(hh_smem + 8u * a.depth * NR * S);
    float* const sums = xs + nblk * HH_BST_XSTRIDE;            // [row][matrix][W]
    const uint32_t nr = w < a.m ? (a.m - w + G - 1) / G : 0;  // this workgroup's rows

    if (wave >= 8) {
        // x -> LDS, 4 elements per lane and step
        float ss = 0.f;
        const float4* x4 = reinterpret_cast<const float4*>(a.x);
#pragma unroll 8
        for (uint32_t i = tid - 512u; i < a.n / 4; i += 256) {
            const float4 v = x4[i];
            *reinterpret_cast<float4*>(xs + (i / 8) * HH_BST_XSTRIDE + (i % 8) * 4) = v;
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
        if (GU && a.norm) {
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) ss += __shfl_xor(ss, o, 64);
            if (lane == 0) ssq[wave - 8] = ss;
            __syncthreads();
            const float inv = 1.0f / sqrtf(((ssq[0] + ssq[1]) + (ssq[2] + ssq[3])) / (float)a.n + a.eps);
            const float4* n4 = reinterpret_cast<const float4*>(a.norm);
#pragma unroll 8
            for (uint32_t i = tid - 512u; i < a.n / 4; i += 256) {
                float4* p = reinterpret_cast<float4*>(xs + (i / 8) * HH_BST_XSTRIDE + (i % 8) * 4);
                const float4 v = *p, g = n4[i];
                *p = make_float4((v.x * inv) * g.x, (v.y * inv) * g.y, (v.z * inv) * g.z, (v.w * inv) * g.w);
            }
        }
        __syncthreads();
    } else {
        const uint32_t T = 8u / W, team = wave / W, slice = wave % W;
        const uint32_t b0 = slice * a.sb, nb = b0 < nblk ? min(a.sb, nblk - b0) : 0u;
        // an item: gate and up of one row (or one of them, wide), or RI rows of the team's
        const uint32_t rows = team < nr ? (nr - team + T - 1) / T : 0;
        const uint32_t items = PAIR ? (rows + RI - 1) / RI : rows * NM;
        const uint32_t D = a.depth;
        char* const ring = hh_smem + wave * D * NR * S;
        const size_t b0_bytes = (size_t)(nb ? b0 : 0u) * F::BB;
        auto row_of = [&](uint32_t k, uint32_t j) {  // index among the workgroup's rows
            if constexpr (PAIR) return min(team + (k * RI + (RI == 2 ? j : 0u)) * T, nr - 1u);
            return team + k / NM * T;
        };
        // slice j of item k: the 16-byte piece that holds its first byte, how far in that is, the
        // whole pieces that cover it, and the bytes of the matrix's end that they leave out
        struct Cover {
            const uint8_t* base;
            uint32_t shift, chunks, left;
        };
        auto cover = [&](uint32_t k, uint32_t j) {
            const bool up = GU && (PAIR ? j == 1 : (k & 1u) != 0);
            const uint8_t* m0 = up ? a.w1 : a.w0;
            const uint8_t* src = m0 + (size_t)(w + row_of(k, j) * G) * a.row_bytes + b0_bytes;
            Cover c;
            c.shift = (uint32_t)(uintptr_t)src & 15u;
            c.base = src - c.shift;
            const size_t rest = (size_t)(m0 + (size_t)a.m * a.row_bytes - c.base);
            c.chunks = (c.shift + max(nb, 1u) * F::BB + 15u) / 16u;
            c.left = 0;
            if (rest < (size_t)c.chunks * 16u) {
                c.chunks = (uint32_t)rest / 16u;
                c.left = (uint32_t)rest & 15u;
            }
            return c;
        };
        // every item is NR * K operations, so that the waits can count them: lane 0 takes part in
        // each, and those past the slice repeat lane 0's part of the last
        auto issue = [&](uint32_t k, char* slot) {
#pragma unroll
            for (uint32_t j = 0; j < NR; j++) {
                const Cover c = cover(k, j);
                const uint32_t last = (c.chunks - 1u) / 64u;
#pragma unroll
                for (uint32_t i = 0; i < K; i++) {
                    const uint32_t p = min(i, last) * 64u + lane;
                    if ((i <= last && p < c.chunks) || lane == 0)
                        __builtin_amdgcn_global_load_lds(
                            (const __attribute__((address_space(1))) void*)(c.base + p * 16u),
                            (__attribute__((address_space(3))) void*)(slot + j * S + min(i, last) * 1024u), 16, 0, 0);
                }
            }
        };
        const uint32_t first = min(D, items);
        for (uint32_t k = 0; k < first; k++) issue(k, ring + k * NR * S);
        if (GU && a.norm) {
            hh_bst_lds_wait();
            __builtin_amdgcn_s_barrier();
        }
        hh_bst_lds_wait();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // the lane's blocks (past the slice: its last, which counts as 0)
        constexpr int NX = PAIR ? 1 : 2;
        float xr[NX][32];
        bool live[NX];
        uint32_t at[NX];  // of the block in its slice
#pragma unroll
        for (uint32_t j = 0; j < NX; j++) {
            const uint32_t b = lane + 64u * j, c = min(b, max(nb, 1u) - 1u);
            live[j] = b < nb;
            const float4* p = reinterpret_cast<const float4*>(xs + (nb ? b0 + c : 0u) * HH_BST_XSTRIDE);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4 v = p[i];
                xr[j][4 * i] = v.x, xr[j][4 * i + 1] = v.y, xr[j][4 * i + 2] = v.z, xr[j][4 * i + 3] = v.w;
            }
            at[j] = c * F::BB;
        }
        char* slot = ring;
        char* const end = ring + D * NR * S;
        for (uint32_t k = 0; k < items; k++) {
            // the items after this one that are on their way
            const uint32_t newer = min(D - 1u, items - 1u - k);
            if (newer == 3)
                hh_bst_wait<3 * NR * K>();
            else if (newer == 2)
                hh_bst_wait<2 * NR * K>();
            else if (newer == 1)
                hh_bst_wait<NR * K>();
            else
                hh_bst_wait<0>();
            uint32_t v[2][F::DW];
#pragma unroll
            for (uint32_t j = 0; j < 2; j++) {
                const Cover c = cover(k, PAIR ? j : 0u);
                char* const in = slot + (PAIR ? j * S : 0u);
                if (c.left) {  // the matrix's last row
                    if (lane < c.left / 2u)
                        *reinterpret_cast<uint16_t*>(in + c.chunks * 16u + lane * 2u) =
                            (uint16_t)hh_ld_u16(c.base + c.chunks * 16u + lane * 2u);
                    hh_bst_lds_wait();
                }
                const uint32_t o = at[PAIR ? 0 : j] + c.shift;
                const uint32_t* q = reinterpret_cast<const uint32_t*>(in + (o & ~3u));
                const uint32_t sh = (o & 2u) * 8u;  // 0 or 16 bits
                uint32_t raw[F::DW];
#pragma unroll
                for (uint32_t i = 0; i < F::DW; i++) raw[i] = q[i];
#pragma unroll
                for (uint32_t i = 0; i < F::DW; i++)
                    v[j][i] = __builtin_amdgcn_alignbit(i + 1 < F::DW ? raw[i + 1] : 0u, raw[i], sh);
            }
            hh_bst_lds_wait();  // the slot's reads are done before it is filled again
            if (k + D < items) issue(k + D, slot);
            slot = slot + NR * S == end ? ring : slot + NR * S;
            float s[2] = {F::dot(v[0], xr[0], live[0]), F::dot(v[1], xr[NX - 1], live[NX - 1])};
            if constexpr (!PAIR) s[0] += s[1];
#pragma unroll
            for (uint32_t j = 0; j < NR; j++) {
                s[j] += hh_dpp<0xB1>(s[j]);
                s[j] += hh_dpp<0x4E>(s[j]);
                s[j] += hh_dpp<0x124>(s[j]);
                s[j] += hh_dpp<0x128>(s[j]);
                s[j] += hh_dpp<0x142, 0xA>(s[j]);
                s[j] += hh_dpp<0x143, 0xC>(s[j]);
                const uint32_t mat = !GU ? 0u : PAIR ? j : (k & 1u);
                if (lane == 63) sums[(row_of(k, j) * NM + mat) * W + slice] = s[j];
            }
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < nr; i += blockDim.x) {
        float v[NM];
#pragma unroll
        for (uint32_t q = 0; q < NM; q++) {
            v[q] = 0.f;
            for (uint32_t k = 0; k < W; k++) v[q] += sums[(i * NM + q) * W + k];
        }
        const uint32_t row = w + i * G;
        if constexpr (GU)
            a.y[row] = hh_act_mul(v[0], v[1], a.act);
        else
            a.y[row] = a.res ? a.res[row] + v[0] : v[0];
    }
}

#define HH_BST_KERNEL(FMT, NAME, GU, PAIR)                                                              \
    extern "C" __global__ void __launch_bounds__(768) hh_bst_##FMT##_##NAME(const hh_bst_args a) {      \
        hh_bst_body<hh_bst_##FMT##_t, GU, PAIR>(a);                                                     \
    }
#define HH_BST_FORMAT(FMT)                        \
    HH_BST_KERNEL(FMT, pair, false, true)         \
    HH_BST_KERNEL(FMT, wide, false, false)        \
    HH_BST_KERNEL(FMT, pair_gu, true, true)       \
    HH_BST_KERNEL(FMT, wide_gu, true, false)
HH_BST_FORMAT(q8_0)
HH_BST_FORMAT(q4_0)
