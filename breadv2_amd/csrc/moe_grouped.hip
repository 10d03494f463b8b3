// moe_grouped.hip — the multi-token MoE path (batched decode, speculative
// verify, prefill chunks): tokens bucketed by expert, the expert products as
// grouped GEMMs on the gfx950 matrix cores with the K-quant weights unpacked
// in registers, and a combine in the reference order.
//
// The reference has no multi-token MoE: prefill runs token by token
// (main.cu:615-639) and speculative verify is sequential
// (main_speculative.cu:477-497).  Per token the result is the MoE block of
// one_layer_forward (one_layer.cu:1800-1986; CPU form 1413-1471).
//
// Numerics.  MFMA operands are fp16 with fp32 accumulation, and every
// product is exact.  A weight enters as its integer part: sc * q (Q4_K,
// <= 63 * 15) or sc * (q - 32) (Q6_K, |.| <= 4096: exact up to 2048 and for
// even values), times a power of two.  Activations are two fp16 terms (hi +
// lo, 23 significant bits at most) after a power-of-two row scale into
// [2^13, 2^14) (exact, undone on the fp32 result).  The superblock scale d,
// and for Q4_K the min term dmin * sum_j m_j * (sum of x over sub-block j),
// are applied to the fp32 sums.
// Layers of the reference GPU path's types round the odd Q6_K integers above
// 2048 to even (7e-5 of a layer's output).  Layers of other types (X), which
// run in fp32 at fewer tokens, carry that rest in a second operand and scale
// the lo terms (LO_EXP): their inputs are off by 2^-23 at most, and with exact
// products the sums come out as near to 64-bit arithmetic as the per-token
// kernels' (27 tokens of hidden 2048, all Q4_K: 5.5e-7 both, all Q6_K: 2.5e-7
// both).
// A row that holds an infinity has NaN terms, so where fp32 sums would give
// some outputs of that token as infinities they are NaN.
//
// Kernels per layer, stream-ordered:
//   k_route_seq   router logits in the reference's sequential order
//                 (route.hip: one lane a token, one or two router rows a wave)
//   k_mt_topk_xprep  one workgroup per token: softmax / top-k /
//                 renormalisation with the host's arithmetic (routing
//                 bit-identical to the reference's), and the activation
//                 preparation: row scale, hi/lo fp16 activations in MFMA
//                 operand order, sub-block sums, shared-gate logit
//   k_mt_bucket   one workgroup: expert histogram, token lists by expert,
//                 tiles of 32 pairs
//   k_gateup_gg   per (tile, 128 rows): gate and up GEMMs and SwiGLU
//   k_down_gg     per (tile, 512 rows): the tile's SwiGLU rows split into hi/lo
//                 fp16 with a row scale, then the down GEMM
//   k_mt_combine  per token: shared expert, then routed experts in rank order
// The shared expert is expert index E with every token, so both GEMMs treat
// it like a routed expert with its own weights.
#include <float.h>

#include "bread_internal.h"
#include "bread_device.h"
#include "quant_dot.h"
#include "route_dev.h"

namespace {

constexpr int MT = 32;           // (token, expert) pairs per tile
constexpr int MAX_INTER = 512;   // largest intermediate size of this path
constexpr int NXCD = 8;          // L2 domains; workgroup L runs on XCD L % 8
constexpr int GG_WAVES = 4;
constexpr int GG_THREADS = GG_WAVES * WAVE;
constexpr int GU_ROWS = 32 * GG_WAVES;       // gate and up rows of a gate/up workgroup
constexpr int DN_WAVES = 8, DN_BLOCKS = 2;   // 32-row blocks of a wave of the down kernel
constexpr int DN_ROWS = 32 * DN_WAVES * DN_BLOCKS;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct MtTile {
    int e;   // expert (E = the shared expert)
    int p0;  // first pair in the sorted pair list
    int nr;  // pairs in the tile (1..MT)
    int pad;
};

__device__ __forceinline__ uint32_t comp(const uint4 &q, int i)
{
    return i == 0 ? q.x : (i == 1 ? q.y : (i == 2 ? q.z : q.w));
}

// Exponent e with max_abs * 2^-e in [2^13, 2^14); 0 for an all-zero or
// non-finite row.
__device__ __forceinline__ int row_exp(float max_abs)
{
    int e = 0;
    if (max_abs > 0.f && max_abs <= FLT_MAX) {
        (void)frexpf(max_abs, &e);
        e -= 14;
    }
    return e;
}

// The lo terms of layers of other types than the reference GPU path's (X
// below) are held times 2^LO_EXP.  A lo term then has its 11 bits wherever the
// hi term has, so a value keeps 23 bits down to 2^-24 of its row's largest;
// unscaled, it runs into the end of fp16's subnormals from 2^-14 on, and a
// channel 10^5 or 10^7 times the others left the rest of a row errors of
// 1.5e-7 or 1.6e-5.  The weights that meet lo terms are times 2^-LO_EXP: 2^10
// is the most at which a Q4_K one (an integer times 2^-14) is an fp16 number.
// The lo terms of the sub-block sums meet integers alone and are held times
// 2^SUM_LO_EXP, the most that fits fp16.  The second operand costs 3 %: 27
// tokens of an all-Q4_K layer 141.5 -> 146 us on MI355X.
constexpr int LO_EXP = 10, SUM_LO_EXP = 13;

// v (already scaled) as hi + lo / ls fp16: hi = fp16(v), lo = fp16((v - hi) ls).
__device__ __forceinline__ void split2(float a, float b, float ls, uint32_t &hi, uint32_t &lo)
{
    const _Float16 ha = (_Float16)a, hb = (_Float16)b;
    const _Float16 la = (_Float16)((a - (float)ha) * ls), lb = (_Float16)((b - (float)hb) * ls);
    hi = (uint32_t)__builtin_bit_cast(uint16_t, ha) | ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
    lo = (uint32_t)__builtin_bit_cast(uint16_t, la) | ((uint32_t)__builtin_bit_cast(uint16_t, lb) << 16);
}

// ---------------------------------------------------------------------------
// Operand order.  v_mfma_f32_32x32x16_f16 with 32 tokens as the M side and 32
// weight rows as the N side: lane (r = lane % 32, g = lane / 32) holds weight
// row r and token r, eight K elements of the step.  K is relabelled so that
// one order serves Q4_K and Q6_K and a lane's bytes are contiguous: lane half
// g takes the elements 128 g .. 128 g + 127 of a superblock, and step s = 8 pp
// + k of 16 takes of those
//   b + {0, 2, 1, 3} and b + 32 + {0, 2, 1, 3},  b = 128 g + 64 pp + 4 k.
// Q4_K: the two quads are the low and high nibbles of one qs dword
// (dequant_q4k_cpu.c:111-121); Q6_K: a nibble each of one dword of the two ql
// ranges with two bits each of one qh dword (dequant_q4k_cpu.c:155-170).
// {0, 2, 1, 3}: a mask with 16-bit period picks bytes 0 and 2 of a dword, the
// same mask 8 bits on bytes 1 and 3.  Unit u = 2 s + g of a superblock holds a
// lane's eight elements of step s.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int unit_base(int u)
{
    return 128 * (u & 1) + 64 * (u >> 4) + 4 * ((u >> 1) & 7);
}

// Eight elements in operand order (a: b .. b + 3, c: b + 32 .. b + 35),
// scaled by 2^-e and split.
__device__ __forceinline__ void split_unit(const float4 &a, const float4 &c, int e, float ls, uint4 &hi, uint4 &lo)
{
    split2(ldexpf(a.x, -e), ldexpf(a.z, -e), ls, hi.x, lo.x);
    split2(ldexpf(a.y, -e), ldexpf(a.w, -e), ls, hi.y, lo.y);
    split2(ldexpf(c.x, -e), ldexpf(c.z, -e), ls, hi.z, lo.z);
    split2(ldexpf(c.y, -e), ldexpf(c.w, -e), ls, hi.w, lo.w);
}

// The same for eight elements already in operand order.
__device__ __forceinline__ void split_unit_op(const float4 &a, const float4 &c, int e, float ls, uint4 &hi, uint4 &lo)
{
    split2(ldexpf(a.x, -e), ldexpf(a.y, -e), ls, hi.x, lo.x);
    split2(ldexpf(a.z, -e), ldexpf(a.w, -e), ls, hi.y, lo.y);
    split2(ldexpf(c.x, -e), ldexpf(c.y, -e), ls, hi.z, lo.z);
    split2(ldexpf(c.z, -e), ldexpf(c.w, -e), ls, hi.w, lo.w);
}

// ---------------------------------------------------------------------------
// Activation preparation: row scale, the row's units (hi then lo per
// superblock, [T][H / 256][2][32]) and the sums over the 32-element
// sub-blocks times 2^-5 (hi and lo unit of eight, [T][H / 256][2]) that the
// Q4_K min term multiplies; the shared-gate logit.
// ---------------------------------------------------------------------------

__device__ __forceinline__ float xor_add(float v, int m)
{
    return v + __shfl_xor(v, m);
}

__device__ __forceinline__ void mt_xprep(int t, const float *__restrict__ x, const uint16_t *__restrict__ shg, int H,
                                         bool scaled_lo, uint4 *__restrict__ xop, uint4 *__restrict__ xsum,
                                         int *__restrict__ xexp, float *__restrict__ gsh)
{
    __shared__ float smax[4], sdot[4];
    const float ls = scaled_lo ? (float)(1 << LO_EXP) : 1.f, ls_sum = scaled_lo ? (float)(1 << SUM_LO_EXP) : 1.f;
    const float *xt = x + (size_t)t * H;
    float mx = 0.f, dot = 0.f;
    for (int i = 4 * (int)threadIdx.x; i < H; i += 1024) {
        const float4 v = *reinterpret_cast<const float4 *>(xt + i);
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        if (shg) {
            const uint2 g = *reinterpret_cast<const uint2 *>(shg + i);
            dot = fmaf(h2f(g.x), v.x, dot);
            dot = fmaf(h2f(g.x >> 16), v.y, dot);
            dot = fmaf(h2f(g.y), v.z, dot);
            dot = fmaf(h2f(g.y >> 16), v.w, dot);
        }
    }
    mx = wave_max(mx);
    dot = wave_sum(dot);
    if (lane_id() == 0) {
        smax[threadIdx.x / WAVE] = mx;
        sdot[threadIdx.x / WAVE] = dot;
    }
    __syncthreads();
    const int e = row_exp(fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3])));
    if (threadIdx.x == 0) {
        xexp[t] = e;
        if (gsh) gsh[t] = shg ? (sdot[0] + sdot[1]) + (sdot[2] + sdot[3]) : 0.f;
    }
    // one unit a thread and pass; H / 8 is a multiple of 32, so the 32 lanes
    // of a superblock are active together
    const int nu = H / 8;
    for (int u = threadIdx.x; u < nu; u += 256) {
        const int sb = u >> 5, b = QK * sb + unit_base(u & 31);
        const float4 a = *reinterpret_cast<const float4 *>(xt + b);
        const float4 c = *reinterpret_cast<const float4 *>(xt + b + 32);
        uint4 h, l;
        split_unit(a, c, e, ls, h, l);
        uint4 *o = xop + ((size_t)t * (H / QK) + sb) * 64;
        o[u & 31] = h;
        o[32 + (u & 31)] = l;
        // sub-blocks j = 4 g + 2 pp (a) and j + 1 (c): sums over k
        float sa = ldexpf((a.x + a.y) + (a.z + a.w), -e - 5), sc = ldexpf((c.x + c.y) + (c.z + c.w), -e - 5);
        sa = xor_add(xor_add(xor_add(sa, 2), 4), 8);
        sc = xor_add(xor_add(xor_add(sc, 2), 4), 8);
        if ((u & 0xE) == 0) {
            uint32_t hh, ll;
            split2(sa, sc, ls_sum, hh, ll);
            uint32_t *so = reinterpret_cast<uint32_t *>(xsum + ((size_t)t * (H / QK) + sb) * 2);
            const int j2 = 2 * (u & 1) + ((u >> 4) & 1);  // j / 2
            so[j2] = hh;
            so[4 + j2] = ll;
        }
    }
}

// Per token, one workgroup: the activation preparation (row scale, operand
// units, shared-gate logit) and, on
// wave 0, softmax / top-k / renormalisation with the host's arithmetic on
// the router logits (route_dev.h topk_wave_exact).
template <int MAXV>
__global__ __launch_bounds__(256) void k_mt_topk_xprep(const float *__restrict__ logits, int E, int K,
                                                       int32_t *__restrict__ idx, float *__restrict__ w,
                                                       const float *__restrict__ x, const uint16_t *__restrict__ shg,
                                                       int H, bool scaled_lo, uint4 *__restrict__ xop,
                                                       uint4 *__restrict__ xsum, int *__restrict__ xexp,
                                                       float *__restrict__ gsh)
{
    __shared__ __attribute__((aligned(16))) float s_e[WAVE * MAXV];
    const int t = (int)blockIdx.x;
    if (wave_id() == 0) {
        int ik;
        float wk;
        topk_wave_exact<MAXV>(logits + (size_t)t * E, E, K, s_e, ik, wk);
        if (lane_id() < K) {
            idx[(size_t)t * K + lane_id()] = ik;
            w[(size_t)t * K + lane_id()] = wk;
        }
    }
    mt_xprep(t, x, shg, H, scaled_lo, xop, xsum, xexp, gsh);
}

// ---------------------------------------------------------------------------
// Bucketing
// ---------------------------------------------------------------------------

// Exclusive prefix sums of two per-thread values over the workgroup.
__device__ __forceinline__ void block_scan2(int a, int b, int *wsa, int *wsb, int &xa, int &xb, int &ta, int &tb)
{
    const int lane = lane_id(), w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    const int ia = wave_scan_incl(a), ib = wave_scan_incl(b);
    if (lane == WAVE - 1) {
        wsa[w] = ia;
        wsb[w] = ib;
    }
    __syncthreads();
    int pa = 0, pb = 0;
    ta = 0;
    tb = 0;
    for (int i = 0; i < nw; i++) {
        if (i < w) {
            pa += wsa[i];
            pb += wsb[i];
        }
        ta += wsa[i];
        tb += wsb[i];
    }
    xa = pa + ia - a;
    xb = pb + ib - b;
}

// Pairs (token t, rank k) sorted by expert; the shared expert's pairs
// (every token in order) follow at T*K.  pos_of[t*K + k] = sorted position
// (-1 for an index outside [0, E), which the combine skips).  Tiles: the
// routed experts' in expert order, then the shared expert's; n_tiles[0] and
// n_tiles[1] are the counts before and with the shared ones.
__global__ __launch_bounds__(1024) void k_mt_bucket(const int32_t *__restrict__ idx, int T, int K, int E,
                                                    int *__restrict__ pair_tok, int *__restrict__ pos_of,
                                                    MtTile *__restrict__ tiles, int *__restrict__ n_tiles)
{
    __shared__ int cnt[1024], base[1024];
    __shared__ int wsa[16], wsb[16];
    const int tid = threadIdx.x;
    cnt[tid] = 0;
    __syncthreads();
    const int P = T * K;
    // PB pairs a thread and pass, an LDS atomic each: its count so far is the
    // pair's place in its expert's list.  The first pass stays in registers,
    // later ones leave the place in pos_of for the second walk.  (A pair at a
    // time, with a second atomic in the second walk, each pair waited for
    // memory twice: 2048 tokens 22 us, now 16 us.)
    constexpr int PB = 16;
    int e[PB], o[PB];
    auto load = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int p = p0 + i * 1024 + tid;
            e[i] = p < P ? idx[p] : -1;
        }
    };
    for (int p0 = (P - 1) / (PB * 1024) * (PB * 1024); p0 >= 0; p0 -= PB * 1024) {
        load(p0);
#pragma unroll
        for (int i = 0; i < PB; i++) {
            o[i] = 0;
            if ((unsigned)e[i] < (unsigned)E) o[i] = atomicAdd(&cnt[e[i]], 1);
        }
        if (p0 == 0) break;
#pragma unroll
        for (int i = 0; i < PB; i++)
            if (p0 + i * 1024 + tid < P) pos_of[p0 + i * 1024 + tid] = o[i];
    }
    __syncthreads();
    const int c = tid < E ? cnt[tid] : 0;
    const int nt = (c + MT - 1) / MT;
    int xc, xt, tc, tt;
    block_scan2(c, nt, wsa, wsb, xc, xt, tc, tt);
    base[tid] = xc;
    __syncthreads();
    for (int p0 = 0; p0 < P; p0 += PB * 1024) {
        if (p0) {
            load(p0);
#pragma unroll
            for (int i = 0; i < PB; i++) o[i] = p0 + i * 1024 + tid < P ? pos_of[p0 + i * 1024 + tid] : 0;
        }
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int p = p0 + i * 1024 + tid;
            if (p >= P) break;
            int pos = -1;
            if ((unsigned)e[i] < (unsigned)E) {
                pos = base[e[i]] + o[i];
                pair_tok[pos] = p / K;
            }
            pos_of[p] = pos;
        }
    }
    for (int i = 0; i < nt; i++) tiles[xt + i] = {tid, xc + i * MT, min(MT, c - i * MT), 0};
    const int nsh = (T + MT - 1) / MT;
    for (int i = tid; i < nsh; i += 1024) tiles[tt + i] = {E, P + i * MT, min(MT, T - i * MT), 0};
    for (int t = tid; t < T; t += 1024) pair_tok[P + t] = t;
    if (tid == 0) {
        n_tiles[0] = tt;
        n_tiles[1] = tt + nsh;
    }
}

// ---------------------------------------------------------------------------
// Raw superblock bytes of a lane: row r, half g of the superblock.
// ---------------------------------------------------------------------------

typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

template <int QT>
struct Raw;

template <>
struct Raw<BREAD_QTYPE_Q4_K> {
    static constexpr uint32_t BYTES = Q4K_BYTES;
    uint4 hd, q[4];  // d, dmin, scales; the half's qs bytes
};

template <>
struct Raw<BREAD_QTYPE_Q6_K> {
    static constexpr uint32_t BYTES = Q6K_BYTES;
    u32x4_a2 l[4], h[2];  // the half's ql and qh bytes
    u32x2_a2 sc;          // its eight scales
    uint32_t d;
};

__device__ __forceinline__ void raw_load(Raw<BREAD_QTYPE_Q4_K> &R, const uint8_t *p, uint32_t off, int g)
{
    R.hd = *reinterpret_cast<const uint4 *>(p + off);
    const uint32_t q = off + 16 + 64 * g;
#pragma unroll
    for (int i = 0; i < 4; i++) R.q[i] = *reinterpret_cast<const uint4 *>(p + (q + 16 * i));
}

// Q6_K superblocks are 2-byte aligned; the loads say so (the target takes
// unaligned vector loads) and stay inside the superblock.
__device__ __forceinline__ void raw_load(Raw<BREAD_QTYPE_Q6_K> &R, const uint8_t *p, uint32_t off, int g)
{
    const uint32_t l = off + 64 * g, h = off + 128 + 32 * g;
#pragma unroll
    for (int i = 0; i < 4; i++) R.l[i] = *reinterpret_cast<const u32x4_a2 *>(p + (l + 16 * i));
    R.h[0] = *reinterpret_cast<const u32x4_a2 *>(p + h);
    R.h[1] = *reinterpret_cast<const u32x4_a2 *>(p + (h + 16));
    R.sc = *reinterpret_cast<const u32x2_a2 *>(p + (off + 192 + 8 * g));
    R.d = *reinterpret_cast<const uint16_t *>(p + (off + 208));
}

// D[32 tokens][32 rows] += X[32][16] * W[16][32]: D register i of lane (r, g)
// holds token 8 (i / 4) + 4 g + i % 4 of row r.
__device__ __forceinline__ f32x16 mfma32(const uint4 &x, const uint4 &w, f32x16 acc)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, x), __builtin_bit_cast(half8, w), acc, 0,
                                                  0, 0);
}

__device__ __forceinline__ f32x16 zero16()
{
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.f;
    return z;
}

__device__ __forceinline__ half2v h2_of(uint32_t v)
{
    return __builtin_bit_cast(half2v, v);
}

__device__ __forceinline__ uint32_t u_of(half2v v)
{
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ half2v dup(half2v v, int i)
{
    return half2v{v[i], v[i]};
}

__device__ __forceinline__ half2v pair(float a, float b)
{
    return half2v{(_Float16)a, (_Float16)b};
}

// Masks and magic numbers in registers: (v & mask) | w is then one
// three-operand instruction (with literals, which that form does not take,
// the compiler makes two).
struct Consts {
    uint32_t lo, hi, q2, magic;  // 0x000F000F, 0x00F000F0, 0x00300030, fp16 1024 twice
    uint32_t sca, scb;           // this lane's half: sc = (s & sca) | ((s0 >> 2) & scb), see Unit
};

__device__ __forceinline__ Consts consts(int g)
{
    Consts c;
    asm("s_mov_b32 %0, 0x000F000F" : "=s"(c.lo));
    asm("s_mov_b32 %0, 0x00F000F0" : "=s"(c.hi));
    asm("s_mov_b32 %0, 0x00300030" : "=s"(c.q2));
    asm("v_mov_b32 %0, 0x64006400" : "=v"(c.magic));
    c.sca = g ? 0x0F0F0F0Fu : 0x3F3F3F3Fu;
    c.scb = g ? 0x30303030u : 0u;
    return c;
}

// Bytes I and J of v (small non-negative integers) as an fp16 pair.
template <int I, int J>
__device__ __forceinline__ half2v pair_u8(uint32_t v)
{
    return h2_of(__builtin_amdgcn_perm(0x64646464u, v, 0x07000700u | I | (J << 16))) - pair(1024.f, 1024.f);
}

// w 2^-EXP: eight weights for lo terms held times 2^EXP.
template <int EXP>
__device__ __forceinline__ uint4 lo_operand(const uint4 &w)
{
    const half2v k = pair(1.f / (1 << EXP), 1.f / (1 << EXP));
    return make_uint4(u_of(h2_of(w.x) * k), u_of(h2_of(w.y) * k), u_of(h2_of(w.z) * k), u_of(h2_of(w.w) * k));
}

// Operand maker of one unit (32 weight rows of one superblock): constants
// from the superblock's header, then a step's eight weights; the scaling of
// the sums.  prepare() sets bad (where `flag`, the layers of the reference GPU
// path's types) for Q4_K |d| >= 64 or |dmin| >= 1024, Q6_K |d sc| >= 2047, or
// NaN: superblocks whose weights fp16 does not hold.  The operands here are
// integers, so finite ones come out right all the same; the flag stays because
// callers know such layers by it (BREAD_DEV_ERR_RANGE).
template <int QT, bool X>
struct Unit;

template <bool X>
struct Unit<BREAD_QTYPE_Q4_K, X> {
    half2v sc[2], ns[X ? 2 : 1];

    // Scales of groups 0, 1 and 2, 3: a pair each.  A masked nibble is the
    // fp16 subnormal q 2^-24 (odd groups: 16 q 2^-24, left in place), and
    //   q 2^-24 * sc 2^10 = sc q 2^-14,
    // or with X fma(q 2^-24, sc 2^10, -8 sc 2^-14) = sc (q - 8) 2^-14, both
    // exact.  The centred form halves the rounding of the sums and with it
    // leaves the layer's error at that of the per-token kernels (5.7e-7
    // against 5.8e-7 over 130 tokens; 6.0e-7 without); it costs gate/up 4 %.
    __device__ __forceinline__ void prepare(const Raw<BREAD_QTYPE_Q4_K> &R, const Consts &C, int g, bool flag, bool &bad)
    {
        const uint32_t s0 = R.hd.y, s2 = R.hd.w;
        if (flag) bad |= !(fabsf(h2f(R.hd.x)) < 64.f && fabsf(h2f(R.hd.x >> 16)) < 1024.f);
        const uint32_t sc4 = ((g ? s2 : s0) & C.sca) | ((s0 >> 2) & C.scb);
        const half2v p0 = pair_u8<0, 1>(sc4), p1 = pair_u8<2, 3>(sc4);
        sc[0] = p0 * pair(1024.f, 64.f);
        sc[1] = p1 * pair(1024.f, 64.f);
        if constexpr (X) {
            ns[0] = p0 * pair(-0x1p-11f, -0x1p-11f);
            ns[1] = p1 * pair(-0x1p-11f, -0x1p-11f);
        }
    }

    // tot += 2^14 d c - sum_j dmin m_j (sum of x over sub-block j), with X +
    // sum_j 8 d sc_j of them: m_0..7 and sc_0..7 against the hi and lo sums.
    // The last two are of one size and cancel, so they meet before the total.
    __device__ __forceinline__ void add(const Raw<BREAD_QTYPE_Q4_K> &R, const uint4 &sums, int g, const f32x16 &c,
                                        f32x16 &tot) const
    {
        const uint32_t s0 = R.hd.y, s1 = R.hd.z, s2 = R.hd.w;
        auto eight = [g](uint32_t lo, uint32_t hi) __attribute__((always_inline)) {
            const uint4 v = make_uint4(u_of(pair_u8<0, 1>(lo)), u_of(pair_u8<2, 3>(lo)), u_of(pair_u8<0, 1>(hi)),
                                       u_of(pair_u8<2, 3>(hi)));
            return X && g ? lo_operand<SUM_LO_EXP>(v) : v;  // lane half 1 meets the lo sums
        };
        const uint4 mv = eight(s1 & 0x3F3F3F3Fu, ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u));
        const f32x16 pm = mfma32(sums, mv, zero16());
        const float d = 16384.f * h2f(R.hd.x), dm = -32.f * h2f(R.hd.x >> 16);
        if constexpr (X) {
            const uint4 sv = eight(s0 & 0x3F3F3F3Fu, (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u));
            const f32x16 ps = mfma32(sums, sv, zero16());
            const float d8 = 256.f * h2f(R.hd.x);
#pragma unroll
            for (int i = 0; i < 16; i++) tot[i] += fmaf(c[i], d, fmaf(pm[i], dm, ps[i] * d8));
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) tot[i] = fmaf(c[i], d, tot[i]);
#pragma unroll
            for (int i = 0; i < 16; i++) tot[i] = fmaf(pm[i], dm, tot[i]);
        }
    }

    __device__ __forceinline__ void step(const Raw<BREAD_QTYPE_Q4_K> &R, const Consts &C, int s, uint4 &w, uint4 &) const
    {
        const int pp = s >> 3;
        const uint32_t v = comp(R.q[s >> 2], s & 3), v8 = v >> 8;
        const half2v se = dup(sc[pp], 0), so = dup(sc[pp], 1);
        const half2v a0 = h2_of(v & C.lo), a1 = h2_of(v8 & C.lo), b0 = h2_of(v & C.hi), b1 = h2_of(v8 & C.hi);
        if constexpr (X) {
            const half2v ne = dup(ns[pp], 0), no = dup(ns[pp], 1);
            w = make_uint4(u_of(__builtin_elementwise_fma(a0, se, ne)), u_of(__builtin_elementwise_fma(a1, se, ne)),
                           u_of(__builtin_elementwise_fma(b0, so, no)), u_of(__builtin_elementwise_fma(b1, so, no)));
        } else {
            w = make_uint4(u_of(a0 * se), u_of(a1 * se), u_of(b0 * so), u_of(b1 * so));
        }
    }
};

template <bool X>
struct Unit<BREAD_QTYPE_Q6_K, X> {
    // scales sc[8 g + 2 q], sc[8 g + 2 q + 1] of group q, elements 0..15 and
    // 16..31, times S: without X an element is the fp16 subnormal q 2^-24 and
    // fma(q 2^-24, 2^8 sc, -32 sc 2^-16) rounds sc (q - 32) 2^-16 once
    static constexpr float S = X ? 1.f : 256.f;
    half2v sc[4], ns[X ? 1 : 4];

    __device__ __forceinline__ void prepare(const Raw<BREAD_QTYPE_Q6_K> &R, const Consts &, int, bool flag, bool &bad)
    {
        const uint32_t a = R.sc[0] ^ 0x80808080u, b = R.sc[1] ^ 0x80808080u;  // sc + 128
        const half2v k = pair(128.f, 128.f);
        sc[0] = pair_u8<0, 1>(a) - k;
        sc[1] = pair_u8<2, 3>(a) - k;
        sc[2] = pair_u8<0, 1>(b) - k;
        sc[3] = pair_u8<2, 3>(b) - k;
        const float d = h2f(R.d);
        if (flag && __builtin_amdgcn_ballot_w64(!(fabsf(d) < 15.9f)) != 0) {
#pragma unroll
            for (int q = 0; q < 8; q++) bad |= !(fabsf(d * (float)sc[q >> 1][q & 1]) < 2047.f);
        }
        if constexpr (!X) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                ns[q] = sc[q] * pair(-0x1p-11f, -0x1p-11f);
                sc[q] = sc[q] * pair(S, S);
            }
        }
    }

    __device__ __forceinline__ void add(const Raw<BREAD_QTYPE_Q6_K> &R, const uint4 &, int, const f32x16 &c,
                                        f32x16 &tot) const
    {
        const float d = (X ? 1.f : 0x1p16f) * h2f(R.d);
#pragma unroll
        for (int i = 0; i < 16; i++) tot[i] = fmaf(c[i], d, tot[i]);
    }

    // w = fp16(sc (q - 32)), times 2^-16 without X; r (X): what that rounds
    // off, 0 or +-1
    __device__ __forceinline__ void step(const Raw<BREAD_QTYPE_Q6_K> &R, const Consts &C, int s, uint4 &w, uint4 &r) const
    {
        const int pp = s >> 3, k = s & 7;
        const uint32_t h = R.h[k >> 2][k & 3];
        uint32_t wv[4], rv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {  // group 2 pp + j / 2, bytes 0 and 2 (j even) or 1 and 3
            const int q = 2 * pp + (j >> 1), lsh = 4 * pp + 8 * (j & 1), hsh = 8 * (j & 1) + 2 * q - 4;
            const uint32_t l = R.l[(j >> 1) * 2 + (k >> 2)][k & 3] >> lsh;
            const uint32_t hb = hsh >= 0 ? h >> hsh : h << -hsh;
            const half2v se = dup(sc[q], k >> 2);
            if constexpr (X) {
                const half2v v = h2_of((hb & C.q2) | ((l & C.lo) | C.magic)) - pair(1056.f, 1056.f);  // q - 32, exact
                const half2v p = v * se;
                wv[j] = u_of(p);
                rv[j] = u_of(__builtin_elementwise_fma(v, se, -p));
            } else {
                wv[j] = u_of(__builtin_elementwise_fma(h2_of((hb & C.q2) | (l & C.lo)), se, dup(ns[q], k >> 2)));
                rv[j] = 0;
            }
        }
        w = make_uint4(wv[0], wv[1], wv[2], wv[3]);
        r = make_uint4(rv[0], rv[1], rv[2], rv[3]);
    }
};

struct GgArgs {
    const uint8_t *w0, *w1;    // routed gate and up (or down), expert e at + e * stride
    uint64_t st0, st1;
    const uint8_t *sw0, *sw1;  // the shared expert's
    uint32_t *err;
    const uint4 *xop, *xsum;   // prepared activations by token
    const int *xexp;
    const int *pair_tok;
    const MtTile *tiles;
    const int *n_tiles;
    float *h;                  // SwiGLU rows by pair [pairs][hstride]
    float *eo;                 // expert outputs by pair [pairs][H]
    int E;
    int nsb, nsb_sh;           // superblocks of the contraction: routed, shared
    int rows, rows_sh;         // rows of an expert
    int hstride;
    int sel;                   // 1: the routed tiles, 2: the shared ones, 3: both
    int flag;                  // report superblocks outside the fp16 range
};

#define CONST_AS __attribute__((address_space(4)))  // read by scalar loads

// The items of a workgroup: (tile, chunk of rows), the chunks of a tile in
// sequence, C a tile (C_sh of the shared expert's, which come last and may have
// another size).  Workgroups go to the 8 XCDs round-robin by linear id and
// each XCD has its own L2, so XCD L % 8 takes a contiguous eighth, where a
// tile's chunks share its activations and an expert's tiles its weights; its
// workgroups take turns.
struct GgItems {
    const MtTile CONST_AS *tiles;
    int routed, first_sh, N, per, j, i, C, C_sh;
    int chunk, e, p0, nr;  // the current item

    __device__ __forceinline__ GgItems(const GgArgs &a, int chunks, int chunks_sh)
    {
        const int CONST_AS *n = (const int CONST_AS *)a.n_tiles;
        tiles = (const MtTile CONST_AS *)a.tiles;
        C = chunks;
        C_sh = chunks_sh;
        first_sh = n[0];
        routed = a.sel & 1 ? n[0] * C : 0;
        N = routed + (a.sel & 2 ? (n[1] - n[0]) * C_sh : 0);
        per = (N + NXCD - 1) / NXCD;
        j = (int)blockIdx.x / NXCD - (int)gridDim.x / NXCD;
        i = ((int)blockIdx.x % NXCD) * per;
    }
    // the next item, false (and the last one kept) past the end
    __device__ __forceinline__ bool next()
    {
        j += (int)gridDim.x / NXCD;
        if (j >= per || i + j >= N) return false;
        const bool sh = i + j >= routed;
        const int k = i + j - (sh ? routed : 0), c = sh ? C_sh : C;
        const int tile = uniform((sh ? first_sh : 0) + k / c);
        chunk = uniform(k % c);
        e = uniform(tiles[tile].e);
        p0 = uniform(tiles[tile].p0);
        nr = uniform(tiles[tile].nr);
        return true;
    }
};

__device__ __forceinline__ void lds_load16(const void *src, void *lds_wave_base)
{
    __builtin_amdgcn_global_load_lds(src, lds_wave_base, 16, 0, 0);
}

// A barrier that publishes the waves' LDS writes and leaves global loads in
// flight (__syncthreads would wait for every one of them).
__device__ __forceinline__ void gg_bar()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// s_waitcnt on the vector memory counter only (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
    __builtin_amdgcn_sched_barrier(0);
}

// Units u = 2 s + g, s = 0 .. 7, of row r in LDS rows of 32 units (16 hi, 16
// lo; half a superblock) or 64 (32 hi, 32 lo): unit u of token n is at u ^ (n
// % 16), so that a read of one unit of 16 tokens covers the banks.  The
// address is made anew each time: the compiler would keep eight of them in
// registers for the whole kernel.
struct XRead {
    const char *p;
    uint32_t a;
    __device__ __forceinline__ XRead(const uint4 *row, int r, int g)
    {
        p = reinterpret_cast<const char *>(row);
        a = (uint32_t)(16 * (g ^ (r & 15)));
        asm volatile("" : "+v"(a));
    }
    __device__ __forceinline__ uint4 operator()(int s, uint32_t off) const
    {
        return *reinterpret_cast<const uint4 *>(p + ((a ^ (uint32_t)(32 * (s & 7))) + off));
    }
};

// ---------------------------------------------------------------------------
// Gate/up: workgroup of 4 waves per (tile, 128 rows); a wave owns 32 gate
// rows and the same 32 up rows, so each activation fragment read from LDS
// meets 64 weight rows and the SwiGLU needs no exchange.
// The workgroups are persistent: the last superblock of an item requests the
// first one of the next.
//
// Everything comes by direct-to-LDS loads whose adjacent lanes read adjacent
// memory: a load whose lanes are 64 rows costs the address unit a cycle a
// lane, and with the weights loaded so (16 bytes of a row a lane) issuing a
// superblock's loads took 2,500-5,000 cycles of an iteration of 8,500.
// Weights: a wave's 2 x 32 rows of a superblock (9 KB) into a buffer of its
// own, moved to registers when the superblock begins, which frees the buffer
// for the next one.  Activations: half a superblock of the tile's 32 rows (16
// KB) into one of two buffers, a half ahead.  A barrier each half; 73 KB of
// LDS, two workgroups a CU, so 256 vector registers a wave: 207 in use, 208
// (Q4_K) to 245 (Q6_K) with X.  20-30 scalar registers spill into vector ones
// in the Q4_K forms, outside the steps.
// Q6_K gate or up (no reference GPU layout) loads its weights straight into
// registers: its 210-byte superblocks are 2-byte aligned.
//
// Measured on MI355X (hidden 2048, intermediate 512, 256 experts, top 8), the
// kernel that dequantised into fp16 d sc q - dmin m operands with a lane a
// weight row / this one: 64 tokens (Zipf) 36 / 28 us, 512 tokens 136 / 110 us,
// 2048 tokens 321 / 253 us.  A superblock (2 x 32 MFMA a wave, 8 waves a CU)
// takes 6,500 cycles against 4,200 of the matrix pipe alone; half the rest is
// issuing the direct-to-LDS loads, and an item's prologue and SwiGLU add
// 6,000.  At 512 tokens (16 pairs an expert) half of a tile's rows are empty.
// ---------------------------------------------------------------------------

constexpr int W_CHUNKS = 32 * Q4K_BYTES / 16;  // 16-byte pieces of a matrix's superblock rows of a wave
constexpr int W_LOADS = (W_CHUNKS + WAVE - 1) / WAVE;
constexpr int W_BUF = W_LOADS * WAVE;  // the last load's idle lanes repeat the last piece

// X: the exact operands of layers of other types than the reference GPU path's
template <int Q0, int Q1, bool X>
__global__ __launch_bounds__(GG_THREADS, 2) void k_gateup_gg(const GgArgs a)
{
    constexpr int Q4 = BREAD_QTYPE_Q4_K;
    constexpr bool X0 = Q0 != Q4, X1 = Q1 != Q4, SUMS = Q0 == Q4 || Q1 == Q4;
    // a variable for each buffer: a read of one that a direct-to-LDS load may
    // write waits for all such loads
    __shared__ uint4 sA0[MT][32], sA1[MT][32], sS[MT][2];
    __shared__ uint4 sW[GG_WAVES][Q0 == Q4 && Q1 == Q4 ? 2 : 1][W_BUF];
    __shared__ int sexp[2][MT];
    const int tid = (int)threadIdx.x, w = wave_id(), lane = lane_id();
    const int g = lane >> 5, r = lane & 31;
    GgItems it(a, a.rows / GU_ROWS, a.rows_sh / GU_ROWS);
    if (!it.next()) return;
    const uint32_t rb0 = (uint32_t)a.nsb * Raw<Q0>::BYTES, rb1 = (uint32_t)a.nsb * Raw<Q1>::BYTES;
    // the item's matrices, from the wave's first row (n0, n1: the next item's)
    const uint8_t *m0, *m1, *n0, *n1;
    auto matrices = [&](const uint8_t *&p, const uint8_t *&q) __attribute__((always_inline)) {
        const uint32_t row0 = (uint32_t)(it.chunk * GU_ROWS + 32 * w);
        p = (it.e == a.E ? a.sw0 : a.w0 + (uint64_t)it.e * a.st0) + (uint64_t)row0 * rb0;
        q = (it.e == a.E ? a.sw1 : a.w1 + (uint64_t)it.e * a.st1) + (uint64_t)row0 * rb1;
    };

    // 16-byte piece c of a matrix's superblock rows: row c / 9, piece c % 9
    uint32_t wo[W_LOADS];
#pragma unroll
    for (int j = 0; j < W_LOADS; j++) {
        const uint32_t c = (uint32_t)min(64 * j + lane, W_CHUNKS - 1);
        wo[j] = (c / 9) * ((uint32_t)a.nsb * Q4K_BYTES) + (c % 9) * 16;
    }
    auto stage_m = [&](const uint8_t *m, int sb, uint4 (&buf)[W_BUF]) __attribute__((always_inline)) {
        const uint8_t *p = m + (uint32_t)sb * Q4K_BYTES;
#pragma unroll
        for (int j = 0; j < W_LOADS; j++)
            lds_load16(p + wo[j], &buf[64 * j]);
    };
    Raw<Q0> R0;
    Raw<Q1> R1;
    constexpr int S1 = Q0 == Q4 ? 1 : 0;  // the up matrix's buffer
    auto stage_w = [&](const uint8_t *p, const uint8_t *q, int sb) __attribute__((always_inline)) {
        if constexpr (Q0 == Q4) stage_m(p, sb, sW[w][0]);
        if constexpr (Q1 == Q4) stage_m(q, sb, sW[w][S1]);
    };
    // the wave's weights of superblock sb into registers: lane (r, g)
    auto take_q4 = [&](Raw<Q4> &R, const uint4 (&buf)[W_BUF]) __attribute__((always_inline)) {
        R.hd = buf[9 * r];
#pragma unroll
        for (int i = 0; i < 4; i++) R.q[i] = buf[9 * r + 1 + 4 * g + i];
    };
    auto take_w = [&](int sb) __attribute__((always_inline)) {
        if constexpr (Q0 == Q4) take_q4(R0, sW[w][0]);
        else raw_load(R0, m0 + (uint32_t)sb * Raw<Q0>::BYTES, (uint32_t)r * rb0, g);
        if constexpr (Q1 == Q4) take_q4(R1, sW[w][S1]);
        else raw_load(R1, m1 + (uint32_t)sb * Raw<Q1>::BYTES, (uint32_t)r * rb1, g);
    };
    constexpr int NW = W_LOADS * ((Q0 == Q4) + (Q1 == Q4));  // loads of stage_w

    // Tokens 2 q and 2 q + 1, q = w, w + 4, ...: an instruction brings half
    // a superblock of both, 16 hi and 16 lo units each (past nr the last
    // token: its results are not stored).  Every wave brings the sums: a
    // branch would blur the wait counts.
    constexpr int NT = MT / (2 * GG_WAVES);
    int tok[NT], tsum;
    const char *xt[NT];
    const uint4 *xs;
    auto tokens = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NT; i++)
            tok[i] = a.pair_tok[it.p0 + min(2 * (w + GG_WAVES * i) + (lane >> 5), it.nr - 1)];
        tsum = a.pair_tok[it.p0 + min(lane >> 1, it.nr - 1)];
    };
    auto pointers = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NT; i++) {
            const int n = 2 * (w + GG_WAVES * i) + (lane >> 5), u = lane & 31;
            xt[i] = reinterpret_cast<const char *>(a.xop + (size_t)tok[i] * a.nsb * 64) + 512 * (u >> 4) +
                    16 * ((u ^ n) & 15);
        }
        xs = a.xsum + (size_t)tsum * a.nsb * 2 + (lane & 1);
    };
    auto stage_x = [&](int sb, int pp, uint4 (&buf)[MT][32]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NT; i++)
            lds_load16(xt[i] + (sb * 1024 + pp * 256), &buf[2 * (w + GG_WAVES * i)][0]);
    };

    const Consts C = consts(g);
    f32x16 t0 = zero16(), t1 = zero16(), c0, c1;
    Unit<Q0, X> U0;
    Unit<Q1, X> U1;
    bool bad = false;
    // steps 8 pp .. 8 pp + 7 of the superblock in R0, R1
    auto compute = [&](const uint4 (&sA)[MT][32], int pp) __attribute__((always_inline)) {
        const XRead x(sA[r], r, g);
        uint4 xh = x(0, 0), xl = x(0, 256), nh, nl;
        uint4 w0, w1, r0, r1, v0, v1, q0, q1;
        U0.step(R0, C, 8 * pp, w0, r0);
        U1.step(R1, C, 8 * pp, w1, r1);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            if (s < 7) {
                nh = x(s + 1, 0);
                nl = x(s + 1, 256);
            }
            c0 = mfma32(xh, w0, c0);
            c1 = mfma32(xh, w1, c1);
            c0 = mfma32(xl, X ? lo_operand<LO_EXP>(w0) : w0, c0);
            c1 = mfma32(xl, X ? lo_operand<LO_EXP>(w1) : w1, c1);
            if (X0) c0 = mfma32(xh, r0, c0);
            if (X1) c1 = mfma32(xh, r1, c1);
            if (X0) c0 = mfma32(xl, lo_operand<LO_EXP>(r0), c0);
            if (X1) c1 = mfma32(xl, lo_operand<LO_EXP>(r1), c1);
            if (s < 7) {
                U0.step(R0, C, 8 * pp + s + 1, v0, q0);
                U1.step(R1, C, 8 * pp + s + 1, v1, q1);
            }
            // an MFMA, then VALU: the next step's operands are made under
            // this one's products
#pragma unroll
            for (int i = 0; i < 4 + 2 * X0 + 2 * X1; i++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, X0 || X1 ? 10 : X ? 6 : 5, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            xh = nh;
            xl = nl;
            w0 = v0;
            w1 = v1;
            r0 = q0;
            r1 = q1;
        }
    };

    matrices(m0, m1);
    tokens();
    pointers();
    stage_x(0, 0, sA0);
    stage_w(m0, m1, 0);
    bool first = true;
    for (int turn = 0;; turn ^= 1, first = false) {
        const int p0 = it.p0, nr = it.nr, row0 = it.chunk * GU_ROWS + 32 * w;
        float *hp = uniform_ptr(a.h + (size_t)p0 * a.hstride);
        const int ex_tok = a.pair_tok[p0 + min(tid & (MT - 1), nr - 1)];
        const bool more = it.next();
        matrices(n0, n1);
        tokens();
        if (tid < MT) sexp[turn][tid] = a.xexp[ex_tok];
        t0 = t1 = zero16();
        for (int sb = 0; sb < a.nsb; sb++) {
            // First half: activations and weights have landed.  The sums and
            // the second half's activations go out, then (behind them, so
            // that the next wait can leave them in flight) the next
            // superblock's weights, at the end the next item's first ones.
            const bool last = sb + 1 == a.nsb;
            if (sb == 0 && !first) wait_vm<16>();  // the last item's 16 stores
            else wait_vm<0>();
            gg_bar();
            take_w(sb);
            if (SUMS) lds_load16(xs + 2 * sb, &sS[0][0]);
            stage_x(sb, 1, sA1);
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's buffer is read
            __builtin_amdgcn_sched_barrier(0);
            stage_w(last ? n0 : m0, last ? n1 : m1, last ? 0 : sb + 1);
            __builtin_amdgcn_sched_barrier(0);
            U0.prepare(R0, C, g, a.flag != 0, bad);
            U1.prepare(R1, C, g, a.flag != 0, bad);
            c0 = c1 = zero16();
            compute(sA0, 0);
            // second half
            wait_vm<NW>();
            gg_bar();
            if (last) pointers();
            stage_x(last ? 0 : sb + 1, 0, sA0);
            compute(sA1, 1);
            uint4 sums = make_uint4(0, 0, 0, 0);
            if (SUMS) sums = sS[r][g];
            U0.add(R0, sums, g, c0, t0);
            U1.add(R1, sums, g, c1, t1);
        }
        // SwiGLU, stored in operand order: row c of a superblock at its
        // unit's place (unit_base), for k_down_gg's loads
        const int c = (row0 + r) & (QK - 1);
        const int u = 2 * (8 * ((c >> 6) & 1) + ((c >> 2) & 7)) + (c >> 7);
        const uint32_t col =
            (uint32_t)(((row0 + r) & ~(QK - 1)) + 8 * u + 4 * ((c >> 5) & 1) + 2 * (c & 1) + ((c >> 1) & 1));
        // rows past nr fall outside the buffer's range: every lane issues all
        // 16 stores, which the next item's first wait leaves in flight
        const __amdgpu_buffer_rsrc_t hb = rsrc(hp, (uint32_t)(nr * a.hstride * 4));
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int n = 8 * (i >> 2) + 4 * g + (i & 3);
            const int ex = sexp[turn][n];
            const float v = silu_mul(ldexpf(t0[i], ex), ldexpf(t1[i], ex));
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), hb,
                                                  4 * (uint32_t)(n * a.hstride) + 4 * col, 0, 0);
        }
        if (!more) break;
        m0 = n0;
        m1 = n1;
    }
    wait_vm<0>();  // (the loads past the end)
    if (a.flag && __builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0)
        __hip_atomic_fetch_or(a.err, BREAD_DEV_ERR_RANGE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Down: workgroup of 8 waves per (tile, 512 output rows), a wave two 32-row
// blocks.  The tile's fp32 SwiGLU rows (operand order) are read once, scaled
// by a power of two per row and split into hi and lo fp16 parts in LDS (64 KB
// for intermediate 512).  A unit is a block's 32 rows of one superblock: its
// bytes come by direct-to-LDS loads of adjacent 16-byte pieces into the wave's
// buffer, from there into registers when the unit begins, which frees the
// buffer for the next one (loads of 16 bytes of a row a lane, 2-byte aligned,
// took the address unit a cycle a lane).  The next item's SwiGLU rows and
// first unit are requested while the last units run.
// Measured as above, a lane a weight row / this: 64 tokens 23 / 21 us, 512
// tokens 98 / 91 us, 2048 tokens 221 / 208 us (a third of the error).  A unit
// of 32 MFMA is bound by the VALU in its steps (a Q6_K operand pair is a mask,
// a merge and a multiply-add on subnormals besides its shifts; with the
// integers biased by 1024 and two more instructions a pair 23 / 100 / 230 us),
// and takes 2,000 cycles in its loads and its move to registers.
// ---------------------------------------------------------------------------

// 16-byte pieces a row of a unit takes in the wave's buffer: a Q4_K superblock
// is 9; a Q6_K one lies in the 14 aligned pieces from the one that holds its
// first byte (inside the expert, whose start and size are 16-byte aligned),
// and a 15th, unused, spreads the rows over the banks.
template <int QT>
constexpr int ROW_CH = QT == BREAD_QTYPE_Q4_K ? 9 : 15;
template <int QT>
constexpr int UNIT_LD = (32 * ROW_CH<QT> + WAVE - 1) / WAVE;  // loads of a unit

// Lane (r, g)'s raw bytes from its buffer row; o: where the superblock starts
// in it (even, below 16).
__device__ __forceinline__ void take_unit(Raw<BREAD_QTYPE_Q4_K> &R, const uint4 *row, int g, uint32_t)
{
    R.hd = row[0];
#pragma unroll
    for (int i = 0; i < 4; i++) R.q[i] = row[1 + 4 * g + i];
}

__device__ __forceinline__ void take_unit(Raw<BREAD_QTYPE_Q6_K> &R, const uint4 *row, int g, uint32_t o)
{
    const uint32_t *p = reinterpret_cast<const uint32_t *>(row) + (o >> 2);
    const uint32_t sh = o & 2;
    auto take = [&](const uint32_t *q, int n, auto &&put) __attribute__((always_inline)) {
        uint32_t a = q[0];
#pragma unroll
        for (int i = 0; i < n; i++) {
            const uint32_t b = q[i + 1];
            put(i, __builtin_amdgcn_alignbyte(b, a, sh));
            a = b;
        }
    };
    take(p + 16 * g, 16, [&](int i, uint32_t v) { R.l[i >> 2][i & 3] = v; });
    take(p + 32 + 8 * g, 8, [&](int i, uint32_t v) { R.h[i >> 2][i & 3] = v; });
    take(p + 48 + 2 * g, 2, [&](int i, uint32_t v) { R.sc[i] = v; });
    R.d = p[52] >> (8 * sh);
}

// X as in k_gateup_gg.  TWO: the shared expert's intermediate size is not the
// routed ones' (the superblocks of an item's rows then come with the item, 0.3
// us of 20 where all have the same).
template <int QT, bool X, bool TWO>
__global__ __launch_bounds__(DN_WAVES * WAVE, 2) void k_down_gg(const GgArgs a)
{
    constexpr int Q4 = BREAD_QTYPE_Q4_K;
    constexpr bool X0 = X && QT != Q4;
    constexpr float LS = X ? (float)(1 << LO_EXP) : 1.f;
    constexpr int NB = MAX_INTER / QK;
    __shared__ uint4 sA[NB][MT][64];
    __shared__ uint32_t sS[QT == Q4 ? NB : 1][MT][2][4];  // sums: hi, lo of eight
    __shared__ uint4 sW[DN_WAVES][UNIT_LD<QT> * WAVE];
    __shared__ int sexp[MT];
    const int tid = (int)threadIdx.x, w = wave_id(), lane = lane_id();
    const int g = lane >> 5, r = lane & 31;
    const int chunks = (a.rows + DN_ROWS - 1) / DN_ROWS;
    GgItems it(a, chunks, chunks);
    if (!it.next()) return;
    // superblocks of `it`'s rows
    auto superblocks = [&]() __attribute__((always_inline)) { return TWO && it.e == a.E ? a.nsb_sh : a.nsb; };
    // the item's matrix from the wave's first row; blocks past the end
    // repeat the last one and are not stored
    auto matrix = [&]() __attribute__((always_inline)) {
        return (it.e == a.E ? a.sw0 : a.w0 + (uint64_t)it.e * a.st0);
    };
    auto block_row = [&](int chunk, int blk) __attribute__((always_inline)) {
        return chunk * DN_ROWS + 32 * (DN_BLOCKS * w + blk);
    };
    // piece 64 j + lane of a unit: its row (its offset unless TWO) and the
    // piece's offset
    uint32_t ro[UNIT_LD<QT>], po[UNIT_LD<QT>];
#pragma unroll
    for (int j = 0; j < UNIT_LD<QT>; j++) {
        const uint32_t c = (uint32_t)min(64 * j + lane, 32 * ROW_CH<QT> - 1);
        ro[j] = c / ROW_CH<QT> * (TWO ? 1u : (uint32_t)a.nsb * Raw<QT>::BYTES);
        po[j] = 16 * min(c % ROW_CH<QT>, (uint32_t)(QT == Q4 ? 8 : 13));
    }
    // unit u: block u / nb, superblock u % nb
    auto stage_w = [&](const uint8_t *m, int chunk, int nb, int u) __attribute__((always_inline)) {
        const int blk = nb == 2 ? u >> 1 : u, b = u - blk * nb;
        const uint32_t rb = (uint32_t)nb * Raw<QT>::BYTES;
        const uint8_t *p = m + (uint64_t)(uint32_t)min(block_row(chunk, blk), a.rows - 32) * rb;
#pragma unroll
        for (int j = 0; j < UNIT_LD<QT>; j++)
            lds_load16(p + ((((TWO ? ro[j] * rb : ro[j]) + (uint32_t)b * Raw<QT>::BYTES) & ~15u) + po[j]),
                       &sW[w][64 * j]);
    };
    // 16 threads a token, each the units q + 16 k of its superblocks
    const int hn = tid >> 4, hq = tid & 15;
    float4 va[2 * NB], vb[2 * NB];
    auto load_h = [&]() __attribute__((always_inline)) {
        const int nb = superblocks();
        const float *hr = a.h + (size_t)(it.p0 + min(hn, it.nr - 1)) * a.hstride + 8 * hq;
#pragma unroll
        for (int k = 0; k < 2 * NB; k++) {
            va[k] = vb[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (k < 2 * nb) {
                va[k] = *reinterpret_cast<const float4 *>(hr + 128 * k);
                vb[k] = *reinterpret_cast<const float4 *>(hr + 128 * k + 4);
            }
        }
    };
    auto split_h = [&](int nb) __attribute__((always_inline)) {
        float mx = 0.f;
#pragma unroll
        for (int k = 0; k < 2 * NB; k++) {
            const float4 x = va[k], y = vb[k];
            mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))),
                                 fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w)))));
        }
        mx = fmaxf(mx, dpp_f<0xB1>(mx));  // the token's 16 lanes
        mx = fmaxf(mx, dpp_f<0x4E>(mx));
        mx = fmaxf(mx, dpp_f<0x141>(mx));
        mx = fmaxf(mx, dpp_f<0x140>(mx));
        const int ex = row_exp(mx);
        if (hq == 0) sexp[hn] = ex;
#pragma unroll
        for (int k = 0; k < 2 * NB; k++) {
            if (k >= 2 * nb) continue;
            const int b = k >> 1, u = hq + 16 * (k & 1);
            uint4 hi, lo;
            split_unit_op(va[k], vb[k], ex, LS, hi, lo);
            sA[b][hn][u ^ (hn & 15)] = hi;
            sA[b][hn][32 + (u ^ (hn & 15))] = lo;
            if (QT == Q4) {
                // sub-blocks 4 g + 2 (k & 1) (x) and the next (y), g = hq & 1:
                // sums over the half's lanes
                const float4 x = va[k], y = vb[k];
                float sx = ldexpf((x.x + x.y) + (x.z + x.w), -ex - 5);
                float sy = ldexpf((y.x + y.y) + (y.z + y.w), -ex - 5);
                sx = xor_add(xor_add(xor_add(sx, 2), 4), 8);
                sy = xor_add(xor_add(xor_add(sy, 2), 4), 8);
                if (hq < 2) {
                    uint32_t h2, l2;
                    split2(sx, sy, X ? (float)(1 << SUM_LO_EXP) : 1.f, h2, l2);
                    sS[b][hn][0][2 * hq + (k & 1)] = h2;
                    sS[b][hn][1][2 * hq + (k & 1)] = l2;
                }
            }
        }
    };

    const Consts C = consts(g);
    f32x16 t = zero16();
    Raw<QT> R;
    Unit<QT, X> U;
    bool bad = false;
    const uint8_t *m = matrix();
    bool stores = false;  // the last unit stored
    load_h();
    stage_w(m, it.chunk, superblocks(), 0);
    for (;;) {
        const int chunk = it.chunk, p0 = it.p0, nr = it.nr, nb = superblocks();
        const uint32_t rb = (uint32_t)nb * Raw<QT>::BYTES;
        const uint8_t *mc = m;
        split_h(nb);
        gg_bar();
        const bool more = it.next();
        m = matrix();
        for (int u = 0; u < DN_BLOCKS * nb; u++) {
            const int blk = nb == 2 ? u >> 1 : u, b = u - blk * nb;
            const int row0 = block_row(chunk, blk);
            if (stores) wait_vm<16>();  // the last unit's 16 stores
            else wait_vm<0>();
            take_unit(R, &sW[w][r * ROW_CH<QT>], g, ((uint32_t)r * rb + (uint32_t)b * Raw<QT>::BYTES) & 15u);
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's buffer is read
            __builtin_amdgcn_sched_barrier(0);
            const bool last = u + 1 == DN_BLOCKS * nb;
            if (last) load_h();
            stage_w(last ? m : mc, last ? it.chunk : chunk, last ? superblocks() : nb, last ? 0 : u + 1);
            __builtin_amdgcn_sched_barrier(0);
            U.prepare(R, C, g, a.flag != 0 && row0 < a.rows, bad);
            f32x16 c0 = zero16(), c1 = zero16();
            const XRead x(sA[b][r], r, g);
            uint4 xh = x(0, 0), xl = x(0, 512), nh, nl;
            uint4 w0, r0, v0, q0;
            U.step(R, C, 0, w0, r0);
#pragma unroll
            for (int s = 0; s < 16; s++) {
                if (s < 15) {
                    nh = x(s + 1, 256 * ((s + 1) >> 3));
                    nl = x(s + 1, 512 + 256 * ((s + 1) >> 3));
                }
                c0 = mfma32(xh, w0, c0);
                c1 = mfma32(xl, w0, c1);
                if (X0) c0 = mfma32(xh, r0, c0);
                if (X0) c1 = mfma32(xl, r0, c1);
                if (s < 15) U.step(R, C, s + 1, v0, q0);
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, QT == Q4 ? 5 : 14, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                xh = nh;
                xl = nl;
                w0 = v0;
                r0 = q0;
            }
#pragma unroll
            for (int i = 0; i < 16; i++) c0[i] = X ? fmaf(c1[i], 1.f / LS, c0[i]) : c0[i] + c1[i];
            uint4 sums = make_uint4(0, 0, 0, 0);
            if (QT == Q4) sums = *reinterpret_cast<const uint4 *>(sS[b][r][g]);
            U.add(R, sums, g, c0, t);
            if (b == nb - 1) {
                // rows past nr (and blocks past the end) fall outside the
                // buffer's range: every lane issues all 16 stores, which the
                // next unit's wait leaves in flight
                const __amdgpu_buffer_rsrc_t ob =
                    rsrc(a.eo + (size_t)p0 * a.rows, row0 < a.rows ? (uint32_t)(nr * a.rows * 4) : 0u);
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int n = 8 * (i >> 2) + 4 * g + (i & 3);
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, ldexpf(t[i], sexp[n])), ob,
                                                          4 * (uint32_t)(n * a.rows + row0 + r), 0, 0);
                    t[i] = 0.f;
                }
                stores = true;
            } else {
                stores = false;
            }
        }
        if (!more) break;
        gg_bar();  // the tile's rows in LDS are read
    }
    wait_vm<0>();  // (the loads past the end)
    if (a.flag && __builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0)
        __hip_atomic_fetch_or(a.err, BREAD_DEV_ERR_RANGE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// hidden[t] += sigmoid(gsh[t]) * shared(t), then += w_k * expert_k(t) for
// k = 0..K-1 (one_layer.cu:1447-1449, 1469), one float4 per thread;
// blockIdx.x = token, blockIdx.y = 1024-column chunk.
__global__ __launch_bounds__(256) void k_mt_combine(const float *__restrict__ eo, const int *__restrict__ pos_of,
                                                    const float *__restrict__ w, const float *__restrict__ gsh,
                                                    float *__restrict__ hidden, int H, int K, int T)
{
#pragma clang fp contract(off)
    const int t = blockIdx.x;
    const int c = 4 * (blockIdx.y * blockDim.x + threadIdx.x);
    if (c >= H) return;
    float4 acc = *reinterpret_cast<const float4 *>(hidden + (size_t)t * H + c);
    const float sg = sigmoidf_ref(gsh[t]);
    const float4 s = *reinterpret_cast<const float4 *>(eo + ((size_t)T * K + t) * H + c);
    acc.x = acc.x + sg * s.x;
    acc.y = acc.y + sg * s.y;
    acc.z = acc.z + sg * s.z;
    acc.w = acc.w + sg * s.w;
#pragma unroll 8
    for (int k = 0; k < K; k++) {
        const int p = pos_of[t * K + k];
        if (p < 0) continue;
        const float wk = w[t * K + k];
        const float4 v = *reinterpret_cast<const float4 *>(eo + (size_t)p * H + c);
        acc.x = acc.x + wk * v.x;
        acc.y = acc.y + wk * v.y;
        acc.z = acc.z + wk * v.z;
        acc.w = acc.w + wk * v.w;
    }
    *reinterpret_cast<float4 *>(hidden + (size_t)t * H + c) = acc;
}

int max_tiles(const bread_moe_shape_t &s, int T)
{
    const int P = T * s.top_k;
    return P / MT + (P < s.n_experts ? P : s.n_experts) + (T + MT - 1) / MT;
}

// Workgroups for the items of at most `tiles` tiles of C chunks: what is
// resident at once, whole XCDs.
dim3 gg_grid(int tiles, int C, int resident)
{
    const int64_t items = (int64_t)tiles * C;
    return dim3((unsigned)(((items < resident ? (int)items : resident) + NXCD - 1) / NXCD * NXCD));
}

// exact: layers of other types than the reference GPU path's (Unit)
void launch_gateup(const GgArgs &a, int tg, int tu, bool exact, int tiles, int cus, hipStream_t st)
{
    constexpr int Q4 = BREAD_QTYPE_Q4_K, Q6 = BREAD_QTYPE_Q6_K;
    const dim3 grid = gg_grid(tiles, max(a.rows, a.rows_sh) / GU_ROWS, 2 * cus), block(GG_THREADS);
    if (!exact) hipLaunchKernelGGL((k_gateup_gg<Q4, Q4, false>), grid, block, 0, st, a);
    else if (tg == Q4 && tu == Q4) hipLaunchKernelGGL((k_gateup_gg<Q4, Q4, true>), grid, block, 0, st, a);
    else if (tg == Q4) hipLaunchKernelGGL((k_gateup_gg<Q4, Q6, true>), grid, block, 0, st, a);
    else if (tu == Q4) hipLaunchKernelGGL((k_gateup_gg<Q6, Q4, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_gateup_gg<Q6, Q6, true>), grid, block, 0, st, a);
}

void launch_down(const GgArgs &a, int td, bool exact, int tiles, int cus, hipStream_t st)
{
    constexpr int Q4 = BREAD_QTYPE_Q4_K, Q6 = BREAD_QTYPE_Q6_K;
    const dim3 grid = gg_grid(tiles, (a.rows + DN_ROWS - 1) / DN_ROWS, cus), block(DN_WAVES * WAVE);
    const bool two = a.nsb != a.nsb_sh;
    const auto kernel = !exact     ? (two ? k_down_gg<Q6, false, true> : k_down_gg<Q6, false, false>)
                        : td == Q4 ? (two ? k_down_gg<Q4, true, true> : k_down_gg<Q4, true, false>)
                                   : (two ? k_down_gg<Q6, true, true> : k_down_gg<Q6, true, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, st, a);
}

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

int bread_grouped_alloc(bread_moe_ctx_t *c)
{
    const bread_moe_shape_t &s = c->shape;
    const size_t T = (size_t)c->max_tokens, K = (size_t)s.top_k, H = (size_t)s.hidden;
    const size_t P = T * (K + 1);
    hipError_t e = hipSuccess;
    bread_grouped_ws &g = c->gws;
    e = hipDeviceGetAttribute(&g.cus, hipDeviceAttributeMultiprocessorCount, c->device);
    if (e == hipSuccess) e = hipMalloc(&g.xop, T * H * 4);
    if (e == hipSuccess) e = hipMalloc(&g.xsum, T * (H / QK) * 32);
    if (e == hipSuccess) e = hipMalloc((void **)&g.xexp, T * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void **)&g.pair_tok, P * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void **)&g.pos_of, T * K * sizeof(int));
    if (e == hipSuccess) e = hipMalloc(&g.tiles, (size_t)max_tiles(s, c->max_tokens) * sizeof(MtTile));
    if (e == hipSuccess) e = hipMalloc((void **)&g.n_tiles, 2 * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void **)&g.eo, P * H * sizeof(float));
    return e == hipSuccess ? BREAD_OK : (e == hipErrorOutOfMemory ? BREAD_ERR_NOMEM : BREAD_ERR_HIP);
}

void bread_grouped_free(bread_moe_ctx_t *c)
{
    bread_grouped_ws &g = c->gws;
    (void)hipFree(g.xop);
    (void)hipFree(g.xsum);
    (void)hipFree(g.xexp);
    (void)hipFree(g.pair_tok);
    (void)hipFree(g.pos_of);
    (void)hipFree(g.tiles);
    (void)hipFree(g.n_tiles);
    (void)hipFree(g.eo);
    g = bread_grouped_ws{};
}

bool bread_grouped_supported(const bread_moe_shape_t &s, const bread_moe_layer_t *L)
{
    if (s.expert_inter > MAX_INTER || s.shared_inter > MAX_INTER) return false;
    // 16-byte aligned down weights, which the down kernel's loads ask for
    const uintptr_t a16 = (uintptr_t)L->down_exps | (uintptr_t)L->down_shexp | L->down_expert_bytes;
    return (a16 & 15) == 0;
}

int bread_launch_moe_grouped(bread_moe_ctx_t *c, const bread_moe_layer_t *L, const float *x, float *hidden, int T,
                             hipStream_t st)
{
    const bread_moe_shape_t &s = c->shape;
    if (!bread_grouped_supported(s, L)) return BREAD_ERR_SHAPE;
    BREAD_REQUIRE(((uintptr_t)hidden & 15) == 0, BREAD_ERR_ALIGN, "hidden must be 16-byte aligned");
    const int H = s.hidden, E = s.n_experts, K = s.top_k;
    const int Imax = s.expert_inter > s.shared_inter ? s.expert_inter : s.shared_inter;
    bread_grouped_ws &g = c->gws;
    bread_clear_stale_error();
    // router logits in the reference's order (route.hip), then per token the
    // exact softmax / top-k with the activation preparation.  The shared-gate
    // score: summed in parallel there, or, for layers that keep the precision
    // of the per-token kernels, in the reference's order too
    const bool standard = bread_standard_qtypes(L);
    const uint16_t *shg = (const uint16_t *)L->shexp_gate;
    float *gsh = standard ? c->gsh : nullptr;
    {
        const int rc = bread_launch_route_logits((const float *)L->router, standard ? nullptr : shg, x, c->logits,
                                                 standard ? nullptr : c->gsh, H, E, T, !standard, st);
        if (rc) return rc;
    }
    if (!standard) shg = nullptr;
    if ((E + WAVE - 1) / WAVE <= 4)
        hipLaunchKernelGGL(k_mt_topk_xprep<4>, dim3(T), dim3(256), 0, st, c->logits, E, K, c->idx, c->w, x, shg, H, !standard,
                           (uint4 *)g.xop, (uint4 *)g.xsum, g.xexp, gsh);
    else
        hipLaunchKernelGGL(k_mt_topk_xprep<16>, dim3(T), dim3(256), 0, st, c->logits, E, K, c->idx, c->w, x, shg, H, !standard,
                           (uint4 *)g.xop, (uint4 *)g.xsum, g.xexp, gsh);
    BREAD_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_mt_bucket, dim3(1), dim3(1024), 0, st, c->idx, T, K, E, g.pair_tok, g.pos_of,
                       (MtTile *)g.tiles, g.n_tiles);
    BREAD_HIP(hipGetLastError());
    const int tiles = max_tiles(s, T);
    GgArgs a;
    a.err = &c->dsync->error.v;
    a.xop = (const uint4 *)g.xop;
    a.xsum = (const uint4 *)g.xsum;
    a.xexp = g.xexp;
    a.pair_tok = g.pair_tok;
    a.tiles = (const MtTile *)g.tiles;
    a.n_tiles = g.n_tiles;
    a.h = c->h;
    a.eo = g.eo;
    a.E = E;
    a.hstride = Imax;
    a.flag = standard ? 1 : 0;
    // one launch takes tiles of one type: the shared expert's ride along with
    // the routed ones' where they agree
    const bool one_gu = L->gate_type == L->gate_shexp_type && L->up_type == L->up_shexp_type;
    const bool one_dn = L->down_type == L->down_shexp_type;
    a.w0 = (const uint8_t *)L->gate_exps;
    a.w1 = (const uint8_t *)L->up_exps;
    a.st0 = L->gate_expert_bytes;
    a.st1 = L->up_expert_bytes;
    a.sw0 = (const uint8_t *)L->gate_shexp;
    a.sw1 = (const uint8_t *)L->up_shexp;
    a.nsb = a.nsb_sh = H / QK;
    a.rows = s.expert_inter;
    a.rows_sh = s.shared_inter;
    a.sel = one_gu ? 3 : 1;
    launch_gateup(a, L->gate_type, L->up_type, !standard, tiles, g.cus, st);
    BREAD_HIP(hipGetLastError());
    if (!one_gu) {
        a.sel = 2;
        launch_gateup(a, L->gate_shexp_type, L->up_shexp_type, !standard, tiles, g.cus, st);
        BREAD_HIP(hipGetLastError());
    }
    a.w0 = a.w1 = (const uint8_t *)L->down_exps;
    a.st0 = a.st1 = L->down_expert_bytes;
    a.sw0 = a.sw1 = (const uint8_t *)L->down_shexp;
    a.nsb = s.expert_inter / QK;
    a.nsb_sh = s.shared_inter / QK;
    a.rows = a.rows_sh = H;
    a.sel = one_dn ? 3 : 1;
    launch_down(a, L->down_type, !standard, tiles, g.cus, st);
    BREAD_HIP(hipGetLastError());
    if (!one_dn) {
        a.sel = 2;
        launch_down(a, L->down_shexp_type, !standard, tiles, g.cus, st);
        BREAD_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_mt_combine, dim3(T, (H / 4 + 255) / 256), dim3(256), 0, st, g.eo, g.pos_of, c->w, c->gsh,
                       hidden, H, K, T);
    BREAD_HIP(hipGetLastError());
    return BREAD_OK;
}
