// sph_mlp.hip - the learned macro-step ("surrogate") of libsph_hip.so.
//
// A particle-interaction network predicts each particle's displacement over
// four plain steps from its neighbourhood at the start of the macro-step:
//
//   edge features  f_ij = (dx/h, dy/h, dvx/5, dvy/5, r/h, 1)   (j within h)
//   edge MLP       e_ij = W2 SiLU(W1 f_ij)      (5 -> 64 -> 64, b1 folded
//                                                into W1 via the constant 1)
//   aggregation    m_i  = sum_j e_ij = W2 S_i + deg_i b2,  S_i = sum_j SiLU(W1 f_ij)
//   node MLP       o_i  = W4 SiLU(W3 [m_i, v_i/5, a_i/10, 1]) + b4   (68 -> 64 -> 2)
//   displacement   d_i  = 4 dt v_i + 10 dt^2 a_i + 0.05 o_i
//
// a_i is the external acceleration (sloshing, -g).  The edge MLP's second
// layer is linear, so it is applied once per particle after the sum: the
// per-edge work is W1 f_ij on MFMA plus one SiLU per hidden unit.
//
// Precision: weights and activations bf16, MFMA 16x16x16 bf16 with fp32
// accumulation, SiLU / sums / losses / Adam in fp32 (fp32 master weights).
//
// Work layout: one wavefront per 16 consecutive particles everywhere (the
// solver context's sorted slots).  The edge passes compact the group's edges
// into LDS, 16 per MFMA tile.  Every product of the node layers is taken with the
// weights as the A operand and the particles as columns, because the
// 16x16x16 MFMA returns, per lane, rows 4 (l / 16) .. + 3 of column l % 16: the
// very layout its B operand takes.  So the layers chain in registers, forward
// and backward, and where a product needs the other layout (the weight
// gradients sum over particles) the values are turned by an MFMA with the
// identity, exactly, on otherwise idle matrix cores.
#include "sph_ctx_internal.h"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <mutex>
#include <new>
#include <vector>

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) short bf16x4;

namespace {

constexpr int kH = 64;      // hidden width
constexpr int kKE = 16;     // edge input width (6 used)
constexpr int kKN = 80;     // node input width (64 + 4 + bias, padded)
constexpr unsigned kGroup = 16;         // consecutive slots per wavefront in the edge passes
constexpr unsigned kEdgeBuf = 176;      // LDS edge rows per wavefront (flushed as it fills)
constexpr unsigned kNoOwner = 16;       // owner of a padding row: no particle of the group
constexpr float kVScale = 0.2f, kAScale = 0.1f, kDScale = 0.05f;
constexpr int kTrendRefresh = 16; // forced plain macro-step per scene every this many

// parameter block (fp32 master copy)
constexpr int oW1 = 0;                  // [64][16]
constexpr int oW2 = oW1 + kH * kKE;     // [64][64]
constexpr int ob2 = oW2 + kH * kH;      // [64]
constexpr int oW3 = ob2 + kH;           // [64][80]
constexpr int oW4 = oW3 + kH * kKN;     // [2][64]
constexpr int ob4 = oW4 + 2 * kH;       // [2]
constexpr int kNParams = ob4 + 2;

// float -> bf16 bits, round to nearest even (v_cvt_pk_bf16_f32 on gfx950)
__device__ __forceinline__ unsigned short f2bf(float f)
{
    return __builtin_bit_cast(unsigned short, (__bf16)f);
}

// Logistic function from the hardware exp2 and reciprocal (1 ulp each): the
// network is trained and run with this definition on both passes.
__device__ __forceinline__ float sigm(float x)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896341f));
}

__device__ __forceinline__ float silu(float x) { return x * sigm(x); }

__device__ __forceinline__ float silu_grad(float x)
{
    const float s = sigm(x);
    return s * (1.0f + x * (1.0f - s));
}

// Two conversions an instruction (the four-wide conversion compiles to one
// each and two byte permutes).
__device__ __forceinline__ bf16x4 pack4(float a, float b, float c, float d)
{
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bfx2;
    const f32x2 lo = {a, b}, hi = {c, d};
    uint2 r;
    r.x = __builtin_bit_cast(unsigned, __builtin_convertvector(lo, bfx2));
    r.y = __builtin_bit_cast(unsigned, __builtin_convertvector(hi, bfx2));
    return __builtin_bit_cast(bf16x4, r);
}

__device__ __forceinline__ bf16x4 pack4(f32x4 v) { return pack4(v[0], v[1], v[2], v[3]); }

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ unsigned lane() { return threadIdx.x & 63u; }

// Particle-level parameters of a scene needed by the network.
struct NodeCtx {
    float h_recip, dt, g_neg, fx;
};

__device__ __forceinline__ NodeCtx node_ctx(const sph_dev_params &P, unsigned long long clock)
{
    NodeCtx c;
    c.h_recip = P.h_recip;
    c.dt = P.dt;
    c.g_neg = P.g_neg;
    c.fx = sph_slosh_accel(P, clock);
    return c;
}

// This wavefront's index in its workgroup, as a scalar: what follows from it
// (the group, its scene's parameters) is uniform and stays in scalar registers.
__device__ __forceinline__ unsigned wave_index()
{
    return (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64u));
}

// LDS edge list of one wavefront's group of kGroup consecutive slots:
// features (dx/h, dy/h, 0.2 dvx, 0.2 dvy, r/h, 1, 0, 0) as two bf16x4, and
// the owning particle (0..15 within the group; kNoOwner for padding rows).
struct EdgeBuf {
    bf16x4 f[kEdgeBuf][2];
    unsigned char owner[kEdgeBuf];
};

__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
}

// Stream every edge of the particles [n0, n0 + 16) through L (one
// wavefront).  Lane l takes every fourth candidate (from l / 16 on) of
// particle l % 16's three candidate rows (cells i-1..i+1 of rows j-1..j+1,
// contiguous in the sorted arrays) taken as one list, so that a wave runs as
// many rounds as its longest list needs; a round's records are loaded one
// round ahead, position and velocity together.  Accepted edges are appended
// to L in arbitrary order; whenever L is nearly full, flush(nedges) consumes
// its first nedges (a multiple of 16) and the remainder moves to the front.
// The final call gets the rest, padded to a multiple of 16 with zero rows of
// no owner.  Returns the degree of particle l % 16.
template <class Flush>
__device__ __forceinline__ float walk_group(unsigned n0, const sph_dev_params &P,
                                            const float2 *__restrict__ POS,
                                            const float2 *__restrict__ VEL,
                                            const unsigned *__restrict__ K,
                                            const unsigned *__restrict__ start, EdgeBuf &L,
                                            Flush &&flush)
{
    const unsigned l = lane(), p = l % 16u, sub = l / 16u;
    const unsigned me = n0 + p;
    const bool valid = me < P.poff + (unsigned)P.n;
    const unsigned mc = valid ? me : n0; // n0 is a live slot
    const float2 a = POS[mc], av = VEL[mc];
    const unsigned key = K[mc] - P.cell_base;
    const unsigned j = key / P.sx, i = key - j * P.sx;
    const unsigned lo = i > 0 ? i - 1 : 0, hi = i + 1 < P.sx ? i + 1 : P.sx - 1;
    unsigned b0[3], n[3]; // begin and length of the candidate rows
#pragma unroll
    for (int dy = 0; dy < 3; dy++) {
        const bool in = valid && (dy == 0 ? j > 0 : dy == 2 ? j + 1 < P.sy : true);
        const unsigned base = P.cell_base + (in ? j + (unsigned)dy - 1u : j) * P.sx;
        const unsigned s0 = start[base + lo], s3 = start[base + hi + 1];
        b0[dy] = s0;
        n[dy] = in ? s3 - s0 : 0u;
    }
    const unsigned n01 = n[0] + n[1], total = n01 + n[2];
    // candidate t of the lane's list (its own slot past the end)
    auto at = [&](unsigned t) {
        unsigned c = b0[0] + t;
        c = t >= n[0] ? b0[1] + (t - n[0]) : c;
        c = t >= n01 ? b0[2] + (t - n01) : c;
        return t < total ? c : mc;
    };
    unsigned count = 0, mine = 0;
    unsigned t = sub, c = at(t);
    float2 q = POS[c], qv = VEL[c];
    while (__ballot(t < total) != 0ull) {
        const unsigned tn = t + 4u, cn = at(tn);
        const float2 qn = POS[cn], qvn = VEL[cn];
        const float dx = q.x - a.x, dy = q.y - a.y;
        const float r2 = dx * dx + dy * dy;
        const bool acc = t < total && c != me && !(r2 > P.h2);
        const unsigned long long m = __ballot(acc);
        const float rr = sph_sqrt(r2);
        if (acc) {
            const unsigned pos =
                __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)m, count));
            L.f[pos][0] = pack4(dx * P.h_recip, dy * P.h_recip, (qv.x - av.x) * kVScale,
                                (qv.y - av.y) * kVScale);
            L.f[pos][1] = pack4(rr * P.h_recip, 1.0f, 0.0f, 0.0f);
            L.owner[pos] = (unsigned char)p;
            mine++;
        }
        count += (unsigned)__popcll(m);
        if (count > kEdgeBuf - 64u) { // the next round might not fit: flush full tiles
            wave_lds_order();
            const unsigned full = count & ~15u, rem = count - full;
            flush(full);
            wave_lds_order();
            bf16x4 f0 = pack4(0, 0, 0, 0), f1 = f0;
            unsigned char ow = kNoOwner;
            if (l < rem) {
                f0 = L.f[full + l][0];
                f1 = L.f[full + l][1];
                ow = L.owner[full + l];
            }
            wave_lds_order();
            if (l < rem) {
                L.f[l][0] = f0;
                L.f[l][1] = f1;
                L.owner[l] = ow;
            }
            count = rem;
        }
        t = tn;
        c = cn;
        q = qn;
        qv = qvn;
    }
    // the rest, padded to a whole 16-edge tile
    const unsigned padded = (count + 15u) & ~15u;
    if (count + l < padded) {
        L.f[count + l][0] = pack4(0, 0, 0, 0);
        L.f[count + l][1] = pack4(0, 0, 0, 0);
        L.owner[count + l] = kNoOwner;
    }
    wave_lds_order();
    if (padded)
        flush(padded);
    float fm = (float)mine;
    fm += __shfl_xor(fm, 16, 64);
    fm += __shfl_xor(fm, 32, 64);
    wave_lds_order();
    return fm;
}

// A operand of an edge tile: lane l holds edge e0 + l%16, features 4*(l/16)
// .. +3.  Features 8..15 are zero in the model; those lanes read the first eight
// again, against weights that w1_bits makes zero.
__device__ __forceinline__ bf16x4 edge_tile_a(const EdgeBuf &L, unsigned e0)
{
    return L.f[e0 + lane() % 16u][(lane() / 16u) & 1u];
}

// Membership of the tile's edges e0 + 4*(l/16) .. +3 in particle l%16 (1 or
// 0): the B operand of the sum over edges.  The four owners are compared as
// one word (they and the particle are at most 16, so no byte carries into the
// next): z has 0x80 in the bytes that match, and 0x3f80, bf16 1, follows from
// it by shifts.
__device__ __forceinline__ bf16x4 member(const EdgeBuf &L, unsigned e0)
{
    const unsigned w = *(const unsigned *)&L.owner[e0 + 4u * (lane() / 16u)];
    const unsigned x = w ^ (lane() % 16u) * 0x01010101u;
    const unsigned z = ((x + 0x7f7f7f7fu) & 0x80808080u) ^ 0x80808080u;
    const unsigned h = (z >> 1) - (z >> 7);
    uint2 r;
    r.x = __builtin_amdgcn_perm(h, z, 0x05010400u);
    r.y = __builtin_amdgcn_perm(h, z, 0x07030602u);
    return __builtin_bit_cast(bf16x4, r);
}

// One-hot A operand of the expansion of particles to a tile's edges: lane l
// holds edge e0 + l%16, particles 4*(l/16) .. +3.
__device__ __forceinline__ bf16x4 one_hot(unsigned own)
{
    const unsigned k = own - 4u * (lane() / 16u); // 0..3 when the owner is one of them
    uint2 r;
    r.x = k < 2u ? 0x3f80u << (16u * k) : 0u;
    r.y = k - 2u < 2u ? 0x3f80u << (16u * (k - 2u)) : 0u;
    return __builtin_bit_cast(bf16x4, r);
}

// The identity as a B operand, and a tile turned by it: x holds, per lane,
// rows 4*(l/16) .. +3 of column l%16; the result columns 4*(l/16) .. +3 of row
// l%16, of the same (bf16) values.
__device__ __forceinline__ bf16x4 identity_b() { return one_hot(lane() % 16u); }

__device__ __forceinline__ bf16x4 turn(bf16x4 x, bf16x4 eye)
{
    f32x4 d = {0, 0, 0, 0};
    return pack4(mfma(x, eye, d));
}

// B operand of W1^T for hidden-unit tile t: B[k][c] = W1[16t + c][k].
__device__ __forceinline__ bf16x4 w1_b(const unsigned short *W1b, int t)
{
    const unsigned c = 16u * t + lane() % 16u, k = 4u * (lane() / 16u);
    return *(const bf16x4 *)(W1b + c * kKE + k);
}

// The edge sums of a group: acc[t] += SiLU(W1 f)^T over the first ne edges,
// per lane hidden units 16t + 4*(l/16) .. +3 of particle l%16.  A tile's four
// pre-activations come first, so that their SiLUs interleave.
__device__ __forceinline__ void edge_sums(const EdgeBuf &L, unsigned ne, const bf16x4 B[4],
                                          f32x4 acc[4])
{
    for (unsigned e0 = 0; e0 < ne; e0 += 16) {
        const bf16x4 a = edge_tile_a(L, e0);
        const bf16x4 mem = member(L, e0);
        const f32x4 zero = {0, 0, 0, 0};
        f32x4 d[4];
#pragma unroll
        for (int t = 0; t < 4; t++)
            d[t] = mfma(a, B[t], zero);
#pragma unroll
        for (int t = 0; t < 4; t++)
            // D (edges 4*(l/16)+q, unit 16t + l%16) is the A layout of the sum
            acc[t] = mfma(pack4(silu(d[t][0]), silu(d[t][1]), silu(d[t][2]), silu(d[t][3])), mem,
                          acc[t]);
    }
}

} // namespace

struct sph_surrogate {
    size_t slots = 0;
    float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
    unsigned short *W1b = nullptr, *W2b = nullptr, *W3b = nullptr;
    float *deg = nullptr, *disp = nullptr, *tgt = nullptr;
    // training, bf16 as the products take them, [group][tile][lane]: the edge
    // sums (particles as columns) and their gradients (particles as rows)
    bf16x4 *S = nullptr, *dS = nullptr;
    float *part = nullptr; // the workgroups' partial gradients
    float *loss = nullptr;
    float2 *tmp2 = nullptr;
    int adam_t = 0;
    bool have_pred = false;
    // judge state (per scene)
    size_t ns = 0;
    float *ref = nullptr, *jsum = nullptr;
    float *jmax = nullptr;
    int *jflags = nullptr;
    const sph_ctx *ref_ctx = nullptr;
    bool ref_ok = false;
    unsigned long long macro = 0; // judged macro-steps so far (the refresh / shadow schedule)
    // shadow judging: 1 of every shadow_every scenes (rotating) also takes
    // the macro-step plainly from the same start; 0 = off
    int shadow_every = 0;
    float *sh_sum = nullptr;              // per scene: the plain shadow's density sum
    float *rho_plain = nullptr, *rho_sur = nullptr; // density by caller index, of
    size_t rho_slots = 0;                           // contexts of up to so many slots
    float *sh_err = nullptr;              // per scene: sum (sur - plain)^2, sum plain^2
    double sh_stats[8] = {0};             // see sph_surrogate_shadow_stats
};

struct sph_trajectory {
    int nscenes = 0, n = 0, frames = 0;
    float4 *data = nullptr;    // [frames][nscenes][n]
    float4 *staging = nullptr; // [cap_samples * n]
    float2 *target = nullptr;  // [cap_samples * n]
    int *idx = nullptr;        // scene[cap], frame[cap]
    int cap = 0, loaded = 0;
};

// ---------------------------------------------------------------------------
// kernels

// MFMA lane-layout self-test: D = A B for fixed small-integer A, B
// (exact in bf16), written row-major as the layout assumed above reads it.
__global__ void k_mfma_selftest(float *D)
{
    const unsigned l = lane();
    bf16x4 a, b;
    for (int q = 0; q < 4; q++) {
        const unsigned row = l % 16u, k = 4u * (l / 16u) + q;
        a[q] = (short)f2bf((float)((int)((row * 16u + k) % 7u) - 3));
        const unsigned kk = 4u * (l / 16u) + q, col = l % 16u;
        b[q] = (short)f2bf((float)((int)((kk * 3u + col) % 5u) - 2));
    }
    f32x4 d = {0, 0, 0, 0};
    d = mfma(a, b, d);
    for (int q = 0; q < 4; q++)
        D[(4u * (l / 16u) + q) * 16u + l % 16u] = d[q];
}

// Edge forward of training: S_i = sum_j SiLU(W1 f_ij) and deg_i.  One
// wavefront per group of 16 slots: the group's edges are compacted into LDS,
// each 16-edge tile runs W1 on MFMA (4 hidden tiles), SiLU, and the
// per-particle sum as a second MFMA against the tile's membership matrix.
// Bound by VALU issue (per tile 16 SiLUs a lane: two transcendentals and three
// instructions each); a launch bound of more than one workgroup keeps the
// MFMA results out of accumulation registers, which cost a read each.  A
// million particles of 17 neighbours: 0.82 -> 0.41 ms.
__global__ void __launch_bounds__(256, 4)
k_edge_fwd(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned slots,
           const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
           const unsigned *__restrict__ K, const unsigned *__restrict__ start,
           const unsigned short *__restrict__ W1b, bf16x4 *__restrict__ S,
           float *__restrict__ deg)
{
    __shared__ __align__(16) EdgeBuf Lb[4];
    const unsigned w = wave_index(), l = lane();
    EdgeBuf &L = Lb[w];
    bf16x4 B[4];
    for (int t = 0; t < 4; t++)
        B[t] = w1_b(W1b, t);
    const unsigned ngroups = slots / kGroup, nw = gridDim.x * 4u;
    for (unsigned g = blockIdx.x * 4u + w; g < ngroups; g += nw) {
        const unsigned n0 = g * kGroup;
        const sph_dev_params P = Pp[BS[n0 / kSphTPB]];
        if (n0 >= P.poff + (unsigned)P.n)
            continue;
        f32x4 acc[4];
        for (int t = 0; t < 4; t++)
            acc[t] = {0, 0, 0, 0};
        const float dg = walk_group(n0, P, POS, VEL, K, start, L,
                                    [&](unsigned ne) { edge_sums(L, ne, B, acc); });
        for (int t = 0; t < 4; t++)
            S[((size_t)g * 4u + t) * 64u + l] = pack4(acc[t]);
        if (l < 16u)
            deg[n0 + l] = dg;
    }
}

namespace {

// Node-layer weights staged in LDS once per workgroup.  A lane reads 8-byte
// pieces of row l%16 of a weight matrix; the rows are 4 shorts longer than the
// matrix, so that a wave's reads fall on different banks.
constexpr unsigned kS2 = kH + 4, kS3 = kKN + 4; // row strides
struct NodeW {
    unsigned short W2[kH * kS2];
    unsigned short W3[kH * kS3];
    float b2[kH], W4[2 * kH], b4[2];
};
// W2 and the first 64 columns of W3 with rows and columns exchanged.
struct NodeWT {
    unsigned short W2[kH * kS2];
    unsigned short W3[kH * kS2];
};

// Ends without a barrier.
__device__ void stage_node_weights(NodeW &sw, const unsigned short *W2b,
                                   const unsigned short *W3b, const float *params)
{
    for (unsigned i = threadIdx.x; i < kH * kH / 4u; i += blockDim.x)
        *(uint2 *)&sw.W2[i / (kH / 4u) * kS2 + i % (kH / 4u) * 4u] = ((const uint2 *)W2b)[i];
    for (unsigned i = threadIdx.x; i < kH * kKN / 4u; i += blockDim.x)
        *(uint2 *)&sw.W3[i / (kKN / 4u) * kS3 + i % (kKN / 4u) * 4u] = ((const uint2 *)W3b)[i];
    for (unsigned i = threadIdx.x; i < kH; i += blockDim.x)
        sw.b2[i] = params[ob2 + i];
    for (unsigned i = threadIdx.x; i < 2u * kH; i += blockDim.x)
        sw.W4[i] = params[oW4 + i];
    if (threadIdx.x < 2u)
        sw.b4[threadIdx.x] = params[ob4 + threadIdx.x];
}

__device__ void stage_turned_weights(NodeWT &sw, const unsigned short *W2b,
                                     const unsigned short *W3b)
{
    for (unsigned i = threadIdx.x; i < kH * kH; i += blockDim.x) {
        const unsigned r = i / kH, c = i % kH;
        sw.W2[c * kS2 + r] = W2b[r * kH + c];
        sw.W3[c * kS2 + r] = W3b[r * kKN + c];
    }
}

// A operand: row 16t + l%16, columns 16kc + 4*(l/16) .. +3.
template <unsigned STRIDE>
__device__ __forceinline__ bf16x4 weight_a(const unsigned short *W, int t, int kc)
{
    return *(const bf16x4 *)(W + (16u * t + lane() % 16u) * STRIDE + 16u * kc +
                             4u * (lane() / 16u));
}

// Four floats of units 16t + 4*(l/16) .. +3.
__device__ __forceinline__ f32x4 unit4(const float *v, int t)
{
    return *(const f32x4 *)(v + 16u * t + 4u * (lane() / 16u));
}

// Node-pass state of one 16-particle group held by one wavefront: per lane
// units 16t + 4*(l/16) .. +3 of particle l%16.
struct NodeTile {
    bf16x4 u[5];   // node input [m, 0.2 v, 0.1 a, 1, 0 ..]
    f32x4 pre3[4];
    float out[2];  // every lane of the particle
};

// The node forward from the edge sums S and degree of particle l%16 (velocity
// v; not ok: no particle, all zero).
__device__ __forceinline__ void node_forward(const bf16x4 S[4], float deg, bool ok, float2 v,
                                             const NodeCtx &nc, const NodeW &sw, NodeTile &T)
{
    const unsigned sub = lane() / 16u;
    // m = W2 S + deg b2
#pragma unroll
    for (int t = 0; t < 4; t++) {
        f32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (int kc = 0; kc < 4; kc++)
            d = mfma(weight_a<kS2>(sw.W2, t, kc), S[kc], d);
        const f32x4 b2 = unit4(sw.b2, t);
        T.u[t] = pack4(ok ? d[0] + deg * b2[0] : 0.0f, ok ? d[1] + deg * b2[1] : 0.0f,
                       ok ? d[2] + deg * b2[2] : 0.0f, ok ? d[3] + deg * b2[3] : 0.0f);
    }
    // node features, bias column, padding
    const bool f0 = ok && sub == 0u;
    T.u[4] = pack4(f0 ? v.x * kVScale : ok && sub == 1u ? 1.0f : 0.0f, f0 ? v.y * kVScale : 0.0f,
                   f0 ? nc.fx * kAScale : 0.0f, f0 ? nc.g_neg * kAScale : 0.0f);
    // pre3 = W3 u; out = W4 SiLU(pre3) + b4
    float o0 = 0.0f, o1 = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        f32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (int kc = 0; kc < 5; kc++)
            d = mfma(weight_a<kS3>(sw.W3, t, kc), T.u[kc], d);
        T.pre3[t] = d;
        const f32x4 w0 = unit4(sw.W4, t), w1 = unit4(sw.W4 + kH, t);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float z = silu(d[q]);
            o0 += z * w0[q];
            o1 += z * w1[q];
        }
    }
    o0 += __shfl_xor(o0, 16, 64);
    o1 += __shfl_xor(o1, 16, 64);
    o0 += __shfl_xor(o0, 32, 64);
    o1 += __shfl_xor(o1, 32, 64);
    T.out[0] = o0 + sw.b4[0];
    T.out[1] = o1 + sw.b4[1];
}

__device__ __forceinline__ float2 ballistic(const NodeCtx &nc, float2 v)
{
    // four steps of v += a dt; x += v dt from rest of interactions
    return make_float2(4.0f * nc.dt * v.x + 10.0f * nc.dt * nc.dt * nc.fx,
                       4.0f * nc.dt * v.y + 10.0f * nc.dt * nc.dt * nc.g_neg);
}

} // namespace

// Inference: the edge pass and the node MLP of each 16-slot group in one
// kernel; everything between the edge list and the displacement stays in
// registers.  Bound by VALU issue, of which the edges' SiLUs are the largest
// part; 64 scenes of 16,384 particles (17 neighbours each) take 0.49 ms, 0.82
// with the layers' values turned through LDS (weight rows on the same banks,
// 32 lane permutes for the output layer), half-width conversions, the MFMA
// results in accumulation registers, two dependent global loads a round, and
// eight groups a wave.
__global__ void __launch_bounds__(256, 3)
k_infer(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned slots,
        const unsigned long long *__restrict__ clock, const float2 *__restrict__ POS,
        const float2 *__restrict__ VEL, const unsigned *__restrict__ K,
        const unsigned *__restrict__ start, const unsigned short *__restrict__ W1b,
        const unsigned short *__restrict__ W2b, const float *__restrict__ params,
        const unsigned short *__restrict__ W3b, float2 *__restrict__ disp)
{
    __shared__ __align__(16) EdgeBuf Lb[4];
    __shared__ __align__(16) NodeW sw;
    stage_node_weights(sw, W2b, W3b, params);
    __syncthreads();
    const unsigned w = wave_index(), l = lane(), p = l % 16u;
    EdgeBuf &L = Lb[w];
    bf16x4 B[4];
    for (int t = 0; t < 4; t++)
        B[t] = w1_b(W1b, t);
    const unsigned ngroups = slots / kGroup, nw = gridDim.x * 4u;
    const unsigned long long ck = *clock;
    for (unsigned g = blockIdx.x * 4u + w; g < ngroups; g += nw) {
        const unsigned n0 = g * kGroup;
        const sph_dev_params P = Pp[BS[n0 / kSphTPB]];
        const unsigned vend = P.poff + (unsigned)P.n;
        if (n0 >= vend)
            continue;
        f32x4 acc[4];
        for (int t = 0; t < 4; t++)
            acc[t] = {0, 0, 0, 0};
        const float dg = walk_group(n0, P, POS, VEL, K, start, L,
                                    [&](unsigned ne) { edge_sums(L, ne, B, acc); });
        bf16x4 S[4];
        for (int t = 0; t < 4; t++)
            S[t] = pack4(acc[t]);
        const bool ok = n0 + p < vend;
        const float2 v = ok ? VEL[n0 + p] : make_float2(0, 0);
        const NodeCtx nc = node_ctx(P, ck);
        NodeTile T;
        node_forward(S, dg, ok, v, nc, sw, T);
        if (l < 16u && ok) {
            const float2 b = ballistic(nc, v);
            disp[n0 + p] = make_float2(b.x + kDScale * T.out[0], b.y + kDScale * T.out[1]);
        }
    }
}

// Node backward: loss, and the gradients of W2, b2, W3, W4, b4 and of the edge
// sums.  One wavefront per group runs the node forward again and the layers
// back, all in registers; the weight gradients dW3 (64x80) = sum dPre3^T U and
// dW2 (64x64) = sum dM^T S sum over particles, so each wave leaves its group's
// four factors, turned, in LDS, and then takes 9 of the 36 output tiles over
// the workgroup's four groups.  (With the factors written to memory, 350 bytes
// a particle, and a second kernel for the products: 0.84 ms for a million
// particles, 0.18 now.)  tgt holds the target displacement per slot.
constexpr int kFactors = 4 + 5 + 4 + 4; // dPre3, U, dM, S tiles of a group
constexpr unsigned kNodeTiles = 36 * 256;    // partial dW3 and dW2 of a workgroup, by tile and lane
constexpr unsigned kNodeRest = 3 * kH + 4;   // dW4 (two rows), db2, db4, loss, 0
constexpr unsigned kNodePart = kNodeTiles + kNodeRest;
__global__ void __launch_bounds__(256, 2)
k_node_grad(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned slots,
            const unsigned long long *__restrict__ clock, const float2 *__restrict__ VEL,
            const bf16x4 *__restrict__ S, const float *__restrict__ deg,
            const unsigned short *__restrict__ W2b, const float *__restrict__ params,
            const unsigned short *__restrict__ W3b, const float2 *__restrict__ tgt, float inv_n,
            bf16x4 *__restrict__ dS, float *__restrict__ part)
{
    __shared__ __align__(16) NodeW sw;
    __shared__ __align__(16) NodeWT st;
    __shared__ bf16x4 fac[4][kFactors][64];
    stage_node_weights(sw, W2b, W3b, params);
    stage_turned_weights(st, W2b, W3b);
    __syncthreads();
    const unsigned w = wave_index(), l = lane(), p = l % 16u, sub = l / 16u;
    const unsigned ngroups = slots / kGroup; // a multiple of 16
    const unsigned long long ck = *clock;
    const bf16x4 eye = identity_b();
    const f32x4 zero = {0, 0, 0, 0};
    f32x4 gW[9]; // output tiles w, w + 4, ...: the first 20 of dW3, the others of dW2
    f32x4 gW4[2][4], gb2[4];
    for (int i = 0; i < 9; i++)
        gW[i] = zero;
    for (int t = 0; t < 4; t++)
        gW4[0][t] = gW4[1][t] = gb2[t] = zero;
    float gb4[2] = {0, 0}, lsum = 0.0f;
    for (unsigned g0 = blockIdx.x * 4u; g0 < ngroups; g0 += gridDim.x * 4u) {
        const unsigned g = g0 + w, n0 = g * kGroup;
        const sph_dev_params P = Pp[BS[n0 / kSphTPB]];
        const unsigned vend = P.poff + (unsigned)P.n;
        const bool any = n0 < vend, ok = n0 + p < vend; // no particles: all factors zero
        bf16x4 Sb[4];
        for (int t = 0; t < 4; t++)
            Sb[t] = any ? S[((size_t)g * 4u + t) * 64u + l] : pack4(zero);
        const float dg = ok ? deg[n0 + p] : 0.0f;
        const float2 v = ok ? VEL[n0 + p] : make_float2(0, 0);
        const float2 y = ok ? tgt[n0 + p] : make_float2(0, 0);
        const NodeCtx nc = node_ctx(P, ck);
        NodeTile T;
        node_forward(Sb, dg, ok, v, nc, sw, T);
        // loss = mean over particles of |d - y|^2 / kDScale^2
        const float2 b = ballistic(nc, v);
        const float ex = (b.x + kDScale * T.out[0] - y.x) / kDScale;
        const float ey = (b.y + kDScale * T.out[1] - y.y) / kDScale;
        const float dout0 = ok ? 2.0f * ex * inv_n : 0.0f, dout1 = ok ? 2.0f * ey * inv_n : 0.0f;
        if (ok && sub == 0u) {
            lsum += (ex * ex + ey * ey) * inv_n;
            gb4[0] += dout0;
            gb4[1] += dout1;
        }
        // dW4, dPre3
        bf16x4 dP[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const f32x4 w0 = unit4(sw.W4, t), w1 = unit4(sw.W4 + kH, t);
            float dp[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float x = T.pre3[t][q], s = sigm(x);
                gW4[0][t][q] += dout0 * (x * s);
                gW4[1][t][q] += dout1 * (x * s);
                dp[q] = (dout0 * w0[q] + dout1 * w1[q]) * (s * (1.0f + x * (1.0f - s)));
            }
            dP[t] = pack4(dp[0], dp[1], dp[2], dp[3]);
        }
        // dm = W3^T dPre3 (the first 64 inputs), db2; dS = W2^T dm
        bf16x4 dM[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            f32x4 d = zero;
#pragma unroll
            for (int kc = 0; kc < 4; kc++)
                d = mfma(weight_a<kS2>(st.W3, t, kc), dP[kc], d);
            for (int q = 0; q < 4; q++)
                gb2[t][q] += dg * d[q];
            dM[t] = pack4(d);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            f32x4 d = zero;
#pragma unroll
            for (int kc = 0; kc < 4; kc++)
                d = mfma(weight_a<kS2>(st.W2, t, kc), dM[kc], d);
            if (any)
                dS[((size_t)g * 4u + t) * 64u + l] = turn(pack4(d), eye);
        }
        // the factors of the weight gradients, units as rows
#pragma unroll
        for (int t = 0; t < 4; t++) {
            fac[w][t][l] = turn(dP[t], eye);
            fac[w][9 + t][l] = turn(dM[t], eye);
            fac[w][13 + t][l] = turn(Sb[t], eye);
        }
#pragma unroll
        for (int t = 0; t < 5; t++)
            fac[w][4 + t][l] = turn(T.u[t], eye);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 9; i++) {
            const unsigned ot = w + 4u * i; // 0..35
            const bool w3 = i < 5;          // ot < 20
            const unsigned fa = w3 ? ot / 5u : 9u + (ot - 20u) / 4u;
            const unsigned fb = w3 ? 4u + ot % 5u : 13u + (ot - 20u) % 4u;
#pragma unroll
            for (int k = 0; k < 4; k++)
                gW[i] = mfma(fac[k][fa][l], fac[k][fb][l], gW[i]);
        }
        __syncthreads(); // the next groups' factors overwrite these
    }
    // this workgroup's partial gradients, to be summed by k_grad_sum
    float *out = part + (size_t)blockIdx.x * kNodePart;
#pragma unroll
    for (int i = 0; i < 9; i++)
        *(f32x4 *)&out[((w + 4u * i) * 64u + l) * 4u] = gW[i];
    // sums over the 16 particles of a row of lanes, then over the waves
    auto over_particles = [](float v) {
        for (int x = 1; x < 16; x <<= 1)
            v += __shfl_xor(v, x, 64);
        return v;
    };
    float(*rest)[kNodeRest] = (float(*)[kNodeRest]) & fac[0][0][0];
    for (int t = 0; t < 4; t++)
        for (int q = 0; q < 4; q++) {
            const float a = over_particles(gW4[0][t][q]), c = over_particles(gW4[1][t][q]);
            const float d = over_particles(gb2[t][q]);
            if (p == 0u) {
                const unsigned unit = 16u * t + 4u * sub + q;
                rest[w][unit] = a;
                rest[w][kH + unit] = c;
                rest[w][2u * kH + unit] = d;
            }
        }
    const float b0 = over_particles(gb4[0]), b1 = over_particles(gb4[1]);
    const float ls = over_particles(lsum);
    if (l < 4u)
        rest[w][3u * kH + l] = l == 0u ? b0 : l == 1u ? b1 : l == 2u ? ls : 0.0f;
    __syncthreads();
    for (unsigned i = threadIdx.x; i < kNodeRest; i += blockDim.x)
        out[kNodeTiles + i] = (rest[0][i] + rest[1][i]) + (rest[2][i] + rest[3][i]);
}

// Edge backward: dW1 += sum over edges of (dS_i * SiLU'(W1 f_ij)) f_ij^T.
// Same groups and tiles as the forward; dS_i is expanded to the tile's edges
// by an MFMA of the one-hot edge->particle matrix with the group's dS, whose
// D layout equals that of the recomputed pre-activations, and the product
// with SiLU' is, in that layout, the A operand of dW1 += dPre1^T F.  The waves
// of a workgroup add their dW1 in LDS and leave it as a partial gradient.  A
// million particles: 0.96 -> 0.57 ms.
constexpr unsigned kEdgePart = kH * 6; // partial dW1 of a workgroup
__global__ void __launch_bounds__(256, 4)
k_edge_bwd(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned slots,
           const float2 *__restrict__ POS, const float2 *__restrict__ VEL,
           const unsigned *__restrict__ K, const unsigned *__restrict__ start,
           const unsigned short *__restrict__ W1b, const bf16x4 *__restrict__ dS,
           float *__restrict__ part)
{
    __shared__ __align__(16) EdgeBuf Lb[4];
    __shared__ float gl[4][kEdgePart];
    const unsigned w = wave_index(), l = lane(), p = l % 16u, sub = l / 16u;
    EdgeBuf &L = Lb[w];
    bf16x4 B[4];
    for (int t = 0; t < 4; t++)
        B[t] = w1_b(W1b, t);
    const bf16x4 eye = identity_b();
    const f32x4 zero = {0, 0, 0, 0};
    f32x4 g[4];
    for (int t = 0; t < 4; t++)
        g[t] = zero;
    const unsigned ngroups = slots / kGroup, nw = gridDim.x * 4u;
    for (unsigned gi = blockIdx.x * 4u + w; gi < ngroups; gi += nw) {
        const unsigned n0 = gi * kGroup;
        const sph_dev_params P = Pp[BS[n0 / kSphTPB]];
        if (n0 >= P.poff + (unsigned)P.n)
            continue;
        bf16x4 Bds[4]; // B operand of the expansion: dS[particle 4*sub+i][unit 16t+p]
        for (int t = 0; t < 4; t++)
            Bds[t] = dS[((size_t)gi * 4u + t) * 64u + l];
        auto tiles = [&](unsigned ne) {
            for (unsigned e0 = 0; e0 < ne; e0 += 16) {
                const bf16x4 a = edge_tile_a(L, e0);
                const bf16x4 oh = one_hot(L.owner[e0 + p]);
                // B operand of the gradient product: F[edge 4*sub+i][feature p]
                const bf16x4 f = turn(a, eye);
                f32x4 d[4], ds[4];
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    d[t] = mfma(a, B[t], zero);
                    ds[t] = mfma(oh, Bds[t], zero);
                }
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    float gp[4];
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        gp[q] = ds[t][q] * silu_grad(d[t][q]);
                    g[t] = mfma(pack4(gp[0], gp[1], gp[2], gp[3]), f, g[t]);
                }
            }
        };
        walk_group(n0, P, POS, VEL, K, start, L, tiles);
    }
    if (p < 6u)
        for (int t = 0; t < 4; t++)
            for (int q = 0; q < 4; q++)
                gl[w][(16u * t + 4u * sub + q) * 6u + p] = g[t][q];
    __syncthreads();
    for (unsigned i = threadIdx.x; i < kEdgePart; i += blockDim.x)
        part[(size_t)blockIdx.x * kEdgePart + i] =
            (gl[0][i] + gl[1][i]) + (gl[2][i] + gl[3][i]);
}

// Sum the partial gradients of `rows` workgroups into grads (and the loss):
// block (x, y) takes 64 columns of four and the rows of chunk y, 16 rows at a
// time, and adds its sums.  A million particles' gradients by atomics straight
// from the workgroups were 4.7 million of them on 9,600 addresses.
template <bool NODE>
__global__ void __launch_bounds__(1024)
k_grad_sum(const float *__restrict__ part, unsigned rows, unsigned chunk,
           float *__restrict__ grads, float *__restrict__ loss)
{
    constexpr unsigned kCols = NODE ? kNodePart : kEdgePart;
    __shared__ f32x4 red[16][64];
    const unsigned c = threadIdx.x % 64u, s = threadIdx.x / 64u;
    const unsigned col = (blockIdx.x * 64u + c) * 4u;
    const unsigned r1 = min(rows, (blockIdx.y + 1u) * chunk);
    f32x4 v = {0, 0, 0, 0};
    if (col < kCols)
        for (unsigned r = blockIdx.y * chunk + s; r < r1; r += 16u)
            v += *(const f32x4 *)&part[(size_t)r * kCols + col];
    red[s][c] = v;
    __syncthreads();
    if (s != 0u || col >= kCols)
        return;
    for (unsigned k = 1; k < 16u; k++)
        v += red[k][c];
    for (unsigned q = 0; q < 4u; q++) {
        const unsigned i = col + q;
        if (!NODE) {
            atomicAdd(&grads[oW1 + i / 6u * kKE + i % 6u], v[q]);
        } else if (i < kNodeTiles) {
            // tile i / 256, lane (i / 4) % 64, register q: the D layout
            const unsigned ot = i / 256u, ln = i / 4u % 64u;
            const unsigned mt = ot < 20u ? ot / 5u : (ot - 20u) / 4u;
            const unsigned nt = ot < 20u ? ot % 5u : (ot - 20u) % 4u;
            const unsigned r = 16u * mt + 4u * (ln / 16u) + q, k = 16u * nt + ln % 16u;
            atomicAdd(&grads[ot < 20u ? oW3 + r * kKN + k : oW2 + r * kH + k], v[q]);
        } else {
            const unsigned k = i - kNodeTiles;
            if (k < 2u * kH)
                atomicAdd(&grads[oW4 + k], v[q]);
            else if (k < 3u * kH)
                atomicAdd(&grads[ob2 + k - 2u * kH], v[q]);
            else if (k < 3u * kH + 2u)
                atomicAdd(&grads[ob4 + k - 3u * kH], v[q]);
            else if (k == 3u * kH + 2u)
                atomicAdd(loss, v[q]);
        }
    }
}

// The bf16 copy of W1's weight i.  The padding columns 8..15 stand against
// repeated features (edge_tile_a) and take no part whatever a caller set them to:
// zero, or NaN where zero times the weight is NaN.  (Here it costs nothing; when
// every wave of the edge kernels did it for its operand, 64 scenes of 16,384
// particles took 887 us to predict instead of 871, 1330 to train instead of 1313.)
__device__ __forceinline__ unsigned short w1_bits(int i, float x)
{
    const unsigned short w = f2bf(x);
    return i % kKE < 8 ? w : (w & 0x7f80u) == 0x7f80u ? 0x7fc0u : 0u;
}

// Adam on the fp32 master weights, then refresh the bf16 copies.  Weights
// of the padding columns (W1 beyond 6 inputs, W3 beyond 69) stay as they are.
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2, unsigned short *__restrict__ W1b,
                       unsigned short *__restrict__ W2b, unsigned short *__restrict__ W3b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    bool live = true;
    if (i >= oW1 && i < oW2)
        live = (i - oW1) % kKE < 6;
    else if (i >= oW3 && i < oW4)
        live = (i - oW3) % kKN < 69;
    float x = p[i];
    if (live) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        x -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        p[i] = x;
    }
    if (i >= oW1 && i < oW2)
        W1b[i - oW1] = w1_bits(i - oW1, x);
    else if (i >= oW2 && i < ob2)
        W2b[i - oW2] = f2bf(x);
    else if (i >= oW3 && i < oW4)
        W3b[i - oW3] = f2bf(x);
}

__global__ void k_to_bf16(const float *__restrict__ p, unsigned short *__restrict__ W1b,
                          unsigned short *__restrict__ W2b, unsigned short *__restrict__ W3b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= oW1 && i < oW2)
        W1b[i - oW1] = w1_bits(i - oW1, p[i]);
    else if (i >= oW2 && i < ob2)
        W2b[i - oW2] = f2bf(p[i]);
    else if (i >= oW3 && i < oW4)
        W3b[i - oW3] = f2bf(p[i]);
}

// by-id (concatenated caller order) -> slot order, and back.
__global__ void k_by_id_to_slot(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                                unsigned slots, const int *__restrict__ ID,
                                const float2 *__restrict__ by_id, float2 *__restrict__ by_slot)
{
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots)
        return;
    const sph_dev_params &P = Pp[BS[s / kSphTPB]];
    if (s < P.poff + (unsigned)P.n)
        by_slot[s] = by_id[P.uoff + (unsigned)ID[s]];
}

__global__ void k_slot_to_by_id(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                                unsigned slots, const int *__restrict__ ID,
                                const float2 *__restrict__ by_slot, float2 *__restrict__ by_id)
{
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots)
        return;
    const sph_dev_params &P = Pp[BS[s / kSphTPB]];
    if (s < P.poff + (unsigned)P.n)
        by_id[P.uoff + (unsigned)ID[s]] = by_slot[s];
}

// Apply a predicted macro-step: x += d (then the box clamp of
// src/fluid.c:729-743), v = d / (4 dt) + 1.5 a dt (the last step's velocity
// under constant acceleration), clamped like src/fluid.c:613-625.
__global__ void k_apply(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS,
                        unsigned slots, const unsigned long long *__restrict__ clock,
                        const float2 *__restrict__ disp, float2 *__restrict__ POS,
                        float2 *__restrict__ VEL)
{
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots)
        return;
    const sph_dev_params &P = Pp[BS[s / kSphTPB]];
    if (s >= P.poff + (unsigned)P.n || P.frozen)
        return;
    const NodeCtx nc = node_ctx(P, *clock);
    const float2 d = disp[s];
    float2 p = POS[s];
    p.x += d.x;
    p.y += d.y;
    if (p.x < P.min_x)
        p.x = P.min_x;
    else if (p.x > P.max_x)
        p.x = P.max_x - 0.001f;
    if (p.y < P.min_y)
        p.y = P.min_y;
    else if (p.y > P.max_y)
        p.y = P.max_y - 0.001f;
    float vx = d.x / (4.0f * nc.dt) + 1.5f * nc.fx * nc.dt;
    float vy = d.y / (4.0f * nc.dt) + 1.5f * nc.g_neg * nc.dt;
    sph_check_velocity(vx, vy);
    POS[s] = p;
    VEL[s] = make_float2(vx, vy);
}

__global__ void k_clock_add(unsigned long long *clock, unsigned long long n)
{
    *clock += n; // one thread: a plain vector load/store pair
}

// Per-scene density sums and maxima of the last density pass: one
// workgroup per scene over its slots, no atomics (deterministic).  A scene's
// range begins at a multiple of 256 slots; a thread takes two particles a
// load and four loads at a time, so that a scene is a few memory round trips:
// 17 us for scenes of 65,536 particles, against 65 with one particle a load
// and 256 threads.
constexpr unsigned kDensityTPB = 1024;
__global__ void __launch_bounds__(kDensityTPB)
k_scene_density(const sph_dev_params *__restrict__ Pp, const float2 *__restrict__ RHO,
                float *__restrict__ sum, float *__restrict__ maxv)
{
    constexpr unsigned kWaves = kDensityTPB / 64u;
    __shared__ float ps[kWaves], pm[kWaves];
    const sph_dev_params &P = Pp[blockIdx.x];
    const unsigned n = (unsigned)P.n;
    const float4 *R = reinterpret_cast<const float4 *>(RHO + P.poff); // two particles
    float t[4] = {0, 0, 0, 0}, m = 0.0f;
    for (unsigned s = threadIdx.x; 2u * s < n; s += 4u * kDensityTPB) {
        float4 r[4];
#pragma unroll
        for (unsigned u = 0; u < 4u; u++) {
            const unsigned i = s + u * kDensityTPB;
            r[u] = 2u * i < n ? R[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            r[u].z = 2u * i + 1u < n ? r[u].z : 0.0f;
        }
#pragma unroll
        for (unsigned u = 0; u < 4u; u++) {
            t[u] += r[u].x + r[u].z;
            m = fmaxf(m, fmaxf(r[u].x, r[u].z));
        }
    }
    float a = (t[0] + t[1]) + (t[2] + t[3]);
    for (int x = 32; x > 0; x >>= 1) {
        a += __shfl_xor(a, x, 64);
        m = fmaxf(m, __shfl_xor(m, x, 64));
    }
    if (lane() == 0) {
        ps[threadIdx.x / 64u] = a;
        pm[threadIdx.x / 64u] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (unsigned w = 1; w < kWaves; w++) {
            a += ps[w];
            m = fmaxf(m, pm[w]);
        }
        sum[blockIdx.x] = a;
        maxv[blockIdx.x] = m;
    }
}

// Density of every particle by caller index (the state is canonical: RHO
// in ID0 order).
__global__ void __launch_bounds__(256)
k_rho_by_id(const sph_dev_params *__restrict__ Pp, const int *__restrict__ BS, unsigned slots,
            const float2 *__restrict__ RHO, const int *__restrict__ ID, float *__restrict__ out)
{
    const unsigned s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots)
        return;
    const sph_dev_params &P = Pp[BS[s / 256u]];
    if (s >= P.poff + (unsigned)P.n)
        return;
    out[P.uoff + (unsigned)ID[s]] = RHO[s].x;
}

// Per shadowed scene (flags[s] != 0): sum over its particles of
// (sur - plain)^2 and of plain^2, for the relative RMS density error.
__global__ void __launch_bounds__(256)
k_shadow_err(const sph_dev_params *__restrict__ Pp, const int *__restrict__ flags,
             const float *__restrict__ plain, const float *__restrict__ sur,
             float *__restrict__ out)
{
    __shared__ float pa[4], pb[4];
    const sph_dev_params &P = Pp[blockIdx.x];
    if (!flags[blockIdx.x])
        return;
    float a = 0.0f, b = 0.0f;
    for (unsigned i = threadIdx.x; i < (unsigned)P.n; i += blockDim.x) {
        const float x = plain[P.uoff + i], y = sur[P.uoff + i];
        a += (y - x) * (y - x);
        b += x * x;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    if (lane() == 0) {
        pa[threadIdx.x / 64u] = a;
        pb[threadIdx.x / 64u] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[2 * blockIdx.x] = (pa[0] + pa[1]) + (pa[2] + pa[3]);
        out[2 * blockIdx.x + 1] = (pb[0] + pb[1]) + (pb[2] + pb[3]);
    }
}

// Judge of a macro-step.  Per scene, ref[s] is the mean density of the
// current state and dref[s] = ref[nscenes + s] the change of the scene's last
// macro-step computed by the plain solver (its density trend).  A predicted
// state passes when its mean density is within tol (relative) of
// ref + dref, the plain solver's trend extrapolated by one macro-step; a
// passing scene takes the new mean as ref.  On input flags[s] = 1 forces a
// re-take (a periodic plain macro-step that refreshes the trend); on output
// flags[s] = 1 for a failed scene, 2 for a forced one.  mode 1 (set) starts
// every scene at the current mean with no trend; mode 2 (after re-takes)
// gives each re-taken scene (flags[s] != 0) the plain change as its trend
// and the plain mean as ref.
__global__ void k_judge(const sph_dev_params *__restrict__ Pp, int nscenes,
                        const float *__restrict__ sum, float *__restrict__ ref, float tol,
                        int mode, int *__restrict__ flags)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nscenes)
        return;
    float *dref = ref + nscenes;
    const int n = Pp[s].n;
    const float mean = n > 0 ? sum[s] / (float)n : 0.0f;
    if (mode == 1) {
        ref[s] = mean;
        dref[s] = 0.0f;
        return;
    }
    if (mode == 2) {
        if (flags[s]) {
            dref[s] = mean - ref[s];
            ref[s] = mean;
        }
        return;
    }
    const float expect = ref[s] + dref[s];
    const bool bad = n > 0 && !(fabsf(mean - expect) <= tol * expect);
    const bool forced = flags[s] != 0;
    flags[s] = forced ? 2 : (bad ? 1 : 0);
    if (!bad && !forced)
        ref[s] = mean;
}

// Trajectory sampling: sample k takes frame f = frame[k] of scene s =
// scene[k]; staging gets its (x, y, v_x, v_y) records, target the 4-step
// displacement to frame f + 1.  data is [frames][nscenes][n] float4.
__global__ void k_traj_sample(const float4 *__restrict__ data, unsigned nscenes, unsigned n,
                              unsigned count, const int *__restrict__ scene,
                              const int *__restrict__ frame, float4 *__restrict__ staging,
                              float2 *__restrict__ target)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)count * n)
        return;
    const unsigned k = (unsigned)(i / n), j = (unsigned)(i % n);
    const size_t src = ((size_t)frame[k] * nscenes + (unsigned)scene[k]) * n + j;
    const float4 a = data[src], b = data[src + (size_t)nscenes * n];
    staging[i] = a;
    target[i] = make_float2(b.x - a.x, b.y - a.y);
}

// ---------------------------------------------------------------------------
// host side

namespace {

thread_local char m_err[256] = "";

int merr(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(m_err, sizeof m_err, fmt, ap);
    va_end(ap);
    return code;
}

#define MCHK(call)                                                                               \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return merr(SPH_EHIP, "%s failed: %s", #call, hipGetErrorString(e_));                \
    } while (0)

template <class T>
int malloc_dev(T **p, size_t n)
{
    if (hipMalloc((void **)p, sizeof(T) * (n ? n : 1)) != hipSuccess) {
        *p = nullptr;
        return merr(SPH_ENOMEM, "hipMalloc of %zu x %zu B failed", n, sizeof(T));
    }
    return SPH_OK;
}

// Workgroups of the passes over groups of 16 slots, one group a wave: groups
// differ in length, and workgroups that end leave their place to the next.
// (2,048 workgroups taking eight groups a wave in turn: 0.56 ms for the edge
// forward of a million particles, against 0.41.)
unsigned group_blocks(unsigned slots) { return slots / (4u * kGroup); }

// The node gradients keep their sums in registers and fit two workgroups per
// CU (256 CUs).
unsigned node_grad_blocks(unsigned slots)
{
    const unsigned n = group_blocks(slots);
    return n < 512u ? n : 512u;
}

size_t part_floats(unsigned slots)
{
    const size_t a = (size_t)node_grad_blocks(slots) * kNodePart;
    const size_t b = (size_t)group_blocks(slots) * kEdgePart;
    return a > b ? a : b;
}

// Sum `rows` partial gradients in chunks of 128.
template <bool NODE>
void grad_sum(sph_surrogate *m, hipStream_t st, unsigned rows)
{
    constexpr unsigned kCols = NODE ? kNodePart : kEdgePart, kChunk = 128;
    k_grad_sum<NODE><<<dim3((kCols + 255u) / 256u, (rows + kChunk - 1u) / kChunk), 1024, 0, st>>>(
        m->part, rows, kChunk, m->grads, m->loss);
}

int ensure_buffers(sph_surrogate *m, size_t slots)
{
    if (m->slots >= slots)
        return SPH_OK;
    void *old[] = {m->S, m->deg, m->dS, m->disp, m->tgt, m->tmp2, m->part};
    for (void *p : old)
        if (p)
            (void)hipFree(p);
    m->deg = m->disp = m->tgt = nullptr;
    m->S = m->dS = nullptr;
    m->tmp2 = nullptr;
    m->part = nullptr;
    int rc = SPH_OK;
    if (!rc) rc = malloc_dev(&m->S, slots * kH / 4);
    if (!rc) rc = malloc_dev(&m->deg, slots);
    if (!rc) rc = malloc_dev(&m->dS, slots * kH / 4);
    if (!rc) rc = malloc_dev(&m->disp, slots * 2);
    if (!rc) rc = malloc_dev(&m->tgt, slots * 2);
    if (!rc) rc = malloc_dev(&m->tmp2, slots);
    if (!rc) rc = malloc_dev(&m->part, part_floats((unsigned)slots));
    m->slots = rc ? 0 : slots;
    return rc;
}

int ensure_judge(sph_surrogate *m, const sph_ctx *c)
{
    const size_t ns = c->sc.size();
    if (m->ns >= ns)
        return SPH_OK;
    void *old[] = {m->ref, m->jsum, m->jmax, m->jflags, m->sh_sum, m->sh_err};
    for (void *p : old)
        if (p)
            (void)hipFree(p);
    m->ref = m->jsum = m->jmax = m->sh_sum = m->sh_err = nullptr;
    m->jflags = nullptr;
    m->ref_ok = false;
    int rc = SPH_OK;
    if (!rc) rc = malloc_dev(&m->ref, 2 * ns); // ref, then the per-scene trend
    if (!rc) rc = malloc_dev(&m->jsum, ns);
    if (!rc) rc = malloc_dev(&m->jmax, ns);
    if (!rc) rc = malloc_dev(&m->jflags, ns);
    if (!rc) rc = malloc_dev(&m->sh_sum, ns);
    if (!rc) rc = malloc_dev(&m->sh_err, 2 * ns);
    m->ns = rc ? 0 : ns;
    return rc;
}

// The shadows' densities, for the largest context so far.
int ensure_shadow(sph_surrogate *m, size_t slots)
{
    if (m->rho_slots >= slots)
        return SPH_OK;
    for (float *p : {m->rho_plain, m->rho_sur})
        if (p)
            (void)hipFree(p);
    m->rho_plain = m->rho_sur = nullptr;
    int rc = malloc_dev(&m->rho_plain, slots);
    if (!rc) rc = malloc_dev(&m->rho_sur, slots);
    m->rho_slots = rc ? 0 : slots;
    return rc;
}

// Per-scene density sums (and maxima) of RHO into m->jsum / m->jmax.
int scene_sums(sph_surrogate *m, sph_ctx *c)
{
    k_scene_density<<<dim3((unsigned)c->sc.size()), kDensityTPB, 0, c->st>>>(c->dP, c->RHO, m->jsum,
                                                                       m->jmax);
    MCHK(hipGetLastError());
    return SPH_OK;
}

// Density of the current (hashed) state into RHO.
int density_now(sph_ctx *c)
{
    if (int rc = sph_internal_canonicalize(c))
        return rc;
    if (!c->lists_valid)
        return merr(SPH_ESTATE, "surrogate: state not hashed");
    if (c->lanes != 16)
        sph_internal_plans(c);
    sph_launch_density(c->st, c->slots, c->bucket_cap != 0, c->dP, c->BS, c->plans, c->POS0, c->K0,
                       c->start, c->RHO, c->MASK, c->dC, c->lanes);
    MCHK(hipGetLastError());
    return SPH_OK;
}

// Prediction of the 4-step displacement of every particle (fused kernel).
int forward(sph_surrogate *m, sph_ctx *c)
{
    if (!c->lists_valid)
        return merr(SPH_ESTATE, "surrogate: the context has no hashed state (step or hash first)");
    if (int rc = ensure_buffers(m, c->slots))
        return rc;
    k_infer<<<dim3(group_blocks(c->slots)), 256, 0, c->st>>>(
        c->dP, c->BS, c->slots, c->dclock, c->POS0, c->VEL, c->K0, c->start, m->W1b, m->W2b,
        m->params, m->W3b, (float2 *)m->disp);
    MCHK(hipGetLastError());
    m->have_pred = true;
    return SPH_OK;
}

// The edge pass of training: per-particle sums S and degrees for the node
// backward (which recomputes the node forward itself).
int forward_edges(sph_surrogate *m, sph_ctx *c)
{
    if (!c->lists_valid)
        return merr(SPH_ESTATE, "surrogate: the context has no hashed state (step or hash first)");
    if (int rc = ensure_buffers(m, c->slots))
        return rc;
    k_edge_fwd<<<dim3(group_blocks(c->slots)), 256, 0, c->st>>>(
        c->dP, c->BS, c->slots, c->POS0, c->VEL, c->K0, c->start, m->W1b, m->S, m->deg);
    MCHK(hipGetLastError());
    return SPH_OK;
}

} // namespace

extern "C" {

const char *sph_surrogate_last_error(void) { return m_err; }

int sph_surrogate_num_params(void) { return kNParams; }

int sph_surrogate_create(sph_surrogate **out, uint64_t seed)
{
    if (!out)
        return merr(SPH_EINVAL, "null output");
    *out = nullptr;
    sph_surrogate *m = new (std::nothrow) sph_surrogate();
    if (!m)
        return merr(SPH_ENOMEM, "host allocation failed");
    int rc = SPH_OK;
    if (!rc) rc = malloc_dev(&m->params, kNParams);
    if (!rc) rc = malloc_dev(&m->grads, kNParams);
    if (!rc) rc = malloc_dev(&m->adam_m, kNParams);
    if (!rc) rc = malloc_dev(&m->adam_v, kNParams);
    if (!rc) rc = malloc_dev(&m->W1b, kH * kKE);
    if (!rc) rc = malloc_dev(&m->W2b, kH * kH);
    if (!rc) rc = malloc_dev(&m->W3b, kH * kKN);
    if (!rc) rc = malloc_dev(&m->loss, 1);
    if (rc) {
        sph_surrogate_destroy(m);
        return rc;
    }
    // Initialisation: uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) from SplitMix64,
    // padding columns zero, the output layer scaled down so the untrained
    // network starts close to the ballistic estimate.
    std::vector<float> p(kNParams, 0.0f);
    uint64_t st = seed;
    auto uni = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (float)(z >> 40) * 0x1p-24f * 2.0f - 1.0f;
    };
    for (int r = 0; r < kH; r++)
        for (int k = 0; k < 6; k++)
            p[oW1 + r * kKE + k] = uni() / sqrtf(6.0f);
    for (int i = 0; i < kH * kH; i++)
        p[oW2 + i] = uni() / sqrtf((float)kH);
    for (int r = 0; r < kH; r++)
        for (int k = 0; k < 69; k++)
            p[oW3 + r * kKN + k] = uni() / sqrtf(69.0f);
    for (int i = 0; i < 2 * kH; i++)
        p[oW4 + i] = 0.1f * uni() / sqrtf((float)kH);
    if (hipMemcpy(m->params, p.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(m->grads, 0, sizeof(float) * kNParams) != hipSuccess ||
        hipMemset(m->adam_m, 0, sizeof(float) * kNParams) != hipSuccess ||
        hipMemset(m->adam_v, 0, sizeof(float) * kNParams) != hipSuccess) {
        sph_surrogate_destroy(m);
        return merr(SPH_EHIP, "surrogate initialisation failed");
    }
    k_to_bf16<<<dim3((kNParams + 255) / 256), 256>>>(m->params, m->W1b, m->W2b, m->W3b);
    if (hipDeviceSynchronize() != hipSuccess) {
        sph_surrogate_destroy(m);
        return merr(SPH_EHIP, "surrogate initialisation failed");
    }
    *out = m;
    return SPH_OK;
}

void sph_surrogate_destroy(sph_surrogate *m)
{
    if (!m)
        return;
    void *ptrs[] = {m->params, m->grads, m->adam_m, m->adam_v, m->W1b, m->W2b, m->W3b, m->S,
                    m->deg,    m->dS,    m->disp,   m->tgt,    m->part,   m->loss,
                    m->tmp2, m->ref, m->jsum, m->jmax, m->jflags, m->sh_sum,
                    m->rho_plain, m->rho_sur, m->sh_err};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
    delete m;
}

int sph_surrogate_get_params(sph_surrogate *m, float *out)
{
    if (!m || !out)
        return merr(SPH_EINVAL, "null argument");
    MCHK(hipDeviceSynchronize());
    MCHK(hipMemcpy(out, m->params, sizeof(float) * kNParams, hipMemcpyDeviceToHost));
    return SPH_OK;
}

int sph_surrogate_set_params(sph_surrogate *m, const float *in)
{
    if (!m || !in)
        return merr(SPH_EINVAL, "null argument");
    MCHK(hipDeviceSynchronize());
    MCHK(hipMemcpy(m->params, in, sizeof(float) * kNParams, hipMemcpyHostToDevice));
    k_to_bf16<<<dim3((kNParams + 255) / 256), 256>>>(m->params, m->W1b, m->W2b, m->W3b);
    MCHK(hipDeviceSynchronize());
    return SPH_OK;
}

int sph_surrogate_get_grads(sph_surrogate *m, float *out)
{
    if (!m || !out)
        return merr(SPH_EINVAL, "null argument");
    MCHK(hipDeviceSynchronize());
    MCHK(hipMemcpy(out, m->grads, sizeof(float) * kNParams, hipMemcpyDeviceToHost));
    return SPH_OK;
}

int sph_surrogate_zero_grads(sph_surrogate *m)
{
    if (!m)
        return merr(SPH_EINVAL, "null argument");
    MCHK(hipMemset(m->grads, 0, sizeof(float) * kNParams));
    return SPH_OK;
}

// Forward on the context's current hashed state; the predicted displacement
// per particle (caller order, 2 floats each) is copied out if disp_by_id.
int sph_surrogate_predict(sph_surrogate *m, sph_ctx *c, float *disp_by_id)
{
    if (!m || !c)
        return merr(SPH_EINVAL, "null argument");
    if (int rc = forward(m, c))
        return rc;
    if (disp_by_id && c->n_total) {
        k_slot_to_by_id<<<dim3(c->slots / 256), 256, 0, c->st>>>(
            c->dP, c->BS, c->slots, c->ID0, (const float2 *)m->disp, m->tmp2);
        if (int rc = sph_internal_fetch(c, disp_by_id, m->tmp2,
                                        sizeof(float2) * (size_t)c->n_total))
            return merr(rc, "%s", sph_last_error());
    }
    return SPH_OK;
}

// One gradient evaluation: forward, loss against target displacements
// (a device buffer in caller order, 2 floats per particle), backward; gradients are accumulated into the gradient
// buffer (zero it with sph_surrogate_zero_grads).  *loss gets the mean of
// |d - target|^2 / 0.05^2 over the particles.
static int backward_dev(sph_surrogate *m, sph_ctx *c, const float2 *target_dev, float *loss)
{
    if (c->n_total == 0)
        return SPH_OK;
    if (int rc = forward_edges(m, c))
        return rc;
    const unsigned S = c->slots;
    k_by_id_to_slot<<<dim3(S / 256), 256, 0, c->st>>>(c->dP, c->BS, S, c->ID0, target_dev,
                                                     (float2 *)m->tgt);
    MCHK(hipMemsetAsync(m->loss, 0, sizeof(float), c->st));
    k_node_grad<<<dim3(node_grad_blocks(S)), 256, 0, c->st>>>(
        c->dP, c->BS, S, c->dclock, c->VEL, m->S, m->deg, m->W2b, m->params, m->W3b,
        (const float2 *)m->tgt, 1.0f / (float)c->n_total, m->dS, m->part);
    grad_sum<true>(m, c->st, node_grad_blocks(S));
    k_edge_bwd<<<dim3(group_blocks(S)), 256, 0, c->st>>>(
        c->dP, c->BS, S, c->POS0, c->VEL, c->K0, c->start, m->W1b, m->dS, m->part);
    grad_sum<false>(m, c->st, group_blocks(S));
    MCHK(hipGetLastError());
    if (loss) {
        MCHK(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, c->st));
        MCHK(hipStreamSynchronize(c->st));
    }
    return SPH_OK;
}

int sph_surrogate_backward(sph_surrogate *m, sph_ctx *c, const float *target_by_id, float *loss)
{
    if (!m || !c || (!target_by_id && c->n_total))
        return merr(SPH_EINVAL, "null argument");
    if (c->n_total == 0)
        return SPH_OK;
    if (int rc = ensure_buffers(m, c->slots))
        return rc;
    MCHK(hipStreamSynchronize(c->st)); // tmp2 may still be read by earlier work
    MCHK(hipMemcpy(m->tmp2, target_by_id, sizeof(float2) * (size_t)c->n_total,
                   hipMemcpyHostToDevice));
    return backward_dev(m, c, m->tmp2, loss);
}

int sph_surrogate_backward_trajectory(sph_surrogate *m, sph_ctx *c, sph_trajectory *tr,
                                      float *loss)
{
    if (!m || !c || !tr)
        return merr(SPH_EINVAL, "null argument");
    if (tr->loaded != (int)c->sc.size() || (long)tr->loaded * tr->n != (long)c->n_total)
        return merr(SPH_ESTATE, "the context does not hold the trajectory's last loaded samples");
    return backward_dev(m, c, tr->target, loss);
}

// ---- trajectory store ------------------------------------------------------

int sph_trajectory_create(sph_trajectory **out, int nscenes, int n, int frames)
{
    if (!out || nscenes <= 0 || n <= 0 || frames < 2)
        return merr(SPH_EINVAL, "sph_trajectory_create: bad sizes");
    *out = nullptr;
    sph_trajectory *t = new (std::nothrow) sph_trajectory();
    if (!t)
        return merr(SPH_ENOMEM, "host allocation failed");
    t->nscenes = nscenes;
    t->n = n;
    t->frames = frames;
    if (int rc = malloc_dev(&t->data, (size_t)frames * nscenes * n)) {
        sph_trajectory_destroy(t);
        return rc;
    }
    *out = t;
    return SPH_OK;
}

void sph_trajectory_destroy(sph_trajectory *t)
{
    if (!t)
        return;
    void *ptrs[] = {t->data, t->staging, t->target, t->idx};
    for (void *p : ptrs)
        if (p)
            (void)hipFree(p);
    delete t;
}

int sph_trajectory_record(sph_trajectory *t, sph_ctx *c, int frame)
{
    if (!t || !c || frame < 0 || frame >= t->frames)
        return merr(SPH_EINVAL, "sph_trajectory_record: bad argument");
    if ((int)c->sc.size() != t->nscenes || (long)c->n_total != (long)t->nscenes * t->n)
        return merr(SPH_EINVAL, "sph_trajectory_record: context is not %d scenes x %d particles",
                    t->nscenes, t->n);
    for (const auto &S : c->sc)
        if (S.n != t->n)
            return merr(SPH_EINVAL, "sph_trajectory_record: scenes of unequal size");
    if (sph_gather_state_dev(c, (float *)(t->data + (size_t)frame * t->nscenes * t->n)))
        return merr(SPH_EHIP, "gather failed: %s", sph_last_error());
    return SPH_OK;
}

int sph_trajectory_read(sph_trajectory *t, int frame, float *out)
{
    if (!t || !out || frame < 0 || frame >= t->frames)
        return merr(SPH_EINVAL, "sph_trajectory_read: bad argument");
    MCHK(hipDeviceSynchronize());
    MCHK(hipMemcpy(out, t->data + (size_t)frame * t->nscenes * t->n,
                   sizeof(float4) * (size_t)t->nscenes * t->n, hipMemcpyDeviceToHost));
    return SPH_OK;
}

int sph_trajectory_load(sph_trajectory *t, sph_ctx *c, int count, const int *scene,
                        const int *frame)
{
    if (!t || !c || !scene || !frame || count <= 0)
        return merr(SPH_EINVAL, "sph_trajectory_load: bad argument");
    if ((int)c->sc.size() != count || (long)c->n_total != (long)count * t->n)
        return merr(SPH_EINVAL, "sph_trajectory_load: context must hold %d scenes of %d particles",
                    count, t->n);
    for (const auto &S : c->sc)
        if (S.n != t->n)
            return merr(SPH_EINVAL, "sph_trajectory_load: scenes of unequal size");
    for (int k = 0; k < count; k++)
        if (scene[k] < 0 || scene[k] >= t->nscenes || frame[k] < 0 || frame[k] + 1 >= t->frames)
            return merr(SPH_EINVAL, "sph_trajectory_load: sample %d (scene %d, frame %d) out of range",
                        k, scene[k], frame[k]);
    if (t->cap < count) {
        void *old[] = {t->staging, t->target, t->idx};
        for (void *p : old)
            if (p)
                (void)hipFree(p);
        t->staging = nullptr;
        t->target = nullptr;
        t->idx = nullptr;
        t->cap = 0;
        int rc = malloc_dev(&t->staging, (size_t)count * t->n);
        if (!rc) rc = malloc_dev(&t->target, (size_t)count * t->n);
        if (!rc) rc = malloc_dev(&t->idx, 2 * (size_t)count);
        if (rc)
            return rc;
        t->cap = count;
    }
    std::vector<int> hidx((size_t)2 * count);
    memcpy(hidx.data(), scene, sizeof(int) * count);
    memcpy(hidx.data() + count, frame, sizeof(int) * count);
    MCHK(hipStreamSynchronize(c->st));
    MCHK(hipMemcpyAsync(t->idx, hidx.data(), sizeof(int) * 2 * count, hipMemcpyHostToDevice, c->st));
    const size_t tot = (size_t)count * t->n;
    k_traj_sample<<<dim3((unsigned)((tot + 255) / 256)), 256, 0, c->st>>>(
        t->data, (unsigned)t->nscenes, (unsigned)t->n, (unsigned)count, t->idx, t->idx + count,
        t->staging, t->target);
    MCHK(hipGetLastError());
    MCHK(hipStreamSynchronize(c->st));
    if (sph_load_state_dev(c, (const float *)t->staging))
        return merr(SPH_EHIP, "load failed: %s", sph_last_error());
    t->loaded = count;
    return SPH_OK;
}

int sph_surrogate_adam(sph_surrogate *m, float lr, float beta1, float beta2, float eps)
{
    if (!m)
        return merr(SPH_EINVAL, "null argument");
    m->adam_t++;
    const float c1 = 1.0f - powf(beta1, (float)m->adam_t);
    const float c2 = 1.0f - powf(beta2, (float)m->adam_t);
    k_adam<<<dim3((kNParams + 255) / 256), 256>>>(m->params, m->grads, m->adam_m, m->adam_v,
                                                  kNParams, lr, beta1, beta2, eps, c1, c2, m->W1b,
                                                  m->W2b, m->W3b);
    MCHK(hipGetLastError());
    MCHK(hipMemset(m->grads, 0, sizeof(float) * kNParams));
    MCHK(hipDeviceSynchronize());
    return SPH_OK;
}

// Apply the last prediction to the context (positions and velocities move
// four steps); frozen scenes are left alone.  The state must be hashed
// again before the next step (the context knows this).
int sph_surrogate_apply(sph_surrogate *m, sph_ctx *c)
{
    if (!m || !c)
        return merr(SPH_EINVAL, "null argument");
    if (!m->have_pred)
        return merr(SPH_ESTATE, "sph_surrogate_apply: no prediction");
    if (m->slots < c->slots)
        return merr(SPH_ESTATE, "sph_surrogate_apply: the prediction is of a smaller context");
    if (int rc = sph_internal_canonicalize(c))
        return rc;
    const unsigned S = c->slots;
    k_apply<<<dim3(S / 256), 256, 0, c->st>>>(c->dP, c->BS, S, c->dclock,
                                             (const float2 *)m->disp, c->POS0, c->VEL);
    MCHK(hipGetLastError());
    k_clock_add<<<1, 1, 0, c->st>>>(c->dclock, 4ull);
    MCHK(hipGetLastError());
    c->lists_valid = false;
    m->have_pred = false;
    return SPH_OK;
}

// One surrogate macro-step (four plain steps of simulated time) of every
// scene, judged by the plain solver.  The predicted state is hashed and its
// density computed; a scene whose mean density is off by more than tol
// (relative) from the plain solver's trend (its mean density plus the change
// of its last plain macro-step) is restored and re-taken with four plain
// steps.  Every scene is also re-taken plainly on its first macro-step and
// then on a fixed schedule, one macro-step in kTrendRefresh (staggered over
// the scenes), which keeps its trend current whatever the failures.
// With shadow judging on (sph_surrogate_set_shadow), one scene in every
// shadow_every (rotating) first takes the macro-step plainly from the same
// start: its surrogate result is then judged against that plain result as
// well (error above tol: re-taken, flag 3), and the error of the steps the
// trend judge accepted is recorded (sph_surrogate_shadow_stats).
// flags (optional, nscenes ints) receives 1 for failed scenes, 2 for
// scheduled re-takes, 3 for shadow failures, 0 for accepted ones;
// *nfallback the number re-taken.
int sph_surrogate_macro_step(sph_surrogate *m, sph_ctx *c, float tol, int *flags, int *nfallback)
{
    if (!m || !c)
        return merr(SPH_EINVAL, "null argument");
    if (!(tol >= 0.0f))
        return merr(SPH_EINVAL, "tolerance must be >= 0");
    const int ns = (int)c->sc.size();
    if (nfallback)
        *nfallback = 0;
    if (c->n_total == 0)
        return SPH_OK;
    if (int rc = ensure_judge(m, c))
        return rc;
    if (!c->lists_valid)
        if (sph_phase_hash(c, 0))
            return merr(SPH_EHIP, "hash failed: %s", sph_last_error());
    const dim3 jg((ns + 255) / 256);
    bool first = false;
    if (!m->ref_ok || m->ref_ctx != c) {
        if (int rc = density_now(c))
            return rc;
        if (int rc = scene_sums(m, c))
            return rc;
        k_judge<<<jg, 256, 0, c->st>>>(c->dP, ns, m->jsum, m->ref, tol, 1, nullptr);
        MCHK(hipGetLastError());
        m->ref_ok = true;
        m->ref_ctx = c;
        first = true;
    }
    const unsigned long long k = m->macro++;
    std::vector<int> hf((size_t)ns), shadow((size_t)ns, 0);
    int nshadow = 0;
    for (int s = 0; s < ns; s++) {
        hf[s] = first || (k + (unsigned)s) % kTrendRefresh == 0 ? 1 : 0;
        if (m->shadow_every > 0 && !hf[s] && (k + (unsigned)s) % (unsigned)m->shadow_every == 0 &&
            c->sc[s].n > 0) {
            shadow[s] = 1;
            nshadow++;
        }
    }
    if (sph_snapshot_save(c))
        return merr(SPH_EHIP, "snapshot failed: %s", sph_last_error());
    const unsigned S = c->slots;
    if (nshadow) { // the shadowed scenes' plain macro-step, then back to the start
        if (int rc = ensure_shadow(m, S))
            return rc;
        std::vector<int> frozen((size_t)ns), none((size_t)ns, 0);
        for (int s = 0; s < ns; s++)
            frozen[s] = shadow[s] ? 0 : 1;
        if (sph_set_scene_frozen(c, frozen.data()) || sph_step(c, 4) ||
            sph_set_scene_frozen(c, none.data()))
            return merr(SPH_EHIP, "shadow step failed: %s", sph_last_error());
        if (int rc = density_now(c))
            return rc;
        k_scene_density<<<dim3((unsigned)ns), kDensityTPB, 0, c->st>>>(c->dP, c->RHO, m->sh_sum,
                                                                       m->jmax);
        k_rho_by_id<<<dim3(S / 256), 256, 0, c->st>>>(c->dP, c->BS, S, c->RHO, c->ID0,
                                                      m->rho_plain);
        MCHK(hipGetLastError());
        if (sph_snapshot_restore(c, shadow.data()))
            return merr(SPH_EHIP, "shadow restore failed: %s", sph_last_error());
    }
    if (int rc = forward(m, c))
        return rc;
    if (int rc = sph_surrogate_apply(m, c))
        return rc;
    if (sph_phase_hash(c, 1))
        return merr(SPH_EHIP, "hash failed: %s", sph_last_error());
    if (int rc = scene_sums(m, c))
        return rc;
    MCHK(hipMemcpyAsync(m->jflags, hf.data(), sizeof(int) * ns, hipMemcpyHostToDevice, c->st));
    k_judge<<<jg, 256, 0, c->st>>>(c->dP, ns, m->jsum, m->ref, tol, 0, m->jflags);
    MCHK(hipGetLastError());
    MCHK(hipMemcpyAsync(hf.data(), m->jflags, sizeof(int) * ns, hipMemcpyDeviceToHost, c->st));
    if (nshadow) {
        std::vector<float> sur((size_t)ns), pl((size_t)ns), err(2 * (size_t)ns);
        k_rho_by_id<<<dim3(S / 256), 256, 0, c->st>>>(c->dP, c->BS, S, c->RHO, c->ID0, m->rho_sur);
        MCHK(hipMemcpyAsync(m->jflags, shadow.data(), sizeof(int) * ns, hipMemcpyHostToDevice,
                            c->st));
        k_shadow_err<<<dim3((unsigned)ns), 256, 0, c->st>>>(c->dP, m->jflags, m->rho_plain,
                                                            m->rho_sur, m->sh_err);
        MCHK(hipGetLastError());
        MCHK(hipMemcpyAsync(sur.data(), m->jsum, sizeof(float) * ns, hipMemcpyDeviceToHost, c->st));
        MCHK(hipMemcpyAsync(pl.data(), m->sh_sum, sizeof(float) * ns, hipMemcpyDeviceToHost, c->st));
        MCHK(hipMemcpyAsync(err.data(), m->sh_err, sizeof(float) * 2 * ns, hipMemcpyDeviceToHost,
                            c->st));
        MCHK(hipStreamSynchronize(c->st));
        for (int s = 0; s < ns; s++) {
            if (!shadow[s])
                continue;
            const double e = ((double)sur[s] - (double)pl[s]) / (double)pl[s];
            const double rms = sqrt((double)err[2 * s] / (double)err[2 * s + 1]);
            m->sh_stats[0] += 1.0;
            if (hf[s] == 0) { // accepted by the trend judge: the error it let through
                m->sh_stats[1] += 1.0;
                m->sh_stats[2] += fabs(e) > tol ? 1.0 : 0.0;
                m->sh_stats[3] += fabs(e);
                m->sh_stats[4] = fmax(m->sh_stats[4], fabs(e));
                m->sh_stats[5] += e;
                m->sh_stats[6] += rms;
                m->sh_stats[7] = fmax(m->sh_stats[7], rms);
                if (fabs(e) > tol)
                    hf[s] = 3;
            }
        }
        // the judge's mean for a shadow failure is the surrogate's; the
        // re-take below replaces it with the plain one (mode 2)
    } else {
        MCHK(hipStreamSynchronize(c->st));
    }
    int nf = 0;
    for (int s = 0; s < ns; s++)
        nf += hf[s] != 0;
    if (nf) {
        std::vector<int> retake((size_t)ns), frozen((size_t)ns), none((size_t)ns, 0);
        for (int s = 0; s < ns; s++) {
            retake[s] = hf[s] ? 1 : 0;
            frozen[s] = hf[s] ? 0 : 1;
        }
        if (sph_snapshot_restore(c, retake.data()) || sph_set_scene_frozen(c, frozen.data()) ||
            sph_step(c, 4) || sph_set_scene_frozen(c, none.data()))
            return merr(SPH_EHIP, "fallback failed: %s", sph_last_error());
        if (int rc = density_now(c))
            return rc;
        if (int rc = scene_sums(m, c))
            return rc;
        MCHK(hipMemcpyAsync(m->jflags, retake.data(), sizeof(int) * ns, hipMemcpyHostToDevice,
                            c->st));
        k_judge<<<jg, 256, 0, c->st>>>(c->dP, ns, m->jsum, m->ref, tol, 2, m->jflags);
        MCHK(hipGetLastError());
        MCHK(hipStreamSynchronize(c->st));
    }
    if (flags)
        memcpy(flags, hf.data(), sizeof(int) * ns);
    if (nfallback)
        *nfallback = nf;
    return SPH_OK;
}

int sph_surrogate_set_shadow(sph_surrogate *m, int every)
{
    if (!m || every < 0)
        return merr(SPH_EINVAL, "sph_surrogate_set_shadow: null model or negative period");
    m->shadow_every = every;
    for (double &x : m->sh_stats)
        x = 0.0;
    return SPH_OK;
}

int sph_surrogate_shadow_stats(sph_surrogate *m, double *out)
{
    if (!m || !out)
        return merr(SPH_EINVAL, "null argument");
    for (int i = 0; i < 8; i++)
        out[i] = m->sh_stats[i];
    return SPH_OK;
}

int sph_surrogate_mfma_selftest(float *out256)
{
    if (!out256)
        return merr(SPH_EINVAL, "null argument");
    float *d = nullptr;
    MCHK(hipMalloc(&d, 256 * sizeof(float)));
    k_mfma_selftest<<<1, 64>>>(d);
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess)
        e = hipMemcpy(out256, d, 256 * sizeof(float), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess)
        return merr(SPH_EHIP, "mfma selftest: %s", hipGetErrorString(e));
    return SPH_OK;
}

// Per-scene mean and maximum density of the last density pass (sph_step's
// or sph_phase_hash(ctx, 1)'s).
int sph_scene_density(sph_ctx *c, float *mean, float *maxv)
{
    if (!c || !mean || !maxv)
        return merr(SPH_EINVAL, "null argument");
    if (int rc = sph_internal_canonicalize(c))
        return rc;
    const size_t ns = c->sc.size();
    float *buf = nullptr;
    if (int rc = malloc_dev(&buf, 2 * ns))
        return rc;
    k_scene_density<<<dim3((unsigned)ns), kDensityTPB, 0, c->st>>>(c->dP, c->RHO, buf, buf + ns);
    hipError_t e = hipGetLastError();
    std::vector<float> h(2 * ns);
    if (e == hipSuccess)
        e = hipStreamSynchronize(c->st);
    if (e == hipSuccess)
        e = hipMemcpy(h.data(), buf, sizeof(float) * 2 * ns, hipMemcpyDeviceToHost);
    (void)hipFree(buf);
    if (e != hipSuccess)
        return merr(SPH_EHIP, "sph_scene_density: %s", hipGetErrorString(e));
    for (size_t s = 0; s < ns; s++) {
        mean[s] = c->sc[s].n ? h[s] / (float)c->sc[s].n : 0.0f;
        maxv[s] = h[ns + s];
    }
    return SPH_OK;
}

} // extern "C"

// ---------------------------------------------------------------------------
// sph_scene_density without allocation.  The per-scene partial results (the
// density sum and maximum of every scene) go to a fixed device array instead
// of a buffer allocated per call.  The array's name is a host-side stand-in
// for its device copy: host code only ever uses the address that
// hipGetSymbolAddress returns for the current device, looked up once per
// device on the first call there.  Every call on a device shares that
// device's array and overwrites the entries it reads back (one sum and one
// maximum per scene, each written by that scene's workgroup), so nothing
// needs clearing; calls that overlap on one device race.

constexpr int kNoAllocMaxScenes = 4096; // 32 KiB of partial results per device
static __device__ __align__(256) float scratch[2 * kNoAllocMaxScenes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float *g_scratch_ptr[kMaxDevices]; // per device: the device address of `scratch`

int scratch_for_current_device(float **out)
{
    int dev = 0;
    MCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return merr(SPH_ENODEV, "sph_scene_density_noalloc: device %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return merr(SPH_EHIP, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                        hipGetErrorString(e));
        g_scratch_ptr[dev] = (float *)p;
    }
    *out = g_scratch_ptr[dev];
    return SPH_OK;
}

} // namespace

extern "C" int sph_scene_density_noalloc(sph_ctx *c, float *mean, float *maxv)
{
    if (!c || !mean || !maxv)
        return merr(SPH_EINVAL, "null argument");
    const size_t ns = c->sc.size();
    if (ns > (size_t)kNoAllocMaxScenes)
        return merr(SPH_EINVAL,
                    "sph_scene_density_noalloc: %zu scenes exceed the fixed scratch of %d scenes "
                    "(use sph_scene_density)",
                    ns, kNoAllocMaxScenes);
    int dev = 0;
    MCHK(hipGetDevice(&dev));
    if (dev != c->device)
        return merr(SPH_EINVAL, "sph_scene_density_noalloc: the context lives on device %d, "
                                "device %d is current", c->device, dev);
    float *buf = nullptr;
    if (int rc = scratch_for_current_device(&buf))
        return rc;
    if (int rc = sph_internal_canonicalize(c))
        return rc;
    k_scene_density<<<dim3((unsigned)ns), kDensityTPB, 0, c->st>>>(c->dP, c->RHO, buf, buf + ns);
    MCHK(hipGetLastError());
    float h[2 * kNoAllocMaxScenes];
    MCHK(hipMemcpyAsync(h, buf, sizeof(float) * 2 * ns, hipMemcpyDeviceToHost, c->st));
    MCHK(hipStreamSynchronize(c->st));
    for (size_t s = 0; s < ns; s++) {
        mean[s] = c->sc[s].n ? h[s] / (float)c->sc[s].n : 0.0f;
        maxv[s] = h[ns + s];
    }
    return SPH_OK;
}
