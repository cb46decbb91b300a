// Key side of the delta rule's backward, chunks of 64 tokens side by side (algebra and names: dfw_chunk_bwd.hip; precision and
// element types: dfw_chunk.hpp).  With the state S0 before a chunk and the adjoint G after it, which the value side leaves
// (store_edge), nothing of the key side is sequential and nothing is inverted: for the chunk's 64 tokens
//   d_query = g S0 + X1 K                                          X1[t][s] = g_t . delta_s   (s < t)
//   d_key   = X1^T Q + Delta G - dU S0 + (X2 + X2^T) K             X2[t][s] = -dU_t . delta_s  (s < t)
// is the block form of 16 with longer sums.  Workgroup = (row, chunk), wave w = tokens 16 w .. 16 w + 15 and all 64 key channels: its
// rows of X1, X1^T and X2 + X2^T come out of the products as ready operands (the accumulator tile of X^T is the operand "rows of
// X") and never leave its registers.  Two phases share the LDS, so that two workgroups (with single operands three, of one value
// block of 16-bit tensors four) fit a CU and one loads while the other computes: first Delta, g and -dU as [64][72] tiles, then K, Q, S0 and G; everything is
// loaded up front, 16 bytes per lane, whole token rows at a time.
//
// Value blocks (several recurrences that share q and k): the workgroup does them one after the other and adds their
// shares up, each rounded to the tensors' type, which is what the shares were stored in when they were summed by a launch of
// their own.
//
// What bounds it: memory.  B = 96, T = 1024, fp32: 5 arrays and two 64 x 64 edges per chunk in, two arrays out, 226 MB in 42 us, 5.4
// TB/s, the rate of a large copy.  Error of d_query and d_key against float64, sequential key side / here: fp32 4.5e-6 / 3.6e-6 and
// 6.7e-6 / 5.9e-6; bf16 with single operands 2.8e-3 / 2.5e-3 and 2.89e-3 / 2.89e-3 (a result is off by what its operands are rounded by,
// a score of two tokens where it was the state that holds one of them).  The sequential key side (two workgroups per row, 64 dependent blocks) took 72 us for it; the
// edges cost the value side 8 us (50 -> 58) and the whole training step goes from 164 to 150 us.  B = 48, T = 777, two value blocks
// of bf16: 32 -> 20 us here, a launch less (6 us), value side 25 -> 31.
#include "common.hpp"
#include "dfw_chunk.hpp"
#include "dfw_scan.hpp"

namespace t2fw {
namespace {

using namespace dfwc;

constexpr int KEY_THREADS = 256;
constexpr int KEY_STRIDE = 72;                            // elements from a row of a tile to the next
constexpr int KEY_PLANE = DCH * KEY_STRIDE;               // elements of a plane (heads or remainders)
template <bool SP> constexpr int KEY_TILE = (SP ? 2 : 1) * KEY_PLANE;
template <bool SP> constexpr int KEY_SMEM = 4 * KEY_TILE<SP> * 2;
static_assert(2 * KEY_SMEM<true> <= 160 * 1024, "two workgroups per CU");

template <bool SP> struct Tile64 {
    u16 *hi;
    __device__ __forceinline__ explicit Tile64(u16 *base) : hi(base) {}
    __device__ __forceinline__ void store4(int row, int col, const Sp2<SP> &v) const {
        *reinterpret_cast<uint2 *>(hi + row * KEY_STRIDE + col) = v.hi;
        if constexpr (SP) *reinterpret_cast<uint2 *>(hi + KEY_PLANE + row * KEY_STRIDE + col) = v.lo;
    }
    // operand "row `row`, columns 32 h + 8 g .. + 7"
    __device__ __forceinline__ Sp4<SP> row(int row, int g, int h) const {
        const u16 *const p = hi + row * KEY_STRIDE + 8 * g + 32 * h;
        Sp4<SP> o;
        o.hi = ld4(p);
        o.lo = SP ? ld4(p + KEY_PLANE) : make_uint4(0u, 0u, 0u, 0u);
        return o;
    }
    // operand "column col0 + r, rows row0 .. row0 + 3 and row1 .. row1 + 3" (transposing LDS reads)
    __device__ __forceinline__ Sp4<SP> column(int row0, int row1, int col0, int r) const {
        const u16 *const p0 = hi + (row0 + (r >> 2)) * KEY_STRIDE + col0 + 4 * (r & 3);
        const u16 *const p1 = hi + (row1 + (r >> 2)) * KEY_STRIDE + col0 + 4 * (r & 3);
        Sp4<SP> o;
        o.hi = bwd::cat(tr4(p0), tr4(p1));
        o.lo = SP ? bwd::cat(tr4(p0 + KEY_PLANE), tr4(p1 + KEY_PLANE)) : make_uint4(0u, 0u, 0u, 0u);
        return o;
    }
    static __device__ __forceinline__ uint2 tr4(const u16 *p) {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_ptr)(p)));
    }
};

// c + a b with the remainders' product too: the matrix cores have the time, and it takes out what the sums of 64 tokens in the place of
// 16 add to the error
template <bool SP> __device__ __forceinline__ floatx4 mma(const Sp4<SP> &a, const Sp4<SP> &b, floatx4 c) {
    if constexpr (SP) c = Bf16::mfma32(a.lo, b.lo, c);
    return mma32(a, b, c);
}

// RAGGED: the last chunk of a sequence that ends within it.  Its edges have no place among its tokens' results: the adjoint after it
// is the final state's own, the state before it comes from the final state by one more product, S0 = S_end - Delta^T K.
template <bool SP, typename E, bool BLOCKS, bool RAGGED> __device__ __forceinline__ void key_chunk(const DfwBwdArgs &p, u16 *lds, int64_t brow, int c) {
    typedef typename E::elem elem;
    typedef typename E::Raw4 Raw4;
    int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tok0 = c * DCH, T = (int)p.T;
    const int blocks = BLOCKS ? p.blocks : 1;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};

    // 64 rows of an array: lane piece i is row (tid + 256 i) / 16, channels 4 (tid % 16) .. + 3
    struct Rows {
        Raw4 v[4];
    };
    auto load_rows = [&](Rows &x, const void *base, int64_t first, u32 stride) {          // the chunk's tokens; those past T are zeroed below
        const elem *const src = reinterpret_cast<const elem *>(base) + first;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = tok0 + (tid >> 4) + 16 * i;
            x.v[i] = *reinterpret_cast<const Raw4 *>(src + (size_t)(RAGGED ? min(t, T - 1) : t) * stride + 4 * (tid & 15));
        }
    };
    auto build = [&](int slot, const Rows &x, float sign, bool tokens = true) {
        const Tile64<SP> tile(lds + slot * KEY_TILE<SP>);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const floatx4 v = E::floats(x.v[i]);
            const bool in = !RAGGED || !tokens || tok0 + (tid >> 4) + 16 * i < T;
            tile.store4((tid >> 4) + 16 * i, 4 * (tid & 15), split4<SP>(in ? sign * v[0] : 0.f, in ? sign * v[1] : 0.f, in ? sign * v[2] : 0.f, in ? sign * v[3] : 0.f));
        }
    };
    // A state or adjoint as the value side left it (store_edge): pieces tid + 256 i
    constexpr int PLANES = SP ? 2 : 1;
    typedef u32 Piece __attribute__((ext_vector_type(4)));
    struct Edge {
        Piece v[2 * PLANES];
    };
    auto load_edge = [&](Edge &x, const void *base, int64_t b) {
        const Piece *const src = reinterpret_cast<const Piece *>(reinterpret_cast<const elem *>(base) + (b * p.T + tok0) * CH_N);
#pragma unroll
        for (int i = 0; i < 2 * PLANES; ++i) x.v[i] = src[tid + KEY_THREADS * i];
    };
    auto build_edge = [&](int slot, const Edge &x) {
#pragma unroll
        for (int i = 0; i < 2 * PLANES; ++i) {
            const int q = tid + KEY_THREADS * (i & 1);                // of plane i / 2
            u16 *const at = lds + slot * KEY_TILE<SP> + (i >> 1) * KEY_PLANE + (16 * (q >> 7) + (q & 15)) * KEY_STRIDE + 32 * ((q >> 6) & 1) + 4 * ((q >> 4) & 3);
            *reinterpret_cast<uint2 *>(at) = make_uint2(x.v[i][0], x.v[i][1]);
            *reinterpret_cast<uint2 *>(at + 16) = make_uint2(x.v[i][2], x.v[i][3]);
        }
    };

    floatx4 sum_q[BLOCKS ? 4 : 1], sum_k[BLOCKS ? 4 : 1];
    if constexpr (BLOCKS)
#pragma unroll
        for (int j = 0; j < 4; ++j) sum_q[j] = sum_k[j] = zero;

    for (int blk = 0; blk < blocks; ++blk) {
        // with several blocks: every address is computed anew, or what the compiler keeps of them over the loop fills the registers
        if constexpr (BLOCKS) asm volatile("" : "+v"(tid));
        const int r = tid & 15, g = (tid >> 4) & 3;
        const int64_t b = brow * blocks + blk;
        const DfwRow<BLOCKS> row(b, p.T, p.blocks);
        Rows dl, go, dv, k, q;
        Edge s0, ge;
        Rows gs;
        load_rows(dl, p.delta, row.value, row.vs);
        load_rows(go, p.g_out, row.value, row.vs);
        load_rows(dv, p.d_v, row.value, row.vs);
        load_rows(k, p.k, row.key, CH_N);
        load_rows(q, p.q, row.key, CH_N);
        if constexpr (RAGGED) {
            const elem *const src = reinterpret_cast<const elem *>(p.g_state) + b * CH_N * CH_N;
#pragma unroll
            for (int i = 0; i < 4; ++i) gs.v[i] = reinterpret_cast<const Raw4 *>(src)[tid + KEY_THREADS * i];
        } else {
            load_edge(s0, p.states, b);
            load_edge(ge, p.adjoints, b);
        }
        if (BLOCKS && blk > 0) __syncthreads();               // the block before has been read
        if constexpr (RAGGED) {
            build(0, dl, -1.f);
            build(1, k, 1.f);
            __syncthreads();
            const Tile64<SP> ND(lds), K(lds + KEY_TILE<SP>), S(lds + 3 * KEY_TILE<SP>);
            const elem *const fin = reinterpret_cast<const elem *>(p.final_state) + (b * CH_N + 16 * w + r) * CH_N + 4 * g;
            const Sp4<SP> d0 = ND.column(8 * g, 8 * g + 4, 16 * w, r), d1 = ND.column(32 + 8 * g, 36 + 8 * g, 16 * w, r);
#pragma unroll
            for (int j = 0; j < 4; ++j) {                     // S0[d = 16 w + r][16 j + 4 g + e]
                floatx4 v = mma(K.column(8 * g, 8 * g + 4, 16 * j, r), d0, E::load4(fin + 16 * j));
                v = mma(K.column(32 + 8 * g, 36 + 8 * g, 16 * j, r), d1, v);
                S.store4(16 * w + r, 16 * j + 4 * g, split4<SP>(v));
            }
            __syncthreads();
        }
        build(0, dl, 1.f);
        build(1, go, 1.f);
        build(2, dv, -1.f);
        __syncthreads();
        // the wave's own rows, and its rows of X1, X1^T and X2 + X2^T against the token tiles a = 0 .. 3: lane (r, g) holds
        // elements 16 a + 4 g + e of row 16 w + r
        Sp4<SP> dl_own[2], go_own[2], nu_own[2];
        Sp2<SP> x1[4], x1t[4], x2[4];
        {
            const Tile64<SP> DL(lds), GO(lds + KEY_TILE<SP>), NU(lds + 2 * KEY_TILE<SP>);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                dl_own[h] = DL.row(16 * w + r, g, h);
                go_own[h] = GO.row(16 * w + r, g, h);
                nu_own[h] = NU.row(16 * w + r, g, h);
            }
            const Sp2<SP> none = split4<SP>(zero);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                floatx4 y = zero;
                x1[a] = x1t[a] = none;
                if (a <= w) {          // tokens before the wave's: [s = 16 a + 4 g + e][t = own r]
                    const Sp4<SP> d0 = DL.row(16 * a + r, g, 0), d1 = DL.row(16 * a + r, g, 1);
                    floatx4 z = mma(d1, go_own[1], mma(d0, go_own[0], zero));
                    floatx4 u = mma(d1, nu_own[1], mma(d0, nu_own[0], zero));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool before = a < w || 4 * g + e < r;
                        z[e] = before ? z[e] : 0.f;
                        y[e] = before ? u[e] : 0.f;
                    }
                    x1[a] = split4<SP>(z);
                }
                if (a >= w) {          // tokens after the wave's: [t = 16 a + 4 g + e][s = own r]
                    floatx4 z = mma(GO.row(16 * a + r, g, 1), dl_own[1], mma(GO.row(16 * a + r, g, 0), dl_own[0], zero));
                    floatx4 u = mma(NU.row(16 * a + r, g, 1), dl_own[1], mma(NU.row(16 * a + r, g, 0), dl_own[0], zero));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool after = a > w || r < 4 * g + e;
                        z[e] = after ? z[e] : 0.f;
                        y[e] = after ? u[e] : y[e];
                    }
                    x1t[a] = split4<SP>(z);
                }
                x2[a] = split4<SP>(y);
            }
        }
        __syncthreads();
        build(0, k, 1.f);
        build(1, q, 1.f);
        if constexpr (RAGGED) {
            build(2, gs, 1.f, false);
        } else {
            build_edge(2, ge);
            build_edge(3, s0);
        }
        __syncthreads();
        const Tile64<SP> K(lds), Q(lds + KEY_TILE<SP>), G(lds + 2 * KEY_TILE<SP>), S(lds + 3 * KEY_TILE<SP>);
        // Pairs of token tiles (2 h, 2 h + 1) make 32-deep sums.  Where a pair's other tile has no part in X1 (X1^T) the zeros
        // there meet the wave's own tile once more: an infinity or a NaN of tokens that a result does not depend on
        // reaches no further than the 16 tokens around it.
#pragma unroll
        for (int j = 0; j < 4; ++j) {          // [channel 16 j + 4 g + e][token r of the wave]
            floatx4 dq = zero, dk = zero;
            const Sp4<SP> s_0 = S.column(8 * g, 8 * g + 4, 16 * j, r), s_1 = S.column(32 + 8 * g, 36 + 8 * g, 16 * j, r);
            dq = mma(s_1, go_own[1], mma(s_0, go_own[0], dq));
            dk = mma(G.column(32 + 8 * g, 36 + 8 * g, 16 * j, r), dl_own[1], mma(G.column(8 * g, 8 * g + 4, 16 * j, r), dl_own[0], dk));
            dk = mma(s_1, nu_own[1], mma(s_0, nu_own[0], dk));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int lo = 32 * h, hi = 32 * h + 16;
                const Sp4<SP> kc = K.column(lo + 4 * g, hi + 4 * g, 16 * j, r);
                dk = mma(kc, cat(x2[2 * h], x2[2 * h + 1]), dk);
                if (2 * h <= w) {              // X1: tiles up to the wave's own
                    const bool both = 2 * h + 1 <= w;
                    const Sp4<SP> kb = both ? kc : K.column(lo + 4 * g, lo + 4 * g, 16 * j, r);
                    dq = mma(kb, cat(x1[2 * h], x1[2 * h + 1]), dq);
                }
                if (2 * h + 1 >= w) {          // X1^T: tiles from the wave's own on
                    const int first = 2 * h >= w ? lo : hi;
                    dk = mma(Q.column(first + 4 * g, hi + 4 * g, 16 * j, r), cat(x1t[2 * h], x1t[2 * h + 1]), dk);
                }
            }
            if constexpr (BLOCKS) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sum_q[j][e] += E::f(E::e(dq[e]));
                    sum_k[j][e] += E::f(E::e(dk[e]));
                }
            } else if (!RAGGED || tok0 + 16 * w + r < T) {
                const int64_t o = row.key + (int64_t)(tok0 + 16 * w + r) * CH_N + 16 * j + 4 * g;
                E::store4(reinterpret_cast<elem *>(p.d_q) + o, dq);
                E::store4(reinterpret_cast<elem *>(p.d_k) + o, dk);
            }
        }
    }
    if constexpr (BLOCKS) {
        const int r = tid & 15, g = (tid >> 4) & 3;
        if (!RAGGED || tok0 + 16 * w + r < T) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t o = (brow * p.T + tok0 + 16 * w + r) * CH_N + 16 * j + 4 * g;
                E::store4(reinterpret_cast<elem *>(p.d_q) + o, sum_q[j]);
                E::store4(reinterpret_cast<elem *>(p.d_k) + o, sum_k[j]);
            }
        }
    }
}

template <bool SP, typename E, bool BLOCKS> __global__ __launch_bounds__(KEY_THREADS, SP ? 2 : 3) void dfw_key_kernel(DfwBwdArgs p, int chunks) {
    extern __shared__ __align__(16) unsigned char smem[];
    u16 *const lds = reinterpret_cast<u16 *>(smem);
    const int brow = (int)blockIdx.x / chunks, c = (int)blockIdx.x - brow * chunks;
    if ((int64_t)(c + 1) * DCH > p.T)
        key_chunk<SP, E, BLOCKS, true>(p, lds, brow, c);
    else
        key_chunk<SP, E, BLOCKS, false>(p, lds, brow, c);
}

template <bool SP, typename E, bool BLOCKS> int launch_key(const DfwBwdArgs &a, hipStream_t stream) {
    auto kern = dfw_key_kernel<SP, E, BLOCKS>;
    const int rc = enable_lds(reinterpret_cast<const void *>(kern), KEY_SMEM<SP>, "hipFuncSetAttribute(delta-rule backward kernel, key side's chunks)");
    if (rc) return rc;
    const int64_t chunks = (a.T + DCH - 1) / DCH, items = a.B / a.blocks * chunks;
    if (items > 0x7fffffffLL) return fail(T2FW_ERR_UNSUPPORTED, "B=%lld T=%lld: too many chunks", (long long)a.B, (long long)a.T);
    hipLaunchKernelGGL(kern, dim3((unsigned)items), dim3(KEY_THREADS), KEY_SMEM<SP>, stream, a, (int)chunks);
    return check_hip(hipGetLastError(), "dfw_key_kernel launch");
}

}  // namespace

int dfw_key_chunks(const DfwBwdArgs &a, int dtype, bool split_operands, hipStream_t stream) {
    if (dtype == T2FW_F32 && split_operands) return a.blocks > 1 ? launch_key<true, ElF32, true>(a, stream) : launch_key<true, ElF32, false>(a, stream);
    if (split_operands) return fail(T2FW_ERR_UNSUPPORTED, "16-bit tensors with split operands have no chunks of the key side");
    switch (dtype) {
    case T2FW_F32: return a.blocks > 1 ? launch_key<false, ElF32, true>(a, stream) : launch_key<false, ElF32, false>(a, stream);
    case T2FW_F16: return a.blocks > 1 ? launch_key<false, El16<Fp16>, true>(a, stream) : launch_key<false, El16<Fp16>, false>(a, stream);
    case T2FW_BF16: return a.blocks > 1 ? launch_key<false, El16<Bf16>, true>(a, stream) : launch_key<false, El16<Bf16>, false>(a, stream);
    default: return fail(T2FW_ERR_UNSUPPORTED, "the block-wise delta-rule kernels take fp32, fp16 and bf16 tensors");
    }
}

}  // namespace t2fw
