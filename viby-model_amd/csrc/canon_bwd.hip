// Canon causal depthwise conv1d for MI355X (gfx950): backward of the prefill
// (dx, and dweight / dbias through partial sets and a fixed-order reduction).
#include "canon_device.h"

namespace canon {

// ---------------------------------------------------------------------------
// backward of the prefill: dx, and per-chunk partial sums of dweight / dbias
//
// Every kernel of this file writes dx and one entry per channel of a partial
// set, partial[(b * nchunk + chunk) * C + c][5] (w0..w3, bias);
// canon_bwd_reduce_kernel sums the sets in a fixed order.
//
// canon_bwd_walk_kernel, the fallback for layouts without a vector kernel
// (any strides): one lane owns a channel and walks a chunk of time steps from
// its END to its start.  dx[t] needs dz[t .. t+W-1] (the three later steps are
// carried in registers), z[t] needs xm[t-3 .. t] (a sliding window refilled
// with one row per step, fetched R rows ahead).  The three dz values just past
// the chunk are recomputed from memory.
//
// With an initial state (a.init) the rows before t = 0 are its last entries
// instead of zeros: they enter the windows (z and dweight) like any other row,
// and the lane that ends at t = 0 also forms their gradient from the three dz
// values it carries out of the loop.
//
// SEQ (packed sequences): the sequence index of every row travels with it
// (window, carried dz values, look-ahead).  A product of a tap with a row of
// another sequence index is dropped wherever it appears: in z, in dx (the dz
// of a later step of another sequence) and in dweight.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float silu_grad(float z)
{
    const float s = __builtin_amdgcn_rcpf(1.0f + __expf(-z));
    return fmaf(s, fmaf(-z, s, z), s);   // s + s * z * (1 - s)
}

template <int DT, int W, bool MASK, int R, bool SEQ>
__global__ __launch_bounds__(256) void canon_bwd_walk_kernel(const BwdArgs a)
{
    constexpr int BY = Elem<DT>::bytes;
    constexpr int E = 1;     // channels per lane
    const uint32_t tid = blockIdx.x * 256u + threadIdx.x;
    if (tid >= a.nthreads) return;
    const uint32_t bc = fdiv(tid, a.div_nvec);
    const uint32_t cv = tid - bc * a.nvec;
    const uint32_t b = fdiv(bc, a.div_nchunk);
    const uint32_t ch = bc - b * a.nchunk;
    const uint32_t c0 = cv * E;

    const char *xb = a.x + ((int64_t)b * a.x_sb + (int64_t)c0 * a.x_sc) * BY;
    const char *gb = a.dy + ((int64_t)b * a.g_sb + (int64_t)c0 * a.g_sc) * BY;
    char *db_ = a.dx + ((int64_t)b * a.d_sb + (int64_t)c0 * a.d_sc) * BY;
    const int64_t xs = a.x_sl * BY, gs = a.g_sl * BY, ds = a.d_sl * BY;
    const int64_t t_begin = (int64_t)ch * a.chunk;
    const int64_t t_stop = t_begin + (int64_t)a.chunk;
    const int64_t t_end = t_stop < (int64_t)a.L ? t_stop : (int64_t)a.L;
    const int64_t Lm1 = (int64_t)a.L - 1;

    RawTaps<E> raw;
    fetch_taps<W, E>(a.weight, a.bias, a.w_sc, a.w_sk, a.w_dtype, false, c0, raw);

    // rows t_end-4 .. t_end+2 of xm (window for the last step + the three steps past the chunk)
    float xr7[7][E], m7[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        const int64_t t = t_end - 4 + j;
        const int64_t tc = t < 0 ? 0 : (t > Lm1 ? Lm1 : t);
        xr7[j][0] = load1<DT>(xb + tc * xs, 0);
        m7[j] = 1.0f;
    }
    float g3[3][E];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int64_t t = t_end + j;
        g3[j][0] = load1<DT>(gb + (t > Lm1 ? Lm1 : t) * gs, 0);
    }
    if constexpr (MASK) load_mask_rows<7>(a.mask, (int64_t)b * a.m_sb, t_end - 4, a.L, a.m_sl, a.mask_dtype, m7);
    // rows before t = 0: entries of the initial state (not masked), zeros without one
    const char *ib = a.init ? a.init + ((int64_t)b * a.i_sb + (int64_t)c0 * a.i_sc + (int64_t)a.S_in * a.i_ss) * BY : nullptr;
    const int64_t is = a.i_ss * BY;
    float h7[7] = {0, 0, 0, 0, 0, 0, 0};
    if (ib && t_end < 4) {
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            const int64_t t = t_end - 4 + j;
            if (t < 0 && t >= -(int64_t)a.S_in) h7[j] = load1<DT>(ib + t * is, 0);
        }
    }
    int32_t q7[7] = {0, 0, 0, 0, 0, 0, 0};   // sequence indices of the same seven rows
    if constexpr (SEQ) load_seq_rows<7>(a.seq, (int64_t)b * a.q_sb, t_end - 4, a.L, a.q_sl, q7);

    float w[E][W], bias[E];
    decode_taps<DT, W, E>(raw, a.w_dtype, false, a.bias != nullptr, w, bias);

#pragma unroll
    for (int j = 0; j < 7; ++j) {
        const int64_t t = t_end - 4 + j;
        const bool inside = t >= 0 && t <= Lm1;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float v = MASK ? mul_round<DT>(xr7[j][e], m7[j]) : xr7[j][e];
            xr7[j][e] = inside ? v : (t < 0 ? h7[j] : 0.0f);
        }
    }
    // dzf[j] = dz[t_end + j]
    float dzf[3][E];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const bool inside = t_end + j <= Lm1;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float z = bias[e];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                const int row = j + 1 + (4 - W) + k;                                   // xm[t_end+j-(W-1)+k]
                const float v = (!SEQ || q7[row] == q7[j + 4]) ? xr7[row][e] : 0.0f;
                z = fmaf(w[e][k], v, z);
            }
            const float d = a.act ? g3[j][e] * silu_grad(z) : g3[j][e];
            dzf[j][e] = inside ? d : 0.0f;
        }
    }
    // xw[k] = xm[t-3+k] for the step being processed, starting with t = t_end - 1
    float xw[4][E];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < E; ++e) xw[k][e] = xr7[k][e];
    // qw[k]: sequence index of xw[k]'s row; qf[j]: of dzf[j]'s step
    int32_t qw[4] = {q7[0], q7[1], q7[2], q7[3]};
    int32_t qf[3] = {q7[4], q7[5], q7[6]};

    float dw[E][W], dbs[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        dbs[e] = 0.0f;
#pragma unroll
        for (int k = 0; k < W; ++k) dw[e][k] = 0.0f;
    }

    for (int64_t t_hi = t_end - 1; t_hi >= t_begin; t_hi -= R) {
        // this batch: steps t_hi, t_hi-1, .., t_hi-R+1; needs dout of those steps and x rows t-4.
        // Rows are kept as loaded (raw) until their step, to keep the register count down.
        float G[R], XN[R], HN[R];
        float mk[R], mn[R];
        int32_t QN[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t t = t_hi - r;
            const int64_t tg = t < 0 ? 0 : t;
            const int64_t tn = t - 4 < 0 ? 0 : t - 4;
            G[r] = load1<DT>(gb + tg * gs, 0);
            XN[r] = load1<DT>(xb + tn * xs, 0);
            HN[r] = (ib && t - 4 < 0 && t - 4 >= -(int64_t)a.S_in) ? load1<DT>(ib + (t - 4) * is, 0) : 0.0f;
            QN[r] = SEQ ? a.seq[(int64_t)b * a.q_sb + tn * a.q_sl] : 0;
            mk[r] = 1.0f;
            mn[r] = 1.0f;
        }
        if constexpr (MASK) {
            // masks of steps t_hi-R+1 .. t_hi (for dx) and of rows t_hi-R-3 .. t_hi-4 (for the window)
            float mm[R + 4];
            load_mask_rows<R + 4>(a.mask, (int64_t)b * a.m_sb, t_hi - R - 3, a.L, a.m_sl, a.mask_dtype, mm);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                mk[r] = mm[R + 3 - r];      // step t_hi - r
                mn[r] = mm[R - 1 - r];      // row  t_hi - r - 4
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t t = t_hi - r;
            if (t < t_begin) break;
            float g[E], xn[E], dz[E], o[E];
            g[0] = G[r];
            xn[0] = XN[r];
            // the window as this step sees it: rows of other sequences read as zero
            float xs_[4][E];
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int e = 0; e < E; ++e) xs_[k][e] = (!SEQ || qw[k] == qw[3]) ? xw[k][e] : 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float z = bias[e];
#pragma unroll
                for (int k = 0; k < W; ++k) z = fmaf(w[e][k], xs_[(4 - W) + k][e], z);
                dz[e] = z;
            }
            if (a.act) {
#pragma unroll
                for (int e = 0; e < E; ++e) dz[e] = g[e] * silu_grad(dz[e]);
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) dz[e] = g[e];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                // dxm[t] = sum_k w[k] * dz[t + (W-1) - k]
                float acc = w[e][W - 1] * dz[e];
                acc = fmaf(w[e][W - 2], (!SEQ || qf[0] == qw[3]) ? dzf[0][e] : 0.0f, acc);
                if constexpr (W >= 3) acc = fmaf(w[e][W - 3], (!SEQ || qf[1] == qw[3]) ? dzf[1][e] : 0.0f, acc);
                if constexpr (W == 4) acc = fmaf(w[e][0], (!SEQ || qf[2] == qw[3]) ? dzf[2][e] : 0.0f, acc);
                o[e] = acc;
#pragma unroll
                for (int k = 0; k < W; ++k) dw[e][k] = fmaf(dz[e], xs_[(4 - W) + k][e], dw[e][k]);
                dbs[e] += dz[e];
                dzf[2][e] = dzf[1][e];
                dzf[1][e] = dzf[0][e];
                dzf[0][e] = dz[e];
            }
            if (a.res_mode == CANON_RESIDUAL_MASKED) {
#pragma unroll
                for (int e = 0; e < E; ++e) o[e] += g[e];
            }
            if (a.dfin && t >= (int64_t)a.L - a.S_out) {
                // this step's masked input was captured into slot t - (L - S_out) of the final state
                o[0] += load1<DT>(a.dfin + ((int64_t)b * a.k_sb + (int64_t)c0 * a.k_sc + (t - ((int64_t)a.L - a.S_out)) * a.k_ss) * BY, 0);
            }
            if constexpr (MASK) {
#pragma unroll
                for (int e = 0; e < E; ++e) o[e] *= mk[r];
            }
            if (a.res_mode == CANON_RESIDUAL_UNMASKED) {
#pragma unroll
                for (int e = 0; e < E; ++e) o[e] += g[e];
            }
            // slide the window one step back: the new oldest row is t - 4
            const bool has_row = t - 4 >= 0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float v = xn[e];
                if constexpr (MASK) v = mul_round<DT>(v, mn[r]);
                xw[3][e] = xw[2][e];
                xw[2][e] = xw[1][e];
                xw[1][e] = xw[0][e];
                xw[0][e] = has_row ? v : HN[r];
            }
            if constexpr (SEQ) {
                qf[2] = qf[1]; qf[1] = qf[0]; qf[0] = qw[3];
                qw[3] = qw[2]; qw[2] = qw[1]; qw[1] = qw[0]; qw[0] = QN[r];
            }
            store1<DT>(db_ + t * ds, 0, o[0]);
        }
    }

    if (a.dinit && ch == 0) {
        // here dzf[i] = dz[i] (zero past the end of the row).  Entry s is the input at t = s - S_in = -d:
        // its gradient is sum_i w[W-1-d-i] * dz[i] over the taps that exist
        char *jb = a.dinit + ((int64_t)b * a.j_sb + (int64_t)c0 * a.j_sc) * BY;
        for (int s = 0; s < a.S_in; ++s) {
            const int d = a.S_in - s;
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int k = W - 1 - d - i;
                if (k >= 0) acc = fmaf(w[0][k], dzf[i][0], acc);
            }
            // a final state longer than the row also captured this entry (input at t = -d) in slot S_out - L - d
            const int64_t slot = (int64_t)a.S_out - (int64_t)a.L - d;
            if (a.dfin && slot >= 0)
                acc += load1<DT>(a.dfin + ((int64_t)b * a.k_sb + (int64_t)c0 * a.k_sc + slot * a.k_ss) * BY, 0);
            store1<DT>(jb + (int64_t)s * a.j_ss * BY, 0, acc);
        }
    }

    float *pp = a.partial + (((int64_t)b * a.nchunk + ch) * a.C + c0) * 5;
#pragma unroll
    for (int e = 0; e < E; ++e) {
#pragma unroll
        for (int k = 0; k < 4; ++k) pp[e * 5 + k] = k < W ? dw[e][k] : 0.0f;
        pp[e * 5 + 4] = dbs[e];
    }
}

// ---------------------------------------------------------------------------
// backward, channel-contiguous tensors ([B, L, C] viewed as [B, C, L]).
//
// A block is four waves; a lane owns two adjacent channels (kBwdLaneChannels),
// a wave a slab of kBwdSlab consecutive time steps of a
// 64-lane channel tile, the four waves four consecutive slabs, and the block
// walks over the `chunk` time steps of its chunk one such 32-step tile at a
// time, keeping its dweight / dbias sums in registers.
//
// Per tile, all rows of x and dout of the slab are requested before anything
// is waited for.  The three rows of x before a slab come from the previous
// wave's slab through LDS (the first wave reads them from memory).  dz of the
// slab's first three steps is computed first and handed to the previous wave
// through LDS (that wave's dx needs dz of the three steps after its slab; the
// last wave recomputes them from three extra rows of x and dout).  The slab is
// then swept from its last step to its first:
//   dz[t] = dout[t] * act'(z[t]),  dx[t] = sum_k w[k] * dz[t + (W-1) - k]
// At the end the four waves' sums are added in a fixed order through LDS and
// written as one partial set entry per channel.
//
// What bounds it: requests in flight.  The sums, taps, window and carried dz
// of a channel stay in registers through the sweep, about thirty of them, so
// the channels a lane owns decide how many waves a CU holds: with four
// channels (8 bytes of a 16-bit row) 170-200 registers, two blocks per CU;
// with two 81-97 without an activation, up to 128 with SiLU or states, four or
// five.  And chunks of 128 steps where the grid alone
// would allow up to 1024: a CU then has new blocks to start while others drain,
// for one partial set (20 bytes per channel) per 768 bytes of rows read and
// written.  With both, us per call with the reduction, four channels -> two,
// L 1024, bf16: B 32 C 3456 masked 145.2 -> 125.2, with SiLU 166.9 -> 128.5;
// B 8 C 3456 38.7 -> 37.6, with SiLU 47.1 -> 41.0; B 16 C 640 L 511 SiLU masked
// 19.0 -> 17.1; B 8 C 640 14.9 -> 12.8; packed rows B 2 C 3456 L 8192 SiLU
// 91.3 -> 77.8; fp32 (two channels before as well) B 8 C 3456 70.1 -> 66.3.
// Chunks of 192 steps: within 1 %; of 256: 2-13 % slower from B 4 C 3456 on.
// ---------------------------------------------------------------------------
// x and dout are read once and dx is written once: streamed (non-temporal) accesses, as in the forward kernels
// (measured at B 8, C 3456, L 1024, bf16: 40.7 -> 37.8 us channel-contiguous, 33.6 -> 30.9 us time-contiguous).
constexpr bool kBwdStream = true;
template <int DT> using BwdIO = VecIO<kBwdLaneChannels * Elem<DT>::bytes>;
template <int DT> using BwdVec = typename BwdIO<DT>::type;   // a lane's piece of one row
template <int DT> __device__ __forceinline__ void unpack_lane(const BwdVec<DT> &v, float *f) { BwdIO<DT>::template unpack<DT>(v, f); }
template <int DT> __device__ __forceinline__ BwdVec<DT> pack_lane(const float *f) { return BwdIO<DT>::template pack<DT>(f); }

// One raw row -> the bits of xm = x * mask in the storage type (zero when the row does not exist)
constexpr uint32_t kMaskOne = 0x3F800000u;   // 1.0f
template <int DT, bool MASK>
__device__ __forceinline__ BwdVec<DT> bwd_mask_row(const BwdVec<DT> &raw, uint32_t m_bits, bool exists)
{
    constexpr int E = kBwdLaneChannels;
    BwdVec<DT> v = raw;
    if constexpr (MASK) {
      // m is the same for the whole wave (its bits are in a scalar register: a scalar branch) and 1 for every valid
      // token of a padded batch: x * 1 is x, bit for bit
      if (m_bits != kMaskOne) {
        const float m = bits_f(m_bits);
        float f[E];
        unpack_lane<DT>(raw, f);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            f[e] *= m;
            if constexpr (DT == CANON_DTYPE_F16) asm volatile("" : "+v"(f[e]));   // see mul_round
        }
        v = pack_lane<DT>(f);
      }
    }
    if (!exists) v = BwdIO<DT>::zero();
    return v;
}

// dz of one step from its window of xm rows and dout
template <int W, int E, bool ACT>
__device__ __forceinline__ void bwd_dz(const float (*w)[W], const float *bias, const float *x0, const float *x1,
                                       const float *x2, const float *x3, const float *g, float *dz)
{
    if constexpr (ACT) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float z = bias[e];
            if constexpr (W == 4) z = fmaf(w[e][0], x0[e], z);
            if constexpr (W >= 3) z = fmaf(w[e][W - 3], x1[e], z);
            z = fmaf(w[e][W - 2], x2[e], z);
            z = fmaf(w[e][W - 1], x3[e], z);
            dz[e] = g[e] * silu_grad(z);
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) dz[e] = g[e];
    }
}

// ... where rows of the window may belong to another packed sequence (keep: whether they belong to this step's)
template <int W, int E, bool ACT>
__device__ __forceinline__ void bwd_dz_gated(const float (*w)[W], const float *bias, const float *x0, const float *x1,
                                             const float *x2, const float *x3, bool keep0, bool keep1, bool keep2,
                                             const float *g, float *dz)
{
    float y[3][E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        y[0][e] = keep0 ? x0[e] : 0.0f;
        y[1][e] = keep1 ? x1[e] : 0.0f;
        y[2][e] = keep2 ? x2[e] : 0.0f;
    }
    bwd_dz<W, E, ACT>(w, bias, y[0], y[1], y[2], x3, g, dz);
}

// The sweep over one slab, last step first.  X / H hold xm in storage bits, dzh the dz of the
// first three steps (already zero past the end of the sequence), dzf the dz of the three steps
// after the slab.  FULL: all R steps exist.  FIN: some steps of the slab were captured into the final state
// (slot t - fin_first for t >= fin_first = L - S_out) and get that slot's gradient, read at `fin` (the lane's
// first channel of slot 0) where it is needed: at most S_out steps per sequence.
// SEQ: rows of several packed sequences in reach; q[j] is the sequence index of slab row j - 3 (rows -3 .. R+2).
// ANY: dx is written through the lane's own pointer `any` (nullptr: a lane without channels), rows a.d_sl apart.
// RES: the residual's gradient is added to dx (1) or is not (0), with nothing between that sum and the store; -1: as the
// arguments say.
template <int DT, int W, bool MASK, bool ACT, bool FULL, bool FIN, int R, int E, bool SEQ = false, bool ANY = false, int RES = -1>
__device__ __forceinline__ void bwd_sweep(const BwdArgs &a, const float (*w)[W], const float *bias, const BwdVec<DT> *X,
                                          const BwdVec<DT> *H, const BwdVec<DT> *G, const uint32_t *mm, const float (*dzh)[E],
                                          float (*dzf)[E], float (*dw)[W], float *dbs, __amdgpu_buffer_rsrc_t rd, uint32_t voff,
                                          uint32_t ds, int rows, const char *fin = nullptr, int64_t fin_first_row = 0,
                                          const int32_t *q = nullptr, char *any = nullptr)
{
    float xw[4][E];   // xm of rows r-3 .. r
#pragma unroll
    for (int k = 0; k < 4; ++k) unpack_lane<DT>(X[R - 4 + k], xw[k]);
    // The residual's gradient is added before the mask multiply (masked residual) or after it (unmasked); with
    // nothing in between the two are the same sum.  Real branches (the empty asm keeps the compiler from turning
    // them into an add and a select per element and mode: 12 of 75 VALU instructions per row).
    const bool res_pre = RES >= 0 ? RES == 1 : a.res_mode == CANON_RESIDUAL_MASKED || (!MASK && !FIN && a.res_mode == CANON_RESIDUAL_UNMASKED);
    const bool res_post = RES < 0 && a.res_mode == CANON_RESIDUAL_UNMASKED && !res_pre;
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
        float g[E], dz[E], o[E];
        unpack_lane<DT>(G[r], g);
        // the window and the three later dz as this row sees them: rows of another sequence read as zero
        float xg[SEQ ? 3 : 1][E], dg[SEQ ? 3 : 1][E];
        if constexpr (SEQ) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const bool before = q[r + k] == q[r + 3], after = q[r + 4 + k] == q[r + 3];
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    xg[k][e] = before ? xw[k][e] : 0.0f;
                    dg[k][e] = after ? dzf[k][e] : 0.0f;
                }
            }
        }
        const float (*xv)[E] = SEQ ? xg : xw;      // rows r-3, r-2, r-1
        const float (*dv)[E] = SEQ ? dg : dzf;     // dz of rows r+1, r+2, r+3
        if (r >= 3 || !ACT) {
            bwd_dz<W, E, ACT>(w, bias, xv[0], xv[1], xv[2], xw[3], g, dz);
            if constexpr (!FULL) {
#pragma unroll
                for (int e = 0; e < E; ++e) dz[e] = r < rows ? dz[e] : 0.0f;
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) dz[e] = dzh[r][e];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float acc = w[e][W - 1] * dz[e];
            acc = fmaf(w[e][W - 2], dv[0][e], acc);
            if constexpr (W >= 3) acc = fmaf(w[e][W - 3], dv[1][e], acc);
            if constexpr (W == 4) acc = fmaf(w[e][0], dv[2][e], acc);
            o[e] = acc;
            // Steps past the end of the sequence have a dz of zero, but their window holds the sequence's last inputs, and
            // 0 * Inf is NaN: the window is zero as well (selects), or the sums are left out (a branch).  By register
            // count: the branch costs the ordinary instances five registers and with SiLU (95 -> 100) a wave per SIMD;
            // the gated sweep holds 107 with it, 128 with the selects, but at width 3 117-122 with the selects and up to 130
            // (fp16: four waves hold 128) with the branch.
            if (!SEQ || W == 3 || r < rows) {
#pragma unroll
                for (int k = 0; k < W - 1; ++k) dw[e][k] = fmaf(dz[e], FULL || (SEQ && W != 3) || r < rows ? xv[(4 - W) + k][e] : 0.0f, dw[e][k]);
                dw[e][W - 1] = fmaf(dz[e], xw[3][e], dw[e][W - 1]);
            }
            dbs[e] += dz[e];
            dzf[2][e] = dzf[1][e];
            dzf[1][e] = dzf[0][e];
            dzf[0][e] = dz[e];
        }
        if (res_pre) {
            if constexpr (RES < 0) asm volatile("");
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] += g[e];
        }
        if constexpr (FIN) {
            // fin_first_row: the slab row of the first captured step (may be negative)
            if (r >= fin_first_row && r < rows) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                    o[e] += load1<DT>(fin, (int64_t)e * a.k_sc + ((int64_t)r - fin_first_row) * a.k_ss);
            }
        }
        if constexpr (MASK) {
            if (mm[3 + r] != kMaskOne) {
#pragma unroll
                for (int e = 0; e < E; ++e) o[e] *= bits_f(mm[3 + r]);
            }
        }
        if (res_post) {
            asm volatile("");
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] += g[e];
        }
        if constexpr (ANY) {
            if ((FULL || r < rows) && any)
                store_any<kBwdLaneChannels * Elem<DT>::bytes>(any + r * a.d_sl * Elem<DT>::bytes, pack_lane<DT>(o));
        } else if (FULL || r < rows) {
            BufIO<kBwdLaneChannels * Elem<DT>::bytes>::template store<kAuxStream>(pack_lane<DT>(o), rd, voff, (uint32_t)r * ds);
        }
        // row by row: interleaved, the eight rows of a slab hold ten more registers and gain nothing
        __builtin_amdgcn_sched_barrier(0);
        if (r > 0) {
            // slide the window one step back: the new oldest row is r - 4
#pragma unroll
            for (int e = 0; e < E; ++e) {
                xw[3][e] = xw[2][e];
                xw[2][e] = xw[1][e];
                xw[1][e] = xw[0][e];
            }
            unpack_lane<DT>(r - 4 >= 0 ? X[r - 4 >= 0 ? r - 4 : 0] : H[r - 1 < 3 ? r - 1 : 0], xw[0]);
        }
    }
}

// STATES: the call has an initial state or the gradient of a captured final state.  Its own instances: as
// run-time branches of one kernel the three pieces of code cost every call 30 registers and 100 scalar spills
// (B 8, C 3456, L 1024 without states: 38 -> 41 us).
//
// SEQ: the call carries sequence indices of packed rows (seq_idx; no states then).  They are staged in LDS like the
// mask.  A slab whose reach (three rows before it to three after) lies in one sequence, which is nearly every slab
// of rows packed from documents of hundreds of tokens, takes the ordinary sweep after one ballot; only a slab with a
// boundary in reach takes the sweep that gates each tap.  The walk kernel, which gates every row and reads two bytes
// per lane, took 192 us at B 2, C 3456, L 8192, bf16, SiLU, this one 74 (profiled; the whole training call 233 us with it, 118 now).
//
// ANY: a channel count, a row pitch or an address off the 8-byte grid.  A lane's channels are independent of every other
// lane's: each takes its two at their elements' alignment through a pointer of its own, the last of an odd count the row's
// last two (the first of which the lane before computes as well, to the same bits).  Such calls took the walk kernel, us
// with the reduction, bf16: B 8, C 961, L 1021 29.6 -> 20.9, with SiLU and a mask 41.9 -> 23.2; B 24, C 1695, L 170 with both
// 33.5 -> 22.0; B 8, C 3455, L 1024 79.1 -> 61.5 (on the grid 36.6: a misaligned four-byte access touches two words).
template <int DT, int W, bool MASK, bool ACT, bool STATES, bool SEQ = false, bool ANY = false>
__global__ __launch_bounds__(256, ACT ? 4 : 1) void canon_bwd_blc_kernel(const BwdArgs a)
{
    static_assert(!(STATES && SEQ), "seq_idx excludes states");
    static_assert(!ANY || !(STATES || SEQ), "neither packed nor with states");
    constexpr int BY = Elem<DT>::bytes;
    constexpr int E = kBwdLaneChannels, VB = E * BY;
    constexpr int R = kBwdSlab, NW = kBwdWaves;
    // which instances take whole slabs through a sweep without branches, and request their first tile ahead of the staged
    // mask and indices (both below): the others hold 82-95 registers and lose a wave per SIMD, or time, to it (ANY with a mask
    // and SiLU, B 8, C 961, L 1021: 24.1 us with its first tile ahead of the mask, 23.3 behind it).
    // kTight: fp16 with SiLU at widths 3 and 4.  Its conversions keep more values alive: with both it spilled 20 registers,
    // 49 with a mask, 62-67 packed, at the 128 that four waves leave it.  With the residual's branch in the sweep's rows
    // (which is what ends each row's live values) and the first tile behind the mask it holds 98-121; us a call before both /
    // with both as they are elsewhere / so: B 8, C 640, L 1024 15.3 / 20.6 / 13.8, with a mask 17.3 / 29.8 / 15.0; B 8, C 3456
    // 41.3 / 73.8 / 40.1, with a mask 44.9 / 118 / 42.4; B 32 134 / 252 / 131, with a mask 145 / 439 / 140; packed B 2,
    // C 3456, L 8192 75 / 161 / 72.3, with a mask 83.5 / 165 / 77.0.  (Ordinary sweeps instead: 43.1 at B 8, masked.)
    // Packed rows with a mask keep the branch in every type: bf16 held 128 and spilled one, now 109: 78.0 -> 77.2 (81.9 before
    // the straight sweep).
    constexpr bool kTight = ACT && !ANY && W > 2 && DT == CANON_DTYPE_F16;
    constexpr bool kStraight = !STATES && (ACT || !(MASK || SEQ));
    constexpr bool kAllAtOnce = !(ANY && MASK) && !kTight && (ACT || !(MASK || SEQ));
    constexpr bool kResBranch = kTight || (SEQ && MASK);
    // With an activation: tailx / headdz, two barriers per tile (dz of a slab's head needs the previous
    // wave's tail first).  Without one dz IS dout, so the head is handed over as raw rows (headg) together
    // with the tail, one barrier per tile, both double-buffered (a fast wave publishes the next tile while
    // a slow one still reads this one).
    // The sums that leave the block after its last tile lie in the same memory: 44 -> 29 KB of LDS with a mask, which
    // lets the register count, not LDS, decide how many blocks a CU holds.
    struct Exchange {
        BwdVec<DT> tailx[ACT ? 1 : 2][NW][3][64];            // last three xm rows of each wave's slab (storage bits)
        float headdz[ACT ? NW : 1][3][ACT ? E : 1][64];  // dz of the first three steps of each wave's slab
        BwdVec<DT> headg[ACT ? 1 : 2][ACT ? 1 : NW][3][64];  // ACT == false: the first three dout rows of each slab
    };
    union Shared {
        Exchange x;
        float red[NW - 1][5 * E][64];                 // dweight / dbias sums of waves 1..3
        // Four blocks a CU instead of the five their registers allow: unmasked launches without an activation, B 8 / 16 / 32,
        // C 3456, L 1024, bf16: 36.2 / 64.0 / 120.5 -> 35.4 / 63.3 / 119.7 us a call (three: 38.5 / 64.6 / 122; with a mask
        // four are 0.4 % slower).  The other instances it holds for, five -> four, B 8 and B 32: fp16 36.5 and 121.0 -> 36.5
        // and 119.9; width 3 36.3 and 121.8 -> 36.6 and 119.9, width 2 36.2 and 123.6 -> 35.9 and 120.3 (fp16 alike); fp32 of
        // widths 2 and 3, B 16 119.3 -> 118.5 (width 4 has four by its registers); off the grid, C 3455 60.9 and 232 -> 61.5
        // and 230; C 640 and 960 within 0.3 % throughout.
        char room[!ACT && !MASK && !SEQ && !STATES ? 33 * 1024 : 16];
    };
    __shared__ Shared shared;
    auto &tailx = shared.x.tailx;
    auto &headdz = shared.x.headdz;
    auto &headg = shared.x.headg;
    auto &red = shared.red;
    // mask entries of steps t_chunk-3 .. t_chunk+chunk+2 as floats.  Staged once per block: inside the
    // time loop (after the first store to dx) the compiler can no longer use scalar loads for them, and
    // as vector loads in the tile's load group they cost 20 % of the kernel.
    __shared__ float smask[MASK ? kBwdMaxChunk + 6 : 1];
    __shared__ int32_t sseq[SEQ ? kBwdMaxChunk + 6 : 1];   // sequence indices of the same steps

    // blockIdx = (b * nchunk + ch) * nct + ct : channel tile fastest, i.e. memory order
    const uint32_t bc = fdiv(blockIdx.x, a.div_nct);
    const uint32_t ct = blockIdx.x - bc * a.nct;
    const uint32_t b = fdiv(bc, a.div_nchunk);
    const uint32_t ch = bc - b * a.nchunk;
    const int lane = threadIdx.x & 63;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t cv = ct * 64u + lane;
    const bool active = cv < a.nvec;
    // idle lanes shadow the last group: loads need no predicate
    const uint32_t c0 = ANY ? (cv < a.nvec - 1u ? cv * E : a.C - E) : (active ? cv : a.nvec - 1u) * E;

    // The wave's rows are reached through buffer resources, one per tensor and tile: the lane is a 32-bit vector offset,
    // the row a scalar one.  (As 64-bit pointers per lane the nineteen row addresses of a tile alone held 38 registers.)
    // Lanes without channels are out of every resource's range: they load zeros and store nothing.
    using IO = BufIO<VB>;
    const uint32_t cv0 = ct * 64u, nl = a.nvec - cv0 < 64u ? a.nvec - cv0 : 64u;
    const uint32_t voff = active ? (uint32_t)lane * VB : 0x80000000u;
    const char *xb0 = a.x + ((int64_t)b * a.x_sb + (int64_t)cv0 * E) * BY;
    const char *gb0 = a.dy + ((int64_t)b * a.g_sb + (int64_t)cv0 * E) * BY;
    char *db0 = a.dx + ((int64_t)b * a.d_sb + (int64_t)cv0 * E) * BY;
    const char *xb = a.x + ((int64_t)b * a.x_sb + c0) * BY;      // this lane's, for the rows past the chunk
    const char *gb = a.dy + ((int64_t)b * a.g_sb + c0) * BY;
    const int64_t xs = a.x_sl * BY, gs = a.g_sl * BY, ds = a.d_sl * BY;
    const uint32_t xs32 = (uint32_t)xs, gs32 = (uint32_t)gs, ds32 = (uint32_t)ds;
    const int64_t Lm1 = (int64_t)a.L - 1;
    const int64_t t_chunk = (int64_t)ch * a.chunk;
    const int ntiles = (int)(a.chunk / (uint32_t)(R * NW));

    // a row of x or dout at this lane's channels
    auto load_row = [](const char *p) {
        if constexpr (ANY) return load_any<VB, false>(p);
        else return BwdIO<DT>::template load<false>(p);
    };
    auto rows_from = [&](int64_t t0) {      // steps of the slab at t0 that exist (wave uniform)
        const int64_t left = (int64_t)a.L - t0;
        return left >= R ? R : (left > 0 ? (int)left : 0);
    };
    // All rows of x and dout of a tile's slab and, for the first wave, the three rows of x before it.  (Requesting the next
    // tile's rows while this one is worked on was measured three times (before, and after, this tile's rows are waited for;
    // with two register sets taken in turn and wait counts that leave the next tile's loads in flight): 3-5 % slower, 40-60
    // more registers.)  The x resource starts three rows before the slab; a row past the end of the sequence is the slab's last
    // row again, loaded and never used, and a slab without rows has resources without a range.
    BwdVec<DT> X[R], G[R], H[3];
    auto request = [&](int it) {
        const int64_t t0 = t_chunk + ((int64_t)it * NW + wv) * R;
        const int rows = rows_from(t0);
        const uint32_t xrec = rows == 0 ? 0u : (uint32_t)(R + 2) * xs32 + nl * VB;
        const uint32_t grec = rows == 0 ? 0u : (uint32_t)(R - 1) * gs32 + nl * VB;
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(xb0 + (t0 - 3) * xs), 0, (int)xrec, kBufFlags);
        const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void *)(gb0 + t0 * gs), 0, (int)grec, kBufFlags);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t rr = r < rows ? (uint32_t)r : (rows > 0 ? (uint32_t)(rows - 1) : 0u);
            if constexpr (ANY) {
                const int64_t t = rows > 0 ? t0 + rr : Lm1;      // (a slab without rows: the sequence's last row, never used)
                X[r] = load_any<VB, true>(xb + t * xs);
                G[r] = load_any<VB, true>(gb + t * gs);
            } else {
                X[r] = IO::template load<kAuxStream>(rx, voff, (rr + 3u) * xs32);
                G[r] = IO::template load<kAuxStream>(rg, voff, rr * gs32);
            }
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) H[j] = BwdIO<DT>::zero();
        if (wv == 0 && t0 > 0) {     // (t0 is a multiple of the tile: all three rows exist)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if constexpr (ANY) H[j] = load_any<VB, false>(xb + ((t0 <= Lm1 ? t0 : Lm1 + 1) - 3 + j) * xs);
                else H[j] = IO::template load<kAuxPlain>(rx, voff, (uint32_t)j * xs32);
            }
        }
    };

    // Everything the block reads before its second tile is requested here, before the first wait: taps, the rows just past
    // the chunk (last wave), the first tile, the staged mask and indices.  One after the other, each behind the barrier or
    // the wait of the one before, they were three memory round trips: B 8, C 640, L 1024, bf16 12.6 -> 12.2 us a call,
    // B 8, C 3456 with SiLU 39.6 -> 38.5; with a mask and no activation 24.0 -> 24.25 (B 16, C 960), so not there.
    RawTaps<E> rawt;
    fetch_taps<W, E, ANY>(a.weight, a.bias, a.w_sc, a.w_sk, a.w_dtype, a.w_vec != 0, c0, rawt);
    const int64_t te = t_chunk + (int64_t)a.chunk;   // first step after the chunk (at least 32)
    BwdVec<DT> XE[ACT ? 6 : 1], GE[3];               // rows te-3 .. te+2 of x (with an activation), te .. te+2 of dout
#pragma unroll
    for (int j = 0; j < (ACT ? 6 : 1); ++j) XE[j] = BwdIO<DT>::zero();
#pragma unroll
    for (int j = 0; j < 3; ++j) GE[j] = BwdIO<DT>::zero();
    if (wv == NW - 1 && te <= Lm1) {
        if constexpr (ACT) {
#pragma unroll
            for (int j = 0; j < 6; ++j) XE[j] = load_row(xb + (te - 3 + j < Lm1 ? te - 3 + j : Lm1) * xs);
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) GE[j] = load_row(gb + (te + j < Lm1 ? te + j : Lm1) * gs);
    }
    if constexpr (kAllAtOnce) request(ntiles - 1);
    if constexpr (MASK || SEQ) {
        for (uint32_t i = threadIdx.x; i < a.chunk + 6u; i += 64u * NW) {
            int64_t t = t_chunk - 3 + (int64_t)i;
            t = t < 0 ? 0 : (t > Lm1 ? Lm1 : t);
            if constexpr (MASK) smask[i] = load_mask(a.mask, (int64_t)b * a.m_sb + t * a.m_sl, a.mask_dtype);
            if constexpr (SEQ) sseq[i] = a.seq[(int64_t)b * a.q_sb + t * a.q_sl];
        }
        __syncthreads();
    }
    if constexpr (!kAllAtOnce) request(ntiles - 1);

    // The tiles are walked from the last to the first, so the dz of the three steps after a tile
    // are the head of the tile done just before (still in headdz[0]).  For the chunk's last tile
    // the last wave computes them here, from six rows of x and three of dout, and leaves them
    // in that slot itself.
    float dzf[3][E];   // dzf[j] = dz[t + 1 + j] for the step t being processed
    float w[E][W], bias[E];
    decode_taps<DT, W, E>(rawt, a.w_dtype, a.w_vec != 0, a.bias != nullptr, w, bias);
    if constexpr (!ACT) {
        // no activation: the three dz after the chunk are three rows of dout, kept by the last wave
#pragma unroll
        for (int j = 0; j < 3; ++j) unpack_lane<DT>(te + j <= Lm1 ? GE[j] : BwdIO<DT>::zero(), dzf[j]);
    } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) dzf[j][e] = 0.0f;
        if (wv == NW - 1) {
            float xt[6][E];
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const uint32_t m = MASK ? f_bits(smask[a.chunk + j]) : kMaskOne;   // steps te-3 .. te+2
                unpack_lane<DT>(bwd_mask_row<DT, MASK>(XE[j], m, te - 3 + j <= Lm1), xt[j]);
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                float g[E], d[E];
                unpack_lane<DT>(GE[j], g);
                if constexpr (SEQ) {
                    const int32_t *q = sseq + a.chunk;      // steps te-3 .. te+2
                    bwd_dz_gated<W, E, ACT>(w, bias, xt[j], xt[j + 1], xt[j + 2], xt[j + 3], q[j] == q[j + 3],
                                            q[j + 1] == q[j + 3], q[j + 2] == q[j + 3], g, d);
                } else {
                    bwd_dz<W, E, ACT>(w, bias, xt[j], xt[j + 1], xt[j + 2], xt[j + 3], g, d);
                }
                const bool inside = te + j <= Lm1;
#pragma unroll
                for (int e = 0; e < E; ++e) headdz[0][j][e][lane] = inside ? d[e] : 0.0f;
            }
        }
    }

    float dw[E][W], dbs[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        dbs[e] = 0.0f;
#pragma unroll
        for (int k = 0; k < W; ++k) dw[e][k] = 0.0f;
    }

    for (int it = ntiles - 1; it >= 0; --it) {
        const int64_t t0 = t_chunk + ((int64_t)it * NW + wv) * R;
        const int rows = rows_from(t0);
        const uint32_t drec = rows == 0 ? 0u : (uint32_t)(R - 1) * ds32 + nl * VB;
        const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void *)(db0 + t0 * ds), 0, (int)drec, kBufFlags);
        if (it != ntiles - 1) request(it);
        bool plain_mask = true;   // every row of the slab and the three before it are valid tokens: x * 1 is x
        uint32_t mm[R + 3];   // mask of steps t0-3 .. t0+R-1 (bits, in scalar registers: one LDS read, then lane by lane)
#pragma unroll
        for (int j = 0; j < R + 3; ++j) mm[j] = kMaskOne;
        if constexpr (MASK) {
            const uint32_t first = ((uint32_t)it * NW + wv) * R;   // index of step t0 - 3 in smask
            const uint32_t m_lane = f_bits(smask[first + (uint32_t)(lane < R + 2 ? lane : R + 2)]);
            // (kTight with states, at its 128 registers, looks at every row of the slab by itself: one spilled with this flag)
            plain_mask = !(STATES && kTight) && __builtin_amdgcn_ballot_w64(m_lane != kMaskOne) == 0;
#pragma unroll
            for (int j = 0; j < R + 3; ++j) mm[j] = (uint32_t)__builtin_amdgcn_readlane((int)m_lane, j);
        }
        // SEQ: indices of steps t0-3 .. t0+R+2, one per lane, and whether they are all the same
        int32_t q_lane = 0;
        bool one_seq = true;
        if constexpr (SEQ) {
            q_lane = sseq[((uint32_t)it * NW + wv) * R + (uint32_t)(lane < R + 6 ? lane : R + 5)];
            one_seq = __builtin_amdgcn_ballot_w64(q_lane != __builtin_amdgcn_readfirstlane(q_lane)) == 0;
        }

        // dz of the three steps after the slab; the last wave's are the previous iteration's head of wave 0
        const int pb = it & 1;   // ACT == false: LDS buffer of this tile
        if constexpr (ACT) {
            if (wv == NW - 1) {
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int e = 0; e < E; ++e) dzf[j][e] = headdz[0][j][e][lane];
            }
        } else {
            if (wv == NW - 1 && it != ntiles - 1) {   // (the chunk's last tile: the rows loaded before the loop)
#pragma unroll
                for (int j = 0; j < 3; ++j) unpack_lane<DT>(headg[pb ^ 1][0][j][lane], dzf[j]);
            }
        }

        // ---- rows become xm (masked, zero where they do not exist), once ----------------
        if (!plain_mask || rows < R) {
#pragma unroll
            for (int r = 0; r < R; ++r) X[r] = bwd_mask_row<DT, MASK>(X[r], mm[3 + r], r < rows);
        }
        if constexpr (MASK) {
            if (wv == 0 && !plain_mask) {
#pragma unroll
                for (int j = 0; j < 3; ++j) H[j] = bwd_mask_row<DT, MASK>(H[j], mm[j], true);   // zero already when t < 0
            }
        }
        if (STATES && a.init && t0 == 0 && wv == 0) {
            // rows before t = 0: entries of the initial state, not masked
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int s_ = a.S_in - 3 + j;
                if (s_ < 0) continue;
                float f[E];
#pragma unroll
                for (int e = 0; e < E; ++e)
                    f[e] = load1<DT>(a.init, (int64_t)b * a.i_sb + (int64_t)(c0 + e) * a.i_sc + (int64_t)s_ * a.i_ss);
                H[j] = pack_lane<DT>(f);
            }
        }
        if constexpr (!ACT) {
            // tail of x and head of dout (zero past the end of the sequence) in one exchange
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                tailx[pb][wv][j][lane] = X[R - 3 + j];
                headg[pb][wv][j][lane] = j < rows ? G[j] : BwdIO<DT>::zero();
            }
            __syncthreads();
            if (wv > 0) {
#pragma unroll
                for (int j = 0; j < 3; ++j) H[j] = tailx[pb][wv - 1][j][lane];
            }
            if (wv < NW - 1) {
#pragma unroll
                for (int j = 0; j < 3; ++j) unpack_lane<DT>(headg[pb][wv + 1][j][lane], dzf[j]);
            }
        }
        float dzh[3][E];
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) dzh[j][e] = 0.0f;   // (unused without an activation)
        if constexpr (ACT) {
#pragma unroll
            for (int j = 0; j < 3; ++j) tailx[0][wv][j][lane] = X[R - 3 + j];
            __syncthreads();
            if (wv > 0) {
#pragma unroll
                for (int j = 0; j < 3; ++j) H[j] = tailx[0][wv - 1][j][lane];
            }

            // ---- dz of the slab's first three steps, handed to the previous wave ---------
            {
                float xq[6][E];   // xm of rows -3 .. 2
#pragma unroll
                for (int k = 0; k < 3; ++k) unpack_lane<DT>(H[k], xq[k]);
#pragma unroll
                for (int k = 0; k < 3; ++k) unpack_lane<DT>(X[k], xq[3 + k]);
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    float g[E];
                    unpack_lane<DT>(G[j], g);
                    if (SEQ && !one_seq) {
                        const int32_t own = __builtin_amdgcn_readlane(q_lane, j + 3);
                        bwd_dz_gated<W, E, ACT>(w, bias, xq[j], xq[j + 1], xq[j + 2], xq[j + 3],
                                                __builtin_amdgcn_readlane(q_lane, j) == own,
                                                __builtin_amdgcn_readlane(q_lane, j + 1) == own,
                                                __builtin_amdgcn_readlane(q_lane, j + 2) == own, g, dzh[j]);
                    } else {
                        bwd_dz<W, E, ACT>(w, bias, xq[j], xq[j + 1], xq[j + 2], xq[j + 3], g, dzh[j]);
                    }
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        dzh[j][e] = j < rows ? dzh[j][e] : 0.0f;
                        headdz[wv][j][e][lane] = dzh[j][e];
                    }
                }
            }
            __syncthreads();
            if (wv < NW - 1) {
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int e = 0; e < E; ++e) dzf[j][e] = headdz[wv + 1][j][e][lane];
            }
        }

        // ---- sweep the slab from its last step to its first --------------------------
        const int64_t fin_first = (int64_t)a.L - a.S_out;   // first captured step (S_out is 0 without dfinal_state)
        if (STATES && a.dfin && t0 + rows > fin_first) {
            // slot 0 of the final state's gradient holds step fin_first
            const char *fin = a.dfin + ((int64_t)b * a.k_sb + (int64_t)c0 * a.k_sc) * BY;
            bwd_sweep<DT, W, MASK, ACT, false, true, R, E>(a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff, ds32, rows,
                                                           fin, fin_first - t0);
        } else if (SEQ && !one_seq) {
            int32_t q[R + 6];
#pragma unroll
            for (int j = 0; j < R + 6; ++j) q[j] = __builtin_amdgcn_readlane(q_lane, j);
            bwd_sweep<DT, W, MASK, ACT, false, false, R, E, SEQ>(a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff, ds32, rows,
                                                                 nullptr, 0, q);
        } else {
            char *dany = ANY && active ? a.dx + ((int64_t)b * a.d_sb + c0) * BY + t0 * ds : nullptr;
            // Whole slabs of valid tokens, which most are, take a sweep without a branch in it: with the residual's and the
            // mask's branches in every row, each a break in the instruction stream, the launches with SiLU were bound by the
            // sweep.  us a call, both changes: C 3456, L 1024, bf16, SiLU B 8 39.5 -> 38.1, with a mask B 32 138.2 -> 133.3;
            // packed rows with SiLU B 2, L 8192 72.5 -> 69.6, B 1, L 4000 25.7 -> 24.2; fp32 B 24, C 2848, L 385 70.6 -> 66.9;
            // (up to 128 registers with SiLU, four waves per SIMD; held to 96 and five it spills: 43-198 us in place of 38-134)
            if (kStraight && rows == R && plain_mask) {
                if (!kResBranch && a.res_mode != CANON_RESIDUAL_NONE)
                    bwd_sweep<DT, W, false, ACT, true, false, R, E, false, ANY, 1>(a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff,
                                                                                   ds32, rows, nullptr, 0, nullptr, dany);
                else
                    bwd_sweep<DT, W, false, ACT, true, false, R, E, false, ANY, kResBranch ? -1 : 0>(
                        a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff, ds32, rows, nullptr, 0, nullptr, dany);
            } else if (rows == R) {
                bwd_sweep<DT, W, MASK, ACT, true, false, R, E, false, ANY>(a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff, ds32,
                                                                           rows, nullptr, 0, nullptr, dany);
            } else {
                bwd_sweep<DT, W, MASK, ACT, false, false, R, E, false, ANY>(a, w, bias, X, H, G, mm, dzh, dzf, dw, dbs, rd, voff, ds32,
                                                                            rows, nullptr, 0, nullptr, dany);
            }
        }
    }

    if (STATES && a.dinit && ch == 0 && wv == 0 && active) {
        // here dzf[i] = dz[i] (zero past the end of the row).  Entry s is the input at t = s - S_in = -d:
        // its gradient is sum_i w[W-1-d-i] * dz[i] over the taps that exist
        for (int s_ = 0; s_ < a.S_in; ++s_) {
            const int d = a.S_in - s_;
            // a final state longer than the row also captured this entry (input at t = -d) in slot S_out - L - d
            const int64_t slot = (int64_t)a.S_out - (int64_t)a.L - d;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                float acc = 0.0f;
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int k = W - 1 - d - i;
                    if (k >= 0) acc = fmaf(w[e][k < 0 ? 0 : k], dzf[i][e], acc);
                }
                if (a.dfin && slot >= 0)
                    acc += load1<DT>(a.dfin, (int64_t)b * a.k_sb + (int64_t)(c0 + e) * a.k_sc + slot * a.k_ss);
                store1<DT>(a.dinit, (int64_t)b * a.j_sb + (int64_t)(c0 + e) * a.j_sc + (int64_t)s_ * a.j_ss, acc);
            }
        }
    }

    // ---- the four waves' sums, added in the order 0, 1, 2, 3 -----------------------------
    __syncthreads();   // (every wave has read its neighbours' rows of the last tile)
    if (wv > 0) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int k = 0; k < W; ++k) red[wv - 1][e * 5 + k][lane] = dw[e][k];
            red[wv - 1][e * 5 + 4][lane] = dbs[e];
        }
    }
    __syncthreads();
    if (wv == 0 && active) {
        float *pp = a.partial + (((int64_t)b * a.nchunk + ch) * a.C + c0) * 5;
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float v = 0.0f;
                if (k < W) {
                    v = dw[e][k < W ? k : 0];
#pragma unroll
                    for (int q = 0; q < NW - 1; ++q) v += red[q][e * 5 + k][lane];
                }
                pp[e * 5 + k] = v;
            }
            float v = dbs[e];
#pragma unroll
            for (int q = 0; q < NW - 1; ++q) v += red[q][e * 5 + 4][lane];
            pp[e * 5 + 4] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// backward, time-contiguous rows ([B, C, L]): one wave owns one segment of one
// (b, c) row, U vectors of E time steps per lane, exactly as the forward
// kernel.  Pass 1 recomputes z and dz = dout * act'(z) for the lane's own
// steps (history from lane l-1 by wave shift) and accumulates the lane's share
// of dweight / dbias; pass 2 forms dx[t] = sum_k w[k] * dz[t+(W-1)-k] with the
// three later dz values taken from lane l+1 (wave shift the other way), from
// the next vector's lane 0, or -- for the last lane of a segment that is not
// the end of the row -- recomputed from memory.  The wave's dweight / dbias
// are reduced across lanes in a fixed butterfly order and written as one
// partial set entry; canon_bwd_reduce_kernel sums the sets.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_shift_down(float v, float last)
{
    // lane i <- lane i+1 across the whole wave; lane 63 <- `last`
    return bits_f((uint32_t)__builtin_amdgcn_update_dpp((int)f_bits(last), (int)f_bits(v),
                                                        0x130 /* wave_shl:1 */, 0xF, 0xF, false));
}

__device__ __forceinline__ float read_lane0(float v)
{
    return bits_f((uint32_t)__builtin_amdgcn_readfirstlane((int)f_bits(v)));
}

__device__ __forceinline__ float wave_sum(float v)
{
    // fixed-order butterfly: every lane ends with the same total
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The scalars in front of the argument block are what a wave needs to request its rows of x and dout; they arrive in
// registers with the wave (kernel-argument preload), so the loads are issued without a read of the argument block in
// front of them, as in the forward kernel.  g_sb / g_sc: the strides of dout when they differ from x's, else a copy
// of x's; `divC_s`: s1 | s2 << 1 of the division by C.
// RAGGED: rows of any length from E and any alignment, as in the forward kernel (`len` is then the length in elements
// and the strides are in elements, else both are in vectors).  Such rows took the walk kernel, whose lanes lie a row
// apart: B 8, C 960, L 1021, bf16 162 -> 12.0 us, as fast as whole vectors (L 1024: 12.5 us with a mask).
template <int DT, int W, int U, bool MASK, bool RAGGED>
__global__ __launch_bounds__(256) void canon_bwd_bcl_kernel(const char *x_base, const char *g_base, uint32_t x_sb32,
                                                            uint32_t x_sc32, uint32_t g_sb32, uint32_t g_sc32,
                                                            uint32_t nthreads, uint32_t nchunk, uint32_t C, uint32_t divC_m,
                                                            uint32_t divC_s, uint32_t len, const BwdArgs a)
{
    constexpr int E = Elem<DT>::per_vec;
    constexpr int BY = Elem<DT>::bytes;
    const int lane = threadIdx.x & 63;
    const uint32_t task = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
    if (task >= nthreads) return;            // nthreads = wave tasks in this kernel
    uint32_t row = task, seg = 0;
    if (nchunk > 1) {                        // nchunk = segments per row
        row = fdiv(task, a.div_nchunk);
        seg = task - row * nchunk;
    }
    const uint32_t b = fdiv(row, FastDiv{C, divC_m, divC_s & 1u, divC_s >> 1});
    const uint32_t c = row - b * C;

    constexpr int UNIT = RAGGED ? BY : 16;   // bytes the strides count in
    const char *xrow = x_base + ((int64_t)b * x_sb32 + (int64_t)c * x_sc32) * UNIT;
    const char *grow = g_base + ((int64_t)b * g_sb32 + (int64_t)c * g_sc32) * UNIT;
    const uint32_t nvec = len;
    char *drow = a.dx + ((int64_t)b * a.d_sb + (int64_t)c * a.d_sc) * BY;
    const uint32_t v0 = seg * (64u * U) + lane;

    uint4 X[U], G[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t v = v0 + u * 64u;
        if constexpr (RAGGED) {
            const int64_t off = (int64_t)row_clamp<E>(v * E, len) * BY;
            X[u] = load_vec_any<kBwdStream>(xrow + off);
            G[u] = load_vec_any<kBwdStream>(grow + off);
        } else {
            const uint32_t vc = v < nvec ? v : nvec - 1u;
            X[u] = load_vec<kBwdStream>(xrow + (int64_t)vc * 16);
            G[u] = load_vec<kBwdStream>(grow + (int64_t)vc * 16);
        }
    }
    RawTaps<1> raw;
    fetch_taps_uniform<W>(a.weight, a.bias, a.w_sc, a.w_sk, a.w_dtype, a.w_vec != 0, a.b_pair != 0, c, raw);
    float M[MASK ? U : 1][E];
    if constexpr (MASK) {
        int64_t mbase[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t v = v0 + u * 64u;
            const uint32_t first = RAGGED ? row_clamp<E>(v * E, len) : (v < nvec ? v : nvec - 1u) * E;
            mbase[u] = b * a.m_sb + (int64_t)first * a.m_sl;
        }
        load_mask_vec<E, U>(a.mask, mbase, a.m_sl, a.mask_dtype, a.m_vec != 0, M);
    }
    if constexpr (RAGGED) {
        // the wave that holds the end of the row undoes the move of its last vectors (zeros past the end)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t gap = row_gap<E>((v0 + u * 64u) * E, len);
            if (__builtin_amdgcn_ballot_w64(gap != 0) != 0) {
                X[u] = shift_down<DT>(X[u], gap);
                G[u] = shift_down<DT>(G[u], gap);
                if constexpr (MASK) shift_down<E>(M[u], gap);
            }
        }
    }
    float w[1][W], bvv[1];
    decode_taps<DT, W, 1>(raw, a.w_dtype, a.w_vec != 0, a.bias != nullptr, w, bvv);
    const float bv = bvv[0];

    // left history of the segment's first vector (lane 0 only), right dz of its last vector (lane 63 only)
    float carry[3] = {0.0f, 0.0f, 0.0f};
    float edge[3] = {0.0f, 0.0f, 0.0f};
    const int64_t t_seg0 = (int64_t)seg * (64 * U) * E;
    const int64_t t_seg1 = t_seg0 + (int64_t)(64 * U) * E;      // first step after the segment
    if (lane == 0 && seg > 0) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            float v = load1<DT>(xrow, t_seg0 - 3 + j);
            if constexpr (MASK) v = mul_round<DT>(v, load_mask(a.mask, b * a.m_sb + (t_seg0 - 3 + j) * a.m_sl, a.mask_dtype));
            carry[j] = v;
        }
    }
    if (lane == 63 && t_seg1 < (int64_t)a.L) {
        // dz[t_seg1 + j], j = 0..2, from x[t_seg1-3 .. t_seg1+2] and dout[t_seg1 .. t_seg1+2]
        float xs6[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int64_t t = t_seg1 - 3 + i;
            float v = 0.0f;
            if (t < (int64_t)a.L) {
                v = load1<DT>(xrow, t);
                if constexpr (MASK) v = mul_round<DT>(v, load_mask(a.mask, b * a.m_sb + t * a.m_sl, a.mask_dtype));
            }
            xs6[i] = v;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int64_t t = t_seg1 + j;
            if (t < (int64_t)a.L) {
                float z = bv;
#pragma unroll
                for (int k = 0; k < W; ++k) z = fmaf(w[0][k], xs6[j + (4 - W) + k], z);
                const float g = load1<DT>(grow, t);
                edge[j] = a.act ? g * silu_grad(z) : g;
            }
        }
    }

    // pass 1: dz of the lane's own steps, and its share of dweight / dbias
    float dz[U][E], gg[U][E];
    float dwl[W], dbl = 0.0f;
#pragma unroll
    for (int k = 0; k < W; ++k) dwl[k] = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t first = (v0 + u * 64u) * E;
        const bool valid = RAGGED ? first + E <= len : v0 + u * 64u < nvec;   // the whole vector
        float xr[E], xm_store[MASK ? E : 1];
        float *xm = MASK ? xm_store : xr;
        unpack_vec<DT>(X[u], xr);
        unpack_vec<DT>(G[u], gg[u]);
        if constexpr (MASK) {
#pragma unroll
            for (int j = 0; j < E; ++j) xm[j] = mul_round<DT>(xr[j], M[u][j]);
        }
        float seq[E + 3];
        seq[0] = wave_shift_up(xm[E - 3], carry[0]);
        seq[1] = wave_shift_up(xm[E - 2], carry[1]);
        seq[2] = wave_shift_up(xm[E - 1], carry[2]);
        if (u + 1 < U) {
            carry[0] = read_lane63(xm[E - 3]);
            carry[1] = read_lane63(xm[E - 2]);
            carry[2] = read_lane63(xm[E - 1]);
        }
#pragma unroll
        for (int j = 0; j < E; ++j) seq[3 + j] = xm[j];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            float z = bv;
#pragma unroll
            for (int k = 0; k < W; ++k) z = fmaf(w[0][k], seq[j + (4 - W) + k], z);
            dz[u][j] = z;
        }
        if (a.act) {
#pragma unroll
            for (int j = 0; j < E; ++j) dz[u][j] = gg[u][j] * silu_grad(dz[u][j]);
        } else {
#pragma unroll
            for (int j = 0; j < E; ++j) dz[u][j] = gg[u][j];
        }
        if (!valid) {
#pragma unroll
            for (int j = 0; j < E; ++j) dz[u][j] = RAGGED && first + j < len ? dz[u][j] : 0.0f;
        }
        // Steps past the end of the row have a dz of zero, but their window reaches back over the row's last inputs, and
        // 0 * Inf is NaN: their window is zero as well.  Whole vectors: selects for every lane (no time measured; a branch
        // around the sums costs up to 5 % at B 8, C 1000, L 1536 with a mask).  Ragged rows, whose last vector has steps
        // on both sides of the end: the selects, one per step and tap, only in the wave that holds the end (B 8, C 960,
        // L 1021 13.5 -> 13.9 us, with SiLU 15.5 -> 15.0, for every lane 16.5; B 32, L 500, where every wave holds one,
        // 21.0 -> 21.5, with SiLU 24.0 -> 25.5).
        if (RAGGED && __builtin_amdgcn_ballot_w64(!valid) == 0) {
#pragma unroll
            for (int j = 0; j < E; ++j)
#pragma unroll
                for (int k = 0; k < W; ++k) dwl[k] = fmaf(dz[u][j], seq[j + (4 - W) + k], dwl[k]);
        } else {
            float win[E + 3];
#pragma unroll
            for (int i = 0; i < E + 3; ++i) win[i] = RAGGED || valid ? seq[i] : 0.0f;
#pragma unroll
            for (int j = 0; j < E; ++j) {
                const bool inside = !RAGGED || first + j < len;
#pragma unroll
                for (int k = 0; k < W; ++k) dwl[k] = fmaf(dz[u][j], inside ? win[j + (4 - W) + k] : 0.0f, dwl[k]);
            }
        }
#pragma unroll
        for (int j = 0; j < E; ++j) dbl += dz[u][j];
    }

    // pass 2: dx
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t v = v0 + u * 64u;
        // the three dz values after this vector: lane l+1 of the same step, for lane 63 lane 0 of the next
        float nx[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float last = (u + 1 < U) ? read_lane0(dz[u + 1 < U ? u + 1 : u][j]) : edge[j];
            nx[j] = wave_shift_down(dz[u][j], last);
        }
        float dq[E + 3];
#pragma unroll
        for (int j = 0; j < E; ++j) dq[j] = dz[u][j];
        dq[E] = nx[0]; dq[E + 1] = nx[1]; dq[E + 2] = nx[2];
        float o[E];
#pragma unroll
        for (int j = 0; j < E; ++j) {
            float acc = w[0][W - 1] * dq[j];
#pragma unroll
            for (int k = W - 2; k >= 0; --k) acc = fmaf(w[0][k], dq[j + (W - 1) - k], acc);
            o[j] = acc;
        }
        if (a.res_mode == CANON_RESIDUAL_MASKED) {
#pragma unroll
            for (int j = 0; j < E; ++j) o[j] += gg[u][j];
        }
        if constexpr (MASK) {
#pragma unroll
            for (int j = 0; j < E; ++j) o[j] *= M[u][j];
        }
        if (a.res_mode == CANON_RESIDUAL_UNMASKED) {
#pragma unroll
            for (int j = 0; j < E; ++j) o[j] += gg[u][j];
        }
        if constexpr (RAGGED) store_row_vec<DT, kBwdStream>(drow, v * E, len, o);
        else if (v < nvec) store_vec<kBwdStream>(drow + (int64_t)v * 16, pack_vec<DT>(o));
    }

    // the wave's dweight / dbias -> partial[(b * nseg + seg) * C + c][5]
    float tot[5];
#pragma unroll
    for (int k = 0; k < 4; ++k) tot[k] = k < W ? wave_sum(dwl[k < W ? k : 0]) : 0.0f;
    tot[4] = wave_sum(dbl);
    if (lane == 0) {
        float *pp = a.partial + (((int64_t)b * a.nchunk + seg) * a.C + c) * 5;
#pragma unroll
        for (int k = 0; k < 5; ++k) pp[k] = tot[k];
    }
}

// Rows of at most 32 vectors, of any length from one vector on and any alignment: as in the forward kernel a row takes
// as many adjacent lanes of a wave as it has vectors, and a wave as many whole rows as fit.
// The three inputs before a lane's vector come from the lane before, the three dz after it from the lane behind, zero at
// the row's ends; a row's sums are added over its lanes in a fixed order and are its partial set entry.
// Leading scalars as in the kernel above (strides in elements); `packed`: vectors per row | gap << 6 | s1, s2 of the
// division by C << 9 | (2^16 / vectors per row, rounded up) << 15 (lane / vectors is a multiply and a shift).
//
// What bounds it is bandwidth once the lanes are full, and the launch.  Such rows took a wave each, most of whose lanes
// then hold nothing, or below 40 steps the walk kernel.  us per call with the reduction, bf16: B 31, C 2848, L 82 with a
// mask 54.4 -> 25.7; B 32, C 3456: L 13 (SiLU, mask) 14.6 -> 11.0, L 39 (SiLU) 48.8 -> 14.6, L 64 47.6 -> 14.8, L 128
// 41.0 -> 23.2, L 129 53.3 -> 31.5 (45.5 with rows in the next power of two of lanes), L 255 57 -> 44, L 256 43.5 -> 40.6
// (27.4 at the plain copy's rate).  A launch of a few rows is one wave's life, which is longer with two to four rows in it
// (B 3, C 96, L 209, SiLU, mask 6.35 -> 7.3): those of 16 vectors and more keep a wave each (few_rows in the planning).
template <int DT, int W, bool MASK>
__global__ __launch_bounds__(256) void canon_bwd_bcl_short_kernel(const char *x_base, const char *g_base, uint32_t x_sb32,
                                                                  uint32_t x_sc32, uint32_t g_sb32, uint32_t g_sc32,
                                                                  uint32_t nrows, uint32_t C, uint32_t divC_m, uint32_t packed,
                                                                  const BwdArgs a)
{
    constexpr int E = Elem<DT>::per_vec;
    constexpr int BY = Elem<DT>::bytes;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4u + (threadIdx.x >> 6));
    const uint32_t nvec = packed & 63u, m = packed >> 15;
    const uint32_t rows = (64u * m) >> 16;                       // rows per wave
    const uint32_t first_row = wave * rows;
    if (first_row >= nrows) return;
    const uint32_t wrow = (lane * m) >> 16;                      // row of the wave
    const uint32_t row = first_row + wrow;
    const bool active = wrow < rows && row < nrows;
    const uint32_t v = active ? lane - wrow * nvec : nvec - 1u;  // vector of the row; idle lanes shadow the end of
    const uint32_t rr = active ? row : first_row;                // the wave's first row: loads need no predicate
    const uint32_t gap = (packed >> 6) & 7u;                     // by how much the last vector's access moves back
    const uint32_t inside = E - gap;                             // its steps before the row's end
    const bool last = v == nvec - 1u;
    const uint32_t first = v * E - (last ? gap : 0u);            // first element of the lane's access
    const uint32_t b = fdiv(rr, FastDiv{C, divC_m, (packed >> 9) & 1u, (packed >> 10) & 31u});
    const uint32_t c = rr - b * C;
    const char *xrow = x_base + ((int64_t)b * x_sb32 + (int64_t)c * x_sc32) * BY;
    const char *grow = g_base + ((int64_t)b * g_sb32 + (int64_t)c * g_sc32) * BY;
    char *drow = a.dx + ((int64_t)b * a.d_sb + (int64_t)c * a.d_sc) * BY;

    uint4 X = load_vec_any<kBwdStream>(xrow + (int64_t)first * BY);
    uint4 G = load_vec_any<kBwdStream>(grow + (int64_t)first * BY);
    RawTaps<1> raw;
    fetch_taps<W, 1>(a.weight, a.bias, a.w_sc, a.w_sk, a.w_dtype, a.w_vec != 0, c, raw);
    float M[1][E];
    if constexpr (MASK) {
        const int64_t mbase[1] = {(int64_t)b * a.m_sb + (int64_t)first * a.m_sl};
        load_mask_vec<E, 1>(a.mask, mbase, a.m_sl, a.mask_dtype, a.m_vec != 0, M);
    }
    float w[1][W], bvv[1];
    decode_taps<DT, W, 1>(raw, a.w_dtype, a.w_vec != 0, a.bias != nullptr, w, bvv);
    const float bv = bvv[0];
    if (gap != 0) {
        X = shift_down<DT>(X, last ? gap : 0u);
        G = shift_down<DT>(G, last ? gap : 0u);
        if constexpr (MASK) {
#pragma unroll
            for (uint32_t n = 1; n < (uint32_t)E; n *= 2) {
                if (gap & n) {
#pragma unroll
                    for (int j = 0; j < E; ++j) M[0][j] = last ? (j + (int)n < E ? M[0][j + (int)n < E ? j + n : 0] : 0.0f) : M[0][j];
                }
            }
        }
    }

    float xr[E], g[E], xm_store[MASK ? E : 1];
    float *xm = MASK ? xm_store : xr;
    unpack_vec<DT>(X, xr);
    unpack_vec<DT>(G, g);
    if constexpr (MASK) {
#pragma unroll
        for (int j = 0; j < E; ++j) xm[j] = mul_round<DT>(xr[j], M[0][j]);
    }
    float seq[E + 3];
    seq[0] = wave_shift_up(xm[E - 3], 0.0f);
    seq[1] = wave_shift_up(xm[E - 2], 0.0f);
    seq[2] = wave_shift_up(xm[E - 1], 0.0f);
#pragma unroll
    for (int j = 0; j < 3; ++j) seq[j] = v == 0 ? 0.0f : seq[j];
#pragma unroll
    for (int j = 0; j < E; ++j) seq[3 + j] = xm[j];

    float dz[E + 3];
#pragma unroll
    for (int j = 0; j < E; ++j) dz[j] = g[j];
    if (a.act) {
#pragma unroll
        for (int j = 0; j < E; ++j) {
            float z = bv;
#pragma unroll
            for (int k = 0; k < W; ++k) z = fmaf(w[0][k], seq[j + (4 - W) + k], z);
            dz[j] = g[j] * silu_grad(z);
        }
    }
    // Steps past the row's end, the last vector's from `inside` on, have no dz, and no window (it reaches back over the
    // row's last inputs, and 0 * Inf is NaN): their terms are summed apart and left out in the lanes that hold the end.
    float dwl[W], past[W], dbl = 0.0f;
#pragma unroll
    for (int k = 0; k < W; ++k) dwl[k] = past[k] = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        if ((uint32_t)j < inside) {
#pragma unroll
            for (int k = 0; k < W; ++k) dwl[k] = fmaf(dz[j], seq[j + (4 - W) + k], dwl[k]);
        } else {
            dz[j] = last ? 0.0f : dz[j];
#pragma unroll
            for (int k = 0; k < W; ++k) past[k] = fmaf(dz[j], seq[j + (4 - W) + k], past[k]);
        }
        dbl += dz[j];
    }
    // dz of the three steps after the vector: the next lane's first, none behind the row's last vector
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float next = wave_shift_down(dz[j], 0.0f);
        dz[E + j] = last ? 0.0f : next;
    }
    float o[E];
#pragma unroll
    for (int j = 0; j < E; ++j) {
        float acc = w[0][W - 1] * dz[j];
#pragma unroll
        for (int k = W - 2; k >= 0; --k) acc = fmaf(w[0][k], dz[j + (W - 1) - k], acc);
        o[j] = acc;
    }
    if (a.res_mode == CANON_RESIDUAL_MASKED) {
#pragma unroll
        for (int j = 0; j < E; ++j) o[j] += g[j];
    }
    if constexpr (MASK) {
#pragma unroll
        for (int j = 0; j < E; ++j) o[j] *= M[0][j];
    }
    if (a.res_mode == CANON_RESIDUAL_UNMASKED) {
#pragma unroll
        for (int j = 0; j < E; ++j) o[j] += g[j];
    }
    uint4 out = pack_vec<DT>(o);
    if (gap != 0) out = row_end_vec<DT>(out, gap, last);
    if (active) store_vec_any<kBwdStream>(drow + (int64_t)first * BY, out);

    float tot[5];
#pragma unroll
    for (int k = 0; k < 4; ++k) tot[k] = k < W && active ? dwl[k < W ? k : 0] + (last ? 0.0f : past[k < W ? k : 0]) : 0.0f;
    tot[4] = active ? dbl : 0.0f;
    // after step n a lane holds the sum of the 2^n lanes from it on, as far as they are of its row
#pragma unroll
    for (uint32_t off = 1; off <= 16; off <<= 1) {
        if (nvec > off) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const float behind = __shfl_down(tot[k], off, 64);
                tot[k] += v + off < nvec ? behind : 0.0f;
            }
        }
    }
    if (v == 0 && active) {
        float *pp = a.partial + (int64_t)rr * 5;      // rows are numbered b * C + c
#pragma unroll
        for (int k = 0; k < 5; ++k) pp[k] = tot[k];
    }
}

// dweight[c, k] / dbias[c] = sum over the partial sets, in a fixed order: a block owns 32 adjacent
// (c, j) columns; its 8 slices each sum every 8th set in set order (fp64), then the slices are added
// in slice order.  Reads are 128 contiguous bytes per set and slice.
//
// U sets a slice are requested together, added in set order: what bounds the kernel is the round trips in a row, not the
// bytes.  Four loads in flight and the sets past the last whole round one by one -> sixteen from 65 sets on, four below, us of the whole
// call: B 8 C 640 L 1024 12.2 -> 11.5, B 16 C 640 L 511 SiLU masked 16.2 -> 15.4, B 4 C 640 9.2 -> 8.5, B 1 C 160 L 896 6.2 ->
// 5.7; from C 3456 on, packed rows included, within 0.5 %.  (Sixteen at B 1 and B 4, C 3456, 8 and 32 sets: 10.0 -> 10.4,
// 20.9 -> 21.4.)
//
// The sum is stored as the caller's gradient type: converting fp32 sums to 16-bit parameters' type in two further
// launches took a training step at B 16, C 640, L 511 (of 33 us on the device) 3.5 us and their host time.
template <typename T> __global__ __launch_bounds__(256) void canon_zero_kernel(T *p, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) p[i] = T(0);
}

__device__ __forceinline__ void store_grad(void *p, uint32_t i, float v, int dtype)
{
    if (dtype == CANON_DTYPE_F32) store1<CANON_DTYPE_F32>(p, i, v);
    else if (dtype == CANON_DTYPE_BF16) store1<CANON_DTYPE_BF16>(p, i, v);
    else store1<CANON_DTYPE_F16>(p, i, v);
}

template <uint32_t U> __global__ __launch_bounds__(256) void canon_bwd_reduce_kernel(const float *partial, void *dweight, void *dbias,
                                                              uint32_t C, uint32_t nsets, int W, int dtype)
{
    __shared__ double part[8][32];
    const uint32_t col = threadIdx.x & 31u, slice = threadIdx.x >> 5;
    const uint32_t ncols = C * 5u;
    const uint32_t i = blockIdx.x * 32u + col;   // (c, j), j in 0..4
    double acc = 0.0;
    if (i < ncols) {
        for (uint32_t s = slice; s < nsets; s += 8u * U) {
            float v[U];   // (past the last set: the round's first again, not added)
#pragma unroll
            for (uint32_t k = 0; k < U; ++k) v[k] = partial[(int64_t)(s + 8u * k < nsets ? s + 8u * k : s) * ncols + i];
#pragma unroll
            for (uint32_t k = 0; k < U; ++k) acc += s + 8u * k < nsets ? (double)v[k] : 0.0;
        }
    }
    part[slice][col] = acc;
    __syncthreads();
    if (slice != 0 || i >= ncols) return;
    double total = part[0][col];
#pragma unroll
    for (int k = 1; k < 8; ++k) total += part[k][col];
    const uint32_t c = i / 5u, j = i - c * 5u;
    if (j < 4) {
        if ((int)j < W) store_grad(dweight, c * W + j, (float)total, dtype);
    } else if (dbias) {
        store_grad(dbias, c, (float)total, dtype);
    }
}

// ---------------------------------------------------------------------------
// backward of one decode step (shift-register state).  A thread owns one
// channel and walks the batch entries of its group in order, so a wave reads
// dense stretches of x / dout / the state and the partial sums of dweight /
// dbias it leaves per group are formed in a fixed order; canon_bwd_reduce_kernel
// then sums the groups.  z is recomputed from the saved state and the token.
// ---------------------------------------------------------------------------
// Taps, window and sums are kept right-aligned in arrays of four (tap k of a width-W filter at index
// 4-W+k, the token's tap always at 3, window entry i = state slot S-3+i), so every register array is
// indexed by compile-time constants whatever W is.
template <int DT>
__device__ __forceinline__ void load_taps_right(const UpdBwdArgs &a, uint32_t c, float *wr, float &bv)
{
    const int lead = 4 - a.W;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        wr[i] = i >= lead ? round_through<DT>(load_w(a.weight, (int64_t)c * a.w_sc + (i - lead) * a.w_sk, a.w_dtype)) : 0.0f;
    bv = a.bias ? round_through<DT>(load_w(a.bias, c, a.w_dtype)) : 0.0f;
}

// one (batch entry, channel): wn[i] = state slot S-3+i (0 where no tap reads it), qr[i] = gradient of the updated
// state at slot S-4+i (qr[3]: the token's own slot).  Returns dz; dx in dxv; adds to the sums.
__device__ __forceinline__ float update_bwd_point(const UpdBwdArgs &a, const float *wr, float bv, const float *wn,
                                                  const float *qr, float xr, float xt, float go, float m, float *dwr,
                                                  float &db, float &dxv)
{
    float dz = go;
    if (a.act) {
        float z = bv;
#pragma unroll
        for (int i = 0; i < 3; ++i) z = fmaf(wr[i], wn[i], z);
        z = fmaf(wr[3], xt, z);
        dz = go * silu_grad(z);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) dwr[i] = fmaf(dz, wn[i], dwr[i]);
    dwr[3] = fmaf(dz, xt, dwr[3]);
    db += dz;
    float dxt = wr[3] * dz;
    if (a.res_mode == CANON_RESIDUAL_MASKED) dxt += go;
    dxt += qr[3];
    dxv = a.tmask ? dxt * m : dxt;
    if (a.res_mode == CANON_RESIDUAL_UNMASKED) dxv += go;
    return dz;
}

__device__ __forceinline__ void store_partial_right(const UpdBwdArgs &a, float *pp, const float *dwr, float db)
{
    const int lead = 4 - a.W;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i - lead == k) v = dwr[i];
        pp[k] = v;
    }
    pp[4] = db;
}

// Ring-buffer mode (seqlens): the forward wrote the token to slot p = seqlens[b] mod S and read the W-1 slots before
// it cyclically, every other slot stayed where it was.  That is the shift register seen through a rotation: entry j
// of the state before the step lives in slot (p + j) mod S, entry i of the state after it in slot (p + 1 + i) mod S,
// so the code below is written in shift-register entries and maps them to slots where it touches memory.
// State-pool mode (indices): batch entry b uses row indices[b] of conv_state / dstate_out / dstate; an entry whose
// index lies outside the pool was skipped by the forward (its output is a constant zero row): dx = 0, nothing else.
// Only the rows the entries name are written: the caller fills dstate with dstate_out (or zeros) beforehand, so that
// the rows no entry used pass their gradient through.
template <int DT>
__global__ __launch_bounds__(256) void canon_update_bwd_kernel(const UpdBwdArgs a)
{
    constexpr int NB = 4;                   // batch entries whose loads are requested together
    const uint32_t c = blockIdx.x * 256u + threadIdx.x;
    if (c >= a.C) return;
    const uint32_t g = blockIdx.y;
    const int S = a.S;
    const int lead = 4 - a.W;               // window entries / taps below this index do not exist
    float wr[4], bv;
    load_taps_right<DT>(a, c, wr, bv);
    float dwr[4] = {0, 0, 0, 0}, db = 0.0f;
    const uint32_t b_begin = g * a.group;
    const uint32_t b_stop = b_begin + a.group < a.B ? b_begin + a.group : a.B;
    for (uint32_t b0 = b_begin; b0 < b_stop; b0 += NB) {
        // every load of the NB entries first (nothing is stored in between, so they are in flight together)
        float xr[NB], go[NB], m[NB], wn[NB][3], qr[NB][4];
        int64_t row[NB];                    // row of the state tensors, -1: entry skipped
        int pos[NB];                        // ring: slot of the token, else -1
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const uint32_t b = b0 + n < b_stop ? b0 + n : b_stop - 1u;
            row[n] = b;
            if (a.indices) {
                const int32_t i = a.indices[b];
                row[n] = (i < 0 || (a.state_rows > 0 && (uint32_t)i >= a.state_rows)) ? -1 : i;
            }
            pos[n] = -1;
            if (a.seqlens) {
                pos[n] = a.seqlens[b] % S;
                if (pos[n] < 0) pos[n] += S;
            }
            const bool live = row[n] >= 0;
            // slots of entry j of the state before the step and of entry e of the state after it
            auto slot = [&](int j) { return pos[n] < 0 ? j : (pos[n] + j) % S; };
            auto slot_after = [&](int e) { return pos[n] < 0 ? e : (pos[n] + 1 + e) % S; };
            xr[n] = load1<DT>(a.x, (int64_t)b * a.x_sb + (int64_t)c * a.x_sc);
            go[n] = live ? load1<DT>(a.dy, (int64_t)b * a.g_sb + (int64_t)c * a.g_sc) : 0.0f;
            m[n] = a.tmask ? load_mask(a.tmask, (int64_t)b * a.m_sb, a.mask_dtype) : 1.0f;
            const int64_t so = row[n] * a.s_sb + (int64_t)c * a.s_sc;
            const int64_t qo = row[n] * a.q_sb + (int64_t)c * a.q_sc;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < 3) wn[n][i] = (live && i >= lead) ? load1<DT>(a.state, so + (int64_t)slot(S - 3 + i) * a.s_ss) : 0.0f;
                qr[n][i] = (live && a.dso && i >= lead && S - 4 + i >= 0) ? load1<DT>(a.dso, qo + (int64_t)slot_after(S - 4 + i) * a.q_ss) : 0.0f;
            }
        }
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const uint32_t b = b0 + n;
            if (b >= b_stop) break;
            if (row[n] < 0) {
                store1<DT>(a.dx, (int64_t)b * a.d_sb + (int64_t)c * a.d_sc, 0.0f);
                continue;
            }
            auto slot = [&](int j) { return pos[n] < 0 ? j : (pos[n] + j) % S; };
            auto slot_after = [&](int e) { return pos[n] < 0 ? e : (pos[n] + 1 + e) % S; };
            const float xt = a.tmask ? mul_round<DT>(xr[n], m[n]) : xr[n];
            float dxv;
            const float dz = update_bwd_point(a, wr, bv, wn[n], qr[n], xr[n], xt, go[n], m[n], dwr, db, dxv);
            store1<DT>(a.dx, (int64_t)b * a.d_sb + (int64_t)c * a.d_sc, dxv);
            if (a.ds) {
                const int64_t ro = row[n] * a.r_sb + (int64_t)c * a.r_sc;
                const int64_t qo = row[n] * a.q_sb + (int64_t)c * a.q_sc;
                // entries no tap reads: the gradient of the updated state one entry earlier (the same slot of a ring)
                for (int j = 0; j < S - 3 + lead; ++j)
                    store1<DT>(a.ds, ro + (int64_t)slot(j) * a.r_ss,
                               (a.dso && j >= 1) ? load1<DT>(a.dso, qo + (int64_t)slot_after(j - 1) * a.q_ss) : 0.0f);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    if (i >= lead) store1<DT>(a.ds, ro + (int64_t)slot(S - 3 + i) * a.r_ss, fmaf(wr[i], dz, qr[n][i]));
            }
        }
    }
    if (a.partial) store_partial_right(a, a.partial + ((int64_t)g * a.C + c) * 5, dwr, db);
}

// The same for a contiguous [B, C, S] state (and state gradients), S = 3 or 4, channel-contiguous token / dout /
// dx: a lane owns E adjacent channels (two of a 16-bit type, one fp32) whose state rows are ONE run of 12 or
// 16 bytes, as in the forward kernel, so every access of a wave is a dense stretch read or written whole.
// The four waves of a block share a 64-lane channel tile and take every fourth batch entry of the block's
// group; their sums are added in wave order through LDS, so a group is 4 x as many entries (a quarter of the
// partial sets) for the same work per wave.
template <int DT, int S>
__global__ __launch_bounds__(256) void canon_update_bwd_vec_kernel(const UpdBwdArgs a)
{
    constexpr int NB = 4;                   // batch entries whose loads are requested together
    constexpr int BY = Elem<DT>::bytes;
    constexpr int E = upd_lane_channels(BY, S);
    constexpr int ND = E * S * BY / 4;      // words of state per lane and batch entry
    static_assert(E * BY == 4 && (S == 3 || S == 4), "one word of token / dout / dx per lane");
    __shared__ float sums[3][64][E * 5 + 1];   // waves 1..3 hand their sums to wave 0 (+1: no bank conflicts)
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t cv = blockIdx.x * 64u + lane;
    const uint32_t c0 = cv * E;
    const bool live = c0 < a.C;
    const uint32_t g = blockIdx.y;
    const int lead = 4 - a.W;
    float wr[E][4], bv[E], dwr[E][4], db[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (live) load_taps_right<DT>(a, c0 + e, wr[e], bv[e]);
        db[e] = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) dwr[e][i] = 0.0f;
    }
    const uint32_t b_begin = g * a.group;
    const uint32_t b_stop = b_begin + a.group < a.B ? b_begin + a.group : a.B;
    // this wave's entries: b_begin + wv, + 4, + 8, ...
    for (uint32_t b0 = b_begin + wv; live && b0 < b_stop; b0 += 4u * NB) {
        uint32_t X[NB], G[NB], ST[NB][ND], Q[NB][ND];
        float m[NB];
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const uint32_t bn = b0 + 4u * n;
            const uint32_t b = bn < b_stop ? bn : b0;
            X[n] = *(const uint32_t *)(a.x + ((int64_t)b * a.x_sb + c0) * BY);
            G[n] = *(const uint32_t *)(a.dy + ((int64_t)b * a.g_sb + c0) * BY);
            load_words<ND>(a.state + ((int64_t)b * a.s_sb + (int64_t)c0 * S) * BY, ST[n]);
            if (a.dso) {
                load_words<ND>(a.dso + ((int64_t)b * a.q_sb + (int64_t)c0 * S) * BY, Q[n]);
            } else {
#pragma unroll
                for (int i = 0; i < ND; ++i) Q[n][i] = 0u;
            }
            m[n] = a.tmask ? load_mask(a.tmask, (int64_t)b * a.m_sb, a.mask_dtype) : 1.0f;
        }
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const uint32_t b = b0 + 4u * n;
            if (b >= b_stop) break;
            uint32_t ox = 0u, DS[ND];
#pragma unroll
            for (int i = 0; i < ND; ++i) DS[i] = 0u;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float xr = Packed<DT>::as_float(Packed<DT>::get(&X[n], e));
                const float go = Packed<DT>::as_float(Packed<DT>::get(&G[n], e));
                const float xt = a.tmask ? mul_round<DT>(xr, m[n]) : xr;
                float wn[3], qr[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (i < 3) wn[i] = i >= lead ? Packed<DT>::as_float(Packed<DT>::get(ST[n], e * S + S - 3 + i)) : 0.0f;
                    qr[i] = (i >= lead && S - 4 + i >= 0) ? Packed<DT>::as_float(Packed<DT>::get(Q[n], e * S + (S - 4 + i >= 0 ? S - 4 + i : 0))) : 0.0f;
                }
                float dxv;
                const float dz = update_bwd_point(a, wr[e], bv[e], wn, qr, xr, xt, go, m[n], dwr[e], db[e], dxv);
                Packed<DT>::put(&ox, e, Packed<DT>::raw_of(dxv));
                // slots no tap reads: the gradient of the updated state shifted by one (raw bits); the others
                // add their tap's share
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    const int i = j - (S - 3);
                    uint32_t raw = j >= 1 ? Packed<DT>::get(Q[n], e * S + (j >= 1 ? j - 1 : 0)) : 0u;
                    if (i >= 0 && i >= lead) raw = Packed<DT>::raw_of(fmaf(wr[e][i >= 0 ? i : 0], dz, qr[i >= 0 ? i : 0]));
                    Packed<DT>::put(DS, e * S + j, raw);
                }
            }
            *(uint32_t *)(a.dx + ((int64_t)b * a.d_sb + c0) * BY) = ox;
            if (a.ds) store_words<ND>(a.ds + ((int64_t)b * a.r_sb + (int64_t)c0 * S) * BY, DS);
        }
    }
    if (!a.partial) return;                 // uniform over the block
    if (wv != 0) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) sums[wv - 1][lane][e * 5 + i] = dwr[e][i];
            sums[wv - 1][lane][e * 5 + 4] = db[e];
        }
    }
    __syncthreads();
    if (wv != 0 || !live) return;
#pragma unroll
    for (int k = 0; k < 3; ++k) {           // wave order: a fixed order of additions
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dwr[e][i] += sums[k][lane][e * 5 + i];
            db[e] += sums[k][lane][e * 5 + 4];
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) store_partial_right(a, a.partial + ((int64_t)g * a.C + c0 + e) * 5, dwr[e], db[e]);
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
namespace {

void launch_reduce(const float *partial, void *dweight, void *dbias, uint32_t C, uint32_t nsets, int W, int dtype, hipStream_t s)
{
    const dim3 g((C * 5u + 31u) / 32u), b(256);
    if (nsets > 64u) hipLaunchKernelGGL((canon_bwd_reduce_kernel<16>), g, b, 0, s, partial, dweight, dbias, C, nsets, W, dtype);
    else hipLaunchKernelGGL((canon_bwd_reduce_kernel<4>), g, b, 0, s, partial, dweight, dbias, C, nsets, W, dtype);
}

template <int DT, int W, bool MASK, bool RAGGED> void launch_bwd_bcl(const BwdPlan &pl, hipStream_t s)
{
    const dim3 g(pl.grid), b(256);
    const BwdArgs &A = pl.args;
    constexpr int64_t EV = RAGGED ? 1 : Elem<DT>::per_vec;   // strides and length in elements, or in vectors
    switch (pl.U) {
#define CANON_BWD_BCL_LAUNCH(UU)                                                                                         \
    hipLaunchKernelGGL((canon_bwd_bcl_kernel<DT, W, UU, MASK, RAGGED>), g, b, 0, s, A.x, A.dy, (uint32_t)(A.x_sb / EV),  \
                       (uint32_t)(A.x_sc / EV), (uint32_t)(A.g_sb / EV), (uint32_t)(A.g_sc / EV), A.nthreads, A.nchunk,  \
                       A.C, A.div_nvec.m, A.div_nvec.s1 | A.div_nvec.s2 << 1, A.L / (uint32_t)EV, A)
    case 4: CANON_BWD_BCL_LAUNCH(4); break;
    case 2: CANON_BWD_BCL_LAUNCH(2); break;
    default: CANON_BWD_BCL_LAUNCH(1); break;
#undef CANON_BWD_BCL_LAUNCH
    }
}

template <int DT, int W, bool MASK> void launch_bwd_m(const BwdPlan &pl, hipStream_t s)
{
    const dim3 g(pl.grid), b(256);
    if (pl.kind == BWD_BCL_VEC) {
        const BwdArgs &A = pl.args;
        if (pl.short_rows)
            hipLaunchKernelGGL((canon_bwd_bcl_short_kernel<DT, W, MASK>), g, b, 0, s, A.x, A.dy, (uint32_t)A.x_sb, (uint32_t)A.x_sc,
                               (uint32_t)A.g_sb, (uint32_t)A.g_sc, A.nthreads, A.C, A.div_nvec.m,
                               A.nvec | (A.nvec * Elem<DT>::per_vec - A.L) << 6 | A.div_nvec.s1 << 9 | A.div_nvec.s2 << 10 | A.chunk << 15, A);
        else if (pl.ragged) launch_bwd_bcl<DT, W, MASK, true>(pl, s);
        else launch_bwd_bcl<DT, W, MASK, false>(pl, s);
    } else if (pl.kind == BWD_BLC_VEC)
    {
        const bool states = pl.args.init != nullptr || pl.args.dfin != nullptr;
        if constexpr (W == 4) {
            if (pl.any) {
                if (pl.args.act) hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, true, false, false, true>), g, b, 0, s, pl.args);
                else hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, false, false, false, true>), g, b, 0, s, pl.args);
                return;
            }
        }
        if (pl.args.seq) {
            if (pl.args.act) hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, true, false, true>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, false, false, true>), g, b, 0, s, pl.args);
        } else if (pl.args.act) {
            if (states) hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, true, true>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, true, false>), g, b, 0, s, pl.args);
        } else {
            if (states) hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, false, true>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_bwd_blc_kernel<DT, W, MASK, false, false>), g, b, 0, s, pl.args);
        }
    }
    else if (pl.args.seq)
        hipLaunchKernelGGL((canon_bwd_walk_kernel<DT, W, MASK, kBwdRows, true>), g, b, 0, s, pl.args);
    else
        hipLaunchKernelGGL((canon_bwd_walk_kernel<DT, W, MASK, kBwdRows, false>), g, b, 0, s, pl.args);
}

template <int DT> void launch_bwd(const BwdPlan &pl, hipStream_t s)
{
    const bool m = pl.args.mask != nullptr;
    switch (pl.args.W) {
    case 2: m ? launch_bwd_m<DT, 2, true>(pl, s) : launch_bwd_m<DT, 2, false>(pl, s); break;
    case 3: m ? launch_bwd_m<DT, 3, true>(pl, s) : launch_bwd_m<DT, 3, false>(pl, s); break;
    default: m ? launch_bwd_m<DT, 4, true>(pl, s) : launch_bwd_m<DT, 4, false>(pl, s); break;
    }
}

}  // namespace

void launch_bwd(const BwdPlan &pl, int x_dtype, hipStream_t s)
{
    switch (x_dtype) {
    case CANON_DTYPE_F32: launch_bwd<CANON_DTYPE_F32>(pl, s); break;
    case CANON_DTYPE_BF16: launch_bwd<CANON_DTYPE_BF16>(pl, s); break;
    default: launch_bwd<CANON_DTYPE_F16>(pl, s); break;
    }
    launch_reduce(pl.args.partial, pl.args.dweight, pl.args.dbias, pl.args.C, pl.args.nsets, pl.args.W, pl.args.grad_dtype, s);
}

void launch_update_bwd(const UpdBwdPlan &pl, int x_dtype, hipStream_t s)
{
    const dim3 g(pl.grid_c, pl.args.ngroups), b(256);   // vec: 64 lanes of channels per block, else 256 channels
    if (pl.vec) {
        const bool s3 = pl.args.S == 3;
        switch (x_dtype) {
        case CANON_DTYPE_F32:
            if (s3) hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_F32, 3>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_F32, 4>), g, b, 0, s, pl.args);
            break;
        case CANON_DTYPE_BF16:
            if (s3) hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_BF16, 3>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_BF16, 4>), g, b, 0, s, pl.args);
            break;
        default:
            if (s3) hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_F16, 3>), g, b, 0, s, pl.args);
            else hipLaunchKernelGGL((canon_update_bwd_vec_kernel<CANON_DTYPE_F16, 4>), g, b, 0, s, pl.args);
            break;
        }
    } else {
        switch (x_dtype) {
        case CANON_DTYPE_F32: hipLaunchKernelGGL((canon_update_bwd_kernel<CANON_DTYPE_F32>), g, b, 0, s, pl.args); break;
        case CANON_DTYPE_BF16: hipLaunchKernelGGL((canon_update_bwd_kernel<CANON_DTYPE_BF16>), g, b, 0, s, pl.args); break;
        default: hipLaunchKernelGGL((canon_update_bwd_kernel<CANON_DTYPE_F16>), g, b, 0, s, pl.args); break;
        }
    }
    if (pl.args.partial)
        launch_reduce(pl.args.partial, pl.args.dweight, pl.args.dbias, pl.args.C, pl.args.ngroups, pl.args.W, CANON_DTYPE_F32, s);
}

// Asking for a kernel's attributes makes the runtime load this file's code object onto the current device.
hipError_t preload_bwd()
{
    hipFuncAttributes attr;
    return hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(&(canon_zero_kernel<float>)));
}

void launch_zero(void *p, uint32_t n, int elem_bytes, hipStream_t s)
{
    if (!n) return;
    const dim3 g((n + 255) / 256), b(256);
    if (elem_bytes == 2) hipLaunchKernelGGL((canon_zero_kernel<uint16_t>), g, b, 0, s, (uint16_t *)p, n);
    else hipLaunchKernelGGL((canon_zero_kernel<float>), g, b, 0, s, (float *)p, n);
}

}  // namespace canon
