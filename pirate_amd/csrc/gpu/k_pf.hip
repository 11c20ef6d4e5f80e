// Peak finding on gfx950 over the subband streams of one output tree.
// Reference semantics: ReferencePeakFindingKernel::apply (src_lib/PeakFindingKernel.cu:252-456):
//
//   boxcars   B_0(e) = x[e-1],  B_l(e) = B_{l-1}(e - 2^(l-1)) + B_{l-1}(e)   (binary-tree sums)
//   candidate (level l, multiplet m, isamp, profile p) ends at e = tout*Dout + (isamp+1)*dt,
//             dt = min(Dcore, 2^l); with x_k = B_l(e - (3-k)*2^l):
//               p=0 (l=0): x3      p=3l+1: x2+x3      p=3l+2: (x1/2 + x2) + x3/2
//               p=3l+3: ((x0/2 + x1) + x2) + x3/2
//   out_max[tout] = max over (l, m, isamp, p) of w[p, n(m)] * y; the first maximum in the loop
//   order (l, m, isamp, p) wins ties; token = t | (p << 8) | (m << 16), t = isamp*dt.
//
// Mapping: one lane per stream (DM row, multiplet m); a block holds 256/M DM rows. Each lane
// walks its stream through time once. Every boxcar level keeps its last values in a register
// window (Wmax and Dout are template parameters, so every shift, sum and candidate of one
// output bin is unrolled at compile time). k_pf_one weights and compares each candidate as it is
// formed (strict '>', candidates visited in (isamp, p) order) and can form the optional
// float64 variances. k_pf keeps the largest value of each profile and finds the token of the
// winning stream in a second step; pf_two_step says where. Either way the multiplets of a DM row are
// reduced in (level, m) order, and the result is the reference's maximum and argmax token, bit
// for bit. Positions before the row start count as zeros, the initial state of the windows.
//
// The chunk's time axis is split into nseg segments (blockIdx.z), one workgroup each, so
// that short chunks still fill the chip. A segment's lanes start from zero windows and run
// the tpad positions before it unevaluated: every window entry at the segment start is a
// sum over at most the last tpad samples (level l holds boxcar sums of 2^l samples ending at
// most 3*2^l positions back, and 4*2^l <= 2*Wmax <= tpad), so the windows, and hence every
// candidate, equal those of one lane walking the whole chunk. The running variance sums
// depend on the order of the bins, so they use one segment.
//
// Rows are [tpad history | Tp samples]; at the end of a chunk the last tpad samples are moved to
// the front for the next chunk.

#include "device_common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace pirate_amd {

static constexpr int kPfThreads = 256;
static constexpr int kPfMaxDout = 32;
static constexpr int kPfLine = 128;      // bytes of a row that one staging tile covers

// k_pf_one's staging tile length (positions) for output time downsampling Dout: whole output
// bins, at least kPfTileMin positions when Dout >= 4, 8 bins below.
static constexpr int kPfTileMin = 16;
__host__ __device__ constexpr int pf_tile_len(int dout)
{
    return (dout >= 4) ? ((dout > kPfTileMin) ? dout : kPfTileMin) : 8 * dout;
}

bool pf_config_supported(int M, int tpad, int Dcore, int Dout, int Tp)
{
    if (M < 1 || M > kPfThreads || Dout < 1 || Dout > kPfMaxDout || (Dout & (Dout - 1)))
        return false;
    if (tpad % 4)
        return false;
    const int dc = (Dout < 8) ? Dout : 8;
    return (Dcore == dc) && (Tp % 32 == 0);
}

template<int LW, int LD>
struct PfShape {
    static constexpr int W = 1 << LW;
    static constexpr int NLEV = (LW > 1) ? LW : 1;
    static constexpr int P = 1 + 3 * LW;
    static constexpr int DOUT = 1 << LD;
    static constexpr int DCORE = (DOUT < 8) ? DOUT : 8;
    static constexpr int TL = pf_tile_len(DOUT);                 // tile length (positions)
    static constexpr int NB = TL / DOUT;                          // output bins per tile
    static constexpr int dt(int l) { return ((1 << l) < DCORE) ? (1 << l) : DCORE; }
    static constexpr int sgrid(int l) { return (1 << l) / dt(l); }   // grid points per 2^l samples
    static constexpr int win(int l) { return 3 * sgrid(l) + 1; }
    static constexpr int woff(int l) { return (l == 0) ? 0 : woff(l - 1) + win(l - 1); }
    static constexpr int WTOT = woff(NLEV);
    static constexpr int WAVES1 = (WTOT + P <= 32 && LD >= 2) ? 4 : 2;     // k_pf_one's waves per SIMD
};

template<typename S, bool VAR>
struct PfLane {
    float w[S::WTOT];          // per level l: w[woff(l) + i] = B_l(e - i*dt(l)), e = newest end
    float bv[S::NLEV];         // per level: best weighted value in the current bin
    unsigned int bc[S::NLEV];  // per level: its code (see code())
    float wt[S::P];            // weights of the current bin, per profile
    // VAR: per profile, the sum of squared weighted candidates in the current bin (bs) and
    // the chunk's running sum of bs / (nt_out * candidates per bin at that level) (acc),
    // in float64 -- the reference peak finder's optional out_var.
    double bs[VAR ? S::P : 1], acc[VAR ? S::P : 1], wv[S::NLEV];

    template<int P>
    __device__ __forceinline__ void sq(float v)
    {
        if constexpr (VAR)
            bs[P] = bs[P] + double(v) * double(v);
    }

    // End of an output bin: fold the bin's sums into the chunk's (same order as the reference).
    __device__ __forceinline__ void fold_var()
    {
        if constexpr (VAR) {
#pragma unroll
            for (int p = 0; p < S::P; p++) {
                acc[p] = acc[p] + bs[p] * wv[(p == 0) ? 0 : (p - 1) / 3];
                bs[p] = 0.0;
            }
        }
    }

    // Candidate codes within a level. Compact codes isamp*4 + q (q = 0 for p = 0, else
    // p - 3l) stay within the hardware's inline-constant range (<= 64) when Dout <= 16, so the
    // per-candidate selects need no literal moves; token() expands them once per bin.
    static constexpr bool COMPACT = (S::DOUT <= 16);

    template<int L>
    static constexpr unsigned int code(int isamp, int q)
    {
        return COMPACT ? unsigned(4 * isamp + q)
                       : (unsigned(isamp * S::dt(L)) | (unsigned(q ? 3 * L + q : 0) << 8));
    }

    template<int L>
    __device__ __forceinline__ unsigned int token(unsigned int c) const
    {
        if constexpr (COMPACT) {
            const unsigned int q = c & 3u, isamp = c >> 2;
            const unsigned int p = q ? (3u * L + q) : 0u;
            return (isamp * unsigned(S::dt(L))) | (p << 8);
        } else {
            return c;
        }
    }

    template<int L>
    __device__ __forceinline__ void push(float v)
    {
        constexpr int o = S::woff(L), n = S::win(L);
#pragma unroll
        for (int i = n - 1; i > 0; i--)
            w[o + i] = w[o + i - 1];
        w[o] = v;
    }

    template<int L, bool FIRST>
    __device__ __forceinline__ void upd(float v, unsigned int code)
    {
        if constexpr (FIRST) {
            bv[L] = v;
            bc[L] = code;
        } else {
            const bool g = v > bv[L];
            bv[L] = g ? v : bv[L];
            bc[L] = g ? code : bc[L];
        }
    }

    template<int L, int POS>
    __device__ __forceinline__ void candidates()
    {
        constexpr int o = S::woff(L), s = S::sgrid(L);
        constexpr int isamp = (POS + 1) / S::dt(L) - 1;
        constexpr bool first = (isamp == 0);
        const float x3 = w[o], x2 = w[o + s], x1 = w[o + 2 * s], x0 = w[o + 3 * s];
        if constexpr (L == 0) {
            const float v0 = wt[0] * x3;
            upd<0, first>(v0, code<0>(isamp, 0));
            sq<0>(v0);
        }
        if constexpr (S::P > 1) {
            constexpr int p = 3 * L + 1;
            const float h3 = 0.5f * x3;
            const float y1 = x2 + x3;
            const float y2 = (0.5f * x1 + x2) + h3;
            const float y3 = ((0.5f * x0 + x1) + x2) + h3;
            const float v1 = wt[p] * y1, v2 = wt[p + 1] * y2, v3 = wt[p + 2] * y3;
            upd<L, first && (L > 0)>(v1, code<L>(isamp, 1));
            upd<L, false>(v2, code<L>(isamp, 2));
            upd<L, false>(v3, code<L>(isamp, 3));
            sq<p>(v1);
            sq<p + 1>(v2);
            sq<p + 2>(v3);
        }
    }

    template<int L, int POS, bool EVAL>
    __device__ __forceinline__ void levels()
    {
        if constexpr (L < S::NLEV) {
            if constexpr ((POS + 1) % S::dt(L) == 0) {
                if constexpr (L > 0) {
                    constexpr int op = S::woff(L - 1), back = S::sgrid(L - 1);
                    push<L>(w[op + back] + w[op]);
                }
                if constexpr (EVAL)
                    candidates<L, POS>();
                levels<L + 1, POS, EVAL>();
            }
        }
    }

    // One output bin (DOUT positions); xs[POS] is the sample at in-bin position POS.
    template<bool EVAL, int POS = 0>
    __device__ __forceinline__ void bin(const float *xs)
    {
        if constexpr (POS < S::DOUT) {
            push<0>(xs[POS]);
            levels<0, POS, EVAL>();
            bin<EVAL, POS + 1>(xs);
        }
    }

    template<int L = 1>
    __device__ __forceinline__ void combine_from(float &V, unsigned int &C) const
    {
        if constexpr (L < S::NLEV) {
            const bool g = bv[L] > V;
            V = g ? bv[L] : V;
            C = g ? token<L>(bc[L]) : C;
            combine_from<L + 1>(V, C);
        }
    }

    // Levels in order, strict '>': the first level with the bin's maximum; C is its token.
    __device__ __forceinline__ void combine(float &V, unsigned int &C) const
    {
        V = bv[0];
        C = token<0>(bc[0]);
        combine_from<1>(V, C);
    }
};

// The same walk without weights or codes: the largest value of every profile in a bin (the
// weight of a profile is constant over a bin, and rounding is monotonic, so the largest
// weighted candidate of a profile is its weight times this value, bit for bit). That needs
// finite values: a candidate that is not finite can be NaN once weighted, and PfLane drops a level
// whose first candidate is NaN (a zero weight times -inf, say), which no maximum shows.
template<typename S>
struct PfMax {
    float w[S::WTOT];          // boxcar windows, as in PfLane
    float mx[S::P];            // per profile: largest value in the current bin

    template<int L, int POS, bool EVAL>
    __device__ __forceinline__ void levels()
    {
        if constexpr (L < S::NLEV) {
            if constexpr ((POS + 1) % S::dt(L) == 0) {
                constexpr int o = S::woff(L), s = S::sgrid(L), n = S::win(L);
                if constexpr (L > 0) {
                    constexpr int op = S::woff(L - 1), back = S::sgrid(L - 1);
#pragma unroll
                    for (int i = n - 1; i > 0; i--)
                        w[o + i] = w[o + i - 1];
                    w[o] = w[op + back] + w[op];
                }
                if constexpr (EVAL) {
                    constexpr bool first = (POS + 1) / S::dt(L) == 1;
                    const float x3 = w[o], x2 = w[o + s], x1 = w[o + 2 * s], x0 = w[o + 3 * s];
                    if constexpr (L == 0)
                        mx[0] = first ? x3 : fmaxf(mx[0], x3);
                    if constexpr (S::P > 1) {
                        constexpr int p = 3 * L + 1;
                        const float h3 = 0.5f * x3;
                        const float y1 = x2 + x3;
                        const float y2 = (0.5f * x1 + x2) + h3;
                        const float y3 = ((0.5f * x0 + x1) + x2) + h3;
                        mx[p] = first ? y1 : fmaxf(mx[p], y1);
                        mx[p + 1] = first ? y2 : fmaxf(mx[p + 1], y2);
                        mx[p + 2] = first ? y3 : fmaxf(mx[p + 2], y3);
                    }
                }
                levels<L + 1, POS, EVAL>();
            }
        }
    }

    template<bool EVAL, int POS = 0>
    __device__ __forceinline__ void bin(const float *xs)
    {
        if constexpr (POS < S::DOUT) {
#pragma unroll
            for (int i = S::win(0) - 1; i > 0; i--)
                w[i] = w[i - 1];
            w[0] = xs[POS];
            levels<0, POS, EVAL>();
            bin<EVAL, POS + 1>(xs);
        }
    }

    // The bin's largest weighted value V and the first level that has it.
    __device__ __forceinline__ void combine(const float (&wt)[S::P], float &V, unsigned int &lev) const
    {
        float v[S::P];
#pragma unroll
        for (int p = 0; p < S::P; p++)
            v[p] = wt[p] * mx[p];
        V = v[0];
        lev = 0;
        if constexpr (S::P > 1) {
            V = fmaxf(fmaxf(fmaxf(V, v[1]), v[2]), v[3]);
#pragma unroll
            for (int l = 1; l < S::NLEV; l++) {
                const float u = fmaxf(fmaxf(v[3 * l + 1], v[3 * l + 2]), v[3 * l + 3]);
                lev = (u > V) ? unsigned(l) : lev;
                V = fmaxf(V, u);
            }
        }
    }
};

// Whether a bin's samples are such that PfMax may not be used for it, nor for the NBACK bins after
// it, whose windows they enter: a candidate adds at most 64 samples (times up to 1), so with
// samples below 1e36 all candidates are finite. One three-operand maximum, which keeps NaN, for
// two samples.
template<int N>
__device__ __forceinline__ bool pf_wild(const float *x)
{
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < N; i++)
        m = __builtin_elementwise_maximum(m, fabsf(x[i]));
    return !(m < 1e36f);
}

__device__ __forceinline__ int pf_level_of_token(unsigned int tok)
{
    const int p = int((tok >> 8) & 0xffu);
    return (p == 0) ? 0 : (p - 1) / 3;
}

// Rotates a workgroup's rows for the next chunk: positions [Tp, Tp + tpad) -> [0, tpad), i.e.
// the rows shift down by Tp. Every load of the rows has completed before the caller's last
// barrier. Done in column blocks of width min(Tp, tpad) in ascending order, with a
// barrier between blocks: within a block the positions read ([c0 + Tp, ...)) and
// written ([c0, c0 + width)) are disjoint, and a later block reads only positions at or
// above every position an earlier block wrote. Segment 0 rotates; the host chooses
// segments of at least nwarm*TL positions, so no other segment reads below tpad, the positions
// written here. A thread issues kRot 4-element loads before their stores: element by element,
// each load waited for the store before it, and segment 0 spent 30-40 memory round trips here.
template<typename Tst>
__device__ __forceinline__ void rotate_rows(Tst *rows, int nstreams, const PfArgs &a)
{
    constexpr int kRot = 8;
    const int wcol = min(a.Tp, a.tpad);          // tpad and Tp are multiples of 4: so is every c0
    for (int c0 = 0; c0 < a.tpad; c0 += wcol) {
        const int ng = min(wcol, a.tpad - c0) >> 2, n = nstreams * ng;
        for (int base = 0; base < n; base += kRot * kPfThreads) {
            rawv_st<Tst, 4> v[kRot];
#pragma unroll
            for (int k = 0; k < kRot; k++) {
                const int idx = min(base + k * kPfThreads + int(threadIdx.x), n - 1);
                const int s = idx / ng, i = c0 + 4 * (idx - s * ng);
                v[k] = ldv_raw<Tst, 4>(rows + long(s) * a.rowlen + a.Tp + i);
            }
#pragma unroll
            for (int k = 0; k < kRot; k++) {
                const int idx = base + k * kPfThreads + int(threadIdx.x);
                const int s = idx / ng, i = c0 + 4 * (idx - s * ng);
                if (idx < n)
                    *reinterpret_cast<rawv_st<Tst, 4> *>(rows + long(s) * a.rowlen + i) = v[k];
            }
        }
        if (c0 + wcol < a.tpad)
            __syncthreads();
    }
}

// The first evaluated tile of time segment z (of nseg) of a chunk of n tiles.
__device__ __forceinline__ int pf_first_tile(int n, int z, int nseg) { return int(long(n) * z / nseg); }

// One step: every candidate is weighted and compared as it is formed, and (VAR) its square summed
// for the float64 out_var.
template<typename Tst, int LW, int LD, bool VAR>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(VAR ? 2 : PfShape<LW, LD>::WAVES1)))
k_pf_one(PfArgs a)
{
    using S = PfShape<LW, LD>;
    constexpr int TL = S::TL, NB = S::NB, STR = TL + 1, VPR = TL / 4;
    __shared__ float tile[kPfThreads * STR];
    __shared__ float rv[kPfThreads * NB];
    __shared__ unsigned int rt[kPfThreads * NB];

    const int tid = threadIdx.x;
    const int M = a.M, N = a.N;
    const int ndpf = kPfThreads / M;
    const int dpf0 = blockIdx.x * ndpf;
    const int b = blockIdx.y;
    const int tile0 = pf_first_tile(a.Tp / TL, blockIdx.z, a.nseg);               // this segment's first tile
    const int ntseg = pf_first_tile(a.Tp / TL, blockIdx.z + 1, a.nseg) - tile0;    // its evaluated tiles
    const int nd = min(ndpf, a.ndm_out - dpf0);
    const int nstreams = nd * M;
    const bool active = tid < nstreams;
    const int dl = tid / M, m = tid - dl * M;

    Tst *rows = reinterpret_cast<Tst *>(a.sb) + long(a.beam0 + b) * a.sb_bstride + long(dpf0) * M * a.rowlen;
    const int Wds = a.ndm_out / a.ndm_wt;
    const int Tds = a.nt_out / a.nt_wt;
    const float *wrow = a.wt + long(b) * a.wt_bstride + long(active ? (dpf0 + dl) / Wds : 0) * a.nt_wt * S::P * N
                        + (active ? a.m_to_n[m] : 0);
    Tst *outm = reinterpret_cast<Tst *>(a.out_max) + long(b) * a.out_bstride;
    unsigned int *outa = a.out_argmax + long(b) * a.out_bstride;

    PfLane<S, VAR> ln;
#pragma unroll
    for (int i = 0; i < S::WTOT; i++)
        ln.w[i] = 0.0f;
    if constexpr (VAR) {
#pragma unroll
        for (int p = 0; p < S::P; p++)
            ln.bs[p] = ln.acc[p] = 0.0;
#pragma unroll
        for (int l = 0; l < S::NLEV; l++)
            ln.wv[l] = 1.0 / double(a.nt_out * (S::DOUT / S::dt(l)));
    }

    const int nwarm = (a.tpad + TL - 1) / TL;
    const int ntiles = nwarm + ntseg;
    const float *xs = tile + tid * STR;

    for (int it = 0; it < ntiles; it++) {
        const int p0 = a.tpad + (tile0 + it - nwarm) * TL;

        // ---- stage [nstreams][TL] samples (4 per load, VPR loads per row segment); a thread
        // issues all of its loads before it converts and stores them (with the conversion at
        // each load, the 16-bit variants waited for each load before issuing the next)
        rawv_st<Tst, 4> raw[VPR];
#pragma unroll
        for (int k = 0; k < VPR; k++) {
            const int idx = tid + k * kPfThreads;
            const int s = idx / VPR, i = (idx - s * VPR) * 4;
            raw[k] = (s < nstreams && p0 + i >= 0) ? ldv_raw<Tst, 4>(rows + long(s) * a.rowlen + p0 + i)
                                                  : rawv_st<Tst, 4>{};
        }
#pragma unroll
        for (int k = 0; k < VPR; k++) {
            const int idx = tid + k * kPfThreads;
            const int s = idx / VPR, i = (idx - s * VPR) * 4;
            if (s < nstreams)
                from_rawv<Tst, 4>(raw[k], tile + s * STR + i);
        }
        __syncthreads();

        if (it < nwarm) {
            if (active) {
#pragma unroll 1
                for (int j = 0; j < NB; j++)
                    ln.template bin<false>(xs + j * S::DOUT);
            }
        } else {
            const int tb0 = (tile0 + it - nwarm) * NB;
            if (active) {
#pragma unroll 1
                for (int j = 0; j < NB; j++) {
                    const float *wp = wrow + long((tb0 + j) / Tds) * S::P * N;
#pragma unroll
                    for (int p = 0; p < S::P; p++)
                        ln.wt[p] = wp[p * N];
                    ln.template bin<true>(xs + j * S::DOUT);
                    ln.fold_var();
                    float V;
                    unsigned int C;
                    ln.combine(V, C);
                    rv[tid * NB + j] = V;
                    rt[tid * NB + j] = C | (unsigned(m) << 16);
                }
            }
        }
        __syncthreads();

        // ---- reduce over multiplets: first (level, m) in loop order with the largest value
        if (it >= nwarm) {
            const int tb0 = (tile0 + it - nwarm) * NB;
            for (int idx = tid; idx < nd * NB; idx += kPfThreads) {
                const int d = idx / NB, j = idx - d * NB;
                const int s0 = d * M;
                float bv = rv[s0 * NB + j];
                unsigned int bt = rt[s0 * NB + j];
                int bk = pf_level_of_token(bt) * M;
                for (int mm = 1; mm < M; mm++) {
                    const float v = rv[(s0 + mm) * NB + j];
                    const unsigned int tk = rt[(s0 + mm) * NB + j];
                    const int key = pf_level_of_token(tk) * M + mm;
                    if (v > bv || (v == bv && key < bk)) {
                        bv = v;
                        bt = tk;
                        bk = key;
                    }
                }
                const long o = long(dpf0 + d) * a.nt_out + tb0 + j;
                st_st(outm + o, bv);
                outa[o] = bt;
            }
        }
    }

    if (VAR && active) {
        double *ov = a.out_var + long(b) * a.ndm_out * M * S::P + (long(dpf0 + dl) * M + m) * S::P;
#pragma unroll
        for (int p = 0; p < S::P; p++)
            ov[p] = ln.acc[p];
    }

    if (blockIdx.z == 0)
        rotate_rows(rows, nstreams, a);
}

// Two steps (bins of 8 and 16 samples; pf_two_step says where). Step 1 walks every stream once and keeps per bin only
// the largest value of each profile (PfMax: about 1.5 maxima per candidate in place of a
// multiply, a compare and two selects), weights these, and leaves the stream's largest value
// and its first level in LDS. Step 2 runs once per kPfBatch bins, one lane per (DM row, bin):
// it picks the winning multiplet (largest value, then first (level, m)) and walks that one
// stream over the bin again with PfLane, which gives the value and the token of the first
// maximum. A DM row has M streams, so step 2 costs (NBACK + 1) / M of a full walk per stream.
// Infinities, NaN and samples that could make a sum overflow (pf_wild): a stream is marked in each
// bin whose windows hold one. A wave with a marked lane walks that bin with PfLane in place of
// PfMax, from the same windows, and leaves value and token for step 2, which then walks nothing
// for a winner that has its token. So data full of NaN costs about what the walk of every candidate
// costs; with all M streams of a marked (DM row, bin) walked by one lane of step 2 it cost up to 4.7
// times that.
//
// Samples reach LDS by direct loads (no registers, no conversion), 128 bytes of a row at a
// time, so that every line is fetched once; a wave stages the 64 rows that its lanes walk, so
// staging needs no barrier: the next tile's loads start when the wave has read the last part of
// this one. One load instruction brings 8 rows x 128 bytes; lane i of the
// instruction writes the i-th 16 bytes, so the 16-byte chunks of a row are permuted on the
// global side (slot s of row r holds chunk s ^ (r & 7)), and the 16-byte reads of 8
// neighbouring rows cover all banks. 51 KB of LDS and 168 VGPRs: three workgroups (12 waves)
// per CU. Bounded by VALU issue (475 instructions per stream and 16-sample bin at Wmax 16, step 2 and
// warm-up included, against 770 with every candidate compared) and, for float32, near half by the row reads.
// 16384 DM rows x 2048 samples x 16 beams, Wmax 16, bins of 16: float32 0.774 -> 0.541 ms,
// float16 0.736 -> 0.423 ms; 36 multiplets, 8 beams of rank 15, float16: 2.28 -> 1.01 ms. No instance
// spills vector registers; all keep 4 to 58 scalars in lanes of one, outside a bin's walk.
// Tried: tiles of 16 positions staged through registers (each 128-byte line fetched twice,
// float32 0.93 ms), two staging buffers and 8 waves per CU (0.68 ms), the walk's float32 loads
// all at once with bins of 16 (31 registers spilled, 1.31 ms).
static constexpr int kPfBatch = 12;

typedef __attribute__((address_space(1))) const void *pf_gptr;
typedef __attribute__((address_space(3))) void *pf_lptr;

template<typename Tst, int LW, int LD>
__global__ void __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(3)))
k_pf(PfArgs a)
{
    using S = PfShape<LW, LD>;
    constexpr int TL = kPfLine / int(sizeof(Tst));                 // positions per tile
    constexpr int CH = 16 / int(sizeof(Tst));                      // positions per 16-byte chunk
    constexpr int SB = (S::DOUT > CH) ? S::DOUT : CH;               // positions read at a time
    constexpr int BPS = SB / S::DOUT;                               // their bins
    constexpr int RVS = kPfThreads + 1, RLS = kPfThreads + 4;      // strides of a batch's bins (banks)
    constexpr int TPAD = (2 * S::W > 4) ? 2 * S::W : 4;             // a.tpad
    constexpr int NBACK = (TPAD + S::DOUT - 1) / S::DOUT;           // bins that reach into a bin's windows
    static_assert(TL % SB == 0 && BPS <= kPfBatch, "whole bins per tile");
    __shared__ __align__(16) unsigned char tile[kPfThreads * kPfLine];
    __shared__ float rv[kPfBatch * RVS];
    __shared__ unsigned short rc[kPfBatch * RLS];     // code: 0x8000 if walked with PfLane | level << 12 | its token
    __shared__ int sn[kPfThreads];               // weight column of each stream

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = a.M, N = a.N;
    const int ndpf = kPfThreads / M;
    const int dpf0 = blockIdx.x * ndpf;
    const int b = blockIdx.y;
    const int tile0 = pf_first_tile(a.Tp / TL, blockIdx.z, a.nseg);               // this segment's first tile
    const int ntseg = pf_first_tile(a.Tp / TL, blockIdx.z + 1, a.nseg) - tile0;    // its evaluated tiles
    const int nd = min(ndpf, a.ndm_out - dpf0);
    const int nstreams = nd * M;
    const bool active = tid < nstreams;
    const int dl = tid / M, m = tid - dl * M;

    Tst *rows = reinterpret_cast<Tst *>(a.sb) + long(a.beam0 + b) * a.sb_bstride + long(dpf0) * M * a.rowlen;
    const int Wds = a.ndm_out / a.ndm_wt;
    const int Tds = a.nt_out / a.nt_wt;
    const float *wbeam = a.wt + long(b) * a.wt_bstride;
    const int wcol = active ? a.m_to_n[m] : 0;
    const float *wrow = wbeam + long(active ? (dpf0 + dl) / Wds : 0) * a.nt_wt * S::P * N + wcol;
    sn[tid] = wcol;
    Tst *outm = reinterpret_cast<Tst *>(a.out_max) + long(b) * a.out_bstride;
    unsigned int *outa = a.out_argmax + long(b) * a.out_bstride;

    PfMax<S> ln;
#pragma unroll
    for (int i = 0; i < S::WTOT; i++)
        ln.w[i] = 0.0f;
    int marked = 0;            // bins, from this one on, whose windows hold a sample that pf_wild rejects

    // The first tile holds the line of position tpad - 1: nwarm tiles reach back to the line of
    // position 0 (rows start 'lead' elements after a line; what lies before position 0 in
    // that line is in the buffer and is older than any window that is evaluated).
    const int nwarm = (a.tpad + TL - 1) / TL;
    const int ntiles = nwarm + ntseg;
    const int srow = 64 * wv + (lane >> 3);                          // row this lane stages, + 8 k
    const Tst *src = rows + long(srow) * a.rowlen + a.tpad + (tile0 - nwarm) * TL + ((lane & 7) ^ (lane >> 3)) * CH;
    auto stage = [&](int it) {
        unsigned char *dst = tile + wv * 64 * kPfLine;
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (srow + 8 * k < nstreams)
                __builtin_amdgcn_global_load_lds((pf_gptr)(src + long(8 * k) * a.rowlen + it * TL),
                                                 (pf_lptr)(dst + k * 8 * kPfLine), 16, 0, 0);
    };

    // step 2's DM rows: the wave's own when whole rows fall into a wave, else the workgroup's
    const bool wave_local = (64 % M) == 0;
    const int d2 = wave_local ? wv * (64 / M) : 0;
    const int nd2 = wave_local ? max(0, min(64 / M, nd - d2)) : nd;

    stage(0);
    int nbatch = 0;            // bins in the batch
    for (int it = 0; it < ntiles; it++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this tile has landed
        const unsigned char *trow = tile + tid * kPfLine;
        const int tb0 = (tile0 + it - nwarm) * (TL / S::DOUT);
#pragma unroll 1
        for (int sb = 0; sb < TL / SB; sb++) {
            float x[SB];
            {
                rawv_st<Tst, CH> r[SB / CH];
#pragma unroll
                for (int c = 0; c < SB / CH; c++)
                    r[c] = *reinterpret_cast<const rawv_st<Tst, CH> *>(trow + (((sb * (SB / CH) + c) ^ (lane & 7)) << 4));
#pragma unroll
                for (int c = 0; c < SB / CH; c++)
                    from_rawv<Tst, CH>(r[c], x + CH * c);
            }
            if (sb + 1 == TL / SB && it + 1 < ntiles) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the wave's reads of this tile are done
                stage(it + 1);
            }
            if (it < nwarm) {
#pragma unroll
                for (int j = 0; j < BPS; j++) {
                    marked = pf_wild<S::DOUT>(x + j * S::DOUT) ? NBACK + 1 : max(marked - 1, 0);
                    ln.template bin<false>(x + j * S::DOUT);
                }
                continue;
            }
            const int tbs = tb0 + sb * BPS;
            if (active) {
#pragma unroll
                for (int j = 0; j < BPS; j++) {
                    const float *wp = wrow + long((tbs + j) / Tds) * S::P * N;
                    marked = pf_wild<S::DOUT>(x + j * S::DOUT) ? NBACK + 1 : max(marked - 1, 0);
                    float V;
                    unsigned int code;
                    // (expected: as equals, the two walks are given registers that spill at Wmax 8 and 32)
                    if (__builtin_expect(!__any(marked > 0), 1)) {
                        // loaded here, used at the end of the bin; kept from bin to bin they would
                        // be live across step 2, which spills
                        float wt[S::P];
#pragma unroll
                        for (int p = 0; p < S::P; p++)
                            wt[p] = wp[p * N];
                        ln.template bin<true>(x + j * S::DOUT);
                        unsigned int lev;
                        ln.combine(wt, V, lev);
                        code = lev << 12;
                    } else {
                        PfLane<S, false> le;
#pragma unroll
                        for (int i = 0; i < S::WTOT; i++)
                            le.w[i] = ln.w[i];
#pragma unroll
                        for (int p = 0; p < S::P; p++)
                            le.wt[p] = wp[p * N];
                        le.template bin<true>(x + j * S::DOUT);
#pragma unroll
                        for (int i = 0; i < S::WTOT; i++)
                            ln.w[i] = le.w[i];
                        unsigned int c;
                        le.combine(V, c);
                        code = 0x8000u | (unsigned(pf_level_of_token(c)) << 12) | c;
                    }
                    rv[(nbatch + j) * RVS + tid] = V;
                    rc[(nbatch + j) * RLS + tid] = (unsigned short)(code);
                }
            }
            nbatch += BPS;
            const bool last = (it + 1 == ntiles && sb + 1 == TL / SB);
            if (nbatch + BPS <= kPfBatch && !last)
                continue;

            // ---- step 2 over the batch's bins
            if (!wave_local)
                __syncthreads();
            const int tbb = tbs + BPS - nbatch;
            for (int idx = wave_local ? lane : tid; idx < nd2 * nbatch; idx += wave_local ? 64 : kPfThreads) {
                const int d = idx / nbatch + d2, j = idx % nbatch;
                const float *pv = rv + j * RVS + d * M;
                const unsigned short *pc = rc + j * RLS + d * M;
                float V = pv[0];
                unsigned int code = pc[0];
                int key = int((code >> 12) & 7) * M, m0 = 0;
#pragma unroll 4
                for (int mm = 1; mm < M; mm++) {
                    const float v = pv[mm];
                    const unsigned int c = pc[mm];
                    const int k = int((c >> 12) & 7) * M + mm;
                    if (v > V || (v == V && k < key)) {
                        V = v;
                        key = k;
                        code = c;
                        m0 = mm;
                    }
                }

                const int tb = tbb + j;
                unsigned int tok = code & 0xfffu;
                if (!(code & 0x8000u)) {
                    const float *wq = wbeam + (long((dpf0 + d) / Wds) * a.nt_wt + tb / Tds) * S::P * N + sn[d * M + m0];
                    PfLane<S, false> pl2;
#pragma unroll
                    for (int i = 0; i < S::WTOT; i++)
                        pl2.w[i] = 0.0f;
#pragma unroll
                    for (int p = 0; p < S::P; p++)
                        pl2.wt[p] = wq[p * N];
                    const Tst *row = rows + long(d * M + m0) * a.rowlen;
                    const int pb = a.tpad + tb * S::DOUT;
                    // groups of 4 samples; those before position 0, which starts a group, read as zeros
                    constexpr int VL = 4, NV = S::DOUT / VL;
                    using Raw = rawv_st<Tst, 4>;
                    auto load_bin = [&](Raw (&r)[NV], int pos) {
#pragma unroll
                        for (int i = 0; i < NV; i++)
                            r[i] = ldv_raw<Tst, 4>(row + max(pos + VL * i, 0));
                    };
                    auto floats = [&](const Raw (&r)[NV], int pos, float (&y)[S::DOUT]) {
#pragma unroll
                        for (int i = 0; i < NV; i++) {
                            from_rawv<Tst, 4>(r[i], y + 4 * i);
#pragma unroll
                            for (int q = 0; q < VL; q++)
                                y[VL * i + q] = (pos + VL * i >= 0) ? y[VL * i + q] : 0.0f;
                        }
                    };
                    float y[S::DOUT];
                    if constexpr ((NBACK + 1) * S::DOUT <= (sizeof(Tst) == 2 ? 64 : 40) && NBACK <= 8) {
                        // all of the walk's loads at once
                        Raw r[NBACK + 1][NV];
#pragma unroll
                        for (int k = 0; k <= NBACK; k++)
                            load_bin(r[k], pb + (k - NBACK) * S::DOUT);
#pragma unroll
                        for (int k = 0; k < NBACK; k++) {
                            floats(r[k], pb + (k - NBACK) * S::DOUT, y);
                            pl2.template bin<false>(y);
                        }
                        floats(r[NBACK], pb, y);
                    } else {
                        Raw r[NV];
#pragma unroll 1
                        for (int k = NBACK; k > 0; k--) {
                            load_bin(r, pb - k * S::DOUT);
                            floats(r, pb - k * S::DOUT, y);
                            pl2.template bin<false>(y);
                        }
                        load_bin(r, pb);
                        floats(r, pb, y);
                    }
                    pl2.template bin<true>(y);
                    pl2.combine(V, tok);
                }
                const long o = long(dpf0 + d) * a.nt_out + tb;
                st_st(outm + o, V);
                outa[o] = tok | (unsigned(m0) << 16);
            }
            nbatch = 0;
            if (!wave_local)
                __syncthreads();       // rv and rc are free
        }
    }

    if (blockIdx.z == 0) {
        __syncthreads();               // step 2 has read the rows
        rotate_rows(rows, nstreams, a);
    }
}

// Output bins that the two-step kernel is built for (see pf_two_step).
static constexpr bool pf_has_two_step(int dout) { return dout == 8 || dout == 16; }

template<typename Tst, int LW>
static void launch_pf_lw(const PfArgs &a, hipStream_t st, dim3 grid)
{
    dim3 block(kPfThreads);
    switch (a.Dout) {
#define PDD_PF(LDV)                                                                \
        case (1 << LDV):                                                           \
            if (a.out_var)                                                         \
                hipLaunchKernelGGL((k_pf_one<Tst, LW, LDV, true>), grid, block, 0, st, a);  \
            else if constexpr (pf_has_two_step(1 << LDV)) {                                      \
                if (a.two_step)                                                    \
                    hipLaunchKernelGGL((k_pf<Tst, LW, LDV>), grid, block, 0, st, a); \
                else                                                               \
                    hipLaunchKernelGGL((k_pf_one<Tst, LW, LDV, false>), grid, block, 0, st, a); \
            } else                                                                 \
                hipLaunchKernelGGL((k_pf_one<Tst, LW, LDV, false>), grid, block, 0, st, a); \
            break;
        PDD_PF(0) PDD_PF(1) PDD_PF(2) PDD_PF(3) PDD_PF(4) PDD_PF(5)
#undef PDD_PF
        default: break;
    }
}

// Two steps or one. Step 2 walks NBACK + 1 bins per output bin, spread over the M multiplets of a DM
// row, so it pays with many multiplets and long bins. One step and two, each at its best segment count, us,
// 2048 samples, float32 and float16:
//   (NBACK + 1) / M                                    float32      float16
//   0.12  (M 16, boxcars up to 4, bins of 16)          101    70     96    60
//   0.31  (M 16, 16, bins of 8)                        122    95    113    86
//   0.62  (M 8, 16, bins of 8)                         117   105    109    98
//   1.12  (M 8, 32, bins of 8)                         130   133    120   119
//   2.25  (M 4, 16, bins of 4)                          80    96     69    80
//   4.25  (M 4, 32, bins of 4)                          91   178     79   125
// Bins of 4 went from 27% slower to 20% faster and seldom occur with 16 multiplets or more; bins of 1
// and 2 were up to 3.2 times slower, and with bins of 32 the unrolled walks spill (up to 7 times slower).
// Small launches are bounded by latency: the tiles of one step are shorter, those of two steps pass
// without a barrier, which counts more the longer the warm-up is. Up to 2^14 positions of a
// workgroup's chunk and boxcars of 2 to 8 samples, one step took 9 to 16 us and two steps 13 to 19;
// with boxcars of 16 and 32 16 and 29 against 14 and 27 (float16 17 and 23). So between 0.7 and 1.15 two steps are
// taken for long boxcars and up to 2^17 positions: 2^15, boxcars of 32, 31 and 27 us (float16 29 and 23); 2^18
// as above; 2^20 455 and 500 us (float16 408 and 425).
static bool pf_two_step(const PfArgs &a, long nblocks, int TL)
{
    if (a.out_var || !pf_has_two_step(a.Dout) || a.Tp % TL != 0 || a.two_step == 0)
        return false;
    if (a.two_step > 0)
        return true;
    const int wmax = 1 << ((a.P - 1) / 3);
    const int bins = (a.tpad + a.Dout - 1) / a.Dout + 1;       // NBACK + 1
    const long work = nblocks * a.Tp;
    return (10 * bins <= 7 * a.M && (wmax >= 16 || work > (1 << 14)))
           || (20 * bins <= 23 * a.M && wmax >= 16 && work <= (1 << 17));
}

// Time segments per chunk, of whole tiles and at least nwarm of them (see rotate_rows). One step: the
// fewest that give at least a.target_blocks workgroups (2048 unless tuned). Two steps: up to that
// number, the count that is done first, a workgroup's time being its tiles and the warm-up's
// times a factor for its company on the CU (three of 768 run there at a time), and rounds of 768 running into
// each other. The factors are fitted to 170 launches of 8 to 2344 workgroups (in one segment) in all types: 1.3% from the best
// count on average, 20% at most. 32 workgroups of 1024 float32
// samples: 16 segments 24 us, 32 (64 positions walked for 32) 33 us; 256 of 1024: 3 segments 77 us, 4 94, 8 88 us;
// 512 of 2048 float16 samples: 1, 2, 4 and 8 segments 264, 240, 224 and 244 us. With out_var, one segment.
static int pf_nseg(const PfArgs &a, bool two_step, long nblocks, int TL)
{
    if (a.out_var)
        return 1;
    const int ntiles = a.Tp / TL, nwarm = (a.tpad + TL - 1) / TL;
    const int most = int(std::min<long>(std::max(1, ntiles / nwarm), (a.target_blocks + nblocks - 1) / nblocks));
    if (!two_step)
        return most;
    int best = 1;
    double cost = 0.0;
    for (int n = 1; n <= most; n++) {
        const long nwg = nblocks * n;
        const double w = nwg / 768.0;
        const double c = ((ntiles + n - 1) / n + nwarm) * ((nwg <= 256) ? 0.6 : (nwg <= 512) ? 0.85 : (nwg <= 768) ? 1.0
                                                           : 0.34 * w + 0.51 * ((nwg + 767) / 768) + 0.21);
        if (n == 1 || c < cost) {
            best = n;
            cost = c;
        }
    }
    return best;
}

template<typename Tst>
static void launch_pf_t(const PfArgs &a0, hipStream_t st)
{
    PfArgs a = a0;
    const int ndpf = kPfThreads / a.M;
    const unsigned nbx = unsigned((a.ndm_out + ndpf - 1) / ndpf);
    constexpr int TL2 = kPfLine / int(sizeof(Tst));      // k_pf's tile
    a.two_step = pf_two_step(a, long(nbx) * a.B, TL2);
    a.nseg = pf_nseg(a, a.two_step, long(nbx) * a.B, a.two_step ? TL2 : pf_tile_len(a.Dout));
    dim3 grid{nbx, unsigned(a.B), unsigned(a.nseg)};
    switch ((a.P - 1) / 3) {
        case 0: launch_pf_lw<Tst, 0>(a, st, grid); break;
        case 1: launch_pf_lw<Tst, 1>(a, st, grid); break;
        case 2: launch_pf_lw<Tst, 2>(a, st, grid); break;
        case 3: launch_pf_lw<Tst, 3>(a, st, grid); break;
        case 4: launch_pf_lw<Tst, 4>(a, st, grid); break;
        case 5: launch_pf_lw<Tst, 5>(a, st, grid); break;
        default: break;
    }
}

void launch_pf(Dtype dt, const PfArgs &a, hipStream_t st)
{
    switch (dt) {
        case Dtype::float32: launch_pf_t<float>(a, st); break;
        case Dtype::float16: launch_pf_t<__half>(a, st); break;
        case Dtype::bfloat16: launch_pf_t<__hip_bfloat16>(a, st); break;
    }
}

}  // namespace pirate_amd
