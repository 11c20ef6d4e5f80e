// Host-visible argument structs and launchers for the gfx950 dedispersion kernels.
// All pointers are device pointers; strides and offsets are in elements.

#ifndef PIRATE_AMD_KERNELS_HPP
#define PIRATE_AMD_KERNELS_HPP

#include <hip/hip_runtime.h>
#include "../host/config.hpp"

namespace pirate_amd {

// ---- tree gridding fused with lagged downsampling ----
// grid[b,n,t] = sum_f w[n,f] in[b,f,t] (CSR weights, ascending f), n < nchan = 2^R, and for
// primary trees p = 1..npri-1: out[p] (B, 2^(R-1), ntime >> p).
static constexpr int kMaxPrimaryTrees = 8;

struct GridLdsArgs {
    const void *in;                      // (B, nfreq, ntime) input slot
    long in_bstride;
    void *grid;                          // (B, nchan, ntime) gridded rows (primary tree 0 input)
    long grid_bstride;
    int B, nchan, nfreq, ntime;
    const int *row_f0;                   // (nchan) first input channel of tree channel n
    const int *row_cnt;                  // (nchan) number of input channels
    const int *row_woff;                 // (nchan) offset into w
    const float *w;                      // overlap weights
    void *out[kMaxPrimaryTrees];         // out[p], p >= 1
    long out_bstride[kMaxPrimaryTrees];
    float *state;                        // per global beam, see lds_state_nelts()
    long state_bstride;
    int npri, s;                         // s = (stage-1 dd_rank of p>=1) + 1
    int xcd_run = 8;                     // consecutive channel pairs per XCD (0: plain order)
    int beam0;                           // global index of the batch's first beam
    long chunk;                          // chunk index (selects the state parity)
    const long *chunk_dev = nullptr;     // if set, the chunk index is read here (graph replay)
};
long lds_state_nelts(int R, int npri, int s);   // per beam
void launch_grid_lds(Dtype dt, const GridLdsArgs &a, hipStream_t st);


// ---- stage-1 tree: (B, 2^amb, 2^dd, Tp) -> lag ring rows (a, dm_brev) ----
struct RingView {
    void *base;               // ring storage of one primary tree
    const long *row_off;      // (nrows) element offset of each row within a beam
    const long *row_cap;      // (nrows) capacity (elements) of each row
    long bstride;             // elements per beam
};

// State blocks, [B beams][2^amb instances] each, that a launch reads and writes: its batch's with one
// time segment. With several, segment 0 reads what the last one writes; then there are nspare more, one per stream.
// Launch n (of the batches in turn, on stream n % nspare) writes the block that the launch nspare before
// it, on the same stream, read, and reads the one written nbatches launches before it.
struct StateBlocks {
    long rd, wr;
};

struct StateArgs {
    float *state;             // phase-A histories and line samples
    long state_bstride;       // per beam
    int nbatches, nspare, batch;
    StateBlocks blocks;       // blocks_of(chunk), unless the chunk index is read on the device
    __host__ __device__ StateBlocks blocks_of(long chunk) const
    {
        const unsigned long launch = (unsigned long) (chunk) * nbatches + batch, n = nbatches + nspare;
        return nspare ? StateBlocks{long((launch + nspare) % n), long(launch % n)} : StateBlocks{batch, batch};
    }
};

struct Stage1Args : StateArgs {
    const void *in;
    long in_bstride;
    RingView ring;
    int B, amb, dd, Tp, beam0;
    int nseg;                 // time segments: tree_segments()
    long chunk;               // chunk index (ring time = chunk*Tp + t)
    const long *chunk_dev = nullptr;   // if set, the chunk index is read here (graph replay)
};


// ---- stage-2 tree + subband streams -> peak-finder input rows ----
// pf_rank = (dd + 1) / 2; band counts and first multiplets per subband level 0..pf_rank.
static constexpr int kMaxPfRank = 4;
struct Stage2Args : StateArgs {
    RingView ring;            // ring of the tree's primary tree
    const int *row_lag;       // (2^dd rows fc, 2^amb j) -> lag, indexed fc*2^amb + j
    void *sb;                 // (B, ndm_out, M, rowlen) peak-finder input rows
    long sb_bstride;
    int rowlen, tpad, M;
    int nband[kMaxPfRank + 1], mband[kMaxPfRank + 1];
    int B, amb, dd, Tp, beam0;
    int nseg;                 // time segments: tree_segments()
    long chunk;
    const long *chunk_dev = nullptr;   // if set, the chunk index is read here (graph replay)
};

// Time segments of a stage with ninst tree instances (2^amb times beams per batch), the same for every
// chunk, and the floats of state per instance.
int tree_segments(int dd, long ninst, int Tp);
long tree_state_nelts(int dd, bool stage2);
// Stage 2 reads a ring row from up to this many samples before the chunk's delayed start (phase
// A's window).
int tree_overlap(int dd);
void launch_stage1(Dtype dt, const Stage1Args &a, hipStream_t st);
void launch_stage2(Dtype dt, const Stage2Args &a, hipStream_t st);


// ---- int4 dequantization: out = scale * value + offset per 256-sample (beam, freq) block ----
// data: nsamples int4 (two per byte, low nibble first); scoff: float16 {scale, offset} pairs.
void launch_dequant(Dtype dt, const void *data, const void *scoff, void *out, long nsamples, hipStream_t st);


// ---- ring-buffer segment copies driven by octuples (device array of 8*noct uint32) ----
// Host spill: appends outbox row i (Tp elements of elt_bytes) of each beam of the batch to
// device ring row rows[i] at ring time chunk * Tp.
void launch_spill_scatter(void *ring, long bstride, int elt_bytes, long outbox_off, const int *rows, long nrows,
                          const long *row_off, const long *row_cap, long Tp, long chunk, int beam0, int B, hipStream_t st);
void launch_ringbuf_copy(void *ringbuf, const uint32_t *octuples, long noct, long seg_bytes, int nbeams,
                         unsigned long long iframe, hipStream_t st);


// ---- peak finder over (B, ndm_out, M, rowlen) rows -> out_max, out_argmax ----
struct PfArgs {
    void *sb;                 // rows [tpad history | Tp]
    long sb_bstride;
    int rowlen, tpad;
    const int *m_to_n;        // (M)
    const float *wt;          // (B, ndm_wt, nt_wt, P, N) non-negative weights
    long wt_bstride;
    void *out_max;            // (B, ndm_out, nt_out), storage dtype
    unsigned int *out_argmax; // (B, ndm_out, nt_out)
    long out_bstride;
    int B, ndm_out, M, N, P, Tp, Dout, Dcore, ndm_wt, nt_wt, nt_out;
    int beam0;                // global index of the batch's first beam (sb rows are per global beam)
    int nseg = 1;             // time segments per chunk (set by launch_pf)
    int two_step = -1;        // two-step kernel: -1 by launch_pf's rule, 0 never, 1 wherever there is one
    long target_blocks = 2048;   // launch_pf picks at most the fewest segments giving this many workgroups
    double *out_var = nullptr;   // optional (B, ndm_out, M, P) float64: per-chunk mean square of each
                                 // (multiplet, profile)'s weighted candidates
};
bool pf_config_supported(int M, int tpad, int Dcore, int Dout, int Tp);
void launch_pf(Dtype dt, const PfArgs &a, hipStream_t st);

}  // namespace pirate_amd

#endif
