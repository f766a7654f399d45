// The chunked form of the linear recurrences (scan_chunks.hip), launched by linear_scan.hip.
#pragma once
#include "common.h"

#define SC_CHUNK 64          // tokens per chunk
#define SC_COLS 16           // columns of S per block
// A chunk's record for a head, in floats: the pairs [64][64] (rows j <= i of them), p_i, d_last,j (pairs and
// d_last,j times the write strengths), and what p_last lost in rounding to 32 bits
#define SC_PRE (SC_CHUNK * SC_CHUNK)
#define SC_SUF (SC_PRE + SC_CHUNK)
#define SC_REST (SC_SUF + SC_CHUNK)
#define SC_RECORD (SC_REST + 4)
// With a decay per key dim: the pairs, q times the decays up to its token [64][D], k times those behind its token [64][D], the
// whole chunk's decays [D] and what their rounding left [D]
#define SC_CHANNEL_Q (SC_CHUNK * SC_CHUNK)
// The delta rule: as without it (no write strengths), then T diag(beta) [64][64] and T diag(beta p) k [64][D]
#define SC_DELTA_T SC_RECORD
#define SC_DELTA_W (SC_DELTA_T + SC_CHUNK * SC_CHUNK)
#define SC_DELTA_RECORD(D) (SC_DELTA_W + SC_CHUNK * (D))
#define SC_CHANNEL_RECORD(D) (SC_CHANNEL_Q + 2 * SC_CHUNK * (D) + 2 * (D))

struct ScanChunks {
    const float* q;
    const float* k;
    const float* v;
    int ldq, ldk, ldv;
    const float* head_decay;     // one of the two
    const float* tok_decay;
    const float* write;          // write strengths per token and head, or null
    int ldg;
    float* state;
    size_t slot_stride;
    const int* seq_q_start;
    const int* seq_q_len;
    const int* seq_slots;
    float* out;
    float* records;
    int n_seqs, min_len, H, G, Dv;
    float o_scale;
    const float* skip;
    const float* chan_decay;     // a decay per token, head and key dim (then neither of the other two, and no write strengths)
    int ldc;
    int corrects;                // the delta rule: u = write (v - S^T k)
};

// Sizes that it takes.
inline bool scan_chunks_takes(int D, int Dv) { return (D == 64 || D == 128 || D == 256) && Dv % SC_COLS == 0; }
// n_chunks: the chunks of all requests of at least min_len tokens, a record each.
void scan_chunks_launch(const ScanChunks& a, int D, int n_chunks, hipStream_t stream);
