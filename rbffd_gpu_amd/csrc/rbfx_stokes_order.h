// The order of an ILU(0) sweep over the velocity block, on the host.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

constexpr int SWEEP_ROWS = 64;     // rows of a chunk, one per lane
constexpr int SWEEP_BLK = 8;       // entries whose products a wave forms together
constexpr int SWEEP_MAX_BLKS = 8;  // up to 64 entries of a row on one side of the diagonal

struct SweepChunk {
    int t0, nr;            // first task, rows
    int base;              // first packed entry, in blocks of 8: rows padded to them may have more than 2^31 entries
    int nblk;              // blocks of 8 entries; bit 8: some entries are older than the ring
    int need[SWEEP_MAX_BLKS];  // chunks that must be done before block b's products
    int unused[4];
};

// One sweep's order on the host: rows level by level, each row's task and chunk, and the chunks
// (up to SWEEP_ROWS rows of a level) with the place of their packed entries.
struct HostSide {
    std::vector<SweepChunk> chunks;
    std::vector<int32_t> rows, task, chunk_of, off;
    size_t n_ent = 0;
};

// lev[r] of n_lev levels; count(r): entries of row r on the sweep's side of the diagonal.
template <typename Fn>
void order_side(const std::vector<int32_t>& lev, int n_lev, const Fn& count, HostSide& D) {
    const int N = (int)lev.size();
    D.off.assign(n_lev + 1, 0);
    for (int r = 0; r < N; r++) D.off[lev[r] + 1]++;
    for (int l = 0; l < n_lev; l++) D.off[l + 1] += D.off[l];
    D.rows.resize(N);
    D.task.resize(N);
    D.chunk_of.resize(N);
    std::vector<int32_t> pos(D.off.begin(), D.off.end() - 1);
    for (int r = 0; r < N; r++) {
        const int t = pos[lev[r]]++;
        D.rows[t] = r;
        D.task[r] = t;
    }
    for (int l = 0; l < n_lev; l++)
        for (int t0 = D.off[l]; t0 < D.off[l + 1]; t0 += SWEEP_ROWS) {
            SweepChunk C = {};
            C.t0 = t0;
            C.nr = std::min(SWEEP_ROWS, D.off[l + 1] - t0);
            C.base = (int)(D.n_ent / SWEEP_BLK);
            int most = 0;
            for (int t = t0; t < t0 + C.nr; t++) {
                const int r = D.rows[t];
                most = std::max(most, count(r));
                D.chunk_of[r] = (int)D.chunks.size();
            }
            C.nblk = (most + SWEEP_BLK - 1) / SWEEP_BLK;
            D.n_ent += (size_t)C.nblk * SWEEP_BLK * C.nr;
            D.chunks.push_back(C);
        }
}
