// SCC launch choices of single-point batches by basis size on MI355X, written
// by qcxms_amd/autotune.py: {max_nao, MFMA eigen refinement, LDS matrices}
// per bin, and {eig, lds} for batches spanning several bins (eig -1: one
// launch per run of systems of one bin).
// Timed with workgroups of 256 threads.  With those of 512 the refinement is no
// longer the faster choice everywhere (1024 uneven systems: 30.2 ms, Jacobi
// alone 25.7 ms); the table stays, because another solver moves the results by
// about 1e-8 relative.
#pragma once

namespace qx {

constexpr int kTuneTable[][3] = {
    {40, 1, 1},
    {56, 0, 1},
    {256, 1, 0},
};
constexpr int kTuneMixed[2] = {1, 1};

}  // namespace qx
