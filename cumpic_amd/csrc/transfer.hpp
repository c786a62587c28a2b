// transfer.hpp -- host arrays in and out of the device planes.
//
// A transfer converts between the caller's AoS arrays (cell-major, nv values per cell) and the SoA
// planes in pieces: device staging buffer, pinned host buffer, caller's memory.  A temporary of the array's
// size on each call cost a hipMalloc and hipFree (which waits for the device) and a copy from or to pageable
// memory at one thread's page-fault rate; here the staging units (2 MiB of either memory) are kept while
// there is a context, and a large transfer runs up to eight of them at once, one host thread each, so that
// conversion, copy and the caller's page faults overlap.  Download of 256^3 (1.7 GB) 166 -> 36 ms, of a 400^2
// box (111 MB, seven planes) 10.0 -> 2.5 ms, of 24^3 202 -> 157 us; upload of 256^3 (1.3 GB) 43 -> 23 ms, of
// 24^3 120 -> 119 us.
#pragma once
#include "ctx.hpp"

// one array of a transfer: nv planes of the layout at `soa`, the caller's AoS array at `host`
struct XferArray {
    double *soa;
    double *host;
    int nv;
};

// The context's stream is idle before the transfer starts and after it returns.
int transfer_in(cumc_ctx *ctx, const XferArray *a, int n);   // host -> planes
int transfer_out(cumc_ctx *ctx, const XferArray *a, int n);  // planes -> host

// contexts that may transfer: the staging units of the process are freed with the last one
void staging_retain();
void staging_release();
