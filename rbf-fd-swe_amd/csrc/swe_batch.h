// What the forecast server asks of libswe_hip beside include/swe_hip.h.
#pragma once

#include "swe_hip.h"

extern "C" {

// Bytes of a batch context that its device bytes leave open: `records` are in
// them but are one copy for all contexts of the mesh; `tiles` may be added to
// them by a later call.
typedef struct swe_hip_batch_bytes {
    long long records, tiles;
} swe_hip_batch_bytes;

// swe_hip_create_ex for a batch that is seldom full.  Where `room` device bytes
// hold them, a tiled fast-mode context gets the matrix-core ensemble kernel's
// records first and the member-lane kernel's tiles with the first
// swe_hip_rk_steps that they are the faster choice for; every launch then runs
// the faster of the two for the active members (the bits are the same).
int swe_hip_batch_create(const swe_hip_static *s, const swe_hip_options *o, long long room,
                         swe_hip_ctx **out, swe_hip_batch_bytes *bytes);
// Whether the device runs nothing beside this context's next launches.
void swe_hip_batch_alone(swe_hip_ctx *ctx, int alone);

}
