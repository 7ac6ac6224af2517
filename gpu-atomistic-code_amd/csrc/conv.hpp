// conv.hpp - FP32 convolution with a mirror-symmetric kernel on meshes of up to
// 128 x 128 x 32 points (k_conv.hip).
#pragma once
#include <array>
#include <memory>

#include "ctx.hpp"

namespace sllg {

struct ConvPlan {
    uint32_t l[3] = {0, 0, 0};    // mesh extents
    uint32_t gx = 0, gy = 0;      // padded extents (powers of two); z: 2 l[2]
    bool dense = false;           // spin i is mesh point i
    DevBuf map;                   // [x][y][z]: device spin or ~0 (not dense)
    DevBuf mu;                    // moment per spin (dipolar)
    DevBuf twx, twy, zt, spec;
    std::shared_ptr<DevBuf> N;    // octant of the transformed kernel
    uint64_t bytes() const {
        return map.bytes + mu.bytes + twx.bytes + twy.bytes + zt.bytes + spec.bytes + (N ? N->bytes : 0);
    }
};

// Whether the mesh and the kernel (the dipolar one, or the FFT exchange fx) take this path.
bool conv_applies(const llg_ctx* c, const llg_dipolar& d, const llg_fftexch* fx);
int conv_create(llg_ctx* c, ConvPlan& p, const llg_dipolar& d, const uint32_t* spin_species, const llg_fftexch* fx,
                bool dip_terms);
// H (SoA) = the convolution of the spins S: SoA, or AoS3 ([3 i + c]).
int conv_apply(llg_ctx* c, const ConvPlan& p, const float* S, bool aos3, float* H);

}  // namespace sllg
