// isect.hpp -- post-step intersection check (internal interface).
#pragma once
#include "lbvh.hpp"
#include "ppf_mi355x.h"

namespace ppf {

// Owns the record buffer. The trees are the narrow phase's, the dynamic ones
// built at the checked positions; cface: the collision mesh's face tree.
class IntersectionCheck {
  public:
    ~IntersectionCheck();
    int run(const BvhView &face, const BvhView &edge, const BvhView &vert,
            const BvhView &cface, const ppf_contact_mesh &m, const ppf_static_mesh *sm,
            const float *vmass, const float *emass, const float *fmass, uint32_t surface_vert_count,
            ppf_isect_record *records, uint32_t cap, uint32_t *count, hipStream_t s,
            uint32_t *scene_count = nullptr);

  private:
    ppf_isect_record *rec_ = nullptr;
    uint32_t rec_cap_ = 0;
    uint32_t *ctr_ = nullptr, *h_ctr_ = nullptr;
    uint32_t ctr_cap_ = 0;
};

} // namespace ppf
