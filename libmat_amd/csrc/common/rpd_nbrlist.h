// The neighbour lists behind an rpd_nbr handle (rpd_prep.h), shared by the
// host builder and the device builder's host side.
#pragma once

#include <stdint.h>

#include <vector>

struct rpd_nbr {
  std::vector<int32_t> valid;
  std::vector<int64_t> offsets;
  std::vector<int32_t> ids;
  int32_t max_degree = 0;
};

// a handle of lists that are symmetric and ascending already
rpd_nbr* rpd_nbr_adopt(std::vector<int32_t>&& valid,
                       std::vector<int64_t>&& offsets,
                       std::vector<int32_t>&& ids);
