// Three-centre classes with la <= 1, (20|c) and (21|c): instantiations of
// df_impl.h, compiled as a separate translation unit.
#include "df_impl.h"

#define ASUKA_DF_P0(X) \
  X(0, 0, 0, 1) X(0, 0, 1, 1) X(0, 0, 2, 1) X(0, 0, 3, 1) \
  X(1, 0, 0, 1) X(1, 0, 1, 1) X(1, 0, 2, 1) X(1, 0, 3, 1) \
  X(1, 1, 0, 1) X(1, 1, 1, 1) X(1, 1, 2, 1) X(1, 1, 3, 2) \
  X(2, 0, 0, 1) X(2, 0, 1, 1) X(2, 0, 2, 1) X(2, 0, 3, 1) \
  X(2, 1, 0, 1) X(2, 1, 1, 1) X(2, 1, 2, 2) X(2, 1, 3, 3)

ASUKA_DF_FIND(find_df_p0, ASUKA_DF_P0)
