// Three-centre classes (22|c), (30|c) and (31|c): instantiations of
// df_impl.h, compiled as a separate translation unit.
#include "df_impl.h"

#define ASUKA_DF_P1(X) \
  X(2, 2, 0, 1) X(2, 2, 1, 2) X(2, 2, 2, 3) X(2, 2, 3, 5) \
  X(3, 0, 0, 1) X(3, 0, 1, 1) X(3, 0, 2, 1) X(3, 0, 3, 2) \
  X(3, 1, 0, 1) X(3, 1, 1, 1) X(3, 1, 2, 3) X(3, 1, 3, 5)

ASUKA_DF_FIND(find_df_p1, ASUKA_DF_P1)
