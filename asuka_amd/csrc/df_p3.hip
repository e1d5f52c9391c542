// Three-centre classes (33|c): instantiations of df_impl.h, compiled as a
// separate translation unit.
#include "df_impl.h"

#define ASUKA_DF_P3(X) X(3, 3, 0, 1) X(3, 3, 1, 3) X(3, 3, 2, 6) X(3, 3, 3, 10)

ASUKA_DF_FIND(find_df_p3, ASUKA_DF_P3)
