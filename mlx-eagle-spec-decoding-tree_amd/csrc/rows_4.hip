// Forms of the rows kernel for 49 .. 64 rows of x (and blocks of 64): tiles of a wave in the first and second half of the waves,
// tiles of x, K parts, chunks requested ahead.
#include "rows.h"

using namespace eagle_rows;

static const RowsForm forms[] = {
    rows_form<1, 1, 4, 1, 4>(),
    rows_form<1, 1, 4, 2, 4>(),
    rows_form<2, 2, 4, 1, 4>(),
    rows_form<3, 3, 4, 1, 2>(),
    rows_form<3, 3, 4, 2, 2>(),
    rows_form<2, 1, 4, 1, 4>(),
    rows_form<3, 2, 4, 1, 2>(),
    rows_form<3, 2, 4, 2, 2>(),
    rows_form<2, 1, 4, 2, 2>(),
};
RowsTable eagle_rows::forms_4() { return {forms, (int)(sizeof(forms) / sizeof(forms[0]))}; }
