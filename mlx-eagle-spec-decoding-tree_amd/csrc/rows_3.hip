// Forms of the rows kernel for 33 .. 48 rows of x (and blocks of 48): tiles of a wave in the first and second half of the waves,
// tiles of x, K parts, chunks requested ahead.
#include "rows.h"

using namespace eagle_rows;

static const RowsForm forms[] = {
    rows_form<1, 1, 3, 1, 4>(),
    rows_form<1, 1, 3, 2, 4>(),
    rows_form<2, 2, 3, 1, 4>(),
    rows_form<3, 3, 3, 1, 2>(),
    rows_form<3, 3, 3, 2, 2>(),
    rows_form<3, 3, 3, 4, 2>(),
    rows_form<5, 5, 3, 1, 2>(),
    rows_form<5, 5, 3, 2, 2>(),
    rows_form<2, 1, 3, 1, 4>(),
    rows_form<3, 2, 3, 1, 2>(),
    rows_form<3, 2, 3, 2, 2>(),
    rows_form<2, 1, 3, 2, 2>(),
};
RowsTable eagle_rows::forms_3() { return {forms, (int)(sizeof(forms) / sizeof(forms[0]))}; }
