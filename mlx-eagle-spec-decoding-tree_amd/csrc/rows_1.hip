// Forms of the rows kernel for 1 .. 16 rows of x: tiles of a wave in the first and second half of the waves,
// tiles of x, K parts, chunks requested ahead.
#include "rows.h"

using namespace eagle_rows;

static const RowsForm forms[] = {
    rows_form<1, 1, 1, 1, 4>(),
    rows_form<1, 1, 1, 2, 4>(),
    rows_form<1, 1, 1, 4, 4>(),
    rows_form<2, 2, 1, 1, 4>(),
    rows_form<3, 3, 1, 1, 4>(),
    rows_form<3, 3, 1, 4, 2>(),
    rows_form<5, 5, 1, 1, 2>(),
    rows_form<5, 5, 1, 4, 2>(),
    rows_form<2, 1, 1, 1, 4>(),
    rows_form<3, 2, 1, 1, 4>(),
    rows_form<3, 2, 1, 2, 4>(),
    rows_form<2, 1, 1, 2, 4>(),
};
RowsTable eagle_rows::forms_1() { return {forms, (int)(sizeof(forms) / sizeof(forms[0]))}; }
