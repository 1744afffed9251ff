"""The JSON line of bench.py keeps to the summary; tables per class, molecule or stage go elsewhere."""
import bench


def test_tables_leave_the_line():
    result = {'metric': 'm', 'value': 1.0, 'class_ms': {'0000': 1.0}, 'roofline': {'kernel': 'k', 'achieved': 2.0},
              'multi_density': {'k4': 3.0, 'classes_one_stream_4_densities': {'0000': {}}},
              'svp32': {'builds_per_s': 5.0, 'autotune': [1], 'class_flops': {}}}
    line, tables = bench.split_tables(result)
    assert line == {'metric': 'm', 'value': 1.0, 'roofline': {'kernel': 'k', 'achieved': 2.0},
                    'multi_density': {'k4': 3.0}, 'svp32': {'builds_per_s': 5.0}}
    assert tables == {'class_ms': {'0000': 1.0}, 'multi_density': {'classes_one_stream_4_densities': {'0000': {}}},
                      'svp32': {'autotune': [1], 'class_flops': {}}}


def test_nested_floats_are_rounded_but_energies():
    assert bench.rounded({'energy': -2430.6301299981697, 'ms': [1.23456789], 'n': 3, 'ok': True}) == {
        'energy': -2430.6301299981697, 'ms': [1.23457], 'n': 3, 'ok': True}
