"""The JSON line of bench.py keeps to the summary; per-class tables go elsewhere."""
import bench


def test_per_class_tables_leave_the_line():
    result = {'metric': 'm', 'value': 1.0, 'class_ms': {'0000': 1.0}, 'roofline': {'kernel': 'k', 'achieved': 2.0},
              'multi_density': {'k4': 3.0, 'classes_one_stream_4_densities': {'0000': {}}},
              'svp32': {'builds_per_s': 5.0, 'autotune': [1], 'class_flops': {}}}
    line, tables = bench.split_class_tables(result)
    assert line == {'metric': 'm', 'value': 1.0, 'roofline': {'kernel': 'k', 'achieved': 2.0},
                    'multi_density': {'k4': 3.0}, 'svp32': {'builds_per_s': 5.0}}
    assert tables == {'class_ms': {'0000': 1.0}, 'multi_density': {'classes_one_stream_4_densities': {'0000': {}}},
                      'svp32': {'autotune': [1], 'class_flops': {}}}
